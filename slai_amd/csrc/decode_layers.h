// What the two launches that keep a model's layers in one kernel share (kernels_decode_small.hip, kernels_decode_mid.hip): workgroups of
// sixteen waves, of which wave 0 moves vectors and the other fifteen multiply.
#pragma once
#include "attention_fast.h"
#include "common.h"
#include "device_util.h"
#include "mfma_q4k.h"
#include "quant_formats.h"

namespace slai {
namespace layers {

constexpr uint32_t NT = 1024, NW = NT / 64, RW = NW - 1;       // threads, waves, waves with rows

// The sum over a wave, in every lane (lane exchanges inside the vector unit: six through LDS take 0.25 us)
__device__ __forceinline__ float sum64(float v) {
    v += mq::dpp<mq::DPP_XOR1>(v); v += mq::dpp<mq::DPP_XOR2>(v); v += mq::dpp<mq::DPP_HALF_MIRROR>(v); v += mq::dpp<mq::DPP_MIRROR>(v);
    const int b = __builtin_bit_cast(int, v);                  // every lane of a row of 16 holds the row's sum
    const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0)), r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32)), r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
    return (r0 + r1) + (r2 + r3);
}

__device__ __forceinline__ float max64(float v) {
    v = fmaxf(v, mq::dpp<mq::DPP_XOR1>(v)); v = fmaxf(v, mq::dpp<mq::DPP_XOR2>(v)); v = fmaxf(v, mq::dpp<mq::DPP_HALF_MIRROR>(v)); v = fmaxf(v, mq::dpp<mq::DPP_MIRROR>(v));
    const int b = __builtin_bit_cast(int, v);
    return fmaxf(fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0)), __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16))),
                 fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32)), __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48))));
}

// Workgroups of `kernel` that a device keeps resident
inline hipError_t resident_workgroups(const void *kernel, int device, uint32_t *resident) {
    int per_cu = 0, cus = 0;
    if (const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, (int)NT, 0)) return e;
    if (const hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device)) return e;
    *resident = (uint32_t)per_cu * (uint32_t)cus;
    return hipSuccess;
}

// The flag of a launch that gave up (the host clears it once it has seen it).  A launch looks at it once, as it starts: a call that cannot have its
// compute units then pays one time limit and not one for every token queued.  (Looking every 64 rounds of a wait as well was 1 us a
// token of 92, for the instructions around its rounds.)
__device__ __forceinline__ void abort_launch(uint32_t *flag) { __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ bool aborted(const uint32_t *flag) { return __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0; }

// The layer table through the scalar cache (it does not change while a kernel runs)
typedef const SmallLayer __attribute__((address_space(4))) LayerEntry;
__device__ __forceinline__ void touch_layers(const SmallLayer *layers, uint32_t n) {
    typedef const uint32_t __attribute__((address_space(4))) word;
    const word *w = (const word *)(uintptr_t)layers;
    const uint32_t words = n * (uint32_t)(sizeof(SmallLayer) / 4);
    for (uint32_t i = 0; i < words; i += 16 * 16) {
        uint32_t any = 0;
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j) any |= w[min(i + 16 * j, words - 1)];
        asm volatile("" : : "s"(any));
    }
}

// Column `col` (a multiple of 4) of the staged input: sixteen and a gap of four, so that lanes that read sixteen each meet no bank twice in a row
__device__ __forceinline__ uint32_t lds_col(uint32_t col) { return col + (col >> 4) * 4u; }

// One head's attention over the cached positions and the new one (batched_multiquery_attention.rs:32-156 with rope.slang:27-84 and the cache
// write): wave 0 takes the fresh query, key and value, the others eight positions a pass each, eight lanes a position for the scores, a lane an
// element for the values; the first rows are requested a step before the query exists.  The result leaves from wave 0.
struct AttnLds { float q[64], k[64], v[64], m[NW], l[NW], o[NW][64]; };

// wave 0, behind the barrier that ends the others' part: element `lane` of the head's result
__device__ __forceinline__ float head_merge(const AttnLds &lds, uint32_t lane) {
    const bool has = lane > 0 && lane < NW;
    const float mw = has ? lds.m[lane] : -FLT_MAX, M = max64(mw);
    const float f = has ? expf(mw - M) : 0.0f, sum = sum64(has ? f * lds.l[lane] : 0.0f);         // a wave that saw no position has sum 0 and outputs 0
    float r = 0.0f;
#pragma unroll
    for (uint32_t w = 1; w < NW; ++w) r = fmaf(lds.o[w][lane], __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), w)), r);
    return r / sum;
}

// the other waves
template <bool F16> struct HeadRows {
    using C = attn::KV<F16>;
    using CT = typename C::T;
    using V8 = attn::Vec8<F16>;
    static constexpr uint32_t PASS = 8 * RW;
    typename V8::Raw kr;
    CT vr[8];
    // (the row being written and rows past it are not read: row 0 stands in and counts as nothing)
    __device__ __forceinline__ void request(const SmallParams &p, const void *kcache, const void *vcache, uint32_t pos, uint32_t h, uint32_t wave, uint32_t lane, uint32_t tb) {
        if (pos == 0) return;
        const uint32_t hs = p.head_size, sub = lane & 7u, piece = sub * 8 < hs ? sub * 8 : 0u, e = lane < hs ? lane : 0u, t0 = tb + (wave - 1) * 8;
        const size_t hoff = (size_t)(h / p.kv_mul) * hs;
        const auto row_of = [&](uint32_t t) { return t < pos ? t : 0u; };
        kr = V8::template load_raw<false>((const CT *)kcache + (size_t)row_of(t0 + (lane >> 3)) * p.kvd + hoff + piece);
#pragma unroll
        for (int j = 0; j < 8; ++j) vr[j] = ((const CT *)vcache)[(size_t)row_of(t0 + j) * p.kvd + hoff + e];
    }
    __device__ __forceinline__ void run(AttnLds &lds, const SmallParams &p, const SmallLayer &L, uint32_t pos, uint32_t h, uint32_t wave, uint32_t lane) {
        const uint32_t hs = p.head_size, sub = lane & 7u, e = lane < hs ? lane : 0u, T = pos + 1;
        const bool inside = sub * 8 < hs;
        lds_barrier();
        float q[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) q[i] = inside ? lds.q[sub * 8 + i] : 0.0f;
        const float root = sqrtf((float)hs);
        float m = -FLT_MAX, l = 0.0f, o = 0.0f;
        for (uint32_t tb = 0; tb < T; tb += PASS) {
            const uint32_t t0 = tb + (wave - 1) * 8, t = t0 + (lane >> 3);
            if (t0 >= T) break;                                // (this wave's positions come to an end first; none in later passes either)
            float k[8] = {}, v[8] = {};
            if (pos) {
                V8::decode(kr, k);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if constexpr (F16) v[j] = attn::h2f((uint16_t)vr[j]);
                    else v[j] = vr[j];
                }
                if (tb + PASS < T) request(p, L.kcache, L.vcache, pos, h, wave, lane, tb + PASS);
            }
            float part = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) part = fmaf(q[i], !inside || t > pos ? 0.0f : t == pos ? lds.k[sub * 8 + i] : k[i], part);
            part += mq::dpp<mq::DPP_XOR1>(part); part += mq::dpp<mq::DPP_XOR2>(part); part += mq::dpp<mq::DPP_HALF_MIRROR>(part);
            const float sc = t < T ? part / root : -FLT_MAX;   // cpu.rs:521 `score /= sqrt(head_size)`
            float mn = m;
#pragma unroll
            for (int j = 0; j < 8; ++j) mn = fmaxf(mn, __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sc), 8 * j)));
            const float resc = expf(m - mn), pr = t < T ? expf(sc - mn) : 0.0f;
            l *= resc; o *= resc;
            m = mn;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float pj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pr), 8 * j));
                l += pj;
                o = fmaf(pj, t0 + j < pos ? v[j] : t0 + j == pos ? lds.v[e] : 0.0f, o);
            }
        }
        if (lane == 0) { lds.m[wave] = m; lds.l[wave] = l; }
        lds.o[wave][lane] = o;
        lds_barrier();
    }
};

}  // namespace layers
}  // namespace slai
