// A token of a small Llama (15 M parameters) as one resident launch on ONE die, gfx950.
//
// The layers of `Llama2::launch` (crates/slai/src/models/llama2/transformer.rs:316-381): norm + q/k/v, attention with rotation and cache
// write, projection into the residual, norm + FFN, projection.  The embedding row, the output matrix and the pick stay launches of
// their own.
//
// Why: such a layer is 1 MB of weights that stay in the 256 MB cache, and a launch between two steps that depend on each other costs
// 3.7 to 5.3 us whatever it does.  The 32 compute units of a die share an L2, so what one of them writes there the others find without
// a trip to memory: a step ends with one atomic per workgroup on a counter in that L2 and the next begins when the counter is full.
//   * 32 workgroups of 16 waves (workgroups i of the grid with i mod 8 equal run on one die; the other seven eighths leave at once).  Wave 0
//     waits for a step's input, normalises it and leaves it in LDS, and writes and reports the step's results; the other fifteen
//     multiply, half a wave a row (a whole one for rows of the FFN's width), a lane one chunk of columns (quant_formats.h), and ask for
//     the next step's weights as soon as they have.  (Every wave reading and normalising the input for itself asked for the same few lines
//     512 times at once: 123 us a token.  A whole wave per row of 18 chunks: 102.)
//   * vectors are handed over in memory of their own per layer and step: no line is read before it is complete, so plain loads do
//     (a compute unit's cache cannot hold an older copy).
//   * every wait is bounded: a workgroup that gives up sets a flag and waits no more, nor does any of a launch that finds the flag set.  The
//     host then repeats the call with launches.
// us a token in the loop, one launch per step / this: Q8_0, f32 cache, position 16: 130.6 / 92.9, 200: 139.6 / 101.3; Q4_0, f16 cache: 143.6 / 104.5.
// A layer takes 11 us (time stamps, position 16): five hand-overs of 0.4 to 0.7 us from the last report to the first workgroup's input, 0.6 to 1.0 to the
// last's, and 1.0 to 1.5 us from input to report, the attention's 1.9 (3.3 at position 200); nothing in it waits for a weight.  GPT-2 small in this form took 321 us a token
// against 328 in launches: seven times the weights are too many instructions for 32 compute units (kernels_decode_mid.hip has the whole device).
#include "common.h"
#include "decode_layers.h"

namespace slai {
namespace {

using namespace layers;
constexpr uint32_t NWG = SMALL_WGS;

// Who waits and reports: wave 0 of each workgroup (its lane 0 looks)
struct Steps {
    uint32_t *abort_flag;
    uint32_t tid, spin_limit;
    bool dead;
    __device__ __forceinline__ void wait(uint32_t *counter, uint32_t target) {        // wave 0 only
        if (tid == 0 && !dead) {
            uint32_t seen = 0, spins = 0;
            do {
                // (a read-modify-write that returns the value executes in the L2; a load could be served by this compute unit's own cache for ever)
                const uint32_t zero = 0;
                asm volatile("global_atomic_add %0, %1, %2, off sc0\n\ts_waitcnt vmcnt(0)" : "=&v"(seen) : "v"(counter), "v"(zero) : "memory");
                ++spins;
            } while (seen < target && spins < spin_limit);
            if (seen < target) { abort_launch(abort_flag); dead = true; }
        }
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void report(uint32_t *counter) const {                 // wave 0 only
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this wave's stores have reached the L2
        if (tid == 0) __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

enum { END_PLAIN, END_SILU };
enum { NORM_NONE, NORM_RMS };
constexpr uint32_t SMALL_WIDEST = 1024;                        // columns: one chunk of sixteen per lane, and what wave 0 stages

// n floats of x (a multiple of 4, at most 256 NJ), normalised, into LDS: wave 0
template <int NJ, int NORM, class Wait>
__device__ __forceinline__ void stage_input(float *xs, const float *x, uint32_t n, const float *nw, float eps, uint32_t lane, Wait &&wait) {
    float4 v[NJ], w[NORM == NORM_NONE ? 1 : NJ];
    const uint32_t n4 = n / 4;
    if constexpr (NORM != NORM_NONE)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const float *e = nw + 4u * min(lane + 64u * j, n4 - 1);      // (norm weights may be any view of a vector)
            w[j] = make_float4(e[0], e[1], e[2], e[3]);
        }
    wait();
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        v[j] = *(const float4 *)(x + 4u * min(lane + 64u * j, n4 - 1));
        if (lane + 64u * j >= n4) v[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    if constexpr (NORM != NORM_NONE) {                         // rms_norm.slang:60-66
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j) { ss = fmaf(v[j].x, v[j].x, ss); ss = fmaf(v[j].y, v[j].y, ss); ss = fmaf(v[j].z, v[j].z, ss); ss = fmaf(v[j].w, v[j].w, ss); }
        const float scale = 1.0f / sqrtf(sum64(ss) / (float)n + eps);
#pragma unroll
        for (int j = 0; j < NJ; ++j) { v[j].x = (v[j].x * scale) * w[j].x; v[j].y = (v[j].y * scale) * w[j].y; v[j].z = (v[j].z * scale) * w[j].z; v[j].w = (v[j].w * scale) * w[j].w; }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        if (lane + 64u * j < n4) *(float4 *)(xs + lds_col(4u * (lane + 64u * j))) = v[j];
}

// A step's rows of one wave: L lanes a row, so 64 / L of the workgroup's rows.  row(r) is the packed row r, row2(r) the same row of the up matrix.
// (L = 32 where a row has that few chunks: with a whole wave per row the fifteen waves were bound by issuing instructions for empty lanes.)
template <int T, int L, bool GATED> struct Rows {
    using F = Chunk<T>;
    typename F::Data d, d2;
    __device__ __forceinline__ static uint32_t at(uint32_t wave, uint32_t lane) { return L == 64 ? wave - 1 : 2 * (wave - 1) + (lane >> 5); }   // the lane's row among the workgroup's
    template <class Row, class Row2>
    __device__ __forceinline__ void request(uint32_t wg, uint32_t wave, uint32_t lane, uint32_t nrows, uint32_t ncols, Row &&row, Row2 &&row2) {
        const uint32_t r = min(nrows * wg / NWG + at(wave, lane), nrows - 1), c = lane & (L - 1), ch = c < F::nchunks(ncols) ? c : 0u;   // (rows past the workgroup's are asked for and not used)
        d = F::load(row(r), ncols / 32, ch);
        if constexpr (GATED) d2 = F::load(row2(r), ncols / 32, ch);
    }
    __device__ __forceinline__ static float row_sum(float v, uint32_t lane) {
        v += mq::dpp<mq::DPP_XOR1>(v); v += mq::dpp<mq::DPP_XOR2>(v); v += mq::dpp<mq::DPP_HALF_MIRROR>(v); v += mq::dpp<mq::DPP_MIRROR>(v);
        const int b = __builtin_bit_cast(int, v);
        const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0)), r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
        const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32)), r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
        return L == 64 ? (r0 + r1) + (r2 + r3) : lane < 32 ? r0 + r1 : r2 + r3;
    }
    // the products with the staged input, by row of the workgroup, into LDS
    __device__ __forceinline__ void multiply(uint32_t wave, uint32_t lane, uint32_t ncols, const float *xs, float *res, float *res2) const {
        const uint32_t c = lane & (L - 1);
        const bool valid = c < F::nchunks(ncols);
        const uint32_t ch = valid ? c : 0u;
        float v[F::E], sums[F::NRUN];
#pragma unroll
        for (int r = 0; r < F::NRUN; ++r) {
            float t = 0.0f;
#pragma unroll
            for (int i = 0; i < F::RUNLEN / 4; ++i) {
                const float4 q = *(const float4 *)(xs + lds_col(F::run_col(ch, r)) + 4 * i);
                float *o = &v[r * F::RUNLEN + 4 * i];
                o[0] = q.x; o[1] = q.y; o[2] = q.z; o[3] = q.w;
                t += (q.x + q.y) + (q.z + q.w);
            }
            sums[r] = t;
        }
        const float t = F::dot(d, ch, v, sums), s = row_sum(valid ? t : 0.0f, lane);
        float s2 = 0.0f;
        if constexpr (GATED) {
            const float t2 = F::dot(d2, ch, v, sums);
            s2 = row_sum(valid ? t2 : 0.0f, lane);
        }
        if (c == 0) {
            res[at(wave, lane)] = s;
            if constexpr (GATED) res2[at(wave, lane)] = s2;
        }
    }
};
constexpr uint32_t MOST = 2 * RW;                              // rows of a workgroup in a step, at most

// Wave 0's part of a step: the input staged, the results of the others finished and written, the step reported
template <int END, int NORM, int NJ, class Wait>
__device__ __forceinline__ void lead_step(Steps &steps, uint32_t *counter, uint32_t wg, uint32_t lane, uint32_t nrows, uint32_t ncols, float *xs, const float *res, const float *res2,
                                          const float *x, const float *nw, float eps, const float *residual, float *out, Wait &&wait) {
    const uint32_t r0 = nrows * wg / NWG, n = nrows * (wg + 1) / NWG - r0;
    const float keep = residual && lane < n ? residual[r0 + lane] : 0.0f;
    stage_input<NJ, NORM>(xs, x, ncols, nw, eps, lane, wait);
    lds_barrier();
    lds_barrier();
    if (lane < n) {
        float val = res[lane];
        if constexpr (END == END_SILU) val = res2[lane] * (val / (1.0f + expf(-val)));        // silu.slang:11-27
        out[r0 + lane] = val + keep;
    }
    steps.report(counter);
}

// wave 0; (c, sn): the rotation of this lane's pair, the same in every layer
template <bool F16, class Wait>
__device__ __forceinline__ void head_lead(Steps &steps, uint32_t *counter, AttnLds &lds, const SmallParams &p, const SmallLayer &L, uint32_t pos, float c, float sn, const float *qkv, float *out, uint32_t h, uint32_t lane,
                                          Wait &&wait) {
    using C = attn::KV<F16>;
    using CT = typename C::T;
    const uint32_t hs = p.head_size;
    const size_t hoff = (size_t)(h / p.kv_mul) * hs;
    CT *kd = (CT *)L.kcache + (size_t)pos * p.kvd + hoff, *vd = (CT *)L.vcache + (size_t)pos * p.kvd + hoff;
    const bool on = lane < hs / 2;
    const uint32_t e0 = p.rope_variant == SLAI_ROPE_NEOX ? lane : 2 * lane, e1 = p.rope_variant == SLAI_ROPE_NEOX ? lane + hs / 2 : 2 * lane + 1;
    float qb0 = 0.0f, qb1 = 0.0f, kb0 = 0.0f, kb1 = 0.0f, vb0 = 0.0f, vb1 = 0.0f;
    if (on) {
        if (L.qb) { qb0 = L.qb[(size_t)h * hs + e0]; qb1 = L.qb[(size_t)h * hs + e1]; }
        if (L.kb) { kb0 = L.kb[hoff + e0]; kb1 = L.kb[hoff + e1]; }
        if (L.vb) { vb0 = L.vb[hoff + e0]; vb1 = L.vb[hoff + e1]; }
    }
    wait();
    float rk0 = 0.0f, rk1 = 0.0f, v0 = 0.0f, v1 = 0.0f;
    if (on) {
        const float *q = qkv + (size_t)h * hs, *kn = qkv + p.dim + hoff, *vn = qkv + p.dim + p.kvd + hoff;
        const float q0 = q[e0] + qb0, q1 = q[e1] + qb1, k0 = kn[e0] + kb0, k1 = kn[e1] + kb1;
        v0 = vn[e0] + vb0; v1 = vn[e1] + vb1;
        const bool rot = p.rope_variant >= 0;
        lds.q[e0] = rot ? c * q0 - sn * q1 : q0; lds.q[e1] = rot ? sn * q0 + c * q1 : q1;
        rk0 = rot ? c * k0 - sn * k1 : k0; rk1 = rot ? sn * k0 + c * k1 : k1;
        lds.k[e0] = C::round(rk0); lds.k[e1] = C::round(rk1);
        lds.v[e0] = C::round(v0); lds.v[e1] = C::round(v1);
    }
    lds_barrier();
    lds_barrier();
    const float r = head_merge(lds, lane);
    if (lane < hs) out[(size_t)h * hs + lane] = r;
    steps.report(counter);
    if (on && h % p.kv_mul == 0) {                             // several query heads share a cache head: the first of the group writes the row (read by later launches only)
        C::store(kd + e0, rk0); C::store(kd + e1, rk1);
        C::store(vd + e0, v0); C::store(vd + e1, v1);
    }
}

template <int T, bool F16>
__global__ void __launch_bounds__(NT) decode_small_kernel(const SmallParams p) {
    touch_kernel_arguments<sizeof(SmallParams)>();
    if ((blockIdx.x & 7u) != p.die) return;
    __shared__ float xs[SMALL_WIDEST / 4 * 5];
    __shared__ AttnLds attn_lds;
    __shared__ float res[MOST], res2[MOST];
    const uint32_t wg = blockIdx.x >> 3, tid = threadIdx.x, lane = tid & 63u, wave = uniform_word(tid >> 6);
    const uint32_t E = p.dim, kvd = p.kvd, H = p.hidden, Q = E + 2 * kvd, pos = uniform_word(*p.pos_ptr);
    const bool has_head = wg < p.n_heads;
    touch_layers(p.layers, p.n_layers);
    const auto layer = [&](uint32_t l) {
        const LayerEntry *le = (const LayerEntry *)(uintptr_t)p.layers + l;
        return SmallLayer{le->q, le->k, le->v, le->o, le->gate, le->up, le->down, le->norm1, le->norm2, le->qb, le->kb, le->vb, nullptr, nullptr, nullptr, nullptr, nullptr, le->kcache, le->vcache};
    };
    if (wave == 0) {
        Steps steps{p.abort_flag, tid, p.spin_limit, aborted(p.abort_flag)};
        float c = 1.0f, sn = 0.0f;                             // rope.slang:36-39: the angle depends on (2*i) mod head_size for both variants
        if (has_head && p.rope_variant >= 0 && lane < p.head_size / 2) sincosf((float)pos * p.rope_theta[lane], &sn, &c);
        const float *x = p.x;
        for (uint32_t l = 0; l < p.n_layers; ++l) {
            const SmallLayer L = layer(l);
            float *qkv = p.work + (size_t)l * p.work_stride, *att = qkv + small_pad(Q), *x1 = att + small_pad(E), *h = x1 + small_pad(E), *x2 = h + small_pad(H);
            if (l + 1 == p.n_layers) x2 = p.x;                 // (read for the last time in layer 0, several hand-overs ago)
            uint32_t *n = p.counters + (size_t)l * SMALL_STEPS * 32;
            lead_step<END_PLAIN, NORM_RMS, 2>(steps, n, wg, lane, Q, E, xs, res, res2, x, L.norm1, p.eps, nullptr, qkv, [&]() { if (l) steps.wait(n - 32, NWG); });
            if (has_head)
                head_lead<F16>(steps, n + 32, attn_lds, p, L, pos, c, sn, qkv, att, wg, lane, [&]() { steps.wait(n, NWG); });
            lead_step<END_PLAIN, NORM_NONE, 2>(steps, n + 64, wg, lane, E, E, xs, res, res2, att, nullptr, 0.0f, x, x1, [&]() { steps.wait(n + 32, p.n_heads); });
            lead_step<END_SILU, NORM_RMS, 2>(steps, n + 96, wg, lane, H, E, xs, res, res2, x1, L.norm2, p.eps, nullptr, h, [&]() { steps.wait(n + 64, NWG); });
            lead_step<END_PLAIN, NORM_NONE, 4>(steps, n + 128, wg, lane, E, H, xs, res, res2, h, nullptr, 0.0f, x1, x2, [&]() { steps.wait(n + 96, NWG); });
            x = x2;
        }
    } else {
        const auto no_row = [](uint32_t) -> const uint8_t * { return nullptr; };
        Rows<T, 32, false> qkv, o;
        Rows<T, 32, true> gate;
        Rows<T, 64, false> down;
        HeadRows<F16> head;
        // (requests follow the barrier behind a step's products: before it wave 0 waited for them to be issued)
        const auto request_qkv = [&](uint32_t l) {
            const SmallLayer L = layer(l);
            qkv.request(wg, wave, lane, Q, E, [&](uint32_t r) { return r < E ? L.q + (size_t)r * p.stride_e : r < E + kvd ? L.k + (size_t)(r - E) * p.stride_e : L.v + (size_t)(r - E - kvd) * p.stride_e; }, no_row);
            if (has_head) head.request(p, L.kcache, L.vcache, pos, wg, wave, lane, 0);
        };
        request_qkv(0);
        for (uint32_t l = 0; l < p.n_layers; ++l) {
            const SmallLayer L = layer(l);
            lds_barrier();
            qkv.multiply(wave, lane, E, xs, res, res2);
            lds_barrier();
            o.request(wg, wave, lane, E, E, [&](uint32_t r) { return L.o + (size_t)r * p.stride_e; }, no_row);
            if (has_head) head.run(attn_lds, p, L, pos, wg, wave, lane);
            lds_barrier();
            o.multiply(wave, lane, E, xs, res, res2);
            lds_barrier();
            gate.request(wg, wave, lane, H, E, [&](uint32_t r) { return L.gate + (size_t)r * p.stride_e; }, [&](uint32_t r) { return L.up + (size_t)r * p.stride_e; });
            lds_barrier();
            gate.multiply(wave, lane, E, xs, res, res2);
            lds_barrier();
            down.request(wg, wave, lane, E, H, [&](uint32_t r) { return L.down + (size_t)r * p.stride_h; }, no_row);
            lds_barrier();
            down.multiply(wave, lane, H, xs, res, res2);
            lds_barrier();
            if (l + 1 < p.n_layers) request_qkv(l + 1);
        }
    }
}

}  // namespace

// One chunk of columns per lane: two rows of the width a wave (32 chunks), one of the FFN's (64); one workgroup per head.
bool small_shape_ok(const SmallParams &p) {
    if ((p.type != T_Q8_0 && p.type != T_Q4_0) || p.n_layers == 0) return false;
    if (p.dim == 0 || p.dim % 32 || Chunk<T_Q8_0>::nchunks(p.dim) > 32 || p.hidden == 0 || p.hidden % 32 || p.hidden > SMALL_WIDEST || p.kvd % 8) return false;
    if (p.n_heads == 0 || p.n_heads > NWG || p.kv_mul == 0 || p.head_size == 0 || p.head_size % 8 || p.head_size > 64 || p.n_heads * p.head_size != p.dim) return false;
    const auto most = [](uint32_t rows) { return (rows + NWG - 1) / NWG; };
    return most(p.dim + 2 * p.kvd) <= 2 * RW && most(p.dim) <= RW && most(p.hidden) <= 2 * RW;
}

// One workgroup per head walks the cache at 11 ns (f32) or 12 (f16) a position and layer; launches split a head over the device and grow by less than one.
// us a token of six layers, launches / this, at positions 500, 700, 900 (the slowest format and cache type of each shape; Q4_0 with an f16 cache):
//   288 wide 154 / 137, 156 / 153, 156 / 166;  480 wide 151 / 135, 151 / 151, 151 / 164;  128 wide 123 / 126, 123 / 140;  64 wide 122 / 126, 123 / 141
// A single layer of up to 128 columns has little to save.  At positions 2, 200, 400: 64 wide 32.5 / 32.3, 33.4 / 34.0, 34.9 / 36.2; with split
// attention (contexts beyond 1024) 34.6 / 32.4, 34.6 / 34.2, 34.6 / 36.4; 128 wide the same; 192 wide 35.5 / 31.9, 36.7 / 34.0, 38.0 / 36.0
uint32_t small_positions(const SmallParams &p, bool split) {
    if (p.dim >= 256) return 672;
    return p.n_layers > 1 || p.dim > 128 ? 448 : split ? 256 : 0;
}

hipError_t small_capacity(const SmallParams &p, int device, uint32_t *resident) {
    const void *kernel = p.type == T_Q8_0 ? (p.kv_f16 ? (const void *)decode_small_kernel<T_Q8_0, true> : (const void *)decode_small_kernel<T_Q8_0, false>)
                                          : (p.kv_f16 ? (const void *)decode_small_kernel<T_Q4_0, true> : (const void *)decode_small_kernel<T_Q4_0, false>);
    if (const hipError_t e = layers::resident_workgroups(kernel, device, resident)) return e;
    *resident /= 8;                                            // (eight dies)
    return hipSuccess;
}

hipError_t launch_decode_small(hipStream_t s, const SmallParams &p) {
    if (!small_shape_ok(p) || p.die > 7 || p.absent >= NWG || !p.layers || !p.work || !p.counters || !p.abort_flag || !p.x || !p.pos_ptr || (p.rope_variant >= 0 && !p.rope_theta)) return hipErrorInvalidValue;
    const dim3 grid((NWG - p.absent) * 8);
    if (p.type == T_Q8_0) {
        if (p.kv_f16) decode_small_kernel<T_Q8_0, true><<<grid, NT, 0, s>>>(p);
        else decode_small_kernel<T_Q8_0, false><<<grid, NT, 0, s>>>(p);
    } else {
        if (p.kv_f16) decode_small_kernel<T_Q4_0, true><<<grid, NT, 0, s>>>(p);
        else decode_small_kernel<T_Q4_0, false><<<grid, NT, 0, s>>>(p);
    }
    return hipGetLastError();
}

}  // namespace slai
