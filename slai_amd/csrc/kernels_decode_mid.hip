// A token of GPT-2 small as one resident launch over the whole device, gfx950.
//
// The layers of the GPT-2 forward pass (crates/slai/src/models/gpt2/cpu.rs:224-383): LayerNorm + q/k/v, attention with cache write,
// projection into the residual, LayerNorm + GELU, projection.  Embedding row, output matrix and pick stay launches of their own.
//
// Why: 63 launches that depend on each other, 5.5 us each, over 90 MB of weights that stay in the 256 MB cache.  Here every compute unit keeps a
// workgroup of sixteen waves: 3 to 12 rows of a step, at most one row a wave.
//   * vectors go through memory with the accesses of device_util.h and are their own flags: a launch starts with all of them FLOW_EMPTY, wave 0
//     of every workgroup asks for the whole vector until none of it is empty, normalises it and leaves it in LDS;
//   * the other fifteen waves multiply (a row of the FFN's width is shared by several, 64 chunks each) and ask for the next step's
//     weights as soon as they have; wave 0 finishes and writes the results;
//   * one workgroup per head takes the attention (decode_layers.h).
// us a token in the loop, launches / this: Q8_0, f32 cache, position 16: 329 / 195, 100: 330 / 201, 900: 429 / 307; Q4_0, f16 cache, 100: 322 / 218.
// A layer takes 12 us (time stamps, position 100): five hand-overs through memory, 0.4 to 1.1 us from the last result to the first workgroup's whole input and 0.8 to
// 1.6 to the last's (the FFN's, four times as wide: 1.6 and 2.2), and 0.6 to 1.1 us from input to result, the attention's 1.7 (10.7 at position 900); on one die (kernels_decode_small.hip) a token took 321 us,
// bound by instructions.  Copies of the matrices as rows are 90 MB of memory.
// Every wait is bounded: a workgroup that gives up sets a flag and waits no more, nor does any of a launch that finds the flag set; the host then
// repeats the call with launches.
#include "common.h"
#include "decode_layers.h"

namespace slai {
namespace {

using namespace layers;
constexpr uint32_t NWG = MID_WGS;

typedef uint32_t u32x4b __attribute__((ext_vector_type(4)));
constexpr int AUX_FLOW = (int)0x80000010u;                    // agent scope (sc1)
// n floats written by other workgroups of this launch (reads past them give zeros)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t flow_rsrc(const float *p, uint32_t n) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), (short)0, (int)(n * 4u), 0x00020000); }
__device__ __forceinline__ bool empty4(u32x4b v) { return v.x == FLOW_EMPTY || v.y == FLOW_EMPTY || v.z == FLOW_EMPTY || v.w == FLOW_EMPTY; }

struct Waits {
    uint32_t *abort_flag;
    uint32_t spin_limit;
    bool dead;
    // whether to look again (`missing`: this lane saw an empty word); the same in every lane
    __device__ __forceinline__ bool again(bool missing, uint32_t &looks) {
        if (dead || __builtin_amdgcn_ballot_w64(missing) == 0) return false;
        if (++looks < spin_limit) return true;
        abort_launch(abort_flag);
        dead = true;
        return false;
    }
};

// n floats of x (a multiple of 4, at most 256 NJ), LayerNorm'ed (ops/layernorm.rs:104-111) where nw is given, into LDS
template <int NJ, bool NORM>
__device__ __forceinline__ void stage_input(Waits &waits, float *xs, const float *x, uint32_t n, const float *nw, const float *nb, float eps, uint32_t lane) {
    u32x4b raw[NJ];
    float4 w[NORM ? NJ : 1], b[NORM ? NJ : 1];
    const uint32_t n4 = n / 4;
    if constexpr (NORM)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const uint32_t at = 4u * min(lane + 64u * j, n4 - 1);
            w[j] = make_float4(nw[at], nw[at + 1], nw[at + 2], nw[at + 3]);
            b[j] = make_float4(nb[at], nb[at + 1], nb[at + 2], nb[at + 3]);
        }
    const __amdgpu_buffer_rsrc_t rs = flow_rsrc(x, n);
    uint32_t looks = 0;
    bool missing;
    do {
        missing = false;
        asm volatile("" ::: "memory");                         // (the loads are made again in every round)
#pragma unroll
        for (int j = 0; j < NJ; ++j) raw[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(16u * (lane + 64u * j)), 0, AUX_FLOW);
#pragma unroll
        for (int j = 0; j < NJ; ++j) missing |= empty4(raw[j]);
    } while (waits.again(missing, looks));
    float4 v[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) v[j] = make_float4(__uint_as_float(raw[j].x), __uint_as_float(raw[j].y), __uint_as_float(raw[j].z), __uint_as_float(raw[j].w));
    if constexpr (NORM) {
        float sm = 0.0f, ss = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j) sm += (v[j].x + v[j].y) + (v[j].z + v[j].w);
        const float mean = sum64(sm) / (float)n;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (lane + 64u * j < n4) { v[j].x -= mean; v[j].y -= mean; v[j].z -= mean; v[j].w -= mean; }
            ss = fmaf(v[j].x, v[j].x, ss); ss = fmaf(v[j].y, v[j].y, ss); ss = fmaf(v[j].z, v[j].z, ss); ss = fmaf(v[j].w, v[j].w, ss);
        }
        const float scale = 1.0f / sqrtf(sum64(ss) / (float)n + eps);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            v[j].x = v[j].x * scale * w[j].x + b[j].x; v[j].y = v[j].y * scale * w[j].y + b[j].y;
            v[j].z = v[j].z * scale * w[j].z + b[j].z; v[j].w = v[j].w * scale * w[j].w + b[j].w;
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        if (lane + 64u * j < n4) *(float4 *)(xs + lds_col(4u * (lane + 64u * j))) = v[j];
}

// One wave's part of a step: chunks 64 part .. + 63 of row (wave - 1) / PARTS of the workgroup's
template <int T, int PARTS> struct RowPart {
    using F = Chunk<T>;
    typename F::Data d;
    __device__ __forceinline__ void request(const uint8_t *W, uint32_t stride, uint32_t wg, uint32_t wave, uint32_t lane, uint32_t nrows, uint32_t ncols) {
        const uint32_t r = min(nrows * wg / NWG + (wave - 1) / PARTS, nrows - 1), c = lane + 64u * ((wave - 1) % PARTS);      // (a wave without a row asks for one it does not use)
        d = F::load(W + (size_t)r * stride, ncols / 32, c < F::nchunks(ncols) ? c : 0u);
    }
    __device__ __forceinline__ void multiply(uint32_t wave, uint32_t lane, uint32_t ncols, const float *xs, float *res) const {
        const uint32_t c = lane + 64u * ((wave - 1) % PARTS);
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
        const float t = F::dot(d, ch, v, sums), s = sum64(valid ? t : 0.0f);
        if (lane == 0) res[wave - 1] = s;
    }
};

// Wave 0's part of a step.  `first`: the residual is the embedding row, which an earlier launch wrote; `last`: the result is read by later launches
template <int NJ, bool NORM, bool GELU, int PARTS>
__device__ __forceinline__ void lead_step(Waits &waits, uint32_t wg, uint32_t lane, uint32_t nrows, uint32_t ncols, float *xs, const float *res, const float *x, const float *nw,
                                          const float *nb, float eps, const float *bias, const float *residual, float *out) {
    const uint32_t r0 = nrows * wg / NWG, n = nrows * (wg + 1) / NWG - r0;
    float b = 0.0f, keep = 0.0f;
    if (lane < n) {
        if (bias) b = bias[r0 + lane];
        if (residual) keep = flow_load(residual + r0 + lane);  // (complete: this workgroup has staged all of it before)
    }
    stage_input<NJ, NORM>(waits, xs, x, ncols, nw, nb, eps, lane);
    lds_barrier();
    lds_barrier();
    if (lane < n) {
        float val = res[lane * PARTS];
#pragma unroll
        for (int q = 1; q < PARTS; ++q) val += res[lane * PARTS + q];
        val += b;
        if constexpr (GELU) val = 0.5f * val * (1.0f + tanhf(0.7978846f * val * (1.0f + 0.044715f * val * val)));       // ops/unary.rs:81-85
        flow_store(out + r0 + lane, val + keep);
    }
}

template <int T, bool F16>
__global__ void __launch_bounds__(NT) decode_mid_kernel(const SmallParams p) {
    touch_kernel_arguments<sizeof(SmallParams)>();
    constexpr int PARTS = T == T_Q8_0 ? 3 : 2;                 // rows of the FFN's width: up to 192 chunks of 16 or 128 of 32
    constexpr int NJH = (PARTS * 64 * Chunk<T>::E + 255) / 256;
    __shared__ float xs[NJH * 256 / 4 * 5];
    __shared__ AttnLds attn_lds;
    __shared__ float res[RW];
    const uint32_t wg = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wave = uniform_word(tid >> 6);
    const uint32_t E = p.dim, H = p.hidden, Q = 3 * E, hs = p.head_size, pos = uniform_word(*p.pos_ptr);
    const bool has_head = wg < p.n_heads;
    touch_layers(p.layers, p.n_layers);
    if (wave == 0) {
        Waits waits{p.abort_flag, p.spin_limit, aborted(p.abort_flag)};
        const float *x = p.x;
        for (uint32_t l = 0; l < p.n_layers; ++l) {
            const LayerEntry *L = (const LayerEntry *)(uintptr_t)p.layers + l;
            float *qkv = p.work + (size_t)l * p.work_stride, *att = qkv + small_pad(Q), *x1 = att + small_pad(E), *h = x1 + small_pad(E), *x2 = h + small_pad(H);
            if (l + 1 == p.n_layers) x2 = p.x;                 // (read for the last time in layer 0, several hand-overs ago)
            lead_step<4, true, false, 1>(waits, wg, lane, Q, E, xs, res, x, L->norm1, L->norm1b, p.eps, L->qb, nullptr, qkv);
            if (has_head) {
                // the fresh query, key and value of this head (one element a lane): LDS, then the cache
                using C = attn::KV<F16>;
                using CT = typename C::T;
                const bool on = lane < hs;
                const float *src = qkv + (size_t)wg * hs + (on ? lane : 0u);
                float q, k, v;
                uint32_t looks = 0;
                bool missing;
                do {
                    q = flow_load(src); k = flow_load(src + E); v = flow_load(src + 2 * E);
                    missing = __float_as_uint(q) == FLOW_EMPTY || __float_as_uint(k) == FLOW_EMPTY || __float_as_uint(v) == FLOW_EMPTY;
                } while (waits.again(missing, looks));
                if (on) { attn_lds.q[lane] = q; attn_lds.k[lane] = C::round(k); attn_lds.v[lane] = C::round(v); }
                lds_barrier();
                lds_barrier();
                const float r = head_merge(attn_lds, lane);
                if (on) {
                    flow_store(att + (size_t)wg * hs + lane, r);
                    C::store((CT *)L->kcache + (size_t)pos * p.kvd + (size_t)wg * hs + lane, k);      // (read by later launches only)
                    C::store((CT *)L->vcache + (size_t)pos * p.kvd + (size_t)wg * hs + lane, v);
                }
            }
            lead_step<4, false, false, 1>(waits, wg, lane, E, E, xs, res, att, nullptr, nullptr, 0.0f, L->ob, x, x1);
            lead_step<4, true, true, 1>(waits, wg, lane, H, E, xs, res, x1, L->norm2, L->norm2b, p.eps, L->upb, nullptr, h);
            lead_step<NJH, false, false, PARTS>(waits, wg, lane, E, H, xs, res, h, nullptr, nullptr, 0.0f, L->downb, x1, x2);
            x = x2;
        }
    } else {
        RowPart<T, 1> qkv, o, up;
        RowPart<T, PARTS> down;
        HeadRows<F16> head;
        const auto request_qkv = [&](uint32_t l) {
            const LayerEntry *L = (const LayerEntry *)(uintptr_t)p.layers + l;
            qkv.request(L->q, p.stride_e, wg, wave, lane, Q, E);
            if (has_head) head.request(p, L->kcache, L->vcache, pos, wg, wave, lane, 0);
        };
        request_qkv(0);
        for (uint32_t l = 0; l < p.n_layers; ++l) {
            const LayerEntry *L = (const LayerEntry *)(uintptr_t)p.layers + l;
            lds_barrier();
            qkv.multiply(wave, lane, E, xs, res);
            lds_barrier();
            o.request(L->o, p.stride_e, wg, wave, lane, E, E);
            if (has_head) {
                SmallLayer caches{};
                caches.kcache = L->kcache; caches.vcache = L->vcache;
                head.run(attn_lds, p, caches, pos, wg, wave, lane);
            }
            lds_barrier();
            o.multiply(wave, lane, E, xs, res);
            lds_barrier();
            up.request(L->up, p.stride_e, wg, wave, lane, H, E);
            lds_barrier();
            up.multiply(wave, lane, E, xs, res);
            lds_barrier();
            down.request(L->down, p.stride_h, wg, wave, lane, E, H);
            lds_barrier();
            down.multiply(wave, lane, H, xs, res);
            lds_barrier();
            if (l + 1 < p.n_layers) request_qkv(l + 1);
        }
    }
}

const void *kernel_of(const SmallParams &p) {
    if (p.type == T_Q8_0) return p.kv_f16 ? (const void *)decode_mid_kernel<T_Q8_0, true> : (const void *)decode_mid_kernel<T_Q8_0, false>;
    return p.kv_f16 ? (const void *)decode_mid_kernel<T_Q4_0, true> : (const void *)decode_mid_kernel<T_Q4_0, false>;
}

}  // namespace

// One row a wave, of at most 64 chunks of columns (the FFN's: of at most PARTS times as many, and PARTS waves a row); one workgroup per head.
bool mid_shape_ok(const SmallParams &p) {
    if ((p.type != T_Q8_0 && p.type != T_Q4_0) || p.n_layers == 0) return false;
    const uint32_t e = p.type == T_Q8_0 ? 16u : 32u, parts = p.type == T_Q8_0 ? 3u : 2u;
    if (p.dim == 0 || p.dim % 32 || p.dim > 1024 || p.dim / e > 64 || p.hidden == 0 || p.hidden % 32 || p.hidden / e > 64 * parts || p.kvd != p.dim || p.kv_mul != 1) return false;
    if (p.n_heads == 0 || p.n_heads > NWG || p.head_size == 0 || p.head_size % 8 || p.head_size > 64 || p.n_heads * p.head_size != p.dim) return false;
    const auto most = [](uint32_t rows) { return (rows + NWG - 1) / NWG; };
    return most(3 * p.dim) <= RW && most(p.hidden) <= RW && most(p.dim) * parts <= RW;
}

// The same walk of the cache as on one die (small_positions), but the launches that it saves are the longer the wider the model is.  us a token of six
// layers, launches / this (Q4_0, f16 cache, the slowest):
//   96 wide, position 250: 132 / 130, 400: 132 / 139;  320, 500: 154 / 151, 700: 155 / 166;  384, 700: 164 / 162;  512, 900: 166 / 172;
//   640, 1100: 189 / 191;  768, 900: 188 / 174, 1100: 188 / 192;  1024, 1000: 178 / 182, Q8_0 181 / 172
// and where contexts of up to 1024 leave the launches' attention whole, two layers at positions 2 and 100: 64 wide 50.3 / 49.1, 50.5 / 50.4; 96 in 12 heads 48.8 / 50.1,
// 48.7 / 51.4, in 3 heads 48.3 / 48.8, 48.5 / 50.0; 128 wide 50.1 / 48.6, 50.1 / 49.9; one layer of 64 34.3 / 34.6, 34.6 / 35.3
uint32_t mid_positions(const SmallParams &p, bool split) {
    if (!split && p.dim < 128 && (p.dim > 64 || p.n_layers == 1)) return 0;
    return min(p.dim * 8 / 5, p.type == T_Q4_0 ? 960u : 1024u);
}

hipError_t mid_capacity(const SmallParams &p, int device, uint32_t *resident) { return resident_workgroups(kernel_of(p), device, resident); }

hipError_t launch_decode_mid(hipStream_t s, const SmallParams &p) {
    if (!mid_shape_ok(p) || p.absent >= NWG || !p.layers || !p.work || !p.abort_flag || !p.x || !p.pos_ptr || p.rope_variant >= 0) return hipErrorInvalidValue;
    if (p.type == T_Q8_0) {
        if (p.kv_f16) decode_mid_kernel<T_Q8_0, true><<<NWG - p.absent, NT, 0, s>>>(p);
        else decode_mid_kernel<T_Q8_0, false><<<NWG - p.absent, NT, 0, s>>>(p);
    } else {
        if (p.kv_f16) decode_mid_kernel<T_Q4_0, true><<<NWG - p.absent, NT, 0, s>>>(p);
        else decode_mid_kernel<T_Q4_0, false><<<NWG - p.absent, NT, 0, s>>>(p);
    }
    return hipGetLastError();
}

}  // namespace slai
