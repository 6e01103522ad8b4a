// Decoder-shell kernels for batch-1 autoregressive decode around the packed
// linears on gfx950 (Qwen3 geometry): embedding gather, residual add +
// RMSNorm, per-head q/k RMSNorm + rotate-half RoPE + KV-cache append,
// split-sequence grouped-query attention, SiLU-gated product, bf16 output
// projection with per-workgroup argmax partials, and greedy selection.
//
// All kernels read the token position from device memory, so one captured
// decode step replays for every position. Every reduction runs in a fixed
// order (wave butterflies, then waves in index order, then sequence blocks in
// index order), so results are identical from run to run.
#include <math.h>

#include "nq_common.h"
#include "../../include/nqamd_shell.h"

namespace {

using nq::f32_to_bf16_bits;

constexpr int kWave = 64;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kSeqBlock = nq::kAttnBlockRows;  // cache rows per attention block
constexpr int kRowThreads = 256;        // per-row kernels
constexpr int kProjWaves = 4;           // output projection: waves per workgroup (2 or 8: 13% slower)
constexpr int kProjLoads = 32;          // 16-byte weight loads per lane in flight

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Wave reductions with DPP row operations and four lane reads (no LDS round
// trips); every lane gets the result, combined in a fixed order.
// Lane value CTRL-permuted within rows; `identity` where a source lane is off.
template <int CTRL>
__device__ __forceinline__ float dpp_src(float x, float identity) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(identity), __float_as_int(x), CTRL, 0xf, 0xf, false));
}

__device__ __forceinline__ float row_lane(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__device__ __forceinline__ float wave_sum(float v) {
    v += dpp_src<0xB1>(v, 0.0f);   // quad_perm [1,0,3,2]
    v += dpp_src<0x4E>(v, 0.0f);   // quad_perm [2,3,0,1]
    v += dpp_src<0x141>(v, 0.0f);  // row_half_mirror
    v += dpp_src<0x140>(v, 0.0f);  // row_mirror
    return (row_lane(v, 0) + row_lane(v, 16)) + (row_lane(v, 32) + row_lane(v, 48));
}

// Max / sum over each row of 16 lanes (every lane of the row gets it).
__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp_src<0xB1>(v, -INFINITY));
    v = fmaxf(v, dpp_src<0x4E>(v, -INFINITY));
    v = fmaxf(v, dpp_src<0x141>(v, -INFINITY));
    return fmaxf(v, dpp_src<0x140>(v, -INFINITY));
}

__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_src<0xB1>(v, 0.0f);
    v += dpp_src<0x4E>(v, 0.0f);
    v += dpp_src<0x141>(v, 0.0f);
    return v + dpp_src<0x140>(v, 0.0f);
}

__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_src<0xB1>(v, -INFINITY));
    v = fmaxf(v, dpp_src<0x4E>(v, -INFINITY));
    v = fmaxf(v, dpp_src<0x141>(v, -INFINITY));
    v = fmaxf(v, dpp_src<0x140>(v, -INFINITY));
    return fmaxf(fmaxf(row_lane(v, 0), row_lane(v, 16)), fmaxf(row_lane(v, 32), row_lane(v, 48)));
}

// Elements [i, i + 8) of a typed buffer as fp32; i % 8 == 0 and the buffer is
// 16-byte aligned (checked on the host).
__device__ __forceinline__ void load8(const void* __restrict__ p, int dtype, int64_t i, float (&v)[8]) {
    if (dtype == NQ_DTYPE_F32) {
        const float4* q = reinterpret_cast<const float4*>(static_cast<const float*>(p) + i);
        const float4 a = q[0], b = q[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        return;
    }
    const uint4 u = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + i);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
    if (dtype == NQ_DTYPE_BF16) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[2 * j] = bf16_lo(w[j]);
            v[2 * j + 1] = bf16_hi(w[j]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[2 * j] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w[j] & 0xffffu)));
            v[2 * j + 1] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w[j] >> 16)));
        }
    }
}

__device__ __forceinline__ uint32_t pack2(int dtype, float a, float b) {
    if (dtype == NQ_DTYPE_BF16) return f32_to_bf16_bits(a) | (static_cast<uint32_t>(f32_to_bf16_bits(b)) << 16);
    const uint16_t ha = __builtin_bit_cast(uint16_t, static_cast<_Float16>(a));
    const uint16_t hb = __builtin_bit_cast(uint16_t, static_cast<_Float16>(b));
    return ha | (static_cast<uint32_t>(hb) << 16);
}

__device__ __forceinline__ void store8(void* __restrict__ p, int dtype, int64_t i, const float (&v)[8]) {
    if (dtype == NQ_DTYPE_F32) {
        float4* q = reinterpret_cast<float4*>(static_cast<float*>(p) + i);
        q[0] = make_float4(v[0], v[1], v[2], v[3]);
        q[1] = make_float4(v[4], v[5], v[6], v[7]);
        return;
    }
    uint4 u;
    u.x = pack2(dtype, v[0], v[1]);
    u.y = pack2(dtype, v[2], v[3]);
    u.z = pack2(dtype, v[4], v[5]);
    u.w = pack2(dtype, v[6], v[7]);
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p) + i) = u;
}

// ---------------------------------------------------------------------------
// Embedding gather.

__global__ __launch_bounds__(kRowThreads) void k_embedding(const int64_t* __restrict__ ids, const void* __restrict__ table,
                                                           int dtype, int64_t vocab, int64_t hidden,
                                                           const float* __restrict__ scale, float* __restrict__ out,
                                                           float* __restrict__ slots) {
    const int64_t t = blockIdx.x;
    const int64_t id = ids[t];
    const bool ok = id >= 0 && id < vocab;
    const float s = scale ? scale[0] : 1.0f;
    for (int64_t i = threadIdx.x * 8; i < hidden; i += kRowThreads * 8) {
        float v[8];
        if (ok) {
            load8(table, dtype, id * hidden + i, v);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = __fmul_rn(v[j], s);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = __builtin_nanf("");
        }
        store8(out, NQ_DTYPE_F32, t * hidden + i, v);
        if (slots) {  // uniform. hidden % 16 == 0: threads 2k and 2k + 1 hold the 16 columns of one slot
            float sq = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) sq = fmaf(v[j], v[j], sq);
            const float pair = sq + __shfl_xor(sq, 1, kWave);
            if ((threadIdx.x & 1) == 0) slots[t * (hidden / 16) + i / 16] = pair;
        }
    }
}

// ---------------------------------------------------------------------------
// Residual add + RMSNorm, one workgroup of kNormThreads per token row. Thread
// i holds elements [8 (i + kNormThreads j), +8) for j < NV in registers, so
// residual, delta and weight are loaded in one round trip; the sum of squares
// goes through wave butterflies and then the wave sums in wave order.

constexpr int kNormThreads = 512;

template <int NV>
__global__ __launch_bounds__(kNormThreads) void k_add_rmsnorm(float* __restrict__ residual, const void* __restrict__ delta,
                                                              int ddt, const void* __restrict__ weight, int wdt,
                                                              float eps, int64_t hidden, void* __restrict__ out, int odt) {
    __shared__ float red[kNormThreads / kWave];
    const int64_t row = static_cast<int64_t>(blockIdx.x) * hidden;
    float v[NV][8], w[NV][8];
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int64_t i = (threadIdx.x + static_cast<int64_t>(kNormThreads) * j) * 8;
        if (i < hidden) {
            load8(residual, NQ_DTYPE_F32, row + i, v[j]);
            load8(weight, wdt, i, w[j]);
            if (delta) {
                float d[8];
                load8(delta, ddt, row + i, d);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[j][e] = __fadd_rn(v[j][e], d[e]);
                store8(residual, NQ_DTYPE_F32, row + i, v[j]);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[j][e] = w[j][e] = 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(v[j][e], v[j][e], ss);
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = ss;
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormThreads / kWave; ++i) total += red[i];
    const float inv = 1.0f / sqrtf(__fadd_rn(total / static_cast<float>(hidden), eps));  // no fma contraction
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int64_t i = (threadIdx.x + static_cast<int64_t>(kNormThreads) * j) * 8;
        if (i < hidden) {
            float o[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = __fmul_rn(w[j][e], __fmul_rn(v[j][e], inv));
            store8(out, odt, row + i, o);
        }
    }
}

// ---------------------------------------------------------------------------
// q/k per-head RMSNorm + rotate-half RoPE + KV-cache append. One wave per
// (token, head); grid.y = q_heads + kv_heads. Lane l holds elements
// d = l + 64 j, so for head_dim >= 128 the rotate-half partner d +- D/2 is
// element j +- E/2 of the same lane; for head_dim 64 it is lane l ^ 32.

// Element i of an F32 / F16 / BF16 buffer from one unconditional 32-bit load
// (the fp32 itself, or the pair of 16-bit elements 2 (i / 2) and 2 (i / 2) + 1,
// counted from the buffer's start: the callers' buffers hold head_dim
// elements, an even count): no branch surrounds the load and nothing is
// derived from it before use, so a wave issues all of them before waiting on
// any.
struct RawHalves {
    uint32_t word, shift;
};

__device__ __forceinline__ RawHalves load_raw(const void* __restrict__ p, int dtype, int64_t i) {
    const bool wide = dtype == NQ_DTYPE_F32;
    RawHalves r;
    r.word = static_cast<const uint32_t*>(p)[wide ? i : i >> 1];
    r.shift = wide ? 0u : static_cast<uint32_t>(i & 1) << 4;
    return r;
}

__device__ __forceinline__ float raw_value(const RawHalves& r, int dtype) {
    const uint32_t half = r.word >> r.shift;
    const float f32 = __uint_as_float(r.word);
    const float bf16 = __uint_as_float(half << 16);
    const float f16 = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(half)));
    return dtype == NQ_DTYPE_F32 ? f32 : (dtype == NQ_DTYPE_BF16 ? bf16 : f16);
}

// The operands of norm_rope_regs for one lane: the head vector's elements
// d = lane + 64 j and the norm weights (loaded from the head vector itself,
// and ignored, when there is no weight).
template <int D>
struct NormRopeIn {
    float x[D / kWave];
    RawHalves w[D / kWave];
};

template <int D>
__device__ __forceinline__ void load_norm_rope_in(NormRopeIn<D>& in, const float* __restrict__ src,
                                                  const void* __restrict__ nw, int ndt, int lane) {
    const void* wp = nw ? nw : static_cast<const void*>(src);
    const int wdt = nw ? ndt : NQ_DTYPE_F32;
#pragma unroll
    for (int j = 0; j < D / kWave; ++j) {
        in.x[j] = src[lane + kWave * j];
        in.w[j] = load_raw(wp, wdt, lane + kWave * j);
    }
}

// norm_rope on loaded operands: cs / sn are the lane's RoPE table entries
// (index d mod D/2 of the position's row).
template <int D>
__device__ __forceinline__ void norm_rope_regs(const NormRopeIn<D>& in, bool has_w, int ndt, float eps,
                                               const float (&cs)[D / kWave], const float (&sn)[D / kWave], int lane,
                                               float (&y)[D / kWave]) {
    constexpr int E = D / kWave;
    constexpr int kHalf = D / 2;
    float x[E];
#pragma unroll
    for (int j = 0; j < E; ++j) x[j] = in.x[j];
    // Branch-free (a branch here would sink the weight loads into it).
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) ss = fmaf(x[j], x[j], ss);
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(__fadd_rn(ss / static_cast<float>(D), eps));  // no fma contraction
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const float normed = __fmul_rn(raw_value(in.w[j], ndt), __fmul_rn(x[j], inv));
        x[j] = has_w ? normed : x[j];
    }
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int d = lane + kWave * j;
        const bool first = d < kHalf;
        float partner;
        if constexpr (E == 1) {
            partner = __shfl_xor(x[0], 32, kWave);
        } else {
            partner = first ? x[j + E / 2] : x[j - E / 2];
        }
        const float rot = first ? -partner : partner;
        y[j] = __fadd_rn(__fmul_rn(x[j], cs[j]), __fmul_rn(rot, sn[j]));
    }
}

// Lane's E = D / 64 elements d = lane + 64 j of one head vector: RMSNorm with
// weight nw (when not NULL), then rotate-half RoPE with the table rows cr/sr
// (the same arithmetic as the fused decode attention, norm_rope_regs).
template <int D>
__device__ __forceinline__ void norm_rope(const float* __restrict__ src, const void* __restrict__ nw, int ndt, float eps,
                                          const float* __restrict__ cr, const float* __restrict__ sr, int lane,
                                          float (&y)[D / kWave]) {
    constexpr int E = D / kWave;
    NormRopeIn<D> in;
    load_norm_rope_in<D>(in, src, nw, ndt, lane);
    float cs[E], sn[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int d = lane + kWave * j;
        const int fi = d < D / 2 ? d : d - D / 2;
        cs[j] = cr[fi];
        sn[j] = sr[fi];
    }
    norm_rope_regs<D>(in, nw != nullptr, ndt, eps, cs, sn, lane, y);
}

// One wave per (token, head), four heads to a workgroup. A head is 512 bytes
// in and 512 or 256 out, so with a workgroup per wave the rate at which
// workgroups start was the bound, not memory: 1531 tokens of 32/8 heads, D 128,
// took 18.8 us (3.7 TB/s over 69 MB), 15.2 with two, four or eight (4.5 TB/s);
// 4096 tokens 42.8 -> 35.2; one token 2.2 either way.
constexpr int kHeadsPerGroup = 4;

template <int D>
__global__ __launch_bounds__(kHeadsPerGroup* kWave) void k_qk_norm_rope_cache(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, int q_heads,
    int kv_heads, const void* __restrict__ q_norm, const void* __restrict__ k_norm, int ndt, float eps,
    const float* __restrict__ cos_table, const float* __restrict__ sin_table, const int32_t* __restrict__ position,
    int64_t max_positions, float* __restrict__ q_out, void* __restrict__ k_cache, void* __restrict__ v_cache, int cdt) {
    constexpr int E = D / kWave;
    const int64_t t = blockIdx.x;
    const int h = blockIdx.y * kHeadsPerGroup + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int64_t pos = static_cast<int64_t>(position[0]) + t;
    if (h >= q_heads + kv_heads || pos < 0 || pos >= max_positions) return;
    const bool is_q = h < q_heads;
    const int g = is_q ? h : h - q_heads;
    const float* src = is_q ? q + (t * q_heads + h) * D : k + (t * kv_heads + g) * D;
    float y[E];
    norm_rope<D>(src, is_q ? q_norm : k_norm, ndt, eps, cos_table + pos * (D / 2), sin_table + pos * (D / 2), lane, y);
    if (is_q) {
        float* dst = q_out + (t * q_heads + h) * D;
#pragma unroll
        for (int j = 0; j < E; ++j) dst[lane + kWave * j] = y[j];
        return;
    }
    const int64_t crow = (static_cast<int64_t>(g) * max_positions + pos) * D;
    const float* vs = v + (t * kv_heads + g) * D;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int d = lane + kWave * j;
        nq::store_f32_as(k_cache, cdt, crow + d, y[j]);
        nq::store_f32_as(v_cache, cdt, crow + d, vs[d]);
    }
}

// ---------------------------------------------------------------------------
// Attention, pass 1: one workgroup per (kv head, block of QT queries,
// 64-row cache block s); wave w serves q head kv_head * G + w. The K rows of
// the block are copied to LDS as stored (16-byte copies, padded rows); lane j
// scores cache row 64 s + j against the query (fp32, in LDS), the wave forms
// its softmax partial (max m, sum l) and lane pairs of dimensions accumulate
// P.V straight from the V rows (all waves of the workgroup read the same rows,
// so they come from cache). The partial goes to the workspace.

template <int CT>
constexpr int cache_bytes() { return CT == NQ_DTYPE_F32 ? 4 : 2; }

template <int D, int CT>
constexpr int k_row_bytes() { return D * cache_bytes<CT>() + 16; }

// k_attention_blocks stages the block's V rows in LDS too when a row is at
// most 256 bytes (the K and V blocks then fit 64 KB with the per-wave rows).
template <int D, int CT>
constexpr bool attention_stages_v() { return D * cache_bytes<CT>() <= 256; }

template <int D, int CT>
constexpr size_t attention_lds(int waves) {
    return static_cast<size_t>(kSeqBlock) * k_row_bytes<D, CT>() +
           (attention_stages_v<D, CT>() ? static_cast<size_t>(kSeqBlock) * D * cache_bytes<CT>() : 0) +
           static_cast<size_t>(waves) * (D + kSeqBlock) * 4;
}

template <int CT>
__device__ __forceinline__ float cache_value(uint32_t bits16) {
    if constexpr (CT == NQ_DTYPE_BF16) return __uint_as_float(bits16 << 16);
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits16)));
}

// Dot product of one staged K row with the query (both D long).
template <int D, int CT>
__device__ __forceinline__ float k_row_dot(const char* __restrict__ kr, const float* __restrict__ qw) {
    // Four accumulators (dimensions d mod 4), combined at the end: four short
    // dependency chains instead of one of length D.
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
    if constexpr (CT == NQ_DTYPE_F32) {
#pragma unroll 8
        for (int d = 0; d < D; d += 4) {
            const float4 kk = *reinterpret_cast<const float4*>(kr + 4 * d);
            const float4 qq = *reinterpret_cast<const float4*>(qw + d);
            a0 = fmaf(kk.x, qq.x, a0);
            a1 = fmaf(kk.y, qq.y, a1);
            a2 = fmaf(kk.z, qq.z, a2);
            a3 = fmaf(kk.w, qq.w, a3);
        }
    } else {
#pragma unroll 4
        for (int d = 0; d < D; d += 8) {
            const uint4 u = *reinterpret_cast<const uint4*>(kr + 2 * d);
            const float4 qa = *reinterpret_cast<const float4*>(qw + d);
            const float4 qb = *reinterpret_cast<const float4*>(qw + d + 4);
            a0 = fmaf(cache_value<CT>(u.x & 0xffffu), qa.x, a0);
            a1 = fmaf(cache_value<CT>(u.x >> 16), qa.y, a1);
            a2 = fmaf(cache_value<CT>(u.y & 0xffffu), qa.z, a2);
            a3 = fmaf(cache_value<CT>(u.y >> 16), qa.w, a3);
            a0 = fmaf(cache_value<CT>(u.z & 0xffffu), qb.x, a0);
            a1 = fmaf(cache_value<CT>(u.z >> 16), qb.y, a1);
            a2 = fmaf(cache_value<CT>(u.w & 0xffffu), qb.z, a2);
            a3 = fmaf(cache_value<CT>(u.w >> 16), qb.w, a3);
        }
    }
    return (a0 + a1) + (a2 + a3);
}

// E consecutive cache elements (E = D / 64, lane's dimensions) as fp32.
template <int E, int CT>
__device__ __forceinline__ void load_v(const char* __restrict__ p, float (&v)[E]) {
    if constexpr (CT == NQ_DTYPE_F32) {
#pragma unroll
        for (int j = 0; j < E; ++j) v[j] = reinterpret_cast<const float*>(p)[j];
    } else if constexpr (E == 1) {
        v[0] = cache_value<CT>(*reinterpret_cast<const uint16_t*>(p));
    } else {
#pragma unroll
        for (int j = 0; j < E; j += 2) {
            const uint32_t u = reinterpret_cast<const uint32_t*>(p)[j / 2];
            v[j] = cache_value<CT>(u & 0xffffu);
            v[j + 1] = cache_value<CT>(u >> 16);
        }
    }
}

__device__ __forceinline__ int64_t attn_part_index(int64_t t, int h, int s, int q_heads, int blocks) {
    return (t * q_heads + h) * blocks + s;
}

template <int D, int CT>
__global__ __launch_bounds__(1024) void k_attention_blocks(const float* __restrict__ q, const char* __restrict__ k_cache,
                                                           const char* __restrict__ v_cache, int64_t tokens,
                                                           int q_heads, int kv_heads, int qt,
                                                           const int32_t* __restrict__ position, int64_t max_positions,
                                                           float scaling, float* __restrict__ part_ml,
                                                           float* __restrict__ part_acc) {
    constexpr int E = D / kWave;
    constexpr int EB = cache_bytes<CT>();
    constexpr int RB = k_row_bytes<D, CT>();
    constexpr int PIECES = D * EB / 16;  // 16-byte pieces per row
    constexpr int U = 8;                 // V rows per unrolled step
    constexpr bool SV = attention_stages_v<D, CT>();
    constexpr int VRB = D * EB;          // V row in LDS
    extern __shared__ float lds_raw[];
    char* klds = reinterpret_cast<char*>(lds_raw);
    char* vlds = klds + kSeqBlock * RB;                                         // [64][D] when SV
    float* qv = reinterpret_cast<float*>(vlds + (SV ? kSeqBlock * VRB : 0));  // [waves][D]
    float* pv = qv + (blockDim.x / kWave) * D;                                  // [waves][64]

    const int group = q_heads / kv_heads;
    const int g = blockIdx.x % kv_heads;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x / kv_heads) * qt;
    const int s = blockIdx.y;
    const int blocks = gridDim.y;
    const int64_t p0 = position[0];
    const int64_t row0 = static_cast<int64_t>(s) * kSeqBlock;
    const int64_t t_end = t0 + qt < tokens ? t0 + qt : tokens;
    // Highest cache row any query of this workgroup may see.
    int64_t last = p0 + t_end - 1;
    if (last >= max_positions) last = max_positions - 1;
    if (p0 < 0 || row0 > last) return;  // uniform: no query of this workgroup reaches row0
    const int rows = static_cast<int>((last - row0 + 1) < kSeqBlock ? (last - row0 + 1) : kSeqBlock);

    // Copy K rows [row0, row0 + rows) of kv head g to LDS as stored, and the
    // V rows too when they fit (every query of the workgroup reads them).
    const int64_t head_row0 = static_cast<int64_t>(g) * max_positions + row0;
    const char* kbase = k_cache + head_row0 * D * EB;
    const char* vbase = v_cache + head_row0 * D * EB;
    for (int i = threadIdx.x; i < rows * PIECES; i += blockDim.x) {
        const int r = i / PIECES, c = i % PIECES;
        const uint4 kq = *reinterpret_cast<const uint4*>(kbase + (static_cast<int64_t>(r) * D) * EB + 16 * c);
        if constexpr (SV) {
            const uint4 vq = *reinterpret_cast<const uint4*>(vbase + (static_cast<int64_t>(r) * D) * EB + 16 * c);
            *reinterpret_cast<uint4*>(vlds + r * VRB + 16 * c) = vq;
        }
        *reinterpret_cast<uint4*>(klds + r * RB + 16 * c) = kq;
    }
    const int w = threadIdx.x / kWave;
    const int lane = threadIdx.x & (kWave - 1);
    const int h = g * group + w;
    float* qw = qv + w * D;
    float* pw = pv + w * kSeqBlock;
    const char* vlane = SV ? vlds + lane * E * EB : v_cache + (head_row0 * D + lane * E) * EB;
    __syncthreads();

    for (int64_t t = t0; t < t_end; ++t) {
        const int64_t pt = p0 + t;
        if (pt < row0 || pt >= max_positions) continue;  // uniform per workgroup
        const float* qs = q + (t * q_heads + h) * D;
#pragma unroll
        for (int j = 0; j < E; ++j) qw[lane + kWave * j] = qs[lane + kWave * j];
        __builtin_amdgcn_wave_barrier();
        const int nvalid = static_cast<int>((pt - row0 + 1) < kSeqBlock ? (pt - row0 + 1) : kSeqBlock);
        const bool valid = lane < nvalid;
        // Lanes past the staged rows score row 0 (always staged) and are masked.
        const float dot = k_row_dot<D, CT>(klds + (lane < rows ? lane : 0) * RB, qw);
        const float score = valid ? dot * scaling : -INFINITY;
        const float m = wave_max(score);
        const float p = valid ? expf(score - m) : 0.0f;
        const float l = wave_sum(p);
        pw[lane] = p;
        __builtin_amdgcn_wave_barrier();
        float acc[E];
#pragma unroll
        for (int j = 0; j < E; ++j) acc[j] = 0.0f;
        for (int r0 = 0; r0 < nvalid; r0 += U) {
            float vv[U][E];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int r = r0 + u < nvalid ? r0 + u : nvalid - 1;  // p is 0 past nvalid
                load_v<E, CT>(vlane + static_cast<int64_t>(r) * D * EB, vv[u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float pr = pw[(r0 + u) & (kSeqBlock - 1)];
#pragma unroll
                for (int j = 0; j < E; ++j) acc[j] = fmaf(pr, vv[u][j], acc[j]);
            }
        }
        const int64_t pi = attn_part_index(t, h, s, q_heads, blocks);
        if (lane == 0) {
            part_ml[2 * pi] = m;
            part_ml[2 * pi + 1] = l;
        }
        float* pa = part_acc + pi * D + lane * E;
#pragma unroll
        for (int j = 0; j < E; ++j) pa[j] = acc[j];
        __builtin_amdgcn_wave_barrier();  // qw / pw are rewritten for the next query
    }
}

// Attention, pass 2: merge the blocks (of block_rows cache rows each) of one
// (token, q head). GROUPS groups of D threads take rounds of ROUND blocks in
// turn and meet in LDS in group order. Bound by latency: every load of a round
// is issued before any use, and the first round before the position is read
// (block indices clamped to the grid's blocks; blocks past the position weigh
// 0). 64 blocks of one token, 32 heads of 128: 3.6 us in eight groups, 7.1 us
// in one (four rounds one after the other).
template <int D, int ROUND, int GROUPS>
__global__ __launch_bounds__(D * GROUPS) void k_attention_merge(
    const float* __restrict__ part_ml, const float* __restrict__ part_acc, int q_heads, int blocks, int block_rows,
    const int32_t* __restrict__ position, int64_t max_positions, void* __restrict__ out, int odt) {
    const int h = blockIdx.x;
    const int64_t t = blockIdx.y;
    const int d = threadIdx.x % D, group = threadIdx.x / D;
    const int64_t o = (t * q_heads + h) * D + d;
    const int64_t p0 = attn_part_index(t, h, 0, q_heads, blocks);
    float mb[ROUND], lb[ROUND], ab[ROUND];
    const auto load_round = [&](const int b0, const int last) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < ROUND; ++i) {
            const int64_t pb = p0 + (b0 + i < last ? b0 + i : last);
            mb[i] = part_ml[2 * pb];
            lb[i] = part_ml[2 * pb + 1];
            ab[i] = part_acc[pb * D + d];
        }
    };
    const int first = group * ROUND;
    load_round(first, blocks - 1);
    const int64_t pt = static_cast<int64_t>(position[0]) + t;
    const bool in_range = pt >= 0 && pt < max_positions;  // uniform
    const int nb = in_range ? static_cast<int>(pt / block_rows) + 1 : 1;
    float mrun = -INFINITY, lsum = 0.0f, acc = 0.0f;
    for (int b0 = first; b0 < nb; b0 += GROUPS * ROUND) {
        if (b0 > first) load_round(b0, nb - 1);
        float mnew = mrun;
#pragma unroll
        for (int i = 0; i < ROUND; ++i) mnew = b0 + i < nb ? fmaxf(mnew, mb[i]) : mnew;
        const float base = mnew == -INFINITY ? 0.0f : mnew;  // every block so far weighs 0 (-inf - -inf is NaN)
        const float keep = nq::merge_exp(mrun - base);  // 0 in the first round
        lsum *= keep;
        acc *= keep;
#pragma unroll
        for (int i = 0; i < ROUND; ++i) {
            if (b0 + i < nb) {  // a select: slots past the position may hold anything
                const float f = nq::merge_exp(mb[i] - base);
                lsum = fmaf(lb[i], f, lsum);
                acc = fmaf(ab[i], f, acc);
            }
        }
        mrun = mnew;
    }
    if constexpr (GROUPS > 1) {
        __shared__ float g_acc[GROUPS][D], g_m[GROUPS], g_l[GROUPS];
        g_acc[group][d] = acc;
        if (d == 0) g_m[group] = mrun, g_l[group] = lsum;
        __syncthreads();
        if (group > 0) return;
        const int groups = nb < (GROUPS - 1) * ROUND + 1 ? (nb + ROUND - 1) / ROUND : GROUPS;  // that hold a block
        float mnew = mrun;
        for (int i = 1; i < groups; ++i) mnew = fmaxf(mnew, g_m[i]);
        mnew = mnew == -INFINITY ? 0.0f : mnew;
        const float keep = nq::merge_exp(mrun - mnew);
        lsum *= keep;
        acc *= keep;
        for (int i = 1; i < groups; ++i) {
            const float f = nq::merge_exp(g_m[i] - mnew);
            lsum = fmaf(g_l[i], f, lsum);
            acc = fmaf(g_acc[i][d], f, acc);
        }
    }
    if (!in_range) acc = 0.0f, lsum = 1.0f;
    nq::store_f32_as(out, odt, o, acc / lsum);
}

// ---------------------------------------------------------------------------
// One-token decode attention on MFMA (head_dim 128, four q heads per kv head,
// 16-bit cache): the same workgroup grid, loads, staging, RoPE / KV append and
// partial output as k_decode_attention below, with the two products on
// v_mfma_f32_16x16x32 (bf16 or f16, the cache's type). The query and the
// softmax weights are fp32; each is split into three 16-bit parts (the
// rounding of the value, of its remainder and of the remainder's remainder),
// which occupy A rows 4h, 4h + 1, 4h + 2 for q head h of the group (row
// 4h + 3 is zero), so the products carry about 24 bits of the fp32 operand
// and K / V (stored 16-bit) are exact. Output rows 4h .. 4h + 3 then sit in
// the four accumulator registers of lane group h.
//   Scores: wave w takes cache rows 16w + n (B columns n; B = K rows from LDS,
//   eight dimensions per lane per step), four steps of 32 dimensions.
//   P.V: wave w takes dimensions 32w + 16u + n (u = 0, 1), two steps of 32
//   cache rows; A = the weights from LDS, B = V rows from LDS.
// The softmax max and sum cross the four waves through LDS; rows past the
// token's position weigh zero (their LDS rows are zero-filled, so 0 * V stays
// 0). Results differ from k_decode_attention only by rounding.
constexpr int kMfmaHeads = 4;

template <int CT>
struct Mfma16 {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
};
template <>
struct Mfma16<NQ_DTYPE_F16> {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
};

typedef float v4f_t __attribute__((ext_vector_type(4)));

template <int CT>
__device__ __forceinline__ v4f_t mfma16(const typename Mfma16<CT>::v8& a, const typename Mfma16<CT>::v8& b,
                                        const v4f_t& c) {
    if constexpr (CT == NQ_DTYPE_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// The 16-bit rounding (nearest-even) of x, and a 16-bit value as fp32.
template <int CT>
__device__ __forceinline__ uint16_t to16(float x) {
    if constexpr (CT == NQ_DTYPE_BF16) return f32_to_bf16_bits(x);
    else return __builtin_bit_cast(uint16_t, static_cast<_Float16>(x));
}

template <int CT>
__device__ __forceinline__ float from16(uint16_t h) {
    if constexpr (CT == NQ_DTYPE_BF16) return __uint_as_float(static_cast<uint32_t>(h) << 16);
    else return static_cast<float>(__builtin_bit_cast(_Float16, h));
}

// The three 16-bit parts of x: the rounding of x, of its remainder and of the
// remainder's remainder (each subtraction is exact in fp32).
template <int CT>
__device__ __forceinline__ void split3(float x, uint16_t (&h)[3]) {
    h[0] = to16<CT>(x);
    const float r1 = x - from16<CT>(h[0]);
    h[1] = to16<CT>(r1);
    h[2] = to16<CT>(r1 - from16<CT>(h[1]));
}

template <int CT>
constexpr size_t decode_attention_mfma_lds() {
    // K and V blocks (plus a scratch row each), the 16-bit parts of q [4][4][128]
    // and of P [4][4][64], maxima and sums [2][4][4].
    return static_cast<size_t>(kSeqBlock + 1) * k_row_bytes<128, CT>() * 2 + kMfmaHeads * 4 * 128 * 2 +
           kMfmaHeads * 4 * kSeqBlock * 2 + 2 * kMfmaHeads * kMfmaHeads * 4;
}

template <int CT, bool HALF>
__global__ __launch_bounds__(kMfmaHeads * kWave) void k_decode_attention_mfma(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, int kv_heads,
    const void* __restrict__ q_norm, const void* __restrict__ k_norm, int ndt, float eps,
    const float* __restrict__ cos_table, const float* __restrict__ sin_table, const int32_t* __restrict__ position,
    int64_t max_positions, char* __restrict__ k_cache, char* __restrict__ v_cache, float scaling,
    float* __restrict__ part_ml, float* __restrict__ part_acc) {
    constexpr int D = 128;
    constexpr int G = kMfmaHeads;
    constexpr int E = D / kWave;
    constexpr int RB = k_row_bytes<D, CT>();  // padded row in LDS (K and V alike)
    constexpr int VRB = D * 2;                // row in the cache
    constexpr int PIECES = VRB / 16;
    constexpr int PER_THREAD = kSeqBlock * PIECES / (G * kWave);
    typedef typename Mfma16<CT>::v8 v8;
    extern __shared__ float lds_raw[];
    char* klds = reinterpret_cast<char*>(lds_raw);
    char* vlds = klds + (kSeqBlock + 1) * RB;
    uint16_t* qs = reinterpret_cast<uint16_t*>(vlds + (kSeqBlock + 1) * RB);  // [G][4 parts][D]
    uint16_t* ps = qs + G * 4 * D;                                             // [G][4 parts][64]
    float* mx = reinterpret_cast<float*>(ps + G * 4 * kSeqBlock);             // [G][4 waves]
    float* ls = mx + G * G;                                                    // [G][4 waves]

    const int g = blockIdx.x;
    const int s = blockIdx.y;
    // gridDim.y, from an argument: gridDim is read from the hidden kernel
    // arguments, one more scalar-cache line before the first load.
    const int blocks = static_cast<int>((max_positions + kSeqBlock - 1) / kSeqBlock);
    const int q_heads = kv_heads * G;
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const int lane = threadIdx.x & (kWave - 1);

    NormRopeIn<D> qin, kin;
    load_norm_rope_in<D>(qin, q + static_cast<int64_t>(g * G + w) * D, q_norm, ndt, lane);
    load_norm_rope_in<D>(kin, k + static_cast<int64_t>(g) * D, k_norm, ndt, lane);
    float vraw[E];
#pragma unroll
    for (int j = 0; j < E; ++j) vraw[j] = v[static_cast<int64_t>(g) * D + lane + kWave * j];

    const int64_t row0 = static_cast<int64_t>(s) * kSeqBlock;
    const int64_t head_row0 = static_cast<int64_t>(g) * max_positions;
    u32x4 kp[PER_THREAD], vp[PER_THREAD];
    const int last_row = static_cast<int>(max_positions - 1 - row0);
    const char* kbase = k_cache + (head_row0 + row0) * VRB;
    const char* vbase = v_cache + (head_row0 + row0) * VRB;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
        const int idx = threadIdx.x + i * G * kWave;
        const int r = idx / PIECES, c = idx % PIECES;
        const int rr = r < last_row ? r : last_row;
        kp[i] = *reinterpret_cast<const u32x4*>(kbase + rr * VRB + 16 * c);
        vp[i] = *reinterpret_cast<const u32x4*>(vbase + rr * VRB + 16 * c);
    }
    __builtin_amdgcn_sched_barrier(0);

    const int64_t pos = position[0];
    const bool live = pos >= 0 && pos < max_positions && row0 <= pos;  // uniform
    const int64_t p = live ? pos : row0;
    const bool owns_p = live && p < row0 + kSeqBlock;
    const int rows = live ? static_cast<int>(owns_p ? p - row0 + 1 : kSeqBlock) : 1;
    const int cached = live ? (owns_p ? rows - 1 : rows) : 0;

    float cs[E], sn[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int d = lane + kWave * j;
        const int fi = d < D / 2 ? d : d - D / 2;
        cs[j] = cos_table[p * (D / 2) + fi];
        sn[j] = sin_table[p * (D / 2) + fi];
    }
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) asm volatile("" : "+v"(kp[i]), "+v"(vp[i]));
    float qy[E];
    norm_rope_regs<D>(qin, q_norm != nullptr, ndt, eps, cs, sn, lane, qy);
    // Cached rows go to their LDS rows; rows past the token's row are zero
    // (their weights are zero, and 0 * V must stay 0); the token's own row is
    // written below, so its staging piece goes to the scratch row.
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
        const int idx = threadIdx.x + i * G * kWave;
        const int r = idx / PIECES, c = idx % PIECES;
        const bool keep = r < cached;
        const int lr = keep || r >= rows ? r : kSeqBlock;
        const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4*>(klds + lr * RB + 16 * c) = keep ? kp[i] : zero;
        *reinterpret_cast<u32x4*>(vlds + lr * RB + 16 * c) = keep ? vp[i] : zero;
    }
#pragma unroll
    for (int j = 0; j < E; ++j) {  // wave w: the parts of q head w (part 3 zero)
        uint16_t h[3];
        split3<CT>(qy[j], h);
        const int d = lane + kWave * j;
#pragma unroll
        for (int part = 0; part < 3; ++part) qs[(w * 4 + part) * D + d] = h[part];
        qs[(w * 4 + 3) * D + d] = 0;
    }
    float ky[E];
    norm_rope_regs<D>(kin, k_norm != nullptr, ndt, eps, cs, sn, lane, ky);
    const int nr = owns_p ? rows - 1 : kSeqBlock;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int d = lane + kWave * j;
        nq::store_f32_as(klds + nr * RB, CT, d, ky[j]);
        nq::store_f32_as(vlds + nr * RB, CT, d, vraw[j]);
    }
    if (owns_p) {
        const int64_t crow = (head_row0 + p) * D;
        if (w == 0) {
#pragma unroll
            for (int j = 0; j < E; ++j) nq::store_f32_as(k_cache, CT, crow + lane + kWave * j, ky[j]);
        }
        if (w == G - 1) {
#pragma unroll
            for (int j = 0; j < E; ++j) nq::store_f32_as(v_cache, CT, crow + lane + kWave * j, vraw[j]);
        }
    }
    __syncthreads();

    // Lane (kg, n): column n of the B operands, q head kg of the A rows
    // (row 4 kg + part, part = n & 3) and of the accumulator rows 4 kg + j.
    const int n = lane & 15, kg = lane >> 4;
    const int arow = lane & 15;  // A row: head arow / 4, part arow % 4 (parts are stored in that order)
    // Scores of cache rows 16w + n.
    v4f_t sc = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int st = 0; st < D / 32; ++st) {
        const int d0 = 32 * st + 8 * kg;
        const v8 a = *reinterpret_cast<const v8*>(qs + arow * D + d0);
        const v8 b = *reinterpret_cast<const v8*>(klds + (16 * w + n) * RB + 2 * d0);
        sc = mfma16<CT>(a, b, sc);
    }
    const int r = 16 * w + n;
    const bool valid = r < rows;
    const float score = valid ? ((sc[0] + sc[1]) + (sc[2] + sc[3])) * scaling : -INFINITY;  // head kg
    const float mw = row16_max(score);
    if (n == 0) mx[kg * G + w] = mw;
    __syncthreads();
    float M = mx[kg * G];
#pragma unroll
    for (int i = 1; i < G; ++i) M = fmaxf(M, mx[kg * G + i]);
    const float pr = valid ? expf(score - M) : 0.0f;
    const float lw = row16_sum(pr);
    {
        uint16_t h[3];
        split3<CT>(pr, h);
#pragma unroll
        for (int part = 0; part < 3; ++part) ps[(kg * 4 + part) * kSeqBlock + r] = h[part];
        ps[(kg * 4 + 3) * kSeqBlock + r] = 0;
    }
    if (n == 0) ls[kg * G + w] = lw;
    __syncthreads();

    // P.V for dimensions 32w + 16u + n.
    v4f_t o[2] = {v4f_t{0.0f, 0.0f, 0.0f, 0.0f}, v4f_t{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int t = 0; t < kSeqBlock / 32; ++t) {
        const int r0 = 32 * t + 8 * kg;
        const v8 a = *reinterpret_cast<const v8*>(ps + arow * kSeqBlock + r0);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            union {
                uint16_t h[8];
                v8 v;
            } b;
            const int d = 32 * w + 16 * u + n;
#pragma unroll
            for (int i = 0; i < 8; ++i) b.h[i] = *reinterpret_cast<const uint16_t*>(vlds + (r0 + i) * RB + 2 * d);
            o[u] = mfma16<CT>(a, b.v, o[u]);
        }
    }
    // A block past the token's row stores the neutral partial (max -inf, sum
    // 0, accumulators 0), which adds nothing to a merge over every block.
    // HALF: the block's output acc / sum as fp16 in place of the accumulators.
    const int64_t pi = attn_part_index(0, g * G + kg, s, q_heads, blocks);
    float l = 0.0f;
#pragma unroll
    for (int i = 0; i < G; ++i) l += ls[kg * G + i];
    const float inv = HALF && live ? 1.0f / l : 0.0f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const float a = (o[u][0] + o[u][1]) + (o[u][2] + o[u][3]);
        if constexpr (HALF)
            reinterpret_cast<_Float16*>(part_acc)[pi * D + 32 * w + 16 * u + n] =
                static_cast<_Float16>(live ? a * inv : 0.0f);
        else
            part_acc[pi * D + 32 * w + 16 * u + n] = live ? a : 0.0f;
    }
    if (w == 0 && n == 0) {
        part_ml[2 * pi] = live ? M : -INFINITY;
        part_ml[2 * pi + 1] = live ? l : 0.0f;
    }
}

// ---------------------------------------------------------------------------
// Prompt attention on MFMA (16-bit cache, two tokens or more, three with
// heads of 256):
// one pass over the cache with a running softmax, so no per-block partials
// leave the chip. A unit is 16 tokens of one q head; a workgroup takes four
// consecutive units of one kv head (the heads of a token tile, or, with fewer
// than four q heads per kv head, further tiles), one wave each, which share
// every K/V tile through LDS. HALVES = 2 adds four waves that take every
// second tile for the same units, merged through LDS at the end.
//   Scores are computed transposed, S^T = K Q^T on v_mfma_f32_16x16x32 (bf16 /
//   f16, the cache's type): A = K rows from LDS (exact), B = the query, split
//   into three 16-bit parts (the rounding of q, of its remainder and of the
//   remainder's remainder: about 24 bits of the fp32 query) held in registers
//   for the whole pass. Lane (kg, n) then holds token n's scores of cache rows
//   16 ct + 4 kg + j: the softmax of a token is a reduction over a lane's
//   registers and its three partner lanes, and the weights, split the same
//   way, are already the B operand of O^T = V^T P^T when k slot 8 kg + e of a
//   32-row step stands for row 16 (e / 4) + 4 kg + e % 4: they never go through LDS.
//   V is staged transposed with its rows in that order (a thread moves 4 rows
//   x 8 dimensions through registers), so an A fragment is one 16-byte read.
// A tile's weighted values are summed on their own (small parts first) and
// join the running output with one rounding: against 64 bits the output is
// 0.9e-7 - 3.6e-7 off (rel-L2; fp16 cache 1.5e-7 - 4.3e-7), 2.6e-7 - 5.8e-7
// with per-block partials.
//   What the parts cannot do as fp32 does: an infinity in the cache (elements
// that come out infinite or NaN are computed again at the end) and, with an
// fp16 cache, magnitudes (the query and each tile's weights are brought to the
// range where three fp16 parts hold 24 bits).
// Bound by the matrix cores and the softmax beside them: 96 MFMAs (16 cycles)
// and about 310 VALU instructions (four) per 16 tokens x 64 rows x 128
// dimensions; 35% of the time is MFMA at 1531 tokens. Measured in a graph, 32 q
// heads, 8 kv heads of 128, bf16 (per-block partials and a merge before): 512
// tokens 21.5 us (56), 1531 tokens after 517 cached 116 us (520), 16 / 8 heads
// 700 after 200 31 us (203), 8 / 4 heads of 256 700 tokens 43 us (176); with an
// fp16 cache 22.6 (45), 124 (406), 32 (184) and 45 us (155). Forming the next
// tile's scores among this tile's softmax was slower (142 against 123 us): the
// registers spill. So were three waves a SIMD (241 us).
constexpr int kFlashTokens = 16;      // tokens per unit (B columns)
constexpr int kFlashUnits = 4;        // units per workgroup

// Cache rows per tile: K and V of a tile take 32 KB of registers in flight
// over 256 threads (half that at head_dim 64).
template <int D>
constexpr int flash_rows() { return D == 256 ? 32 : 64; }

template <int CT>
__device__ __forceinline__ uint32_t pack16(float a, float b) {
    if constexpr (CT == NQ_DTYPE_BF16) {
        typedef float v2f __attribute__((ext_vector_type(2)));
        typedef __bf16 v2b __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{a, b}, v2b));
    } else {
        return to16<CT>(a) | (static_cast<uint32_t>(to16<CT>(b)) << 16);
    }
}

// split3 of two values, part by part as packed pairs.
template <int CT>
__device__ __forceinline__ void split3_pair(float a, float b, uint32_t (&h)[3]) {
    h[0] = pack16<CT>(a, b);
    a -= from16<CT>(static_cast<uint16_t>(h[0])), b -= from16<CT>(static_cast<uint16_t>(h[0] >> 16));
    h[1] = pack16<CT>(a, b);
    a -= from16<CT>(static_cast<uint16_t>(h[1])), b -= from16<CT>(static_cast<uint16_t>(h[1] >> 16));
    h[2] = pack16<CT>(a, b);
}

// Max / sum over lanes n, n + 16, n + 32, n + 48 (every one of them gets it).
__device__ __forceinline__ float column_max(float v) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ float column_sum(float v) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

struct FlashArgs {
    const float* q;
    const char* k_cache;
    const char* v_cache;
    int64_t tokens;
    int64_t max_positions;
    const int32_t* position;
    int q_heads, kv_heads;
    int quads;             // workgroups per kv head and split
    int tiles_per_split;
    int splits;            // grid y; more than one leaves partials for k_attention_merge
    float scaling;
    void* out;
    int odt;
    int vec_out;           // out allows the four-element stores
    float* part_ml;
    float* part_acc;
};

// One query against cache rows [begin, end) in fp32, by one wave, 64 rows at a
// time: the running max of the scaled scores, the sum of the weights and the
// weighted values of dimensions (D / 64) lane + [0, D / 64). `q` is uniform.
template <int D, int CT>
__device__ void fp32_attention_row(const float* __restrict__ q, const char* __restrict__ k_head,
                                   const char* __restrict__ v_head, int begin, int end, float scaling, int lane,
                                   float& m, float& l, float (&acc)[D / kWave]) {
    constexpr int E = D / kWave, U = 8;
    m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) acc[j] = 0.0f;
    for (int r0 = begin; r0 < end; r0 += kWave) {
        const int rows = end - r0 < kWave ? end - r0 : kWave;
        const int64_t r = r0 + (lane < rows ? lane : rows - 1);
        const float score = lane < rows ? k_row_dot<D, CT>(k_head + r * (2 * D), q) * scaling : -INFINITY;
        const float mx = fmaxf(m, wave_max(score));
        const float base = mx == -INFINITY ? 0.0f : mx;  // no score above -inf yet: their weights are 0
        const float keep = m == -INFINITY ? 0.0f : expf(m - base);
        const float w = lane < rows ? expf(score - base) : 0.0f;
        m = mx;
        l = l * keep + wave_sum(w);
#pragma unroll
        for (int j = 0; j < E; ++j) acc[j] *= keep;
        for (int i0 = 0; i0 < rows; i0 += U) {
            float vv[U][E];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t i = r0 + (i0 + u < rows ? i0 + u : rows - 1);
                load_v<E, CT>(v_head + (i * D + lane * E) * 2, vv[u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i0 + u < rows) {
#pragma unroll
                    for (int j = 0; j < E; ++j) acc[j] = fmaf(row_lane(w, i0 + u), vv[u][j], acc[j]);
                }
        }
    }
}

template <int D, int CT, int HALVES>
__global__ __launch_bounds__(HALVES * 256, 2) void k_prompt_attention(const FlashArgs g) {
    constexpr int R = flash_rows<D>();
    constexpr int KB = 2 * D + 16;               // padded K row in LDS, bytes
    constexpr int VS = R + 8;                    // 16-bit values per transposed V row
    constexpr int kTileBytes = R * KB + D * VS * 2;
    constexpr int kMergeBytes = HALVES == 2 ? (D / 4 + 2) * 256 * 4 : 0;
    constexpr int kLds = HALVES * kTileBytes > kMergeBytes ? HALVES * kTileBytes : kMergeBytes;
    constexpr int NS = D / 32;                   // 32-dimension steps of the scores
    constexpr int NC = R / 16;                   // 16-row score tiles
    constexpr int ND = D / 16;                   // 16-dimension output tiles
    constexpr int KPT = R * D / 8 / 256;         // 16-byte K pieces per thread
    constexpr int kQuads = R / 4 * (D / 8);      // V patches (4 rows x 8 dimensions)
    static_assert(kQuads <= 256, "one V patch per thread");
    typedef typename Mfma16<CT>::v8 v8;
    union Frag {
        uint32_t u[4];
        v8 v;
    };
    __shared__ __attribute__((aligned(16))) char lds[kLds];
    __shared__ int wild[HALVES];  // a V value that is not finite, in a row some token of the tile may not see

    const int group = g.q_heads / g.kv_heads;
    const int kvh = static_cast<int>(blockIdx.x) % g.kv_heads;
    // The longest units first: what is left at the end is short.
    const int quad = g.quads - 1 - static_cast<int>(blockIdx.x) / g.kv_heads;
    const int split = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const int lane = threadIdx.x & (kWave - 1);
    const int n = lane & 15, kg = lane >> 4;
    const int half = wave >> 2;
    const int ht = threadIdx.x & 255;  // thread within the half
    const int units = static_cast<int>((g.tokens + kFlashTokens - 1) / kFlashTokens) * group;
    const int unit0 = quad * kFlashUnits;
    const int unit_last = unit0 + kFlashUnits - 1 < units ? unit0 + kFlashUnits - 1 : units - 1;
    const bool unit_ok = unit0 + (wave & 3) <= unit_last;
    const int unit = unit_ok ? unit0 + (wave & 3) : unit_last;
    const int h = kvh * group + unit % group;
    const int64_t t0 = static_cast<int64_t>(unit / group) * kFlashTokens;
    const int64_t t = t0 + n;
    const int64_t p0 = g.position[0];
    const int64_t pt = p0 + t;  // the last row token n sees
    constexpr uint32_t kExp = CT == NQ_DTYPE_BF16 ? 0x7f80u : 0x7c00u;  // exponent of an infinity or NaN
    const int64_t t_first = static_cast<int64_t>(unit0 / group) * kFlashTokens;
    const int64_t t_end = (static_cast<int64_t>(unit_last / group) + 1) * kFlashTokens;
    int64_t last_row = p0 + (t_end < g.tokens ? t_end : g.tokens) - 1;
    last_row = last_row < g.max_positions ? last_row : g.max_positions - 1;
    // The last row that any token of the workgroup sees and that every one
    // does (the host bounds the cache below 2^22 rows).
    const int last = static_cast<int>(last_row), first = static_cast<int>(p0 + t_first);
    int tile = split * g.tiles_per_split;
    int tile_end = p0 < 0 || p0 + t_first >= g.max_positions ? 0 : static_cast<int>(last / R) + 1;
    tile_end = tile_end < tile + g.tiles_per_split ? tile_end : tile + g.tiles_per_split;

    char* const klds = lds + half * kTileBytes;
    uint16_t* const vt = reinterpret_cast<uint16_t*>(klds + R * KB);
    const int64_t head0 = static_cast<int64_t>(kvh) * g.max_positions;
    const char* const k_head = g.k_cache + head0 * (2 * D);
    const char* const v_head = g.v_cache + head0 * (2 * D);

    // Query operand: token n, dimensions 32 st + 8 kg + [0, 8), in three parts.
    // fp16 parts hold 24 bits only between 2^-11 and 65504, so the token's
    // query is first brought to [2^14, 2^15) by a power of two, which goes into
    // the factor of its scores.
    Frag qa[3][NS];
    float c = g.scaling * 1.4426950408889634f;  // weights are 2^(c s - c max)
    {
        const float* qp = g.q + ((t < g.tokens ? t : g.tokens - 1) * g.q_heads + h) * D + 8 * kg;
        float x[NS][8];
#pragma unroll
        for (int st = 0; st < NS; ++st) {
            const float4 a = *reinterpret_cast<const float4*>(qp + 32 * st);
            const float4 b = *reinterpret_cast<const float4*>(qp + 32 * st + 4);
            x[st][0] = a.x, x[st][1] = a.y, x[st][2] = a.z, x[st][3] = a.w;
            x[st][4] = b.x, x[st][5] = b.y, x[st][6] = b.z, x[st][7] = b.w;
        }
        if constexpr (CT == NQ_DTYPE_F16) {
            float top = 0.0f;
#pragma unroll
            for (int st = 0; st < NS; ++st)
#pragma unroll
                for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(x[st][e]));
            const int shift = 141 - static_cast<int>(__float_as_uint(column_max(top)) >> 23);
            const int k = shift < 100 ? shift : 100;  // a query below 2^-86 stays smaller than that
            const float up = __uint_as_float(static_cast<uint32_t>(127 + k) << 23);
            c *= __uint_as_float(static_cast<uint32_t>(127 - k) << 23);
#pragma unroll
            for (int st = 0; st < NS; ++st)
#pragma unroll
                for (int e = 0; e < 8; ++e) x[st][e] *= up;
        }
#pragma unroll
        for (int st = 0; st < NS; ++st)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t hh[3];
                split3_pair<CT>(x[st][2 * e], x[st][2 * e + 1], hh);
#pragma unroll
                for (int p = 0; p < 3; ++p) qa[p][st].u[e] = hh[p];
            }
    }

    // This thread's V patch: rows 4 vq + [0, 4), dimensions 8 vc + [0, 8); the
    // rows' slots within the 32-row step t are 8 kg + 4 eh + [0, 4).
    const int vq = ht % (R / 4), vc = ht / (R / 4);
    const int v_slot = 32 * (vq >> 3) + 8 * (vq & 3) + 4 * ((vq >> 2) & 1);
    const bool v_on = kQuads == 256 || ht < kQuads;
    u32x4 kp[KPT], vp[4];
    const auto load_tile = [&](int kt) __attribute__((always_inline)) {
        const int row0 = kt * R;
#pragma unroll
        for (int i = 0; i < KPT; ++i) {
            const int piece = ht + 256 * i;
            const int r = row0 + piece / (D / 8);
            kp[i] = *reinterpret_cast<const u32x4*>(
                k_head + (static_cast<uint32_t>(r < last ? r : last) * (2 * D) + 16 * (piece % (D / 8))));
        }
        if (v_on) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = row0 + 4 * vq + i;
                vp[i] = *reinterpret_cast<const u32x4*>(
                    v_head + (static_cast<uint32_t>(r < last ? r : last) * (2 * D) + 16 * vc));
            }
        }
    };
    // Rows past `last` are stored as zeros: their weights are zero, and 0 * V
    // must stay 0. So are infinities and NaNs in the rows that not every token
    // of the workgroup sees: the loop below adds those where they belong.
    const auto store_tile = [&](int kt) __attribute__((always_inline)) {
        const int row0 = kt * R;
#pragma unroll
        for (int i = 0; i < KPT; ++i) {
            const int piece = ht + 256 * i;
            *reinterpret_cast<u32x4*>(klds + (piece / (D / 8)) * KB + 16 * (piece % (D / 8))) = kp[i];
        }
        if (v_on) {
            if (row0 + R - 1 > first) {
                bool bad = false;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = row0 + 4 * vq + i;
                    if (r > last) vp[i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool lo = (vp[i][e] & kExp) == kExp, hi = ((vp[i][e] >> 16) & kExp) == kExp;
                        bad |= r > first && (lo || hi);
                        if (r > first) vp[i][e] &= (lo ? 0u : 0xffffu) | (hi ? 0u : 0xffff0000u);
                    }
                }
                if (bad) wild[half] = 1;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;
                uint2 w;
                w.x = __builtin_amdgcn_perm(vp[1][e >> 1], vp[0][e >> 1], sel);
                w.y = __builtin_amdgcn_perm(vp[3][e >> 1], vp[2][e >> 1], sel);
                *reinterpret_cast<uint2*>(vt + (8 * vc + e) * VS + v_slot) = w;
            }
        }
    };

    if (threadIdx.x < HALVES) wild[threadIdx.x] = 0;
    v4f_t o[ND];
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) o[dt] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, mc = 0.0f, l = 0.0f;  // running max of s, c * max (0 before any row), this lane's sum
    if (tile + half < tile_end) load_tile(tile + half);
    for (; tile < tile_end; tile += HALVES) {
        const int kt = tile + half;
        const bool on = kt < tile_end;  // uniform per wave
        __syncthreads();
        if (on) store_tile(kt);
        __syncthreads();
        if (kt + HALVES < tile_end) load_tile(kt + HALVES);
        if (!on) continue;
        const int row0 = kt * R;
        if (row0 > p0 + t0 + kFlashTokens - 1) continue;  // uniform per wave: no token of the unit reaches the tile
        const bool edge = row0 + R - 1 > p0 + t0;          // some token does not see every row
        // The query's high part and its small parts in sums of their own: a
        // score takes NS + 1 roundings at its own size instead of 3 NS.
        // Consecutive MFMAs add to different accumulators.
        v4f_t s[NC], lo[NC];
#pragma unroll
        for (int ct = 0; ct < NC; ++ct) s[ct] = lo[ct] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int st = 0; st < NS; ++st) {
            v8 a[NC];
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
                a[ct] = *reinterpret_cast<const v8*>(klds + (16 * ct + n) * KB + 64 * st + 16 * kg);
#pragma unroll
            for (int p = 2; p >= 0; --p)
#pragma unroll
                for (int ct = 0; ct < NC; ++ct) {
                    v4f_t& sum = p == 0 ? s[ct] : lo[ct];
                    sum = mfma16<CT>(a[ct], qa[p][st].v, sum);
                }
        }
#pragma unroll
        for (int ct = 0; ct < NC; ++ct) s[ct] += lo[ct];
        if (edge) {
            const int seen = static_cast<int>(pt - row0 < R ? pt - row0 : R);
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
#pragma unroll
                for (int j = 0; j < 4; ++j) s[ct][j] = 16 * ct + 4 * kg + j <= seen ? s[ct][j] : -INFINITY;
        }
        // The weights are relative to the running max; with an fp16 cache to
        // the tile's own, where it is 2^15, and the tile joins by the factor
        // `join`: fp16 parts hold 24 bits of what is above 2^-26 of that (2^-11
        // of the row's largest weight otherwise), and 2^-40 of it below.
        constexpr bool kOwnMax = CT == NQ_DTYPE_F16;
        constexpr float kTop = kOwnMax ? 15.0f : 0.0f;
        float mx = kOwnMax ? -INFINITY : m;
#pragma unroll
        for (int ct = 0; ct < NC; ++ct)
#pragma unroll
            for (int j = 0; j < 4; ++j) mx = fmaxf(mx, s[ct][j]);
        mx = column_max(mx);
        const float mc_tile = mx == -INFINITY ? 0.0f : fmaf(mx, c, -kTop);
        const float mc_new = kOwnMax && m > mx ? mc : mc_tile;
        const float keep = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mc - mc_new);
        const float join = kOwnMax && mx != -INFINITY ? __builtin_amdgcn_exp2f(mc_tile - mc_new) : 1.0f;
        m = kOwnMax ? fmaxf(m, mx) : mx;
        mc = mc_new;
        float lt = 0.0f;
#pragma unroll
        for (int ct = 0; ct < NC; ++ct)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s[ct][j] = __builtin_amdgcn_exp2f(fmaf(s[ct][j], c, -mc_tile));
                lt += s[ct][j];
            }
        l = fmaf(l, keep, kOwnMax ? lt * join : lt);
        Frag pa[3][R / 32];
#pragma unroll
        for (int ks = 0; ks < R / 32; ++ks)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t hh[3];
                split3_pair<CT>(s[2 * ks + (e >> 1)][2 * (e & 1)], s[2 * ks + (e >> 1)][2 * (e & 1) + 1], hh);
#pragma unroll
                for (int p = 0; p < 3; ++p) pa[p][ks].u[e] = hh[p];
            }
        // A tile's products on their own, small parts first, then one rounding
        // into the running output.
#pragma unroll
        for (int d0 = 0; d0 < ND; d0 += 4) {
            v4f_t y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int p = 2; p >= 0; --p)
#pragma unroll
                for (int ks = 0; ks < R / 32; ++ks)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const v8 a = *reinterpret_cast<const v8*>(vt + (16 * (d0 + i) + n) * VS + 32 * ks + 8 * kg);
                        y[i] = mfma16<CT>(a, pa[p][ks].v, y[i]);
                    }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    o[d0 + i][j] = fmaf(o[d0 + i][j], keep, kOwnMax ? y[i][j] * join : y[i][j]);
        }
        if (row0 + R - 1 > first && wild[half]) {
            // The values that store_tile left out, for the tokens that see their rows (also in a
            // tile whose rows all of this unit's tokens see).
            const int r_end = last < row0 + R - 1 ? last : row0 + R - 1;
            for (int r = row0 > first ? row0 : first + 1; r <= r_end; ++r) {
                const int rr = r - row0;
                float w = 0.0f;
#pragma unroll
                for (int ct = 0; ct < NC; ++ct)
#pragma unroll
                    for (int j = 0; j < 4; ++j) w = rr >> 4 == ct && (rr & 3) == j ? s[ct][j] : w;
                w = __shfl(w, 16 * ((rr >> 2) & 3) + n, kWave) * join;
                const uint16_t* vr = reinterpret_cast<const uint16_t*>(v_head) + static_cast<uint32_t>(r) * D + 4 * kg;
#pragma unroll
                for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t x = vr[16 * dt + i];
                        if (r <= pt && (x & kExp) == kExp)
                            o[dt][i] = fmaf(w, from16<CT>(static_cast<uint16_t>(x)), o[dt][i]);
                    }
            }
        }
    }

    if constexpr (HALVES == 2) {
        // The second half's max, sum and sums join the first's, lane by lane.
        float* const mg = reinterpret_cast<float*>(lds) + ht;
        __syncthreads();
        if (half == 1) {
            mg[0] = m;
            mg[256] = mc;
#pragma unroll
            for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) mg[(2 + 4 * dt + i) * 256] = o[dt][i];
        }
        __shared__ float l_other[256];
        if (half == 1) l_other[ht] = l;
        __syncthreads();
        if (half == 1) return;
        const float m2 = mg[0], mc2 = mg[256];
        const float mcn = m2 > m ? mc2 : mc;
        const float f1 = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mc - mcn);
        const float f2 = m2 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mc2 - mcn);
        l = l * f1 + l_other[ht] * f2;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[dt][i] = o[dt][i] * f1 + mg[(2 + 4 * dt + i) * 256] * f2;
        m = m2 > m ? m2 : m;
        mc = mcn;
    }
    l = column_sum(l);
    const int64_t split_row0 = static_cast<int64_t>(split) * g.tiles_per_split * R;
    const bool ours = unit_ok && t < g.tokens;
    const bool in_range = p0 >= 0 && pt < g.max_positions;  // tokens outside the cache: zero
    const bool live = ours && in_range && pt >= split_row0;
    if (g.splits > 1) {
        if (live) {
            const int64_t pi = attn_part_index(t, h, split, g.q_heads, g.splits);
#pragma unroll
            for (int dt = 0; dt < ND; ++dt) *reinterpret_cast<v4f_t*>(g.part_acc + pi * D + 16 * dt + 4 * kg) = o[dt];
            if (kg == 0) {
                g.part_ml[2 * pi] = m == -INFINITY ? m : mc * 0.69314718055994531f;
                g.part_ml[2 * pi + 1] = l;
            }
        }
    } else if (ours) {
        const int64_t out0 = (t * g.q_heads + h) * D + 4 * kg;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {
            v4f_t y;
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = in_range ? o[dt][i] / l : 0.0f;
            const int64_t oi = out0 + 16 * dt;
            if (g.odt == NQ_DTYPE_F32) {
                float* const dst = static_cast<float*>(g.out) + oi;
                if (g.vec_out) *reinterpret_cast<v4f_t*>(dst) = y;
                else dst[0] = y[0], dst[1] = y[1], dst[2] = y[2], dst[3] = y[3];
            } else {
                uint16_t* const dst = static_cast<uint16_t*>(g.out) + oi;
                uint2 w;
                w.x = pack2(g.odt, y[0], y[1]);
                w.y = pack2(g.odt, y[2], y[3]);
                if (g.vec_out) {
                    *reinterpret_cast<uint2*>(dst) = w;
                } else {
                    dst[0] = static_cast<uint16_t>(w.x), dst[1] = static_cast<uint16_t>(w.x >> 16);
                    dst[2] = static_cast<uint16_t>(w.y), dst[3] = static_cast<uint16_t>(w.y >> 16);
                }
            }
        }
    }

    // An infinity in the cache meets parts of a query or of a weight that have
    // the other sign or are zero, so it ends as NaN where fp32 arithmetic has
    // a weight of zero (a score of -inf) or an infinite output. Elements that
    // came out infinite or NaN are computed once more in fp32; all others keep
    // what they have. Nothing of this is in the loop above (testing every
    // value of V there costs 48 VALU instructions a tile and wave).
    float z = 0.0f;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) z = fmaf(o[dt][i], 0.0f, z);
    const uint64_t odd = __ballot(live && z != z);
    if (odd == 0) return;  // uniform per wave
    uint32_t odd_lo = 0, odd_hi = 0;  // this lane's elements: bit 4 dt + i
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t bit = o[dt][i] * 0.0f != 0.0f ? 1u << ((4 * dt + i) & 31) : 0u;
            if (dt < 8) odd_lo |= bit;
            else odd_hi |= bit;
        }
    __threadfence();  // the stores above are done before others go to the same places
    constexpr int E = D / kWave;
    const int split_end = split_row0 + g.tiles_per_split * R < g.max_positions
                              ? static_cast<int>(split_row0) + g.tiles_per_split * R : static_cast<int>(g.max_positions);
    for (uint32_t rest = static_cast<uint32_t>((odd | odd >> 16 | odd >> 32 | odd >> 48) & 0xffff); rest; rest &= rest - 1) {
        const int nn = __builtin_ctz(rest);
        const int64_t tt = t0 + nn;
        const float* const qr = g.q + (tt * g.q_heads + h) * D;
        float qz = 0.0f;
#pragma unroll
        for (int j = 0; j < E; ++j) qz = fmaf(qr[lane + kWave * j], 0.0f, qz);
        if (__ballot(qz != qz)) continue;  // no finite score: NaN throughout, as it is
        const int end = p0 + tt + 1 < split_end ? static_cast<int>(p0 + tt) + 1 : split_end;
        float m1, l1, acc[E];
        fp32_attention_row<D, CT>(qr, k_head, v_head, static_cast<int>(split_row0), end, g.scaling, lane, m1, l1, acc);
        const float l0 = __shfl(l, nn, kWave);
        const bool whole = l0 * 0.0f != 0.0f;  // the sum is NaN, so every element is
        const int64_t pi = attn_part_index(tt, h, split, g.q_heads, g.splits);
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const int d = lane * E + j, src = 16 * ((d >> 2) & 3) + nn, at = 4 * (d >> 4) + (d & 3);
            const uint32_t lo_bits = __shfl(odd_lo, src, kWave), hi_bits = __shfl(odd_hi, src, kWave);
            if (!((at < 32 ? lo_bits : hi_bits) >> (at & 31) & 1)) continue;
            // Beside a sum and a max that stand, the element in their units.
            if (g.splits > 1) g.part_acc[pi * D + d] = whole ? acc[j] : acc[j] / l1 * l0;
            else nq::store_f32_as(g.out, g.odt, (tt * g.q_heads + h) * D + d, acc[j] / l1);
        }
        if (g.splits > 1 && whole && lane == 0) g.part_ml[2 * pi] = m1, g.part_ml[2 * pi + 1] = l1;
    }
}

// ---------------------------------------------------------------------------
// One-token decode attention with the q/k RMSNorm + RoPE + KV append fused in
// (pass 1; k_attention_merge is pass 2). Workgroup (kv head g, 64-row cache
// block s), one wave per q head of the group:
//   - every load is issued first: the block's K and V rows below the token's
//     row p (coalesced 16-byte pieces), each wave's raw q head, and, in the
//     block that holds p, the raw k and v of head g;
//   - K and V rows go to LDS as stored; wave w normalises and rotates q head
//     g * G + w into LDS; in p's block wave 0 rotates k and wave G - 1 (wave 0
//     when G == 1) copies v into LDS row p - 64 s and into cache row p;
//   - after one barrier lane j scores row 64 s + j (K row from LDS, q
//     broadcast), the wave forms its softmax partial and lanes over
//     dimensions accumulate P.V from LDS; the partial goes to the workspace.
// Used when head_dim * element bytes <= 256 (the staged block fits LDS
// twice) and G is 1, 2, 4 or 8.

template <int D, int CT, int G>
constexpr size_t decode_attention_lds() {
    return static_cast<size_t>(kSeqBlock + 1) * k_row_bytes<D, CT>() +
           static_cast<size_t>(kSeqBlock + 1) * D * cache_bytes<CT>() + static_cast<size_t>(G) * (D + kSeqBlock) * sizeof(float);
}

template <int D, int CT, int G, bool HALF>
__global__ __launch_bounds__(G * kWave) void k_decode_attention(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, int kv_heads,
    const void* __restrict__ q_norm, const void* __restrict__ k_norm, int ndt, float eps,
    const float* __restrict__ cos_table, const float* __restrict__ sin_table, const int32_t* __restrict__ position,
    int64_t max_positions, char* __restrict__ k_cache, char* __restrict__ v_cache, float scaling,
    float* __restrict__ part_ml, float* __restrict__ part_acc) {
    constexpr int E = D / kWave;
    constexpr int EB = cache_bytes<CT>();
    constexpr int RB = k_row_bytes<D, CT>();   // padded K row in LDS
    constexpr int VRB = D * EB;                // V row in LDS
    constexpr int PIECES = D * EB / 16;        // 16-byte pieces per row
    constexpr int PER_THREAD = kSeqBlock * PIECES / (G * kWave);
    extern __shared__ float lds_raw[];
    char* klds = reinterpret_cast<char*>(lds_raw);   // kSeqBlock rows + one scratch row
    char* vlds = klds + (kSeqBlock + 1) * RB;
    float* qs = reinterpret_cast<float*>(vlds + (kSeqBlock + 1) * VRB);  // [G][D]
    float* ps = qs + G * D;                                             // [G][64]

    const int g = blockIdx.x;
    const int s = blockIdx.y;
    // gridDim.y, from an argument: gridDim is read from the hidden kernel
    // arguments, one more scalar-cache line before the first load.
    const int blocks = static_cast<int>((max_positions + kSeqBlock - 1) / kSeqBlock);
    const int q_heads = kv_heads * G;
    const int w = threadIdx.x / kWave;
    const int lane = threadIdx.x & (kWave - 1);

    // Loads that do not need the position go first: this wave's q head and
    // the k and v of head g, with their norm weights (no branch on the dtype).
    NormRopeIn<D> qin, kin;
    load_norm_rope_in<D>(qin, q + static_cast<int64_t>(g * G + w) * D, q_norm, ndt, lane);
    load_norm_rope_in<D>(kin, k + static_cast<int64_t>(g) * D, k_norm, ndt, lane);
    float vraw[E];
#pragma unroll
    for (int j = 0; j < E; ++j) vraw[j] = v[static_cast<int64_t>(g) * D + lane + kWave * j];

    // The block's K and V rows, loaded whatever the position (rows past the
    // cache's end reload its last row); rows at or past `cached` go to the
    // scratch row. The position and its RoPE entries follow the barrier;
    // nothing is used before all are issued.
    const int64_t row0 = static_cast<int64_t>(s) * kSeqBlock;
    const int64_t head_row0 = static_cast<int64_t>(g) * max_positions;
    u32x4 kp[PER_THREAD], vp[PER_THREAD];
    const int last_row = static_cast<int>(max_positions - 1 - row0);  // >= 0: the block starts in the cache
    const char* kbase = k_cache + (head_row0 + row0) * VRB;
    const char* vbase = v_cache + (head_row0 + row0) * VRB;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
        const int idx = threadIdx.x + i * G * kWave;
        const int r = idx / PIECES, c = idx % PIECES;
        const int rr = r < last_row ? r : last_row;
        kp[i] = *reinterpret_cast<const u32x4*>(kbase + rr * VRB + 16 * c);
        vp[i] = *reinterpret_cast<const u32x4*>(vbase + rr * VRB + 16 * c);
    }
    __builtin_amdgcn_sched_barrier(0);

    // No early exit (it would sink the loads above below the wait for the
    // position): a block past the position runs the arithmetic of a one-row
    // block at row0 and stores nothing; the merge ignores it. The position is
    // read after the scheduling barrier, so every load above is issued before
    // its (scalar) wait.
    const int64_t pos = position[0];
    const bool live = pos >= 0 && pos < max_positions && row0 <= pos;  // uniform
    const int64_t p = live ? pos : row0;
    const bool owns_p = live && p < row0 + kSeqBlock;
    const int rows = live ? static_cast<int>(owns_p ? p - row0 + 1 : kSeqBlock) : 1;  // rows scored
    const int cached = live ? (owns_p ? rows - 1 : rows) : 0;                         // rows read from the cache

    float cs[E], sn[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int d = lane + kWave * j;
        const int fi = d < D / 2 ? d : d - D / 2;
        cs[j] = cos_table[p * (D / 2) + fi];
        sn[j] = sin_table[p * (D / 2) + fi];
    }
    // Pin the block loads here: all of them are issued before the first wait.
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) asm volatile("" : "+v"(kp[i]), "+v"(vp[i]));
    float qy[E];
    norm_rope_regs<D>(qin, q_norm != nullptr, ndt, eps, cs, sn, lane, qy);
    // Stage K and V rows below p (the others to the scratch row).
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
        const int idx = threadIdx.x + i * G * kWave;
        const int r = idx / PIECES, c = idx % PIECES;
        const int lr = r < cached ? r : kSeqBlock;
        *reinterpret_cast<u32x4*>(klds + lr * RB + 16 * c) = kp[i];
        *reinterpret_cast<u32x4*>(vlds + lr * VRB + 16 * c) = vp[i];
    }
#pragma unroll
    for (int j = 0; j < E; ++j) qs[w * D + lane + kWave * j] = qy[j];
    // Row p's k and v: every wave forms them (identical values) and writes
    // them to LDS row rows - 1 when this block holds p, else to the scratch
    // row (no branch, so their loads stay ahead of the position wait); wave 0
    // appends k and wave G - 1 appends v to the cache.
    float ky[E];
    norm_rope_regs<D>(kin, k_norm != nullptr, ndt, eps, cs, sn, lane, ky);
    const int nr = owns_p ? rows - 1 : kSeqBlock;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int d = lane + kWave * j;
        nq::store_f32_as(klds + nr * RB, CT, d, ky[j]);
        nq::store_f32_as(vlds + nr * VRB, CT, d, vraw[j]);
    }
    if (owns_p) {
        const int64_t crow = (head_row0 + p) * D;
        if (w == 0) {
#pragma unroll
            for (int j = 0; j < E; ++j) nq::store_f32_as(k_cache, CT, crow + lane + kWave * j, ky[j]);
        }
        if (w == G - 1) {
#pragma unroll
            for (int j = 0; j < E; ++j) nq::store_f32_as(v_cache, CT, crow + lane + kWave * j, vraw[j]);
        }
    }
    __syncthreads();

    // Scores, softmax partial, P.V for q head g * G + w.
    const bool valid = lane < rows;
    const float dot = k_row_dot<D, CT>(klds + (valid ? lane : 0) * RB, qs + w * D);
    const float score = valid ? dot * scaling : -INFINITY;
    const float m = wave_max(score);
    const float pj = valid ? expf(score - m) : 0.0f;
    const float l = wave_sum(pj);
    float* pw = ps + w * kSeqBlock;
    pw[lane] = pj;
    __builtin_amdgcn_wave_barrier();
    // P.V over the scored rows in groups of four, one accumulator per row of
    // the group (four short dependency chains), combined at the end; rows past
    // `rows` read row 0 with weight 0.
    float acc4[4][E];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < E; ++e) acc4[u][e] = 0.0f;
    for (int r0 = 0; r0 < rows; r0 += 4) {
        float pr[4], vv[4][E];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int r = r0 + u < rows ? r0 + u : 0;
            pr[u] = r0 + u < rows ? pw[r] : 0.0f;
            load_v<E, CT>(vlds + r * VRB + lane * E * EB, vv[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < E; ++e) acc4[u][e] = fmaf(pr[u], vv[u][e], acc4[u][e]);
    }
    float acc[E];
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] = (acc4[0][e] + acc4[1][e]) + (acc4[2][e] + acc4[3][e]);
    // A block past the token's row stores the neutral partial (max -inf, sum
    // 0, accumulators 0), which adds nothing to a merge over every block.
    // HALF: the block's output acc / sum as fp16 in place of the accumulators.
    const int h = g * G + w;
    const int64_t pi = attn_part_index(0, h, s, q_heads, blocks);
    if (lane == 0) {
        part_ml[2 * pi] = live ? m : -INFINITY;
        part_ml[2 * pi + 1] = live ? l : 0.0f;
    }
    const float inv = HALF && live ? 1.0f / l : 0.0f;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if constexpr (HALF)
            reinterpret_cast<_Float16*>(part_acc)[pi * D + lane * E + e] =
                static_cast<_Float16>(live ? acc[e] * inv : 0.0f);
        else
            part_acc[pi * D + lane * E + e] = live ? acc[e] : 0.0f;
    }
}

// ---------------------------------------------------------------------------
// SiLU-gated product.

__global__ __launch_bounds__(kRowThreads) void k_silu_mul(const float* __restrict__ gate, const float* __restrict__ up,
                                                          int64_t n, void* __restrict__ out, int odt) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * kRowThreads + threadIdx.x) * 8;
    if (i >= n) return;
    float gv[8], uv[8];
    load8(gate, NQ_DTYPE_F32, i, gv);
    load8(up, NQ_DTYPE_F32, i, uv);
#pragma unroll
    for (int j = 0; j < 8; ++j) gv[j] = __fmul_rn(gv[j] / (1.0f + expf(-gv[j])), uv[j]);
    store8(out, odt, i, gv);
}

// ---------------------------------------------------------------------------
// Output projection: logits = W x for one token, W bf16 [vocab, hidden].
// Wave w of workgroup b owns RW = kProjLoads / NCH consecutive rows; lane l
// reads 8-element chunk k * 64 + l of each row for k < NCH, so all of a
// wave's RW * NCH 16-byte loads are issued before the first is used. x is
// staged in LDS as fp32. Each workgroup also writes its best (logit, index)
// as one orderable 64-bit key.

__device__ __forceinline__ uint64_t argmax_key(float v, uint32_t idx) {
    uint32_t u = __float_as_uint(v == 0.0f ? 0.0f : v);
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return (static_cast<uint64_t>(u) << 32) | static_cast<uint64_t>(0xffffffffu - idx);
}

template <int NCH>
__global__ __launch_bounds__(kProjWaves * kWave) void k_output_projection(const void* __restrict__ x, int xdt,
                                                                          const uint16_t* __restrict__ weight,
                                                                          int64_t vocab, int64_t hidden,
                                                                          float* __restrict__ logits,
                                                                          uint64_t* __restrict__ partial) {
    constexpr int RW = kProjLoads / NCH;
    __shared__ float xs[NCH * kWave * 8];
    __shared__ uint64_t best[kProjWaves];
    const int lane = threadIdx.x & (kWave - 1);
    const int w = threadIdx.x / kWave;
    const int64_t chunks = hidden / 8;
    const int64_t row0 = (static_cast<int64_t>(blockIdx.x) * kProjWaves + w) * RW;

    // Weight loads first (clamped rows and chunks; masked in the arithmetic),
    // nontemporal: the matrix streams through once per token. Measured on
    // MI355X at 151936 x 4096: 193 us (6.4 TB/s) against 215 us with plain
    // loads, the same logits bit for bit.
    uint4 wv[RW][NCH];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int64_t row = row0 + r < vocab ? row0 + r : vocab - 1;
#pragma unroll
        for (int kk = 0; kk < NCH; ++kk) {
            const int64_t c = kk * kWave + lane;
            const int64_t cc = c < chunks ? c : chunks - 1;
            const u32x4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(weight + row * hidden + cc * 8));
            wv[r][kk] = make_uint4(t.x, t.y, t.z, t.w);
        }
    }
    for (int64_t i = threadIdx.x * 8; i < static_cast<int64_t>(NCH) * kWave * 8; i += kProjWaves * kWave * 8) {
        float v[8];
        if (i < hidden) {
            load8(x, xdt, i, v);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = 0.0f;
        }
        float4* d = reinterpret_cast<float4*>(&xs[i]);
        d[0] = make_float4(v[0], v[1], v[2], v[3]);
        d[1] = make_float4(v[4], v[5], v[6], v[7]);
    }
    __syncthreads();

    float acc[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int kk = 0; kk < NCH; ++kk) {
        const int64_t c = kk * kWave + lane;
        const float4 xa = *reinterpret_cast<const float4*>(&xs[c * 8]);
        const float4 xb = *reinterpret_cast<const float4*>(&xs[c * 8 + 4]);
        const bool live = c < chunks;
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            const uint4 u = wv[r][kk];
            float a = acc[r];
            a = fmaf(bf16_lo(u.x), xa.x, a);
            a = fmaf(bf16_hi(u.x), xa.y, a);
            a = fmaf(bf16_lo(u.y), xa.z, a);
            a = fmaf(bf16_hi(u.y), xa.w, a);
            a = fmaf(bf16_lo(u.z), xb.x, a);
            a = fmaf(bf16_hi(u.z), xb.y, a);
            a = fmaf(bf16_lo(u.w), xb.z, a);
            a = fmaf(bf16_hi(u.w), xb.w, a);
            acc[r] = live ? a : acc[r];
        }
    }
    uint64_t key = 0;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const float sum = wave_sum(acc[r]);
        const int64_t row = row0 + r;
        if (row < vocab) {
            if (lane == r) logits[row] = sum;
            const uint64_t kr = argmax_key(sum, static_cast<uint32_t>(row));
            key = kr > key ? kr : key;
        }
    }
    if (lane == 0) best[w] = key;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t b = best[0];
#pragma unroll
        for (int i = 1; i < kProjWaves; ++i) b = best[i] > b ? best[i] : b;
        partial[blockIdx.x] = b;
    }
}

__global__ __launch_bounds__(1024) void k_greedy_select(const uint64_t* __restrict__ partial, int64_t count,
                                                        int64_t* __restrict__ token_out, int64_t* __restrict__ history,
                                                        int64_t history_capacity, int32_t* __restrict__ step,
                                                        int32_t* __restrict__ position) {
    constexpr int kThreads = 1024;  // the launch's block size
    constexpr int kRound = 16;      // loads in flight per thread
    __shared__ uint64_t red[kThreads / kWave];
    // Rounds of kRound independent loads per thread (indices clamped to the
    // last partial, whose repeats do not change the maximum), so a round
    // costs one memory round trip: 9496 partials for a 151936-row vocabulary
    // are one round instead of ten dependent loads.
    uint64_t key = 0;
    for (int64_t base = threadIdx.x; base < count; base += static_cast<int64_t>(kThreads) * kRound) {
        uint64_t v[kRound];
#pragma unroll
        for (int j = 0; j < kRound; ++j) {
            const int64_t i = base + static_cast<int64_t>(j) * kThreads;
            v[j] = partial[i < count ? i : count - 1];
        }
#pragma unroll
        for (int j = 0; j < kRound; ++j) key = v[j] > key ? v[j] : key;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t lo = __shfl_xor(static_cast<uint32_t>(key), o, kWave);
        const uint32_t hi = __shfl_xor(static_cast<uint32_t>(key >> 32), o, kWave);
        const uint64_t other = (static_cast<uint64_t>(hi) << 32) | lo;
        key = other > key ? other : key;
    }
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = key;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t b = red[0];
        for (int i = 1; i < kThreads / kWave; ++i) b = red[i] > b ? red[i] : b;
        const int64_t token = static_cast<int64_t>(0xffffffffu - static_cast<uint32_t>(b & 0xffffffffu));
        token_out[0] = token;
        if (history && step) {
            const int32_t k = step[0];
            if (k >= 0 && k < history_capacity) history[k] = token;
            step[0] = k + 1;
        }
        if (position) position[0] += 1;
    }
}

// ---------------------------------------------------------------------------
// Host helpers.

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool float_code(int d) { return nq::is_float_dtype(d); }
hipStream_t as_stream(void* s) { return static_cast<hipStream_t>(s); }

int proj_chunks_per_lane(int64_t hidden) {
    for (int n : {1, 2, 4, 8, 16})
        if (static_cast<int64_t>(n) * kWave * 8 >= hidden) return n;
    return 0;
}

int64_t proj_workgroups(int64_t vocab, int64_t hidden) {
    const int nch = proj_chunks_per_lane(hidden);
    if (nch == 0) return -1;
    const int64_t rows = static_cast<int64_t>(kProjWaves) * (kProjLoads / nch);
    return (vocab + rows - 1) / rows;
}

int attention_blocks(int64_t max_positions) { return static_cast<int>((max_positions + kSeqBlock - 1) / kSeqBlock); }

// How a prompt attention of `groups` workgroups (four units each) over up to
// `tiles` cache tiles of `rows` rows is laid out.
struct FlashPlan {
    int halves;
    int64_t splits, tiles_per_split;
};

// Fewer than 128 workgroups leave most of the chip idle: their cache goes to
// several, which pays for the merge where it is long enough: up to 32
// workgroups 64 rows each or more (as the workspace holds), 256 workgroups in
// all; from eight tiles on, up to 128 workgroups, two tiles each or more, 512 in
// all; 16 parts at most. Not split and split, bf16, 32 / 8 heads of 128 where
// not said: 17 tokens after 100 with 16 / 4 heads (8 workgroups) 10.8 and 9.5
// us, after 300 (16) 15.8 and 10.5; 64 after 250 (32) 16.2 and 12.8; 33 after
// 300 with 16 / 8 16.4 and 10.6; 100 after none (56, 300-row cache) 10.7 and
// 11.4; 128 after 3000 (64) 75 and 39; 256 after 1000 (128) 35 either way. Two
// tiles a part and one: 17 after 1000 with 16 / 4 13.4 and 12.2, but 33 after
// 500 with 64 / 8 (48, of which 480) 15.5 and 18.3. Below 512 workgroups that
// are not split, eight waves share a workgroup's cache between them where it
// has two tiles (17 after 1000: 30 us against 35 in four; 1024 tokens, 512
// workgroups: 44 either way; 17 of one tile 13.0 against 11.2).
FlashPlan flash_plan(int64_t groups, int64_t tiles, int64_t rows) {
    FlashPlan p;
    const auto least = [](int64_t a, int64_t b) { return a < b ? a : b; };
    const int64_t ones = groups <= 32 ? least(256 / groups, tiles * rows / kSeqBlock) : 1;
    const int64_t twos = groups < 128 && tiles >= 8 ? least(512 / groups, tiles / 2) : 1;
    const int64_t want = least(ones > twos ? ones : twos, 16);
    p.tiles_per_split = want > 1 ? (tiles + want - 1) / want : tiles;
    p.splits = (tiles + p.tiles_per_split - 1) / p.tiles_per_split;
    p.halves = groups < 512 && p.splits == 1 && tiles > 1 ? 2 : 1;
    return p;
}

// Prompt attention over a 16-bit cache. The grid is four units (16 tokens of a
// q head) a workgroup.
template <int D, int CT>
int launch_prompt_attention(const float* q, const void* kc, const void* vc, int64_t tokens, int q_heads, int kv_heads,
                            const int32_t* position, int64_t max_positions, float scaling, void* out, int odt,
                            float* ws, hipStream_t st) {
    constexpr int R = flash_rows<D>();
    const int group = q_heads / kv_heads;
    const int64_t units = (tokens + kFlashTokens - 1) / kFlashTokens * group;
    const int64_t quads = (units + kFlashUnits - 1) / kFlashUnits;
    const int64_t groups = quads * kv_heads;
    if (groups > 0x7fffffff) return NQ_ERR_SHAPE;
    const int64_t tiles = (max_positions + R - 1) / R;
    const FlashPlan plan = flash_plan(groups, tiles, R);
    FlashArgs a;
    a.q = q;
    a.k_cache = static_cast<const char*>(kc);
    a.v_cache = static_cast<const char*>(vc);
    a.tokens = tokens;
    a.max_positions = max_positions;
    a.position = position;
    a.q_heads = q_heads;
    a.kv_heads = kv_heads;
    a.quads = static_cast<int>(quads);
    a.tiles_per_split = static_cast<int>(plan.tiles_per_split);
    a.splits = static_cast<int>(plan.splits);
    a.scaling = scaling;
    a.out = out;
    a.odt = odt;
    a.vec_out = aligned16(out) ? 1 : 0;
    a.part_acc = ws;
    a.part_ml = ws + tokens * q_heads * plan.splits * D;
    const dim3 grid(static_cast<unsigned>(groups), static_cast<unsigned>(plan.splits));
    if (plan.halves == 2)
        hipLaunchKernelGGL((k_prompt_attention<D, CT, 2>), grid, dim3(512), 0, st, a);
    else
        hipLaunchKernelGGL((k_prompt_attention<D, CT, 1>), grid, dim3(256), 0, st, a);
    if (plan.splits > 1) {
        if (hipGetLastError() != hipSuccess) return NQ_ERR_LAUNCH;
        hipLaunchKernelGGL((k_attention_merge<D, 4, 1>), dim3(q_heads, static_cast<unsigned>(tokens)), dim3(D), 0, st,
                           a.part_ml, a.part_acc, q_heads, a.splits, a.tiles_per_split * R, position, max_positions,
                           out, odt);
    }
    return nq::launch_status();
}

// Merge of the 64-row blocks' partials. One token has few (token, head) rows,
// so more than one round of blocks goes to several groups of threads.
template <int D>
int launch_merge(const float* ml, const float* acc, int64_t tokens, int q_heads, int blocks, const int32_t* position,
                 int64_t max_positions, void* out, int odt, hipStream_t st) {
    constexpr int kGroups = 1024 / D;
    const dim3 grid(static_cast<unsigned>(q_heads), static_cast<unsigned>(tokens));
    if (tokens == 1 && blocks > 16)
        hipLaunchKernelGGL((k_attention_merge<D, 8, kGroups>), grid, dim3(D * kGroups), 0, st, ml, acc, q_heads, blocks,
                           kSeqBlock, position, max_positions, out, odt);
    else
        hipLaunchKernelGGL((k_attention_merge<D, 16, 1>), grid, dim3(D), 0, st, ml, acc, q_heads, blocks, kSeqBlock,
                           position, max_positions, out, odt);
    return nq::launch_status();
}

template <int D, int CT>
int launch_attention(const float* q, const void* kc, const void* vc, int64_t tokens, int q_heads, int kv_heads,
                     const int32_t* position, int64_t max_positions, float scaling, void* out, int odt, float* ml,
                     float* acc, hipStream_t st) {
    if constexpr (CT != NQ_DTYPE_F32) {
        // One token, and two with heads of 256 (8 / 4 heads, after 40, 500 and
        // 2000: 10.7, 16.3 and 20.8 us in one pass, 9.2, 15.9 and 17.6 in
        // blocks; of 128, 32 / 8 heads, after 500 9.1 and 10.8), take the blocks.
        if (tokens > (D == 256 ? 2 : 1))
            return launch_prompt_attention<D, CT>(q, kc, vc, tokens, q_heads, kv_heads, position, max_positions,
                                                  scaling, out, odt, ml, st);
    }
    const int group = q_heads / kv_heads;
    const int blocks = attention_blocks(max_positions);
    const int qt = tokens == 1 ? 1 : 16;
    const int64_t qblocks = (tokens + qt - 1) / qt;
    const size_t lds = attention_lds<D, CT>(group);
    if (lds > 64 * 1024) return NQ_ERR_UNSUPPORTED;
    if (qblocks * kv_heads > 0x7fffffff) return NQ_ERR_SHAPE;
    dim3 grid(static_cast<unsigned>(qblocks * kv_heads), static_cast<unsigned>(blocks));
    hipLaunchKernelGGL((k_attention_blocks<D, CT>), grid, dim3(group * kWave), lds, st, q,
                       static_cast<const char*>(kc), static_cast<const char*>(vc), tokens, q_heads, kv_heads, qt,
                       position, max_positions, scaling, ml, acc);
    if (hipGetLastError() != hipSuccess) return NQ_ERR_LAUNCH;
    return launch_merge<D>(ml, acc, tokens, q_heads, blocks, position, max_positions, out, odt, st);
}

template <int D>
int launch_attention_for(int cdt, const float* q, const void* kc, const void* vc, int64_t tokens, int q_heads,
                         int kv_heads, const int32_t* position, int64_t max_positions, float scaling, void* out,
                         int odt, float* ml, float* acc, hipStream_t st) {
    switch (cdt) {
        case NQ_DTYPE_F32:
            return launch_attention<D, NQ_DTYPE_F32>(q, kc, vc, tokens, q_heads, kv_heads, position, max_positions,
                                                     scaling, out, odt, ml, acc, st);
        case NQ_DTYPE_F16:
            return launch_attention<D, NQ_DTYPE_F16>(q, kc, vc, tokens, q_heads, kv_heads, position, max_positions,
                                                     scaling, out, odt, ml, acc, st);
        case NQ_DTYPE_BF16:
            return launch_attention<D, NQ_DTYPE_BF16>(q, kc, vc, tokens, q_heads, kv_heads, position, max_positions,
                                                      scaling, out, odt, ml, acc, st);
        default:
            return NQ_ERR_DTYPE;
    }
}

bool decode_fast_path(int head_dim, int cdt, int group) {
    const int eb = cdt == NQ_DTYPE_F32 ? 4 : 2;
    return head_dim * eb <= 256 && (group == 1 || group == 2 || group == 4 || group == 8);
}

int64_t round16(int64_t bytes) { return (bytes + 15) / 16 * 16; }

template <int D, int CT, int G>
int launch_decode_attention_g(const float* q, const float* k, const float* v, int kv_heads, const void* qn,
                              const void* kn, int ndt, float eps, const float* cs, const float* sn,
                              const int32_t* position, int64_t max_positions, void* kc, void* vc, float scaling,
                              void* out, int odt, float* ml, float* acc, bool merge, hipStream_t st) {
    const int blocks = attention_blocks(max_positions);
    // The partials form (no merge here) stores each block's output in fp16 for
    // the projection input that merges them; the merge below reads fp32 sums.
    if constexpr (D == 128 && G == kMfmaHeads && CT != NQ_DTYPE_F32) {
        if (merge)
            hipLaunchKernelGGL((k_decode_attention_mfma<CT, false>), dim3(kv_heads, blocks), dim3(G * kWave),
                               decode_attention_mfma_lds<CT>(), st, q, k, v, kv_heads, qn, kn, ndt, eps, cs, sn,
                               position, max_positions, static_cast<char*>(kc), static_cast<char*>(vc), scaling, ml,
                               acc);
        else
            hipLaunchKernelGGL((k_decode_attention_mfma<CT, true>), dim3(kv_heads, blocks), dim3(G * kWave),
                               decode_attention_mfma_lds<CT>(), st, q, k, v, kv_heads, qn, kn, ndt, eps, cs, sn,
                               position, max_positions, static_cast<char*>(kc), static_cast<char*>(vc), scaling, ml,
                               acc);
    } else {
        const size_t lds = decode_attention_lds<D, CT, G>();
        if (lds > 64 * 1024) return NQ_ERR_UNSUPPORTED;
        if (merge)
            hipLaunchKernelGGL((k_decode_attention<D, CT, G, false>), dim3(kv_heads, blocks), dim3(G * kWave), lds,
                               st, q, k, v, kv_heads, qn, kn, ndt, eps, cs, sn, position, max_positions,
                               static_cast<char*>(kc), static_cast<char*>(vc), scaling, ml, acc);
        else
            hipLaunchKernelGGL((k_decode_attention<D, CT, G, true>), dim3(kv_heads, blocks), dim3(G * kWave), lds,
                               st, q, k, v, kv_heads, qn, kn, ndt, eps, cs, sn, position, max_positions,
                               static_cast<char*>(kc), static_cast<char*>(vc), scaling, ml, acc);
    }
    if (hipGetLastError() != hipSuccess) return NQ_ERR_LAUNCH;
    if (!merge) return NQ_OK;  // the partials stay in the workspace
    return launch_merge<D>(ml, acc, 1, kv_heads * G, blocks, position, max_positions, out, odt, st);
}

template <int D, int CT>
int launch_decode_attention_ct(int group, const float* q, const float* k, const float* v, int kv_heads, const void* qn,
                               const void* kn, int ndt, float eps, const float* cs, const float* sn,
                               const int32_t* position, int64_t max_positions, void* kc, void* vc, float scaling,
                               void* out, int odt, float* ml, float* acc, bool merge, hipStream_t st) {
#define NQ_DA(G)                                                                                                   \
    return launch_decode_attention_g<D, CT, G>(q, k, v, kv_heads, qn, kn, ndt, eps, cs, sn, position, max_positions, \
                                               kc, vc, scaling, out, odt, ml, acc, merge, st)
    switch (group) {
        case 1: NQ_DA(1);
        case 2: NQ_DA(2);
        case 4: NQ_DA(4);
        case 8: NQ_DA(8);
        default: return NQ_ERR_UNSUPPORTED;
    }
#undef NQ_DA
}

}  // namespace

extern "C" int nq_embedding(const int64_t* ids, int64_t tokens, const void* table, int32_t table_dtype, int64_t vocab,
                            int64_t hidden, const float* scale, float* out, void* stream) {
    if (!ids || !table || !out) return NQ_ERR_ARGUMENT;
    if (!float_code(table_dtype)) return NQ_ERR_DTYPE;
    if (tokens <= 0 || tokens > 0x7fffffff || vocab <= 0 || hidden <= 0 || hidden % 8) return NQ_ERR_SHAPE;
    if (!aligned16(table) || !aligned16(out)) return NQ_ERR_ALIGNMENT;
    hipLaunchKernelGGL(k_embedding, dim3(static_cast<unsigned>(tokens)), dim3(kRowThreads), 0, as_stream(stream), ids,
                       table, table_dtype, vocab, hidden, scale, out, nullptr);
    return nq::launch_status();
}

extern "C" int nq_embedding_slots(const int64_t* ids, int64_t tokens, const void* table, int32_t table_dtype,
                                  int64_t vocab, int64_t hidden, const float* scale, float* out, float* slots,
                                  void* stream) {
    if (!ids || !table || !out || !slots) return NQ_ERR_ARGUMENT;
    if (!float_code(table_dtype)) return NQ_ERR_DTYPE;
    if (tokens <= 0 || tokens > 0x7fffffff || vocab <= 0 || hidden <= 0 || hidden % 16) return NQ_ERR_SHAPE;
    if (!aligned16(table) || !aligned16(out)) return NQ_ERR_ALIGNMENT;
    hipLaunchKernelGGL(k_embedding, dim3(static_cast<unsigned>(tokens)), dim3(kRowThreads), 0, as_stream(stream), ids,
                       table, table_dtype, vocab, hidden, scale, out, slots);
    return nq::launch_status();
}

extern "C" int nq_add_rmsnorm(float* residual, const void* delta, int32_t delta_dtype, const void* weight,
                              int32_t weight_dtype, float eps, int64_t tokens, int64_t hidden, void* out,
                              int32_t out_dtype, void* stream) {
    if (!residual || !weight || !out) return NQ_ERR_ARGUMENT;
    if ((delta && !float_code(delta_dtype)) || !float_code(weight_dtype) || !float_code(out_dtype)) return NQ_ERR_DTYPE;
    if (tokens <= 0 || tokens > 0x7fffffff || hidden <= 0 || hidden % 8 || hidden > kNormThreads * 32)
        return NQ_ERR_SHAPE;
    if (!(eps >= 0.0f)) return NQ_ERR_ARGUMENT;
    if (!aligned16(residual) || (delta && !aligned16(delta)) || !aligned16(weight) || !aligned16(out))
        return NQ_ERR_ALIGNMENT;
    const dim3 grid(static_cast<unsigned>(tokens)), block(kNormThreads);
    hipStream_t st = as_stream(stream);
    if (hidden <= kNormThreads * 8) {
        hipLaunchKernelGGL(k_add_rmsnorm<1>, grid, block, 0, st, residual, delta, delta_dtype, weight, weight_dtype,
                           eps, hidden, out, out_dtype);
    } else if (hidden <= kNormThreads * 16) {
        hipLaunchKernelGGL(k_add_rmsnorm<2>, grid, block, 0, st, residual, delta, delta_dtype, weight, weight_dtype,
                           eps, hidden, out, out_dtype);
    } else {
        hipLaunchKernelGGL(k_add_rmsnorm<4>, grid, block, 0, st, residual, delta, delta_dtype, weight, weight_dtype,
                           eps, hidden, out, out_dtype);
    }
    return nq::launch_status();
}

extern "C" int nq_qk_norm_rope_cache(const float* q, const float* k, const float* v, int64_t tokens, int32_t q_heads,
                                     int32_t kv_heads, int32_t head_dim, const void* q_norm, const void* k_norm,
                                     int32_t norm_dtype, float eps, const float* cos_table, const float* sin_table,
                                     const int32_t* position, int64_t max_positions, float* q_out, void* k_cache,
                                     void* v_cache, int32_t cache_dtype, void* stream) {
    if (!q || !k || !v || !cos_table || !sin_table || !position || !q_out || !k_cache || !v_cache)
        return NQ_ERR_ARGUMENT;
    if (((q_norm || k_norm) && !float_code(norm_dtype)) || !float_code(cache_dtype)) return NQ_ERR_DTYPE;
    if (tokens <= 0 || tokens > 0x7fffffff || q_heads <= 0 || kv_heads <= 0 || q_heads + kv_heads > 65535 ||
        max_positions <= 0)
        return NQ_ERR_SHAPE;
    if (!(eps >= 0.0f)) return NQ_ERR_ARGUMENT;
    const int groups = (q_heads + kv_heads + kHeadsPerGroup - 1) / kHeadsPerGroup;
    dim3 grid(static_cast<unsigned>(tokens), static_cast<unsigned>(groups));
    hipStream_t st = as_stream(stream);
#define NQ_QKR(D)                                                                                                     \
    hipLaunchKernelGGL(k_qk_norm_rope_cache<D>, grid, dim3(kHeadsPerGroup * kWave), 0, st, q, k, v, q_heads, kv_heads, \
                       q_norm, k_norm, norm_dtype, eps, cos_table, sin_table, position, max_positions, q_out, k_cache,  \
                       v_cache, cache_dtype)
    switch (head_dim) {
        case 64: NQ_QKR(64); break;
        case 128: NQ_QKR(128); break;
        case 256: NQ_QKR(256); break;
        default: return NQ_ERR_SHAPE;
    }
#undef NQ_QKR
    return nq::launch_status();
}

extern "C" int64_t nq_attention_workspace_bytes(int64_t tokens, int32_t q_heads, int32_t head_dim,
                                                int64_t max_positions) {
    if (tokens <= 0 || q_heads <= 0 || head_dim <= 0 || max_positions <= 0) return -1;
    const int64_t parts = tokens * q_heads * attention_blocks(max_positions);
    return parts * (2 + head_dim) * static_cast<int64_t>(sizeof(float));
}

extern "C" int nq_attention(const float* q, const void* k_cache, const void* v_cache, int32_t cache_dtype,
                            int64_t tokens, int32_t q_heads, int32_t kv_heads, int32_t head_dim,
                            const int32_t* position, int64_t max_positions, float scaling, void* out, int32_t out_dtype,
                            void* workspace, int64_t workspace_bytes, void* stream) {
    if (!q || !k_cache || !v_cache || !position || !out || !workspace) return NQ_ERR_ARGUMENT;
    if (!float_code(cache_dtype) || !float_code(out_dtype)) return NQ_ERR_DTYPE;
    if (tokens <= 0 || tokens > 65535 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads ||
        q_heads / kv_heads > 16 || max_positions <= 0 || attention_blocks(max_positions) > 65535)
        return NQ_ERR_SHAPE;
    if (!(scaling > 0.0f)) return NQ_ERR_ARGUMENT;
    if (!aligned16(k_cache) || !aligned16(v_cache) || !aligned16(workspace)) return NQ_ERR_ALIGNMENT;
    const int64_t need = nq_attention_workspace_bytes(tokens, q_heads, head_dim, max_positions);
    if (need < 0) return NQ_ERR_SHAPE;
    if (workspace_bytes < need) return NQ_ERR_WORKSPACE;
    const int64_t parts = tokens * q_heads * attention_blocks(max_positions);
    float* ml = static_cast<float*>(workspace);
    float* acc = ml + 2 * parts;
    hipStream_t st = as_stream(stream);
    switch (head_dim) {
        case 64:
            return launch_attention_for<64>(cache_dtype, q, k_cache, v_cache, tokens, q_heads, kv_heads, position,
                                            max_positions, scaling, out, out_dtype, ml, acc, st);
        case 128:
            return launch_attention_for<128>(cache_dtype, q, k_cache, v_cache, tokens, q_heads, kv_heads, position,
                                             max_positions, scaling, out, out_dtype, ml, acc, st);
        case 256:
            return launch_attention_for<256>(cache_dtype, q, k_cache, v_cache, tokens, q_heads, kv_heads, position,
                                             max_positions, scaling, out, out_dtype, ml, acc, st);
        default:
            return NQ_ERR_SHAPE;
    }
}

extern "C" int nq_silu_mul(const float* gate, const float* up, int64_t n, void* out, int32_t out_dtype, void* stream) {
    if (!gate || !up || !out) return NQ_ERR_ARGUMENT;
    if (!float_code(out_dtype)) return NQ_ERR_DTYPE;
    if (n <= 0 || n % 8) return NQ_ERR_SHAPE;
    if (!aligned16(gate) || !aligned16(up) || !aligned16(out)) return NQ_ERR_ALIGNMENT;
    const int64_t groups = (n / 8 + kRowThreads - 1) / kRowThreads;
    if (groups > 0x7fffffff) return NQ_ERR_SHAPE;
    hipLaunchKernelGGL(k_silu_mul, dim3(static_cast<unsigned>(groups)), dim3(kRowThreads), 0, as_stream(stream), gate,
                       up, n, out, out_dtype);
    return nq::launch_status();
}

extern "C" int64_t nq_output_projection_workspace_bytes(int64_t vocab, int64_t hidden) {
    if (vocab <= 0 || hidden <= 0 || hidden % 8) return -1;
    const int64_t wgs = proj_workgroups(vocab, hidden);
    return wgs < 0 ? -1 : wgs * static_cast<int64_t>(sizeof(uint64_t));
}

extern "C" int nq_output_projection(const void* x, int32_t x_dtype, const void* weight, int64_t vocab, int64_t hidden,
                                    float* logits, void* workspace, int64_t workspace_bytes, void* stream) {
    if (!x || !weight || !logits || !workspace) return NQ_ERR_ARGUMENT;
    if (x_dtype != NQ_DTYPE_F32 && x_dtype != NQ_DTYPE_BF16) return NQ_ERR_DTYPE;
    if (vocab <= 0 || vocab > 0x7fffffffLL || hidden <= 0 || hidden % 8 || hidden > 16 * kWave * 8)
        return NQ_ERR_SHAPE;
    if (!aligned16(x) || !aligned16(weight) || !aligned16(workspace)) return NQ_ERR_ALIGNMENT;
    const int64_t need = nq_output_projection_workspace_bytes(vocab, hidden);
    if (need < 0) return NQ_ERR_SHAPE;
    if (workspace_bytes < need) return NQ_ERR_WORKSPACE;
    const int64_t wgs = proj_workgroups(vocab, hidden);
    hipStream_t st = as_stream(stream);
    const uint16_t* w = static_cast<const uint16_t*>(weight);
    uint64_t* part = static_cast<uint64_t*>(workspace);
    const dim3 grid(static_cast<unsigned>(wgs)), block(kProjWaves * kWave);
    switch (proj_chunks_per_lane(hidden)) {
        case 1: hipLaunchKernelGGL(k_output_projection<1>, grid, block, 0, st, x, x_dtype, w, vocab, hidden, logits, part); break;
        case 2: hipLaunchKernelGGL(k_output_projection<2>, grid, block, 0, st, x, x_dtype, w, vocab, hidden, logits, part); break;
        case 4: hipLaunchKernelGGL(k_output_projection<4>, grid, block, 0, st, x, x_dtype, w, vocab, hidden, logits, part); break;
        case 8: hipLaunchKernelGGL(k_output_projection<8>, grid, block, 0, st, x, x_dtype, w, vocab, hidden, logits, part); break;
        case 16: hipLaunchKernelGGL(k_output_projection<16>, grid, block, 0, st, x, x_dtype, w, vocab, hidden, logits, part); break;
        default: return NQ_ERR_SHAPE;
    }
    return nq::launch_status();
}

extern "C" int nq_greedy_select(const void* workspace, int64_t vocab, int64_t hidden, int64_t* token_out,
                                int64_t* history, int64_t history_capacity, int32_t* step, int32_t* position,
                                void* stream) {
    if (!workspace || !token_out) return NQ_ERR_ARGUMENT;
    if ((history != nullptr) != (step != nullptr) || history_capacity < 0) return NQ_ERR_ARGUMENT;
    const int64_t wgs = vocab > 0 && vocab <= 0x7fffffffLL && hidden > 0 && hidden % 8 == 0 ? proj_workgroups(vocab, hidden) : -1;
    if (wgs <= 0) return NQ_ERR_SHAPE;
    hipLaunchKernelGGL(k_greedy_select, dim3(1), dim3(1024), 0, as_stream(stream),
                       static_cast<const uint64_t*>(workspace), wgs, token_out, history, history_capacity, step,
                       position);
    return nq::launch_status();
}

extern "C" int64_t nq_decode_attention_workspace_bytes(int32_t q_heads, int32_t kv_heads, int32_t head_dim,
                                                       int32_t cache_dtype, int64_t max_positions) {
    if (q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads || head_dim <= 0 || max_positions <= 0) return -1;
    if (decode_fast_path(head_dim, cache_dtype, q_heads / kv_heads))
        return nq_attention_workspace_bytes(1, q_heads, head_dim, max_positions);
    const int64_t attn = nq_attention_workspace_bytes(1, q_heads, head_dim, max_positions);
    return attn < 0 ? -1 : round16(static_cast<int64_t>(q_heads) * head_dim * 4) + attn;
}

namespace {

// nq_decode_attention (merge) and nq_decode_attention_partials (!merge: pass 1
// only, out unused).
int decode_attention(const float* q, const float* k, const float* v, int32_t q_heads, int32_t kv_heads,
                     int32_t head_dim, const void* q_norm, const void* k_norm, int32_t norm_dtype, float eps,
                     const float* cos_table, const float* sin_table, const int32_t* position, int64_t max_positions,
                     void* k_cache, void* v_cache, int32_t cache_dtype, float scaling, void* out, int32_t out_dtype,
                     bool merge, void* workspace, int64_t workspace_bytes, void* stream) {
    if (!q || !k || !v || !cos_table || !sin_table || !position || !k_cache || !v_cache || (merge && !out) || !workspace)
        return NQ_ERR_ARGUMENT;
    if (((q_norm || k_norm) && !float_code(norm_dtype)) || !float_code(cache_dtype) || (merge && !float_code(out_dtype)))
        return NQ_ERR_DTYPE;
    if (q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads || max_positions <= 0 ||
        attention_blocks(max_positions) > 65535)
        return NQ_ERR_SHAPE;
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return NQ_ERR_SHAPE;
    if (!(eps >= 0.0f) || !(scaling > 0.0f)) return NQ_ERR_ARGUMENT;
    if (!aligned16(k_cache) || !aligned16(v_cache) || !aligned16(workspace)) return NQ_ERR_ALIGNMENT;
    const int64_t need = nq_decode_attention_workspace_bytes(q_heads, kv_heads, head_dim, cache_dtype, max_positions);
    if (need < 0) return NQ_ERR_SHAPE;
    if (workspace_bytes < need) return NQ_ERR_WORKSPACE;
    hipStream_t st = as_stream(stream);
    const int group = q_heads / kv_heads;
    if (!decode_fast_path(head_dim, cache_dtype, group)) {
        if (!merge) return NQ_ERR_UNSUPPORTED;  // the partials exist only in the one-pass form
        // Unfused: rotate q into the workspace and append k/v, then attend.
        float* q_rot = static_cast<float*>(workspace);
        char* attn_ws = static_cast<char*>(workspace) + round16(static_cast<int64_t>(q_heads) * head_dim * 4);
        int rc = nq_qk_norm_rope_cache(q, k, v, 1, q_heads, kv_heads, head_dim, q_norm, k_norm, norm_dtype, eps,
                                       cos_table, sin_table, position, max_positions, q_rot, k_cache, v_cache,
                                       cache_dtype, stream);
        if (rc != NQ_OK) return rc;
        return nq_attention(q_rot, k_cache, v_cache, cache_dtype, 1, q_heads, kv_heads, head_dim, position,
                            max_positions, scaling, out, out_dtype, attn_ws,
                            workspace_bytes - round16(static_cast<int64_t>(q_heads) * head_dim * 4), stream);
    }
    float* ml = static_cast<float*>(workspace);
    float* acc = ml + 2 * static_cast<int64_t>(q_heads) * attention_blocks(max_positions);
#define NQ_DAC(D, CT)                                                                                             \
    return launch_decode_attention_ct<D, CT>(group, q, k, v, kv_heads, q_norm, k_norm, norm_dtype, eps, cos_table, \
                                             sin_table, position, max_positions, k_cache, v_cache, scaling, out,   \
                                             out_dtype, ml, acc, merge, st)
    if (head_dim == 64) {
        if (cache_dtype == NQ_DTYPE_F32) NQ_DAC(64, NQ_DTYPE_F32);
        if (cache_dtype == NQ_DTYPE_F16) NQ_DAC(64, NQ_DTYPE_F16);
        NQ_DAC(64, NQ_DTYPE_BF16);
    }
    if (cache_dtype == NQ_DTYPE_F16) NQ_DAC(128, NQ_DTYPE_F16);
    NQ_DAC(128, NQ_DTYPE_BF16);
#undef NQ_DAC
}

}  // namespace

extern "C" int nq_decode_attention(const float* q, const float* k, const float* v, int32_t q_heads, int32_t kv_heads,
                                   int32_t head_dim, const void* q_norm, const void* k_norm, int32_t norm_dtype,
                                   float eps, const float* cos_table, const float* sin_table, const int32_t* position,
                                   int64_t max_positions, void* k_cache, void* v_cache, int32_t cache_dtype,
                                   float scaling, void* out, int32_t out_dtype, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
    return decode_attention(q, k, v, q_heads, kv_heads, head_dim, q_norm, k_norm, norm_dtype, eps, cos_table,
                            sin_table, position, max_positions, k_cache, v_cache, cache_dtype, scaling, out, out_dtype,
                            true, workspace, workspace_bytes, stream);
}

extern "C" int nq_decode_attention_partials(const float* q, const float* k, const float* v, int32_t q_heads,
                                            int32_t kv_heads, int32_t head_dim, const void* q_norm,
                                            const void* k_norm, int32_t norm_dtype, float eps,
                                            const float* cos_table, const float* sin_table,
                                            const int32_t* position, int64_t max_positions, void* k_cache,
                                            void* v_cache, int32_t cache_dtype, float scaling, void* workspace,
                                            int64_t workspace_bytes, void* stream) {
    return decode_attention(q, k, v, q_heads, kv_heads, head_dim, q_norm, k_norm, norm_dtype, eps, cos_table,
                            sin_table, position, max_positions, k_cache, v_cache, cache_dtype, scaling, nullptr,
                            NQ_DTYPE_F32, false, workspace, workspace_bytes, stream);
}
