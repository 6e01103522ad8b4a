// Decode calls of 9 to 16 tokens: the two GEMMs on fp6 activation planes and
// fp4 signs (nq_planes.h) with v_mfma_scale_f32_16x16x128_f8f6f4.
//
// Five planes, 25 bits below the largest of 32 columns: the int8 digits of the
// calls of up to eight tokens hold 24 bits of the largest of 512, so no row
// keeps fewer here, with outlier channels either (4 planes, 20 bits, did:
// 4096 columns, one of them a thousand times the others, 2.1e-6 rel-L2 in
// digits, 3.0e-6 in four planes, 1.4e-7 in five; 64 columns 2.0e-7, 1.8e-6,
// 7e-8; normal rows of 4096 1.6e-5, 1.5e-6, 1.0e-7, the digits' rank
// intermediate taking its exponent from a bound). The operand of 16 rows and a
// 128-column block is, per plane, 64 lanes' first 16 bytes and then their last
// 8 (lane 16 g + row holds lane group g's 32 columns); exponents
// [kb / 4][lane][kb % 4].
//
// k_planes_gemm16: a workgroup takes 32 NG sign rows and its eight waves share
// the K blocks out in chunks of four (a lane's sign words of a chunk are one
// 16-byte load). With 32 sign rows all of a chunk's loads are issued before its
// first MFMA, by a scheduling barrier: left alone the compiler interleaves them
// to save registers, and a chunk takes several round trips (16 tokens, us: 4096
// -> 4096 r1638 16.9 and 14.4 with it, 10240 -> 2560 r1536 24.7 and 18.6). With
// 64 the registers that takes halve the workgroups of a CU, which costs more
// (4096 -> 2 x 12288 r3072 21.5 with it, 19.9 without). A wave reads an
// operand fragment once for all of its 2 NG tiles, straight from memory:
// nothing is shared between waves until their sums meet in LDS, added in wave
// order. GEMM 1's tiles are cut across the sign tiles so that two of them hold
// one exponent group of the rank intermediate (rows 16 m + 4 g + b of a
// 128-row block, m < 4 and m >= 4), which the workgroup then converts.
// Bound by latency (three launches, a chunk or two per wave) and, for long
// rows, by every workgroup reading the whole operand. Against the int8 stages
// at 16 tokens (us a call): 4096 -> 4096 r1638 14.4 and 28.5, 4096 -> 2 x 12288
// r3072 19.9 and 27.6, 10240 -> 2560 r1536 18.6 and 22.2, 14336 -> 4096 r2549
// 22.7 and 28.1. GEMM 1 forming its operand from x itself, without
// k_planes_prep16, was slower: every workgroup repeats the conversion.
#include "nq_decode_planes.h"
#include "nq_planes.h"

namespace {

constexpr int kP = 5;          // planes
constexpr int kWaves = 8;
constexpr int kM = 16;         // token rows

int64_t a256(int64_t n) { return (n + 255) & ~int64_t(255); }

template <int ADT, int SDT, bool VEC>
__global__ __launch_bounds__(kBlock) void k_planes_prep16(const PrepBatch batch) {
    const PrepArgs& pa = batch.p[blockIdx.y];
    const int lane = threadIdx.x & 63;
    const int64_t row = lane & 15, kb = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (kb >= pa.nkb || row >= pa.tokens) return;
    v16f half[2];
    GroupLoad<ADT, SDT, VEC> raw;
    raw.load(pa, row, kb, lane >> 4);
    raw.values(pa, row, kb, lane >> 4, half);
    store_planes<kP>(pa.out.planes + kb * (kP * kPlaneBytes), lane, pa.out.exps + (kb >> 2) * 256 + 4 * lane + (kb & 3),
                     half[0], half[1]);
}

// Plane PL's product of K block I of a chunk: B scales 2^(-5 PL) are the bytes of `eb` and `eb4`.
template <int PL, int I>
__device__ __forceinline__ v4f mfma16_plane(const v8i& a, const v8i& b, const v4f& c, int ea, int eb, int eb4) {
    if constexpr (PL < 4) return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 2, 4, I, ea, PL, eb);
    else return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 2, 4, I, ea, 0, eb4);
}

template <int NG>
__global__ __launch_bounds__(kWaves * 64, 2) void k_planes_gemm16(const GemmBatch batch) {
    constexpr int T = 2 * NG;                  // 16-row tiles
    constexpr int Q = 4 * T;                   // sums per lane
    constexpr int kParkStride = 32 * NG + 4;
    __shared__ __attribute__((aligned(16))) float red[kWaves * Q * 64];
    const int member = batch_member(batch, static_cast<int>(blockIdx.x));
    const GemmArgs& g = batch.p[member];
    const int ct = static_cast<int>(blockIdx.x) - batch.begin[member];
    const int lane = threadIdx.x & 63, n = lane & 15, kg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const bool mid = g.mid.planes != nullptr;
    const int nsc = static_cast<int>(g.nb);
    // Sign row of lane column n in tile t (clamped: past the last, its sums are not stored).
    const auto column = [&](int t) __attribute__((always_inline)) {
        if (!mid) return ct * (32 * NG) + 16 * t + n;
        const int grp = ct * NG + (t >> 1);
        return 128 * (grp >> 2) + 16 * (4 * (t & 1) + (n >> 2)) + 4 * (grp & 3) + (n & 3);
    };
    const int rows = static_cast<int>(g.n);
    uint32_t tile_at[T];
    int wl[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int c = column(t) < rows ? column(t) : rows - 1;
        tile_at[t] = static_cast<uint32_t>(c >> 4) * nsc * 64;
        wl[t] = 16 * kg + (c & 15);
    }
    // Planes 2 to 4 sum up apart from the two coarse ones, as in k_sign_gemm
    // (the matrix core truncates what it adds to an accumulator).
    v4f acc[2][T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[0][t] = acc[1][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t sign_mask = 0x88888888u, fp4_one = 0x22222222u;
    constexpr int kE = kPlaneBits;
    int eb = 127 | (127 - kE) << 8 | (127 - 2 * kE) << 16 | (127 - 3 * kE) << 24, eb4 = 127 - 4 * kE;
    asm volatile("" : "+v"(sign_mask), "+v"(fp4_one), "+v"(eb), "+v"(eb4));  // keep them in VGPRs
    for (int chunk = wave; 4 * chunk < nsc; chunk += kWaves) {
        const int dw = nsc - 4 * chunk < 4 ? nsc - 4 * chunk : 4;
        // A narrow last chunk's words lie closer; the load runs into what follows them, not used.
        WordRun<4> w[T];
#pragma unroll
        for (int t = 0; t < T; ++t)
            w[t] = *reinterpret_cast<const WordRun<4>*>(g.tiles + tile_at[t] + (chunk * 256 + wl[t] * dw));
        uint4 lo[4][kP];
        uint2 hi[4][kP];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint8_t* p = g.a.planes + static_cast<int64_t>(4 * chunk + (i < dw ? i : 0)) * (kP * kPlaneBytes);
#pragma unroll
            for (int f = 0; f < kP; ++f) {
                lo[i][f] = *reinterpret_cast<const uint4*>(p + f * kPlaneBytes + 16 * lane);
                hi[i][f] = *reinterpret_cast<const uint2*>(p + f * kPlaneBytes + 1024 + 8 * lane);
            }
        }
        const int ea = *reinterpret_cast<const int*>(g.a.exps + chunk * 256 + 4 * lane);
        if constexpr (NG == 1) __builtin_amdgcn_sched_barrier(0);
        each(std::make_integer_sequence<int, 4>{}, [&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            if (i >= dw) return;  // uniform
            v8i b[T];
#pragma unroll
            for (int t = 0; t < T; ++t) b[t] = expand_signs(w[t].w[i], sign_mask, fp4_one);
            each(std::make_integer_sequence<int, kP>{}, [&](auto f_) __attribute__((always_inline)) {
                constexpr int f = decltype(f_)::value;
                const uint4 l = lo[i][f];
                const uint2 u = hi[i][f];
                const v8i a = v8i{static_cast<int>(l.x), static_cast<int>(l.y), static_cast<int>(l.z),
                                  static_cast<int>(l.w), static_cast<int>(u.x), static_cast<int>(u.y), 0, 0};
#pragma unroll
                for (int t = 0; t < T; ++t)
                    acc[f > 1][t] = mfma16_plane<f, i>(a, b[t], acc[f > 1][t], ea, eb, eb4);
            });
        });
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) red[(wave * Q + 4 * t + j) * 64 + lane] = acc[0][t][j] + acc[1][t][j];
    __syncthreads();
    // Wave w finishes sums [w NG, + NG): token 4 kg + j of tile t, q = 4 t + j.
    const int t_own = wave * NG / 4;  // NG <= 2: one tile
    const int64_t col = column(t_own), col_c = col < g.n ? col : g.n - 1;
    const Raw2 cs_raw = load_raw2(g.col_scale, g.col_scale_dtype, col_c);
    const Raw2 bias_raw =
        load_raw2(g.bias ? g.bias : g.col_scale, g.bias ? g.bias_dtype : g.col_scale_dtype, col_c);
    const float cs = raw2_value(cs_raw, g.col_scale_dtype);
    float v[NG];
    int row[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int q = wave * NG + i;
        row[i] = 4 * kg + (q & 3);
        v[i] = 0.0f;
#pragma unroll
        for (int k = 0; k < kWaves; ++k) v[i] += red[(k * Q + q) * 64 + lane];
        v[i] *= cs;
    }
    if (mid) {
        __syncthreads();  // every sum is read
#pragma unroll
        for (int i = 0; i < NG; ++i) red[row[i] * kParkStride + 16 * t_own + n] = col < g.n ? v[i] : 0.0f;
        __syncthreads();
        const int task = threadIdx.x, trow = task & 15, grp = ct * NG + (task >> 4), kb = grp >> 2;
        if (task >= 16 * NG || trow >= g.m || kb >= g.mid_blocks) return;
        v16f half[2];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const v4f x = *reinterpret_cast<const v4f*>(red + trow * kParkStride + 32 * (task >> 4) + 4 * i);
#pragma unroll
            for (int b = 0; b < 4; ++b) half[i >> 2][4 * (i & 3) + b] = x[b];
        }
        const int ml = 16 * (grp & 3) + trow;
        store_planes<kP>(g.mid.planes + static_cast<int64_t>(kb) * (kP * kPlaneBytes), ml,
                         g.mid.exps + (kb >> 2) * 256 + 4 * ml + (kb & 3), half[0], half[1]);
        return;
    }
    if (col >= g.n) return;
    if (g.bias) {
#pragma unroll
        for (int i = 0; i < NG; ++i) v[i] += raw2_value(bias_raw, g.bias_dtype);
    }
    for (int64_t k = 0; k < g.salient_count; ++k) {
        float wk = nq::load_f32(g.salient_values, g.salient_dtype, col * g.salient_count + k);
        if (g.salient_scales) wk *= nq::load_f32(g.salient_scales, g.scale_dtype, k);
        const int64_t idx = g.salient_indices[k];
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int64_t t = row[i] < g.m ? row[i] : g.m - 1;
            v[i] += wk * nq::load_f32(g.x, g.x_dtype, t * g.in + idx);
        }
    }
#pragma unroll
    for (int i = 0; i < NG; ++i)
        if (row[i] < g.m) nq::store_f32_as(g.out, g.out_dtype, row[i] * g.n + col, v[i]);
}

// One GEMM phase of a batch. 32 sign rows a workgroup keep most CUs busy; a wide
// phase takes 64, which read the operand half as often (2 x 12288 sign rows at
// 16 tokens, the call: 19.9 us with 64, 23.7 with 32, 22.4 with 128).
void launch_phase16(GemmArgs* p, int count, hipStream_t stream) {
    int64_t groups = 0;
    for (int i = 0; i < count; ++i) groups += (p[i].n + 31) / 32;
    const int ng = groups >= 256 ? 2 : 1;
    GemmBatch gb;
    int64_t x = 0;
    for (int i = 0; i < kPrefillBatch; ++i) {
        gb.begin[i] = i < count ? static_cast<int32_t>(x) : INT32_MAX;
        gb.p[i] = i < count ? p[i] : GemmArgs{};
        // GEMM 1 writes every group of its operand, the ones past the rank too (zeros).
        if (i < count) x += p[i].mid.planes ? (4 * p[i].mid_blocks + ng - 1) / ng : (p[i].n + 32 * ng - 1) / (32 * ng);
    }
    const dim3 grid(static_cast<unsigned>(x)), block(kWaves * 64);
    if (ng == 2)
        hipLaunchKernelGGL(k_planes_gemm16<2>, grid, block, 0, stream, gb);
    else
        hipLaunchKernelGGL(k_planes_gemm16<1>, grid, block, 0, stream, gb);
}

// Planes and exponents of 16 rows of nkb 128-column blocks.
int64_t operand_bytes(int64_t nkb) { return a256(nkb * kP * kPlaneBytes) + a256((nkb + 3) / 4 * 256); }

Operand operand_at(uint8_t* ws, int64_t nkb) { return Operand{ws, ws + a256(nkb * kP * kPlaneBytes), 1}; }

}  // namespace

namespace nq {

int64_t decode_planes_bytes(const nq_linear_desc* d) {
    return operand_bytes((d->in_features + kBK - 1) / kBK) + operand_bytes((d->rank + kBK - 1) / kBK);
}

int launch_decode_planes(const nq_linear_desc* const* descs, int count, const void* const* xs, int x_dtype,
                         int64_t tokens, void* const* ys, int y_dtype, void* const* scratch, hipStream_t stream) {
    if (count < 1 || count > kPrefillBatch || tokens < 1 || tokens > kM) return NQ_ERR_SHAPE;
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const int64_t header = tiles_header_words();
    PrepBatch pb{};
    GemmArgs g1[kPrefillBatch], g2[kPrefillBatch];
    bool vec = true;
    int64_t nkb_max = 0;
    for (int i = 0; i < count; ++i) {
        const nq_linear_desc* d = descs[i];
        if (decode_planes_bytes(d) > decode_scratch_bytes(d, tokens)) return NQ_ERR_WORKSPACE;
        const int64_t nb1 = (d->in_features + kBK - 1) / kBK, nb2 = (d->rank + kBK - 1) / kBK;
        const int64_t v_words = (d->rank + kTileRows - 1) / kTileRows * nb1 * 64;
        uint8_t* const ws = static_cast<uint8_t*>(scratch[i]);
        PrepArgs& pa = pb.p[i];
        pa = PrepArgs{xs[i], d->scale_pre, x_dtype, d->scale_dtype, tokens, d->in_features, nb1, operand_at(ws, nb1)};
        vec = vec && d->in_features % 4 == 0 && aligned(xs[i]) && aligned(d->scale_pre);
        nkb_max = nb1 > nkb_max ? nb1 : nkb_max;
        g1[i] = GemmArgs{};
        g1[i].a = pa.out;
        g1[i].m = tokens;
        g1[i].tiles = static_cast<const uint32_t*>(d->tiles) + header;
        g1[i].n = d->rank;
        g1[i].nb = nb1;
        g1[i].col_scale = d->scale_mid;
        g1[i].col_scale_dtype = d->scale_dtype;
        g1[i].mid = operand_at(ws + operand_bytes(nb1), nb2);
        g1[i].mid_blocks = nb2;
        g2[i] = GemmArgs{};
        g2[i].a = g1[i].mid;
        g2[i].m = tokens;
        g2[i].tiles = g1[i].tiles + v_words;
        g2[i].n = d->out_features;
        g2[i].nb = nb2;
        g2[i].col_scale = d->scale_post;
        g2[i].col_scale_dtype = d->scale_dtype;
        g2[i].x = xs[i];
        g2[i].x_dtype = x_dtype;
        g2[i].in = d->in_features;
        g2[i].salient_count = d->salient_count;
        g2[i].salient_indices = d->salient_indices;
        g2[i].salient_values = d->salient_values;
        g2[i].salient_dtype = d->salient_dtype;
        g2[i].salient_scales = d->salient_scales;
        g2[i].scale_dtype = d->scale_dtype;
        g2[i].bias = d->bias;
        g2[i].bias_dtype = d->bias_dtype;
        g2[i].out = ys[i];
        g2[i].out_dtype = y_dtype;
    }
    const dim3 rows(static_cast<unsigned>((nkb_max + 3) / 4), static_cast<unsigned>(count));
    const int sdt = descs[0]->scale_dtype;
    bool prepped = false;
#define NQ_PREP(ADT, SDT)                                                                                   \
    if (vec && x_dtype == ADT && sdt == SDT) {                                                              \
        hipLaunchKernelGGL((k_planes_prep16<ADT, SDT, true>), rows, dim3(kBlock), 0, stream, pb);            \
        prepped = true;                                                                                     \
    }
#define NQ_PREP_S(ADT) NQ_PREP(ADT, NQ_DTYPE_F16) NQ_PREP(ADT, NQ_DTYPE_BF16) NQ_PREP(ADT, NQ_DTYPE_F32)
    NQ_PREP_S(NQ_DTYPE_BF16) NQ_PREP_S(NQ_DTYPE_F16) NQ_PREP_S(NQ_DTYPE_F32)
#undef NQ_PREP_S
#undef NQ_PREP
    if (!prepped) hipLaunchKernelGGL((k_planes_prep16<0, 0, false>), rows, dim3(kBlock), 0, stream, pb);
    launch_phase16(g1, count, stream);
    launch_phase16(g2, count, stream);
    return launch_status();
}

}  // namespace nq
