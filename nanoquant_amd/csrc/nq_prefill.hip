// Prefill path (tokens > 16) for the packed binary low-rank linear on gfx950:
// two dense sign GEMMs on v_mfma_scale_f32_32x32x64_f8f6f4 (activations as
// fp6, signs as fp4).
//
//   k_prep_rows:  planes of x * s_in                 (6-bit values, below)
//   GEMM 1:       planes of lm[t, r] = s_mid[r] * (x s_in · V±1ᵀ)[t, r]
//   GEMM 2:       y[t, o] = s_out[o] * (lm · U±1ᵀ)[t, o]
//                           + Σ_k x[t, idx_k] W_sal[o, k] (* scale_k) + bias[o]
//
// The operands' form and why: nq_planes.h.
//
// Activation operand in memory, in the order the MFMA and LDS want it: per
// 128-column block kb and group of 32 rows, for each 64-column step and plane
// the 64 lanes' first 16 bytes and then their last 8 (1536 bytes): a K step of
// a block tile is one run of bytes, moved into LDS linearly by
// global_load_lds_dwordx4 and read back without bank conflicts. Exponents:
// [kb][row group][lane][step], one byte each, read from global memory.
//
// Block tile up to 128 (tokens) x 256 (sign rows), four waves in a 2 x 2 grid
// of 64 x 128 (each expanded sign fragment feeds 2 x P MFMAs, each A fragment
// four). The next 128-column step moves into the idle LDS buffer during the
// current one's MFMAs; one barrier per step orders the swap. Within a step the
// 2 P (64-column step, plane) phases are software-pipelined.
//
// Split K: when a GEMM has too few (token, sign-row) tiles to fill the GPU,
// its K blocks are split into slices, each workgroup writes its raw fp32
// accumulators to partial[slice][t][n], and a reduction sums them in slice
// order (deterministic) and applies the epilogue. A batched call runs up to
// eight GEMMs of one phase in one launch, their (column block, slice) ranges
// concatenated along grid x.
#include "nq_planes.h"
#include "nq_prefill.h"

namespace {

// planes of act * colscale, zero past the last column. Grid: 16-row groups,
// four 128-column blocks (one per wave), members; lane 16 g + r takes row r and
// columns 16 m + 4 g + [0, 4). Bound by memory and launch.
// Written and read once, 2048 x 14336 bf16 moves 126 MB in 23.5 us (5.4 TB/s;
// fp16 operands with a scale per row: 19.4 us for 117 MB); 61 x 4096 4.6 us.
template <int ADT, int SDT, int P, bool VEC>
__global__ __launch_bounds__(kBlock) void k_prep_rows(const PrepBatch batch) {
    const PrepArgs& pa = batch.p[blockIdx.z];
    const int lane = threadIdx.x & 63, g = lane >> 4;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 16 + (lane & 15);
    const int64_t kb = static_cast<int64_t>(blockIdx.y) * 4 + (threadIdx.x >> 6);
    if (kb >= pa.nkb || row >= pa.tokens) return;
    v16f half[2];
    GroupLoad<ADT, SDT, VEC> raw;
    raw.load(pa, row, kb, g);
    raw.values(pa, row, kb, g, half);
    store_group<P>(pa.out, row, kb, g, half[0], half[1]);
}

// One plane's product of a 64-column step: A fp6 (format 2) with its row
// groups' exponents (byte STEP of `ea`), B fp4 (format 4) with the plane's.
template <int STEP, int PL>
__device__ __forceinline__ v16f mfma_plane(const v8i& a, const v8i& b, const v16f& c, int ea, int eb, int eb4) {
    if constexpr (PL < 4) return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 2, 4, STEP, ea, PL, eb);
    else return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 2, 4, STEP, ea, 0, eb4);
}

// The LDS byte address of a shared pointer, for M0.
__device__ __forceinline__ uint32_t lds_address(char* p) {
    typedef __attribute__((address_space(3))) char lds_char_t;
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char_t*)p));
}

// Block shapes, as (WR wave rows, II 32-row A fragments and JJ 32-column B
// fragments per wave): WR = 2: the four waves form a 2 x 2 grid; WR = 1: they
// sit side by side. P planes.
template <int WR, int II, int JJ, int P>
__global__ __launch_bounds__(kBlock, 2) void k_sign_gemm(const GemmBatch batch) {
    constexpr int RG = WR * II;                  // row groups per block
    constexpr int BM = kRows * RG;               // token rows per block
    constexpr int BN = (4 / WR) * 32 * JJ;       // sign rows per block
    constexpr int kGroupBytes = 2 * P * kPlaneBytes;  // a row group's K step
    // In LDS a group is 64 bytes longer: the compiler would pair two groups'
    // 8-byte reads (their distance a multiple of 512), which puts them in
    // registers the MFMA cannot take and costs four moves a phase.
    constexpr int kGroupLds = kGroupBytes + 64;
    constexpr int kStepBytes = RG * kGroupLds;
    constexpr int NI = RG * kGroupBytes / 1024;  // LDS transfers per K step (64 lanes x 16 bytes)
    constexpr int NL = (NI + 3) / 4;             // and per wave
    constexpr int kParkStride = BN + 16;         // floats per parked row (GEMM 1's epilogue)
    constexpr int kParkBytes = WR * kRows * kParkStride * 4;
    // Blocks of 32 and 64 rows (JJ = 1) have little work per step, so they keep
    // NB - 1 steps in flight and move sign words and exponents through LDS
    // too: a load the compiler tracks would be waited for together with every
    // transfer issued before it.
    constexpr bool kRing = JJ == 1;
    constexpr int NB = !kRing ? 2 : (RG == 1 ? 4 : (P == kPlanes ? 3 : 2));
    constexpr int kExpBytes = kRing ? 256 : 0;
    constexpr int kWordBytes = kRing ? BN / kTileRows * 1024 : 0;  // a four-block chunk of the block's tiles
    constexpr int kRingBytes = NB * (kStepBytes + kExpBytes) + 2 * kWordBytes;
    constexpr int kLds = kRingBytes > kParkBytes ? kRingBytes : kParkBytes;
    static_assert(!kRing || RG <= 2, "one transfer moves the exponents");
    constexpr int kSalient = 8;                  // salient columns staged at a time
    constexpr int W = JJ == 4 ? 2 : 4;           // blocks whose sign words one load moves
    constexpr bool kSignsAhead = JJ < 4;         // both by the registers JJ = 4 leaves
    static_assert(BN % 128 == 0 && kSalient * BM * 4 <= kLds, "epilogue tiles");
    const int member = batch_member(batch, static_cast<int>(blockIdx.x));
    const GemmArgs& g = batch.p[member];
    const int local = static_cast<int>(blockIdx.x) - batch.begin[member];
    const int col_blocks = static_cast<int>(g.col_blocks);
    const int slice = local / col_blocks;
    const int col_block = local - slice * col_blocks;
    __shared__ __attribute__((aligned(16))) char lds[kLds];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wm = WR == 2 ? wave >> 1 : 0;  // wave row
    const int wn = WR == 2 ? wave & 1 : wave;  // wave column
    const int h = lane >> 5;   // K half of the operands
    const int r = lane & 31;   // A row / B column within a 32-wide fragment
    const int64_t row_block = static_cast<int64_t>(blockIdx.z) * kRowsPerGridZ + blockIdx.y;
    const int64_t m0 = row_block * BM;
    if (m0 >= g.m) return;  // uniform
    const int64_t n0 = static_cast<int64_t>(col_block) * BN;
    const int64_t rt_count = (g.n + kTileRows - 1) / kTileRows;

    // The matrix core truncates what it adds to an accumulator. Two planes of
    // five bits sum up exactly or nearly so within an accumulator's 24 bits, so
    // with split operands planes 2 to 4 take one of their own (one for all
    // five: 1.0e-7 to 3.0e-7 rel-L2 against 7.5e-8 to 9.1e-8).
    constexpr int NA = P > 3 ? 2 : 1;
    v16f sums[NA][II][JJ];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int i = 0; i < II; ++i)
#pragma unroll
            for (int j = 0; j < JJ; ++j) sums[a][i][j] = v16f{};
    v16f (&acc)[II][JJ] = sums[0];

    // Activation steps: transfer i of a step fills LDS bytes [1024 i, + 1024).
    // Row groups past the last one read the last (their rows are not stored).
    // What the K loop uses of the arguments is taken once: loads from the
    // argument segment would be repeated (and waited for) in every step.
    const int nsc = static_cast<int>(g.nb);
    const int64_t groups = g.a.row_groups, rg0 = row_block * RG;
    const int rg_max = static_cast<int>(groups - rg0 < RG ? groups - rg0 : RG) - 1;
    const int k_begin = slice * static_cast<int>(g.k_per_split);
    const int k_end = k_begin + static_cast<int>(g.k_per_split) < nsc ? k_begin + static_cast<int>(g.k_per_split) : nsc;
    const uint64_t plane_stride = groups * kGroupBytes, exp_stride = groups * 128;  // from block to block
    uint64_t plane_at = uniform64(reinterpret_cast<uint64_t>(g.a.planes) + (k_begin * groups + rg0) * kGroupBytes);
    uint64_t exp_at = uniform64(reinterpret_cast<uint64_t>(g.a.exps) + (k_begin * groups + rg0) * 128);
    uint32_t a_src[NL];  // from the step's first row group (below 2^31: at most four groups)
    uint32_t a_dst[NL];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        // A wave without a transfer of its own repeats the last one.
        const int i = 4 * j + wave < NI ? 4 * j + wave : NI - 1, rg = i / (kGroupBytes / 1024);
        a_src[j] = (rg < rg_max ? rg : rg_max) * kGroupBytes + (i % (kGroupBytes / 1024)) * 1024 + 16 * lane;
        a_dst[j] = __builtin_amdgcn_readfirstlane(lds_address(lds) + rg * 64 + i * 1024);
    }
    // The transfer is issued as inline asm with its LDS address in M0: the
    // compiler then does not track it, so the fragment reads of the current
    // buffer wait only on themselves instead of on the tile in flight.
    // Completion is this kernel's own business: a transfer only targets a
    // buffer no wave reads in that step, and every step ends with a wait and a
    // barrier before the next buffer is read. Steps are moved in order;
    // `more`: there is another one (past the last, its tile is moved again).
    const auto load_a = [&](int buf, bool more) __attribute__((always_inline)) {
        const uint64_t base = plane_at;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            // s_nop: one wait state between the M0 write and the LDS transfer.
            asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(a_src[j]), "s"(base),
                         "{m0}"(a_dst[j] + buf * kStepBytes)
                         : "memory");
        }
        plane_at = uniform64(more ? base + plane_stride : base);
    };
    // Ring form: exponents of a step (lane i: bytes 4 i of the two row groups'
    // 256) and the sign words of a chunk (1 KB a tile: 64 lanes x 4 blocks;
    // lanes past a narrow last chunk read its first bytes again).
    const uint32_t exp_lds = lds_address(lds) + NB * kStepBytes, word_lds = exp_lds + NB * kExpBytes;
    const uint32_t exp_src = ((lane >> 5) < rg_max ? (lane >> 5) : rg_max) * 128 + 4 * (lane & 31);
    const auto load_exps_ring = [&](int buf, bool more) __attribute__((always_inline)) {
        const uint64_t base = exp_at;
        if (wave == 0)
            asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(exp_src), "s"(base),
                         "{m0}"(exp_lds + buf * kExpBytes)
                         : "memory");
        exp_at = uniform64(more ? base + exp_stride : base);
    };
    constexpr int NT = kRing ? BN / kTileRows / 4 : 1;  // sign tiles a wave moves
    uint64_t word_at[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int64_t rt = n0 / kTileRows + 4 * j + wave;
        word_at[j] = uniform64(reinterpret_cast<uint64_t>(g.tiles + (rt < rt_count ? rt : rt_count - 1) * nsc * 64));
    }
    const auto load_words_ring = [&](int chunk) __attribute__((always_inline)) {
        const int rem = nsc - 4 * chunk;
        const uint32_t src = 1024 * chunk + (rem >= 4 || lane < 16 * rem ? 16 * lane : 0);
#pragma unroll
        for (int j = 0; j < NT; ++j)
            asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(src), "s"(word_at[j]),
                         "{m0}"(word_lds + (chunk & 1) * kWordBytes + (4 * j + wave) * 1024)
                         : "memory");
    };
    // B fragment jj covers sign rows n0 + 32 JJ wn + 32 jj + [0, 32): lane r
    // reads row r & 15 of tile r >> 4 of that pair, the words of lane groups h
    // and 2 + h. Tiles past the last one read it (their columns are not stored).
    const int64_t rt0 = n0 / kTileRows + 2 * JJ * wn + (r >> 4);
    const int wl0 = 16 * h + (r & 15), wl1 = wl0 + 32;
    const uint32_t* bt[JJ];
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj) {
        const int64_t rt = rt0 + 2 * jj < rt_count ? rt0 + 2 * jj : rt_count - 1;
        bt[jj] = g.tiles + rt * nsc * 64;
    }
    uint32_t et[II];
#pragma unroll
    for (int ii = 0; ii < II; ++ii) {
        const int rg = II * wm + ii < rg_max ? II * wm + ii : rg_max;
        et[ii] = rg * 128 + 2 * lane;
    }
    // A lane's words of W consecutive blocks of a chunk lie side by side: one
    // load moves them (a dword load costs the texture path as much as a
    // 16-byte one here, lanes lying 16 bytes apart). Slices begin at multiples
    // of W; a load may run past a narrow last chunk (not used; the buffer has a
    // 256-byte tail).
    uint32_t words[JJ][2][W], next_words[JJ][2][W];
    int ea[II], next_ea[II];
    const auto load_words = [&](int sc) __attribute__((always_inline)) {
        const int rem_ = nsc - (sc & ~3);
        const int dw_ = rem_ < 4 ? rem_ : 4;
        const int64_t off_ = static_cast<int64_t>(sc >> 2) * 256 + (sc & 3);
#pragma unroll
        for (int jj = 0; jj < JJ; ++jj) {
            const WordRun<W> a = *reinterpret_cast<const WordRun<W>*>(bt[jj] + off_ + wl0 * dw_);
            const WordRun<W> b = *reinterpret_cast<const WordRun<W>*>(bt[jj] + off_ + wl1 * dw_);
#pragma unroll
            for (int i = 0; i < W; ++i) next_words[jj][0][i] = a.w[i], next_words[jj][1][i] = b.w[i];
        }
    };
    const auto load_exps = [&](bool more) __attribute__((always_inline)) {
        const uint8_t* const base = reinterpret_cast<const uint8_t*>(exp_at);
#pragma unroll
        for (int ii = 0; ii < II; ++ii) next_ea[ii] = *reinterpret_cast<const uint16_t*>(base + et[ii]);
        exp_at = uniform64(more ? exp_at + exp_stride : exp_at);
    };
    // Ring form: the two words of block sc for this lane, from LDS.
    const auto read_words = [&](int sc, uint32_t (&w)[2]) __attribute__((always_inline)) {
        const int rem = nsc - (sc & ~3), dw = rem < 4 ? rem : 4;
        const uint32_t* p = reinterpret_cast<const uint32_t*>(lds + NB * (kStepBytes + kExpBytes) +
                                                              ((sc >> 2) & 1) * kWordBytes) +
                            (2 * wn + (r >> 4)) * 256 + (sc & 3);
        w[0] = p[wl0 * dw], w[1] = p[wl1 * dw];
    };
    const auto take_words = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int jj = 0; jj < JJ; ++jj)
#pragma unroll
            for (int i = 0; i < W; ++i)
                words[jj][0][i] = next_words[jj][0][i], words[jj][1][i] = next_words[jj][1][i];
    };
    const auto take_exps = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int ii = 0; ii < II; ++ii) ea[ii] = next_ea[ii];
    };
    // Step s computes on buffer s & 1 while the tile of step s + 1 moves into
    // the other; a wait for this wave's transfers and one barrier per step
    // make every wave's part of the next tile visible before it is read.
    // Ring: step s computes on buffer s % NB while the next NB - 1 steps move;
    // the wait leaves the transfers of the youngest NB - 2 in flight (counted
    // as the fewest a wave issues per step).
    constexpr int kInFlight = (NB - 2) * NL;
    uint32_t ring_words[2];
    if constexpr (kRing) {
        load_words_ring(k_begin >> 2);
#pragma unroll
        for (int i = 0; i < NB - 1; ++i) {
            load_exps_ring(i, k_begin + i + 1 < k_end);
            load_a(i, k_begin + i + 1 < k_end);
        }
        __builtin_amdgcn_s_waitcnt(wait_vmcnt(kInFlight));
        __syncthreads();
        read_words(k_begin, ring_words);
    } else {
        load_a(0, k_begin + 1 < k_end);
        load_words(k_begin);
        load_exps(k_begin + 1 < k_end);
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        __syncthreads();
        take_words();
        take_exps();
    }
    int buf = 0;
    uint32_t sign_mask = 0x88888888u, fp4_one = 0x22222222u;
    // B scales 2^(-5p) of planes 0-3 (one byte each) and 4.
    constexpr int kE = kPlaneBits;
    int eb = 127 | (127 - kE) << 8 | (127 - 2 * kE) << 16 | (127 - 3 * kE) << 24, eb4 = 127 - 4 * kE;
    asm volatile("" : "+v"(sign_mask), "+v"(fp4_one), "+v"(eb), "+v"(eb4));  // keep them in VGPRs
    // One K step, block sc, word `wi` of the run.
    const auto step = [&](int sc, auto wi_) __attribute__((always_inline)) {
        constexpr int wi = decltype(wi_)::value;
        const bool more = sc + NB < k_end;
        if constexpr (kRing) {
            if (wi == 0 && sc + W < k_end) load_words_ring((sc >> 2) + 1);
            const int idle = buf == 0 ? NB - 1 : buf - 1;
            load_exps_ring(idle, more);
            load_a(idle, more);
            words[0][0][wi] = ring_words[0], words[0][1][wi] = ring_words[1];
#pragma unroll
            for (int ii = 0; ii < II; ++ii)
                ea[ii] = *reinterpret_cast<const uint16_t*>(lds + NB * kStepBytes + buf * kExpBytes + 128 * ii + 2 * lane);
        } else {
            load_a(buf ^ 1, more);
            if constexpr (wi == 0) load_words(sc + W < k_end ? sc + W : sc);
            load_exps(more);
        }
        // The sign words of the next steps are issued here, ahead of the
        // MFMAs; left to itself the scheduler sinks them to the step's end,
        // where the wait before the barrier would take their whole latency.
        __builtin_amdgcn_sched_barrier(0);
        const char* const a_lds = lds + buf * kStepBytes + II * wm * kGroupLds;
        const auto read_a = [&](int phase, v8i (&a)[II]) __attribute__((always_inline)) {
#pragma unroll
            for (int ii = 0; ii < II; ++ii) {
                const char* p = a_lds + ii * kGroupLds + phase * kPlaneBytes;
                const uint4 lo = *reinterpret_cast<const uint4*>(p + 16 * lane);
                const uint2 hi = *reinterpret_cast<const uint2*>(p + 1024 + 8 * lane);
                a[ii] = v8i{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z),
                            static_cast<int>(lo.w), static_cast<int>(hi.x), static_cast<int>(hi.y), 0, 0};
            }
        };
        // Software pipeline over the 2 P phases: a phase's MFMAs issue while
        // the next one's A fragments are read and, in the first step's last
        // phases, the second step's signs are expanded.
        v8i a_cur[II], b_cur[JJ], b_nxt[JJ];
        read_a(0, a_cur);
        if constexpr (kRing) read_words(sc + 1 < k_end ? sc + 1 : sc, ring_words);  // a chunk lands within its predecessor
#pragma unroll
        for (int jj = 0; jj < JJ; ++jj) b_cur[jj] = expand_signs(words[jj][0][wi], sign_mask, fp4_one);
        each(std::make_integer_sequence<int, 2 * P>{}, [&](auto phase_) __attribute__((always_inline)) {
            constexpr int kPhase = decltype(phase_)::value, kStep = kPhase / P, kPl = kPhase % P;
            constexpr int kSum = NA > 1 && kPl > 1 ? 1 : 0;
            __builtin_amdgcn_sched_barrier(0);
            v8i a_nxt[II];
            if constexpr (kPhase + 1 < 2 * P) read_a(kPhase + 1, a_nxt);
            if constexpr (kPhase == P - 1 && kSignsAhead) {
#pragma unroll
                for (int jj = 0; jj < JJ; ++jj) b_nxt[jj] = expand_signs(words[jj][1][wi], sign_mask, fp4_one);
            }
            if constexpr (kPhase == P && !kSignsAhead) {
#pragma unroll
                for (int jj = 0; jj < JJ; ++jj) b_cur[jj] = expand_signs(words[jj][1][wi], sign_mask, fp4_one);
            }
#pragma unroll
            for (int ii = 0; ii < II; ++ii)
#pragma unroll
                for (int jj = 0; jj < JJ; ++jj)
                    sums[kSum][ii][jj] = mfma_plane<kStep, kPl>(a_cur[ii], b_cur[jj], sums[kSum][ii][jj], ea[ii], eb, eb4);
            if constexpr (kPhase + 1 < 2 * P) {
                __builtin_amdgcn_sched_group_barrier(0x100, 2 * II, 0);  // LDS reads of the next phase
#pragma unroll
                for (int q = 0; q < II * JJ; ++q) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // a part of the expansion
                }
#pragma unroll
                for (int ii = 0; ii < II; ++ii) a_cur[ii] = a_nxt[ii];
            }
            if constexpr (kPhase == P - 1 && kSignsAhead) {
#pragma unroll
                for (int jj = 0; jj < JJ; ++jj) b_cur[jj] = b_nxt[jj];
            }
        });
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kRing) {
            __builtin_amdgcn_s_waitcnt(wait_vmcnt(kInFlight));
            __syncthreads();
            buf = buf + 1 < NB ? buf + 1 : 0;
        } else {
            take_exps();
            __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
            __syncthreads();
            buf ^= 1;
        }
    };
    for (int sc = k_begin; sc < k_end; sc += W) {
        each(std::make_integer_sequence<int, W>{}, [&](auto wi) __attribute__((always_inline)) {
            if (sc + decltype(wi)::value < k_end) step(sc + decltype(wi)::value, wi);  // uniform
        });
        if constexpr (!kRing) take_words();
    }
    if constexpr (kRing) {  // the transfers past the last step, before LDS is used again
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        __syncthreads();
    }
    if constexpr (NA > 1) {
#pragma unroll
        for (int ii = 0; ii < II; ++ii)
#pragma unroll
            for (int jj = 0; jj < JJ; ++jj) acc[ii][jj] += sums[1][ii][jj];
    }
    // Lane (h, r) holds D[8 (q / 4) + 4 h + q % 4][r] of each 32 x 32 tile; a
    // store is 32 columns of two rows.
    const int64_t row_w = m0 + kRows * II * wm, col_w = n0 + 32 * JJ * wn + r;
    const auto store = [&](auto* out, int64_t ld, auto convert) __attribute__((always_inline)) {
        const int64_t row0 = row_w + 4 * h;
        const bool all = row_w + kRows * II <= g.m;  // uniform per wave
        auto* const o = out + row0 * ld + col_w;
#pragma unroll
        for (int jj = 0; jj < JJ; ++jj) {
            if (col_w + 32 * jj >= g.n) continue;
            if (all) {
#pragma unroll
                for (int ii = 0; ii < II; ++ii)
#pragma unroll
                    for (int q = 0; q < 16; ++q)
                        o[(kRows * ii + 8 * (q >> 2) + (q & 3)) * ld + 32 * jj] = convert(acc[ii][jj][q]);
            } else {
#pragma unroll
                for (int ii = 0; ii < II; ++ii)
#pragma unroll
                    for (int q = 0; q < 16; ++q) {
                        const int row = kRows * ii + 8 * (q >> 2) + (q & 3);
                        if (row0 + row < g.m) o[row * ld + 32 * jj] = convert(acc[ii][jj][q]);
                    }
            }
        }
    };
    if (g.partial) {
        store(g.partial + static_cast<int64_t>(slice) * g.m * part_ld(g.n), part_ld(g.n), [](float v) { return v; });
        return;
    }
    float cs[JJ], bias[JJ];
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj) {
        const int64_t col = col_w + 32 * jj < g.n ? col_w + 32 * jj : g.n - 1;
        cs[jj] = nq::load_f32(g.col_scale, g.col_scale_dtype, col);
        bias[jj] = g.bias ? nq::load_f32(g.bias, g.bias_dtype, col) : 0.0f;
    }
    if (g.mid.planes) {
        // The rank intermediate as planes: one row group of every wave at a
        // time goes through LDS, so that a thread has the 32 columns that
        // share an exponent. Columns past n are zero.
        float* const park = reinterpret_cast<float*>(lds);
        each(std::make_integer_sequence<int, II>{}, [&](auto ii_) __attribute__((always_inline)) {
            constexpr int ii = decltype(ii_)::value;
            if constexpr (ii > 0) __syncthreads();  // the rows before are read
#pragma unroll
            for (int jj = 0; jj < JJ; ++jj) {
                const bool in = col_w + 32 * jj < g.n;
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    park[(kRows * wm + 8 * (q >> 2) + 4 * h + (q & 3)) * kParkStride + 32 * JJ * wn + 32 * jj + r] =
                        in ? acc[ii][jj][q] * cs[jj] : 0.0f;
            }
            __syncthreads();
            for (int task = threadIdx.x; task < WR * kRows * (BN / kBK) * 4; task += kBlock) {
                const int grp = (task >> 4) & 3, rest = task >> 6;
                const int prow = 16 * (rest % (2 * WR)) + (task & 15), kbl = rest / (2 * WR);
                const int64_t row = m0 + kRows * (II * (prow >> 5) + ii) + (prow & 31);
                const int64_t kb = n0 / kBK + kbl;
                if (row >= g.m || kb >= g.mid_blocks) continue;
                const float* src = park + prow * kParkStride + kbl * kBK + 4 * grp;
                v16f half[2];
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    const v4f v = *reinterpret_cast<const v4f*>(src + 16 * m);
#pragma unroll
                    for (int b = 0; b < 4; ++b) half[m >> 2][4 * (m & 3) + b] = v[b];
                }
                store_group<P>(g.mid, row, kb, grp, half[0], half[1]);
            }
        });
        return;
    }
#pragma unroll
    for (int ii = 0; ii < II; ++ii)
#pragma unroll
        for (int jj = 0; jj < JJ; ++jj)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[ii][jj][q] = acc[ii][jj][q] * cs[jj] + bias[jj];
    // Salient columns (none for most layers), kSalient at a time in index
    // order: x of the block's rows goes through LDS.
    float* const sx = reinterpret_cast<float*>(lds);  // [kSalient][BM]
    for (int64_t k0 = 0; k0 < g.salient_count; k0 += kSalient) {
        const int count = static_cast<int>(g.salient_count - k0 < kSalient ? g.salient_count - k0 : kSalient);
        if (k0 > 0) __syncthreads();
        for (int i = threadIdx.x; i < count * BM; i += kBlock) {
            const int64_t row = m0 + i % BM < g.m ? m0 + i % BM : g.m - 1;
            sx[i] = nq::load_f32(g.x, g.x_dtype, row * g.in + g.salient_indices[k0 + i / BM]);
        }
        __syncthreads();
        for (int k = 0; k < count; ++k) {
            float w[JJ];
#pragma unroll
            for (int jj = 0; jj < JJ; ++jj) {
                const int64_t col = col_w + 32 * jj < g.n ? col_w + 32 * jj : g.n - 1;
                w[jj] = nq::load_f32(g.salient_values, g.salient_dtype, col * g.salient_count + k0 + k);
                if (g.salient_scales) w[jj] *= nq::load_f32(g.salient_scales, g.scale_dtype, k0 + k);
            }
#pragma unroll
            for (int ii = 0; ii < II; ++ii)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const v4f xr = *reinterpret_cast<const v4f*>(sx + k * BM + kRows * (II * wm + ii) + 8 * i + 4 * h);
#pragma unroll
                    for (int jj = 0; jj < JJ; ++jj)
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[ii][jj][4 * i + j] += w[jj] * xr[j];
                }
        }
    }
    switch (g.out_dtype) {
        case NQ_DTYPE_F32:
            store(static_cast<float*>(g.out), g.n, [](float v) { return v; });
            break;
        case NQ_DTYPE_F16:
            store(static_cast<_Float16*>(g.out), g.n, [](float v) { return static_cast<_Float16>(v); });
            break;
        case NQ_DTYPE_BF16:
            store(static_cast<uint16_t*>(g.out), g.n, [](float v) { return nq::f32_to_bf16_bits(v); });
            break;
        default:
            break;
    }
}

// A GEMM of few tokens and few sign rows: a workgroup takes 32 sign rows and
// its eight waves share the K blocks out (chunks of four, dealt in turn), so
// that even a small matrix keeps most of the chip busy without a second launch
// for partial sums. Nothing is shared between the waves until their sums meet
// in LDS (added in wave order): A fragments go straight from memory (the
// operand's order is the fragment's) to registers, a step ahead. GEMM 1 takes
// the 32 rows of one exponent group of the rank intermediate: tile rows
// 16 m + 4 g + b of its 128-column block, in lane 4 m + b. Bound by latency.
// Calls with both GEMMs here and on k_sign_gemm: 4096 -> 4096 r1638 at 24
// tokens 15.9 and 24.6 us, at 61 16.9 and 26.4; at 128 23.6 and 27.8.
constexpr int kFewWaves = 8;

template <int II, int P>
__global__ __launch_bounds__(kFewWaves * 64, 2) void k_sign_gemm_few(const GemmBatch batch) {
    constexpr int Q = 16 * II;                // sums per lane
    constexpr int kOwn = Q / kFewWaves;       // of which a wave finishes
    constexpr int kParkStride = 36;
    __shared__ __attribute__((aligned(16))) float red[kFewWaves * Q * 64];
    const int member = batch_member(batch, static_cast<int>(blockIdx.x));
    const GemmArgs& g = batch.p[member];
    const int ct = static_cast<int>(blockIdx.x) - batch.begin[member];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int h = lane >> 5, r = lane & 31;
    const int64_t row_block = static_cast<int64_t>(blockIdx.z) * kRowsPerGridZ + blockIdx.y;
    const int64_t m0 = row_block * (kRows * II);
    if (m0 >= g.m) return;  // uniform
    const bool mid = g.mid.planes != nullptr;
    const int64_t col = mid ? static_cast<int64_t>(ct >> 2) * 128 + 16 * (r >> 2) + 4 * (ct & 3) + (r & 3)
                            : static_cast<int64_t>(ct) * 32 + r;
    const int64_t col_c = col < g.n ? col : g.n - 1;  // its words feed sums that are not stored
    const int nsc = static_cast<int>(g.nb);
    const int64_t groups = g.a.row_groups, rg0 = row_block * II;
    const uint32_t* const bt = g.tiles + (col_c >> 4) * nsc * 64;
    const int wl = 16 * h + static_cast<int>(col_c & 15);
    const uint8_t* at[II];
    const uint8_t* et[II];
#pragma unroll
    for (int ii = 0; ii < II; ++ii) {
        const int64_t rg = rg0 + ii < groups ? rg0 + ii : groups - 1;
        at[ii] = g.a.planes + rg * (2 * P * kPlaneBytes);
        et[ii] = g.a.exps + rg * 128 + 2 * lane;
    }
    constexpr int NA = P > 3 ? 2 : 1;  // as in k_sign_gemm
    v16f sums[NA][II];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int ii = 0; ii < II; ++ii) sums[a][ii] = v16f{};
    uint32_t sign_mask = 0x88888888u, fp4_one = 0x22222222u;
    constexpr int kE = kPlaneBits;
    int eb = 127 | (127 - kE) << 8 | (127 - 2 * kE) << 16 | (127 - 3 * kE) << 24, eb4 = 127 - 4 * kE;
    asm volatile("" : "+v"(sign_mask), "+v"(fp4_one), "+v"(eb), "+v"(eb4));  // keep them in VGPRs
    struct Step {
        uint4 lo[II][2 * P];
        uint2 hi[II][2 * P];
        int ea[II];
    };
    const auto load = [&](int sc, Step& s) __attribute__((always_inline)) {
#pragma unroll
        for (int ii = 0; ii < II; ++ii) {
            const uint8_t* p = at[ii] + sc * groups * (2 * P * kPlaneBytes);
#pragma unroll
            for (int f = 0; f < 2 * P; ++f) {
                s.lo[ii][f] = *reinterpret_cast<const uint4*>(p + f * kPlaneBytes + 16 * lane);
                s.hi[ii][f] = *reinterpret_cast<const uint2*>(p + f * kPlaneBytes + 1024 + 8 * lane);
            }
            s.ea[ii] = *reinterpret_cast<const uint16_t*>(et[ii] + sc * groups * 128);
        }
    };
    for (int chunk = wave; 4 * chunk < nsc; chunk += kFewWaves) {
        const int dw = nsc - 4 * chunk < 4 ? nsc - 4 * chunk : 4;
        // Four words side by side (a narrow last chunk's load runs into what follows it, not used).
        const WordRun<4> w0 = *reinterpret_cast<const WordRun<4>*>(bt + chunk * 256 + wl * dw);
        const WordRun<4> w1 = *reinterpret_cast<const WordRun<4>*>(bt + chunk * 256 + (wl + 32) * dw);
        Step cur, nxt;
        load(4 * chunk, cur);
        each(std::make_integer_sequence<int, 4>{}, [&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            if (i >= dw) return;  // uniform
            if (i + 1 < 4) load(4 * chunk + (i + 1 < dw ? i + 1 : i), nxt);
            __builtin_amdgcn_sched_barrier(0);  // the next step's loads stay ahead of this one's MFMAs
            each(std::make_integer_sequence<int, 2 * P>{}, [&](auto f_) __attribute__((always_inline)) {
                constexpr int f = decltype(f_)::value, kStep = f / P, kPl = f % P;
                constexpr int kSum = NA > 1 && kPl > 1 ? 1 : 0;
                const v8i b = expand_signs(kStep ? w1.w[i] : w0.w[i], sign_mask, fp4_one);
#pragma unroll
                for (int ii = 0; ii < II; ++ii) {
                    const uint4 lo = cur.lo[ii][f];
                    const uint2 hi = cur.hi[ii][f];
                    const v8i a = v8i{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z),
                                      static_cast<int>(lo.w), static_cast<int>(hi.x), static_cast<int>(hi.y), 0, 0};
                    sums[kSum][ii] = mfma_plane<kStep, kPl>(a, b, sums[kSum][ii], cur.ea[ii], eb, eb4);
                }
            });
            cur = nxt;
        });
    }
#pragma unroll
    for (int ii = 0; ii < II; ++ii) {
        if constexpr (NA > 1) sums[0][ii] += sums[1][ii];
#pragma unroll
        for (int q = 0; q < 16; ++q) red[(wave * Q + 16 * ii + q) * 64 + lane] = sums[0][ii][q];
    }
    __syncthreads();
    // Wave w finishes sums [w kOwn, + kOwn): rows 32 ii + 8 (q / 4) + 4 h + q % 4.
    const Raw2 cs_raw = load_raw2(g.col_scale, g.col_scale_dtype, col_c);
    const Raw2 bias_raw =
        load_raw2(g.bias ? g.bias : g.col_scale, g.bias ? g.bias_dtype : g.col_scale_dtype, col_c);
    const float cs = raw2_value(cs_raw, g.col_scale_dtype);
    float v[kOwn];
    int row[kOwn];
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
        const int q = wave * kOwn + i;
        row[i] = kRows * (q >> 4) + 8 * ((q & 15) >> 2) + 4 * h + (q & 3);
        v[i] = 0.0f;
#pragma unroll
        for (int k = 0; k < kFewWaves; ++k) v[i] += red[(k * Q + q) * 64 + lane];
        v[i] *= cs;
    }
    if (mid) {
        __syncthreads();  // every sum is read
#pragma unroll
        for (int i = 0; i < kOwn; ++i) red[row[i] * kParkStride + r] = col < g.n ? v[i] : 0.0f;
        __syncthreads();
        const int t = threadIdx.x;
        if (t >= kRows * II || m0 + t >= g.m) return;
        v16f half[2];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const v4f x = *reinterpret_cast<const v4f*>(red + t * kParkStride + 4 * i);
#pragma unroll
            for (int b = 0; b < 4; ++b) half[i >> 2][4 * (i & 3) + b] = x[b];
        }
        store_group<P>(g.mid, m0 + t, ct >> 2, ct & 3, half[0], half[1]);
        return;
    }
    if (col >= g.n) return;
    if (g.bias) {
#pragma unroll
        for (int i = 0; i < kOwn; ++i) v[i] += raw2_value(bias_raw, g.bias_dtype);
    }
    for (int64_t k = 0; k < g.salient_count; ++k) {
        float w = nq::load_f32(g.salient_values, g.salient_dtype, col * g.salient_count + k);
        if (g.salient_scales) w *= nq::load_f32(g.salient_scales, g.scale_dtype, k);
        const int64_t idx = g.salient_indices[k];
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            const int64_t t = m0 + row[i] < g.m ? m0 + row[i] : g.m - 1;
            v[i] += w * nq::load_f32(g.x, g.x_dtype, t * g.in + idx);
        }
    }
#pragma unroll
    for (int i = 0; i < kOwn; ++i)
        if (m0 + row[i] < g.m) nq::store_f32_as(g.out, g.out_dtype, (m0 + row[i]) * g.n + col, v[i]);
}

// Split-K epilogue of GEMM 2, one thread per output element (t, c), grid (the
// members' column blocks, token rows; t = blockIdx.y + kRowsPerGridZ *
// blockIdx.z): out[t, c] = (Σ_z partial[z][t][c]) * col_scale[c] + bias +
// salient columns, the slices summed in z order. The column's scale and bias
// and the first eight partials are loaded before any is used.
__global__ __launch_bounds__(kBlock) void k_reduce_splits(const GemmBatch batch) {
    const int member = batch_member(batch, static_cast<int>(blockIdx.x));
    const GemmArgs& ga = batch.p[member];
    const int splits = static_cast<int>(ga.splits);
    // Every argument the kernel reads is loaded in one batch: the empty asm
    // needs them all at one point, instead of one round trip per branch.
    GemmArgs g;
    g.m = ga.m;
    g.n = ga.n;
    g.out = ga.out;
    g.out_dtype = ga.out_dtype;
    g.partial = ga.partial;
    g.col_scale = ga.col_scale;
    g.col_scale_dtype = ga.col_scale_dtype;
    g.bias = ga.bias;
    g.bias_dtype = ga.bias_dtype;
    g.salient_count = ga.salient_count;
    asm volatile("" ::"s"(g.m), "s"(g.n), "s"(g.out), "s"(g.out_dtype), "s"(g.partial), "s"(g.col_scale),
                 "s"(g.col_scale_dtype), "s"(g.bias), "s"(g.bias_dtype), "s"(g.salient_count), "s"(splits));
    g.salient_values = ga.salient_values;
    g.salient_dtype = ga.salient_dtype;
    g.salient_scales = ga.salient_scales;
    g.scale_dtype = ga.scale_dtype;
    g.salient_indices = ga.salient_indices;
    g.x = ga.x;
    g.x_dtype = ga.x_dtype;
    g.in = ga.in;
    const int64_t c = static_cast<int64_t>(static_cast<int>(blockIdx.x) - batch.begin[member]) * kBlock + threadIdx.x;
    const int64_t t = static_cast<int64_t>(blockIdx.z) * kRowsPerGridZ + blockIdx.y;
    if (splits <= 1 || c >= g.n || t >= g.m) return;  // members without a split have no partials
    const int64_t plane = g.m * part_ld(g.n);
    const int64_t pi = t * part_ld(g.n) + c;
    const Raw2 cs_raw = load_raw2(g.col_scale, g.col_scale_dtype, c);
    const Raw2 bias_raw = load_raw2(g.bias ? g.bias : g.col_scale, g.bias ? g.bias_dtype : g.col_scale_dtype, c);
    float part[8];
    float v = 0.0f;
    for (int z0 = 0; z0 < splits; z0 += 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) part[j] = z0 + j < splits ? g.partial[(z0 + j) * plane + pi] : 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) v += part[j];
    }
    v *= raw2_value(cs_raw, g.col_scale_dtype);
    if (g.bias) v += raw2_value(bias_raw, g.bias_dtype);
    for (int64_t k = 0; k < g.salient_count; ++k) {
        float w = nq::load_f32(g.salient_values, g.salient_dtype, c * g.salient_count + k);
        if (g.salient_scales) w *= nq::load_f32(g.salient_scales, g.scale_dtype, k);
        v += w * nq::load_f32(g.x, g.x_dtype, t * g.in + g.salient_indices[k]);
    }
    nq::store_f32_as(g.out, g.out_dtype, t * g.n + c, v);
}

// Split-K epilogue of GEMM 1: planes of (Σ_z partial[z][t][c]) * col_scale[c],
// zero past the last column. A workgroup takes one 128-column block of 16 rows
// (16-row groups blockIdx.y + kRowsPerGridZ * blockIdx.z): lane 16 g + r has the
// 32 columns of row r that share an exponent, wave w sums slices w, w + 4, ...
// (bound by latency: every load of a slice is issued at once), and the waves
// meet in LDS in order.
template <int P>
__global__ __launch_bounds__(kBlock) void k_reduce_mid(const GemmBatch batch) {
    __shared__ float sum[3][32][64];
    const int member = batch_member(batch, static_cast<int>(blockIdx.x));
    const GemmArgs& g = batch.p[member];
    const int splits = static_cast<int>(g.splits);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, grp = lane >> 4;
    const int64_t kb = static_cast<int>(blockIdx.x) - batch.begin[member];
    const int64_t row = (static_cast<int64_t>(blockIdx.z) * kRowsPerGridZ + blockIdx.y) * 16 + (lane & 15);
    const int64_t c0 = kb * kBK + 4 * grp, ld = part_ld(g.n), plane = g.m * ld;
    const float* src = g.partial + (row < g.m ? row : g.m - 1) * ld + wave * plane;
    Raw2 cs[32];
    if (wave == 0) {
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const int64_t c = c0 + 16 * (i >> 2) + (i & 3);
            cs[i] = load_raw2(g.col_scale, g.col_scale_dtype, c < g.n ? c : g.n - 1);
        }
    }
    v16f half[2] = {v16f{}, v16f{}};
    for (int z = wave; z < splits; z += 4, src += 4 * plane) {
        v4f v[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) v[m] = *reinterpret_cast<const v4f*>(src + (c0 + 16 * m < g.n ? c0 + 16 * m : 0));
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int b = 0; b < 4; ++b) half[m >> 2][4 * (m & 3) + b] += v[m][b];
    }
    if (wave > 0) {
#pragma unroll
        for (int i = 0; i < 32; ++i) sum[wave - 1][i][lane] = half[i >> 4][i & 15];
    }
    __syncthreads();
    if (wave > 0 || row >= g.m) return;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const int64_t c = c0 + 16 * (i >> 2) + (i & 3);
        const float v = ((half[i >> 4][i & 15] + sum[0][i][lane]) + sum[1][i][lane]) + sum[2][i][lane];
        half[i >> 4][i & 15] = c < g.n ? v * raw2_value(cs[i], g.col_scale_dtype) : 0.0f;
    }
    store_group<P>(g.mid, row, kb, grp, half[0], half[1]);
}

// Tile counts and 128-column block counts of V [rank, in] and U [out, rank]
// (the same geometry as the decode tiles).
struct Geometry {
    int64_t rt1, nsc1, rt2, nsc2, v_words, u_words;
};

Geometry geometry(const nq_linear_desc* d) {
    Geometry g{};
    g.rt1 = (d->rank + kTileRows - 1) / kTileRows;
    g.nsc1 = (d->in_features + kBK - 1) / kBK;
    g.rt2 = (d->out_features + kTileRows - 1) / kTileRows;
    g.nsc2 = (d->rank + kBK - 1) / kBK;
    g.v_words = g.rt1 * g.nsc1 * 64;
    g.u_words = g.rt2 * g.nsc2 * 64;
    return g;
}

int64_t a256(int64_t n) { return (n + 255) & ~int64_t(255); }

// Block shapes of k_sign_gemm: tokens x sign rows, and for three and five
// planes the time of a K step of a workgroup that has its CU to itself and
// what each of several sharing the CU adds (us, fitted to the sweeps below).
struct Shape {
    int64_t rows, cols;
    double alone[2], shared[2];
};
enum ShapeId { kShape32x128, kShape64x128, kShape64x256, kShape128x128, kShape128x256, kShapes, kFew32, kFew64 };
constexpr Shape kShape[kShapes] = {{32, 128, {0.45, 0.60}, {0.33, 0.44}},
                                   {64, 128, {0.62, 0.85}, {0.52, 0.80}},
                                   {64, 256, {0.00, 1.30}, {0.00, 1.15}},   // five planes only
                                   {128, 128, {1.10, 0.00}, {0.80, 0.00}},  // three planes only
                                   {128, 256, {1.90, 0.00}, {1.55, 0.00}}};

// Block shape (or k_sign_gemm_few's rows) and K slices of one phase's launch.
struct Plan {
    int shape;
    int64_t k_per_split[kPrefillBatch], slices[kPrefillBatch];
};

// Plan of a phase: the shape and split with the least time by a model of its K
// steps, (steps + 2) x the step's time at the CU's average load, plus a
// reduction where K is split. Narrow shapes win while the grid is small: a
// step's time is mostly its own chain (barrier, LDS reads, dependent MFMAs).
// Measured on whole calls (us; every GEMM on one shape, no split: 32 x 128, 64
// x 128, 128 x 128, 128 x 256; then this plan): 4096 -> 4096 r1638 at 512
// tokens 34, 40, 55, 80; 34. 4096 -> 2 x 14336 r2549 at 512 126, 106, 108, 118;
// 90-102. 4096 -> 2 x 12288 r3072 at 2048 452, 374, 346, 322; 318-335. Splits
// pay only for few tokens of long rows (14336 -> 4096 r2549 at 61: 58 us
// unsplit, 34 with GEMM 1 in eight slices).
// A small grid goes to k_sign_gemm_few, without a search: at most 256
// workgroups (one a CU) of 32 sign rows and 32 tokens, or else 64 tokens, which
// read the signs half as often (32 against 64 tokens a workgroup where both
// fit: 4096 -> 4096 r1638 at 61 tokens 16.9 and 22.2 us, Q/K/V of 4096 21.4 and
// 24.7, 1152 -> 6912 r768 at 200 17.3 and 18.6). Beyond, every workgroup reading
// all of A costs more (2 x 12288 sign rows, 768 workgroups, at 24 tokens: 27 us
// against 24). More than 48 K blocks go there up to 64 tokens of three planes
// (against split K: 10240 -> 2560 r1536 at 24 tokens 23.1 and 26.9, at 61 22.1
// and 26.2, 9000 -> 300 r240 19.6 and 21.6; five planes 28.8 and 26.8 at 17, 26.5
// and 23.5 the other way).
constexpr int64_t kFewWgs = 256, kFewBlocks = 48, kFewTokens = 64;
constexpr double kCus = 256.0;
constexpr int64_t kMinSliceBlocks = 4;
constexpr double kReduceUs = 5.0;
constexpr double kPartialBytesPerUs = 4.0e6;

Plan plan_phase(int count, const int64_t* k_blocks, const int64_t* n, const int64_t* cap, int64_t tokens, int planes) {
    Plan best{};
    double best_us = -1.0;
    const int wide = planes == kPlanesSplit ? 1 : 0;
    int64_t kb_max = 1;
    for (int i = 0; i < count; ++i) kb_max = k_blocks[i] > kb_max ? k_blocks[i] : kb_max;
    int64_t few_wgs = 0;
    for (int i = 0; i < count; ++i) few_wgs += (n[i] + 31) / 32;
    const int64_t few32_wgs = few_wgs * ((tokens + 31) / 32);
    const bool few64 = few32_wgs > kFewWgs && planes == kPlanes;  // five planes of 64 rows would spill
    if ((few64 ? few_wgs * ((tokens + 63) / 64) : few32_wgs) <= kFewWgs &&
        (kb_max <= kFewBlocks || (tokens <= kFewTokens && planes == kPlanes && !few64))) {
        best.shape = few64 ? kFew64 : kFew32;
        for (int i = 0; i < count; ++i) best.k_per_split[i] = k_blocks[i], best.slices[i] = 1;
        return best;
    }
    for (int id = 0; id < kShapes; ++id) {
        const Shape& sh = kShape[id];
        if (sh.alone[wide] == 0.0 || (id > 0 && tokens <= kShape[id].rows / 2)) continue;
        const int64_t mt = (tokens + sh.rows - 1) / sh.rows;
        for (int64_t kmax = kb_max; kmax >= 1; --kmax) {
            Plan p{};
            p.shape = id;
            int64_t wgs = 0, steps = 0, partial_elems = 0;
            for (int i = 0; i < count; ++i) {
                const int64_t most_k = k_blocks[i] / kMinSliceBlocks > 1 ? k_blocks[i] / kMinSliceBlocks : 1;
                const int64_t most_cap = cap[i] / (tokens * part_ld(n[i])) > 1 ? cap[i] / (tokens * part_ld(n[i])) : 1;
                int64_t sl = (k_blocks[i] + kmax - 1) / kmax;
                sl = sl < most_k ? sl : most_k;
                sl = sl < most_cap ? sl : most_cap;
                p.k_per_split[i] = ((k_blocks[i] + sl - 1) / sl + 3) / 4 * 4;  // sign words load in runs of four
                p.slices[i] = (k_blocks[i] + p.k_per_split[i] - 1) / p.k_per_split[i];
                wgs += mt * ((n[i] + sh.cols - 1) / sh.cols) * p.slices[i];
                const int64_t own = p.k_per_split[i] < k_blocks[i] ? p.k_per_split[i] : k_blocks[i];
                steps = own > steps ? own : steps;
                if (p.slices[i] > 1) partial_elems += p.slices[i] * tokens * n[i];
            }
            const double per_cu = static_cast<double>(wgs) / kCus;
            const double whole = static_cast<double>(static_cast<int64_t>((wgs + 255) / 256));
            const double busy = (per_cu + whole) / 2 * sh.shared[wide];
            double us = static_cast<double>(steps + 2) * (per_cu > 1.0 && busy > sh.alone[wide] ? busy : sh.alone[wide]);
            if (partial_elems > 0) us += kReduceUs + 2.0 * static_cast<double>(partial_elems * 4) / kPartialBytesPerUs;
            if (best_us < 0.0 || us < best_us) best = p, best_us = us;
        }
    }
    return best;
}

// NQ_ERR_LAUNCH for a shape that the operands have no kernel for (kShape's zeros keep plans off them).
template <int P>
int launch_gemm(int shape, dim3 grid, hipStream_t stream, const GemmBatch& gb) {
    switch (shape) {
        case kShape32x128: hipLaunchKernelGGL((k_sign_gemm<1, 1, 1, P>), grid, dim3(kBlock), 0, stream, gb); return NQ_OK;
        case kShape64x128: hipLaunchKernelGGL((k_sign_gemm<1, 2, 1, P>), grid, dim3(kBlock), 0, stream, gb); return NQ_OK;
        case kFew32:
            hipLaunchKernelGGL((k_sign_gemm_few<1, P>), grid, dim3(kFewWaves * 64), 0, stream, gb);
            return NQ_OK;
        default: break;
    }
    if constexpr (P == kPlanesSplit) {
        if (shape != kShape64x256) return NQ_ERR_LAUNCH;
        hipLaunchKernelGGL((k_sign_gemm<1, 2, 2, P>), grid, dim3(kBlock), 0, stream, gb);
    } else {
        if (shape == kShape128x128)
            hipLaunchKernelGGL((k_sign_gemm<2, 2, 2, P>), grid, dim3(kBlock), 0, stream, gb);
        else if (shape == kShape128x256)
            hipLaunchKernelGGL((k_sign_gemm<2, 2, 4, P>), grid, dim3(kBlock), 0, stream, gb);
        else if (shape == kFew64)
            hipLaunchKernelGGL((k_sign_gemm_few<2, P>), grid, dim3(kFewWaves * 64), 0, stream, gb);
        else
            return NQ_ERR_LAUNCH;
    }
    return NQ_OK;
}

// One launch of a phase's GEMMs and, when any member's K is split, one launch
// of the reductions.
template <int P>
int launch_phase(GemmArgs* p, const Plan& plan, int count, int64_t tokens, hipStream_t stream) {
    const bool few = plan.shape >= kShapes;
    const int64_t rows = few ? (plan.shape == kFew32 ? 32 : 64) : kShape[plan.shape].rows;
    GemmBatch gb;
    GemmBatch rb;
    int64_t x = 0, rx = 0;
    const bool mid = p[0].mid.planes != nullptr;
    for (int i = 0; i < kPrefillBatch; ++i) {
        if (i >= count) {
            gb.begin[i] = rb.begin[i] = INT32_MAX;
            gb.p[i] = rb.p[i] = GemmArgs{};
            continue;
        }
        p[i].k_per_split = plan.k_per_split[i];
        p[i].splits = plan.slices[i];
        if (p[i].splits == 1) p[i].partial = nullptr;
        const int64_t cols = few ? 32 : kShape[plan.shape].cols;
        p[i].col_blocks = few && mid ? 4 * p[i].mid_blocks : (p[i].n + cols - 1) / cols;
        gb.begin[i] = static_cast<int32_t>(x);
        rb.begin[i] = static_cast<int32_t>(rx);
        gb.p[i] = rb.p[i] = p[i];
        x += p[i].col_blocks * p[i].splits;
        if (p[i].splits > 1) rx += mid ? p[i].mid_blocks : (p[i].n + kBlock - 1) / kBlock;
    }
    const auto grid_of = [](int64_t cols, int64_t rows) {
        return dim3(static_cast<unsigned>(cols), static_cast<unsigned>(rows < kRowsPerGridZ ? rows : kRowsPerGridZ),
                    static_cast<unsigned>((rows + kRowsPerGridZ - 1) / kRowsPerGridZ));
    };
    const int st = launch_gemm<P>(plan.shape, grid_of(x, (tokens + rows - 1) / rows), stream, gb);
    if (st != NQ_OK || rx == 0) return st;
    const dim3 grid = grid_of(rx, mid ? (tokens + 15) / 16 : tokens);
    if (mid)
        hipLaunchKernelGGL(k_reduce_mid<P>, grid, dim3(kBlock), 0, stream, rb);
    else
        hipLaunchKernelGGL(k_reduce_splits, grid, dim3(kBlock), 0, stream, rb);
    return NQ_OK;
}

int planes_of(const nq_linear_desc* d) {
    return d->prefill_operands == NQ_PREFILL_FP16_SPLIT ? kPlanesSplit : kPlanes;
}

struct Scratch {
    int64_t planes1, exps1, planes2, exps2, partial, total;
    int64_t partial_elems;  // fp32 elements of the partial buffer
};

// Workspace sizes are those of 16-bit operands (two per value when split),
// their rows' scales and partials for a split of 128 x 128 blocks (64-row up to
// 64 tokens) by a latency model of K steps of 1 us (0.5), 512 resident
// workgroups (1024), a reduction of 6 us (3) and 8 TB/s: callers size buffers
// and nq_linear_static takes or refuses calls by them. Where the planes take
// more than the 16-bit operands, the sizes grow so that the partials keep
// theirs; where they take less, what they leave holds more partials.
int64_t reserved_slices(int64_t tokens, int64_t k_blocks, int64_t n) {
    const bool small = tokens <= 64;
    const int64_t tiles = (tokens + 127) / 128 * ((n + 127) / 128);
    int64_t best = 1;
    double best_ns = -1.0;
    const int64_t most = k_blocks / 2 > 1 ? k_blocks / 2 : 1;
    for (int64_t want = 1; want <= most; ++want) {
        const int64_t per = (k_blocks + want - 1) / want, slices = (k_blocks + per - 1) / per;
        const int64_t resident = small ? 1024 : 512;
        const int64_t rounds = (tiles * slices + resident - 1) / resident;
        double ns = static_cast<double>(rounds * (per + 1)) * (small ? 500.0 : 1000.0);
        if (slices > 1) ns += (small ? 3000.0 : 6000.0) + 2.0 * static_cast<double>(slices * tokens * n * 4) / 8000.0;
        if (best_ns < 0.0 || ns < best_ns) best = slices, best_ns = ns;
    }
    return best;
}

int64_t reserved_partial_bytes(const nq_linear_desc* d, int64_t tokens) {
    const Geometry g = geometry(d);
    const int64_t s1 = reserved_slices(tokens, g.nsc1, d->rank), s2 = reserved_slices(tokens, g.nsc2, d->out_features);
    const int64_t p1 = s1 > 1 ? s1 * tokens * d->rank : 0, p2 = s2 > 1 ? s2 * tokens * d->out_features : 0;
    return a256(4 * (p1 > p2 ? p1 : p2));
}

// Everything else that is reserved: the fp32 rank intermediate, 16-bit operands, row scales.
int64_t reserved_operand_bytes(const nq_linear_desc* d, int64_t tokens) {
    const Geometry g = geometry(d);
    const int64_t parts = d->prefill_operands == NQ_PREFILL_FP16_SPLIT ? 2 : 1;
    return a256(tokens * d->rank * 4) + a256(tokens * g.nsc1 * kBK * 2 * parts) +
           a256(tokens * g.nsc2 * kBK * 2 * parts) + 2 * a256(tokens * 4);
}

Scratch scratch_layout(const nq_linear_desc* d, int64_t tokens) {
    const Geometry g = geometry(d);
    const int64_t groups = (tokens + kRows - 1) / kRows, bytes = 2 * planes_of(d) * kPlaneBytes;
    Scratch s{};
    s.planes1 = 0;
    s.exps1 = s.planes1 + a256(g.nsc1 * groups * bytes);
    s.planes2 = s.exps1 + a256(g.nsc1 * groups * 128);
    s.exps2 = s.planes2 + a256(g.nsc2 * groups * bytes);
    s.partial = s.exps2 + a256(g.nsc2 * groups * 128);
    // Room for the reserved partials beside the planes, which take more than
    // 16-bit operands where few tokens fill whole groups of 32 rows (without
    // it 9000 -> 300 r240 at 33 tokens had no room to split K: 36 us, 20 with).
    const int64_t operands = reserved_operand_bytes(d, tokens);
    s.total = (s.partial > operands ? s.partial : operands) + reserved_partial_bytes(d, tokens);
    s.partial_elems = (s.total - s.partial) / 4;
    return s;
}

}  // namespace

namespace nq {

int64_t prefill_reserved_bytes(const nq_linear_desc* d, int64_t tokens) {
    if (!d->tiles) return a256(tokens * d->rank * 4);
    return reserved_operand_bytes(d, tokens) + reserved_partial_bytes(d, tokens);
}

int64_t prefill_scratch_bytes(const nq_linear_desc* d, int64_t tokens) {
    return d->tiles ? scratch_layout(d, tokens).total : prefill_reserved_bytes(d, tokens);
}

bool prefill_path_applies(const nq_linear_desc* d, int64_t tokens) {
    return d->tiles != nullptr && tokens > 16 && tokens <= 65535 * int64_t(128);
}

}  // namespace nq

namespace {

template <int P>
int launch_prefill_planes(const nq_linear_desc* const* descs, int count, const void* const* xs, int x_dtype,
                          int64_t tokens, void* const* ys, int y_dtype, void* const* scratch, hipStream_t stream) {
    const int64_t header_words = nq::tiles_header_words();
    auto aligned = [](const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
    Geometry geo[kPrefillBatch];
    Scratch sl[kPrefillBatch];
    Operand mid[kPrefillBatch];
    PrepBatch pb{};
    bool all_vec = true;
    int64_t nkb_max = 0;
    for (int i = 0; i < count; ++i) {
        const nq_linear_desc* d = descs[i];
        geo[i] = geometry(d);
        if (d->tiles_bytes < (header_words + geo[i].v_words + geo[i].u_words) * 4) return NQ_ERR_ARGUMENT;
        if (d->prefill_operands != descs[0]->prefill_operands) return NQ_ERR_ARGUMENT;
        // The planes and partials are written and read by 16-byte accesses.
        if (!aligned(scratch[i], 16)) return NQ_ERR_ALIGNMENT;
        sl[i] = scratch_layout(d, tokens);
        uint8_t* ws = static_cast<uint8_t*>(scratch[i]);
        const int64_t groups = (tokens + kRows - 1) / kRows;
        PrepArgs& pa = pb.p[i];
        pa.act = xs[i];
        pa.act_dtype = x_dtype;
        pa.colscale = d->scale_pre;
        pa.colscale_dtype = d->scale_dtype;
        pa.tokens = tokens;
        pa.cols = d->in_features;
        pa.nkb = geo[i].nsc1;
        pa.out = Operand{ws + sl[i].planes1, ws + sl[i].exps1, groups};
        mid[i] = Operand{ws + sl[i].planes2, ws + sl[i].exps2, groups};
        all_vec = all_vec && d->in_features % 4 == 0 && aligned(xs[i], 16) && aligned(d->scale_pre, 16) &&
                  d->scale_dtype == descs[0]->scale_dtype;
        nkb_max = pa.nkb > nkb_max ? pa.nkb : nkb_max;
    }

    // Row passes: one launch.
    const dim3 rows(static_cast<unsigned>((tokens + 15) / 16), static_cast<unsigned>((nkb_max + 3) / 4),
                    static_cast<unsigned>(count));
    const int sdt = descs[0]->scale_dtype;
    bool prepped = false;
#define NQ_PREP(ADT, SDT)                                                                                  \
    if (all_vec && x_dtype == ADT && sdt == SDT) {                                                         \
        hipLaunchKernelGGL((k_prep_rows<ADT, SDT, P, true>), rows, dim3(kBlock), 0, stream, pb);            \
        prepped = true;                                                                                    \
    }
#define NQ_PREP_S(ADT) NQ_PREP(ADT, NQ_DTYPE_F16) NQ_PREP(ADT, NQ_DTYPE_BF16) NQ_PREP(ADT, NQ_DTYPE_F32)
    NQ_PREP_S(NQ_DTYPE_BF16) NQ_PREP_S(NQ_DTYPE_F16) NQ_PREP_S(NQ_DTYPE_F32)
#undef NQ_PREP_S
#undef NQ_PREP
    if (!prepped) hipLaunchKernelGGL((k_prep_rows<0, 0, P, false>), rows, dim3(kBlock), 0, stream, pb);

    int64_t kb[kPrefillBatch], n[kPrefillBatch], cap[kPrefillBatch];
    GemmArgs g[kPrefillBatch];

    // GEMM 1: the rank intermediate.
    for (int i = 0; i < count; ++i) {
        const nq_linear_desc* d = descs[i];
        kb[i] = geo[i].nsc1;
        n[i] = d->rank;
        cap[i] = sl[i].partial_elems;
        GemmArgs& a = g[i];
        a = GemmArgs{};
        a.a = pb.p[i].out;
        a.m = tokens;
        a.tiles = static_cast<const uint32_t*>(d->tiles) + header_words;
        a.n = d->rank;
        a.nb = geo[i].nsc1;
        a.col_scale = d->scale_mid;
        a.col_scale_dtype = d->scale_dtype;
        a.mid = mid[i];
        a.mid_blocks = geo[i].nsc2;
        a.partial = reinterpret_cast<float*>(static_cast<uint8_t*>(scratch[i]) + sl[i].partial);
    }
    const int st = launch_phase<P>(g, plan_phase(count, kb, n, cap, tokens, P), count, tokens, stream);
    if (st != NQ_OK) return st;

    // GEMM 2: y = s_out * (lm · U±1ᵀ) + salient columns + bias.
    for (int i = 0; i < count; ++i) {
        const nq_linear_desc* d = descs[i];
        kb[i] = geo[i].nsc2;
        n[i] = d->out_features;
        GemmArgs& a = g[i];
        a = GemmArgs{};
        a.a = mid[i];
        a.m = tokens;
        a.tiles = static_cast<const uint32_t*>(d->tiles) + header_words + geo[i].v_words;
        a.n = d->out_features;
        a.nb = geo[i].nsc2;
        a.col_scale = d->scale_post;
        a.col_scale_dtype = d->scale_dtype;
        a.x = xs[i];
        a.x_dtype = x_dtype;
        a.in = d->in_features;
        a.salient_count = d->salient_count;
        a.salient_indices = d->salient_indices;
        a.salient_values = d->salient_values;
        a.salient_dtype = d->salient_dtype;
        a.salient_scales = d->salient_scales;
        a.scale_dtype = d->scale_dtype;
        a.bias = d->bias;
        a.bias_dtype = d->bias_dtype;
        a.out = ys[i];
        a.out_dtype = y_dtype;
        a.partial = reinterpret_cast<float*>(static_cast<uint8_t*>(scratch[i]) + sl[i].partial);
    }
    const int st2 = launch_phase<P>(g, plan_phase(count, kb, n, cap, tokens, P), count, tokens, stream);
    return st2 != NQ_OK ? st2 : nq::launch_status();
}

}  // namespace

namespace nq {

int launch_prefill_batch(const nq_linear_desc* const* descs, int count, const void* const* xs, int x_dtype,
                         int64_t tokens, void* const* ys, int y_dtype, void* const* scratch, hipStream_t stream) {
    if (count < 1 || count > kPrefillBatch) return NQ_ERR_SHAPE;
    if (descs[0]->prefill_operands == NQ_PREFILL_FP16_SPLIT)
        return launch_prefill_planes<kPlanesSplit>(descs, count, xs, x_dtype, tokens, ys, y_dtype, scratch, stream);
    return launch_prefill_planes<kPlanes>(descs, count, xs, x_dtype, tokens, ys, y_dtype, scratch, stream);
}

int launch_prefill(const nq_linear_desc* d, const void* x, int x_dtype, int64_t tokens, void* y, int y_dtype,
                   void* scratch, hipStream_t stream) {
    return launch_prefill_batch(&d, 1, &x, x_dtype, tokens, &y, y_dtype, &scratch, stream);
}

}  // namespace nq
