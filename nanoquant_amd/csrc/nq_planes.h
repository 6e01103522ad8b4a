// fp6 activation planes and fp4 signs: what the prefill GEMMs (nq_prefill.hip)
// and the GEMMs of 9 to 16 tokens (nq_decode_planes.hip) share.
//
// Activation operands. A group of 32 columns of a row shares a power of two
// 2^e (its largest value lies in [2, 4) of it); a value is the sum of P fp6
// (e2m3) numbers, each the rounding of what the ones before left over, plane p
// in units of 2^(e - 5p). A plane takes a value below 4 to a remainder of at
// most 1/8, which the next plane, 32 times finer, sees below 4 again, so every
// plane adds five bits and P of them leave at most 2^(1 - 5 P) of the group's
// largest value: 2^-14 for P = 3 (default operands), 2^-24 for P = 5 (split
// operands, NQ_PREFILL_FP16_SPLIT, and 9 to 16 tokens). That is a share of the
// largest, not of each value: where fp16 kept 11 bits of a value a thousandth of
// its group's largest, three planes keep 4. The error of a product fell all the
// same in every form measured (rel-L2, fp16 and three planes, worst of 35 to
// 4096 columns: normal rows 3.4e-4 and 5.2e-5, one channel 30 times the others
// 4.6e-4 and 1.0e-4, a thousand times 4.6e-4 and 1.1e-4, the same with rows that
// fp16 holds exactly 2.4e-4 and 5.8e-5; split operands 4.6e-7 and 1.4e-7), the
// rounding of the largest having been the larger part. Exponents go from 2^-127
// up; a value of 3.3e38 or more (31/32 of fp32's range) may round to infinity.
// The group's exponent is the MFMA's A scale and the plane's 2^-5p its B scale, so no
// pass over the row is needed for a scale of its own, the rank intermediate is
// formed from its own values (no bound), and the sums come out unscaled. A
// group that holds a NaN or an infinity has the NaN scale: every output of the
// token is NaN, as the reference's fp32 forward yields (a non-finite
// activation reaches every rank value with both signs; reference.py:208-217).
//
// Why fp6 planes. The signs are exact in fp4 (+-1), the products exact, and
// the matrix cores take fp6 x fp4 at four times the fp16 rate (register-only
// loops on this chip: 4.1 - 6.7 PFLOP/s against 1.28 - 1.85, held down by
// power either way), so three planes cost 3/4 of one fp16 pass and five planes
// 5/8 of the two of split fp16 operands. Expanding signs costs one shift and
// one and-or for eight of them instead of three instructions for four.
//
// Sign operand, straight from the decode tile layout (16-row tiles; in
// 128-column block kb = 4c + d a lane's word d of chunk c holds, at bit 8b + m,
// column 128kb + 16m + 4g + b for lane group g). A 32 x 32 x 64 MFMA takes, in
// lane 32h + r, 32 k slots of B column r: exactly one word, that of lane group
// g = 2 step + h for 64-column step `step`. Slot 8s + j is the nibble j of
// dword s, sign bit 4j + s of the word: column 16 (4 (j & 1) + s) + 4g + (j >> 1).
// The columns of one word are the 32-column group that shares a scale.
#pragma once

#include <utility>

#include "nq_common.h"

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef uint32_t v6u __attribute__((ext_vector_type(6)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

constexpr int kBlock = 256;
constexpr int kBK = 128;                 // columns per K step
constexpr int kTileRows = 16;
constexpr int kRows = 32;                // rows of an operand group
constexpr int kPlaneBytes = 1536;        // 32 rows x 64 columns of 6 bits
constexpr int kPlaneBits = 5;            // what a plane adds
constexpr int kPrefillBatch = 8;         // members of one batched call
constexpr int kPlanes = 3, kPlanesSplit = 5;
constexpr int64_t kRowsPerGridZ = 65535;  // grid y's limit; rows beyond it go to grid z
// s_waitcnt vmcnt(n) expcnt(7) lgkmcnt(15): wait until this wave has at most n
// vector memory operations in flight (gfx9 encoding), as a builtin the
// compiler's own wait tracking takes into account.
constexpr int wait_vmcnt(int n) { return (n & 15) | 0x0F70 | (n >> 4) << 14; }
constexpr int kWaitVmcnt0 = wait_vmcnt(0);

__device__ __forceinline__ float exp2i(int e) { return __uint_as_float(static_cast<uint32_t>(e + 127) << 23); }

// An activation matrix as fp6 planes: rows in groups of 32 (row_groups of
// them; the rows past the last token hold anything), nkb 128-column blocks.
struct Operand {
    uint8_t* planes;     // [nkb][row_groups][2][P][1536]
    uint8_t* exps;       // [nkb][row_groups][64][2]
    int64_t row_groups;
};

// 32 values of a row that share an exponent, a[4 m + b] = column 16 m + 4g + b
// of their block and c the same for m + 4, as P planes of 24 bytes; returns
// the exponent's byte.
template <int P>
__device__ __forceinline__ int make_planes(v16f a, v16f c, v6u (&w)[P]) {
    uint32_t top = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t x = __float_as_uint(a[i]) & 0x7fffffffu, y = __float_as_uint(c[i]) & 0x7fffffffu;
        top = top > x ? top : x;
        top = top > y ? top : y;
    }
    const bool finite = top < 0x7f800000u;
    int e = static_cast<int>(top >> 23) - 128;  // 2^e: half the largest value's binade
    e = e < -127 ? -127 : (finite ? e : 0);     // the scale's smallest exponent
    // A small group is cut from its values times 2^64 (exact), so that the last
    // plane's unit is a normal number too.
    const bool small = e < -64;
    if (small) {
        const float up = exp2i(64);
#pragma unroll
        for (int i = 0; i < 16; ++i) a[i] *= up, c[i] *= up;
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const float unit = exp2i((small ? e + 64 : e) - kPlaneBits * p);
        w[p] = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(a, c, unit);
        // The conversion's operands outlive it, or the compiler lets its result
        // overlap them, and what is written first is read again (seen in the
        // last plane: 5.7e-6 rel-L2 with five).
        asm volatile("" : "+v"(w[p]) : "v"(a), "v"(c), "v"(unit));
        if (p + 1 < P) {
            v32f got = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(w[p], unit);
            asm volatile("" : "+v"(got) : "v"(w[p]), "v"(unit));
#pragma unroll
            for (int i = 0; i < 16; ++i) a[i] -= got[2 * i], c[i] -= got[2 * i + 1];  // exact
        }
    }
    return finite ? e + 127 : 255;
}

// The same into memory: lane `lane`'s 24 bytes at dst (kPlaneBytes from plane
// to plane), the exponent at *exp.
template <int P>
__device__ __forceinline__ void store_planes(uint8_t* dst, int lane, uint8_t* exp, const v16f& a, const v16f& c) {
    v6u w[P];
    *exp = static_cast<uint8_t>(make_planes<P>(a, c, w));
#pragma unroll
    for (int p = 0; p < P; ++p) {
        *reinterpret_cast<uint4*>(dst + p * kPlaneBytes + 16 * lane) = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
        *reinterpret_cast<uint2*>(dst + p * kPlaneBytes + 1024 + 8 * lane) = make_uint2(w[p][4], w[p][5]);
    }
}

// The group of lane group g of 128-column block kb of a row.
template <int P>
__device__ __forceinline__ void store_group(const Operand& op, int64_t row, int64_t kb, int g, const v16f& a,
                                            const v16f& c) {
    const int64_t at = kb * op.row_groups + (row >> 5);
    const int lane = 32 * (g & 1) + static_cast<int>(row & 31);
    store_planes<P>(op.planes + (at * 2 + (g >> 1)) * (P * kPlaneBytes), lane, op.exps + (at * 64 + lane) * 2 + (g >> 1),
                    a, c);
}

// Four elements of a buffer: one load (the host checked alignment), and their
// values as fp32.
template <int DT>
struct Raw4 {
    uint2 w;
    __device__ __forceinline__ void load(const void* __restrict__ p, int64_t i) {
        w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p) + i);
    }
    __device__ __forceinline__ float get(int b) const {
        const uint32_t u = (b < 2 ? w.x : w.y) >> (16 * (b & 1));
        if constexpr (DT == NQ_DTYPE_BF16) return __uint_as_float(u << 16);
        return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(u)));
    }
};
template <>
struct Raw4<NQ_DTYPE_F32> {
    v4f w;
    __device__ __forceinline__ void load(const void* __restrict__ p, int64_t i) {
        w = *reinterpret_cast<const v4f*>(static_cast<const float*>(p) + i);
    }
    __device__ __forceinline__ float get(int b) const { return w[b]; }
};

// Row pass of one member of a batched call.
struct PrepArgs {
    const void* act;                 // [tokens, cols] activations
    const void* colscale;            // [cols] s_in
    int act_dtype, colscale_dtype;
    int64_t tokens, cols, nkb;
    Operand out;
};

struct PrepBatch {
    PrepArgs p[kPrefillBatch];
};

// act * colscale of the group (row, kb, g), zero past the last column. VEC
// reads four elements per load (cols % 4 == 0, aligned, typed), issued by
// load(); the other form takes any type, alignment and width, in values().
template <int ADT, int SDT, bool VEC>
struct GroupLoad {
    Raw4<ADT> x[8];
    Raw4<SDT> s[8];
    __device__ __forceinline__ void load(const PrepArgs& pa, int64_t row, int64_t kb, int g) {
        if constexpr (VEC) {
            const int64_t c0 = kb * kBK + 4 * g, at = row * pa.cols + c0;
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                // Past the row: its first columns, dropped in values().
                const int64_t back = c0 + 16 * m < pa.cols ? 16 * m : -c0;
                x[m].load(pa.act, at + back);
                s[m].load(pa.colscale, c0 + back);
            }
        }
    }
    __device__ __forceinline__ void values(const PrepArgs& pa, int64_t row, int64_t kb, int g, v16f (&half)[2]) const {
        const int64_t c0 = kb * kBK + 4 * g, at = row * pa.cols + c0;
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int64_t c = 16 * m + b;
                float v = 0.0f;
                if constexpr (VEC) {
                    v = c0 + 16 * m < pa.cols ? x[m].get(b) * s[m].get(b) : 0.0f;
                } else if (c0 + c < pa.cols) {
                    v = nq::load_f32(pa.act, pa.act_dtype, at + c) * nq::load_f32(pa.colscale, pa.colscale_dtype, c0 + c);
                }
                half[m >> 2][4 * (m & 3) + b] = v;
            }
    }
};

// Signs of one word as the B operand (32 fp4 values of +-1): nibble j of dword
// s takes sign bit 4j + s.
__device__ __forceinline__ v8i expand_signs(uint32_t w, uint32_t mask, uint32_t one) {
    // The masks come in registers: a VOP3 instruction cannot take two literals.
    v8i b = {};
    b[0] = static_cast<int>(((w << 3) & mask) | one);
    b[1] = static_cast<int>(((w << 2) & mask) | one);
    b[2] = static_cast<int>(((w << 1) & mask) | one);
    b[3] = static_cast<int>((w & mask) | one);
    return b;
}

// A wave-uniform value, in scalar registers.
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    return static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32))) << 32 |
           static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}

template <typename F, int... I>
__device__ __forceinline__ void each(std::integer_sequence<int, I...>, const F& f) {
    (f(std::integral_constant<int, I>{}), ...);
}

template <int W>
struct __attribute__((packed, aligned(4))) WordRun {
    uint32_t w[W];
};

struct GemmArgs {
    Operand a;                // [m] rows of nb 128-column blocks
    int64_t m;                // tokens
    const uint32_t* tiles;    // sign tiles [rt][nb * 64] (chunked, see above)
    int64_t n;                // sign rows (rank or out)
    int64_t nb;               // 128-column blocks
    const void* col_scale;    // [n] s_mid or s_out
    int col_scale_dtype;
    // GEMM 1: the rank intermediate's operand (planes set); GEMM 2: y and what joins it
    Operand mid;
    int64_t mid_blocks;       // 128-column blocks of `mid`
    const void* x;
    int x_dtype;
    int64_t in;
    int64_t salient_count;
    const int32_t* salient_indices;
    const void* salient_values;
    int salient_dtype;
    const void* salient_scales;
    int scale_dtype;
    const void* bias;
    int bias_dtype;
    void* out;                // [M, n]
    int out_dtype;
    int64_t k_per_split;      // K blocks per K slice
    int64_t splits;           // K slices (1: no split)
    int64_t col_blocks;       // column blocks at the launch's block width
    float* partial;           // [splits][M][part_ld(n)] raw accumulators, or null (direct epilogue)
};

// Floats per row of the partials: rows begin at multiples of 16 bytes.
__host__ __device__ constexpr int64_t part_ld(int64_t n) { return (n + 3) & ~int64_t(3); }

// Up to kPrefillBatch GEMMs of one phase (the members of a batched call share
// the token count) in one launch. Grid x concatenates the members' ranges:
// member i owns [begin[i], begin[i + 1]) (k_sign_gemm: col_blocks * splits
// workgroups, slice-major; the reductions: their column blocks, none for a
// member without a split); begin[i] = INT32_MAX past the last member.
struct GemmBatch {
    int32_t begin[kPrefillBatch];
    GemmArgs p[kPrefillBatch];
};

// The member whose range holds grid-x index x: the last one beginning at or
// before it (a member with an empty range shares its begin with the next).
__device__ __forceinline__ int batch_member(const GemmBatch& b, int x) {
    int m = 0;
#pragma unroll
    for (int i = 1; i < kPrefillBatch; ++i) m = x >= b.begin[i] ? i : m;
    return m;
}

// Element i of an F32 / F16 / BF16 buffer from two unconditional 16-bit
// loads (the halves of an fp32, or the same half twice), decoded by a
// uniform select: no branch surrounds the loads, so they issue together.
struct Raw2 {
    uint32_t lo, hi;
};

__device__ __forceinline__ Raw2 load_raw2(const void* __restrict__ p, int dtype, int64_t i) {
    const uint16_t* h = static_cast<const uint16_t*>(p);
    const bool wide = dtype == NQ_DTYPE_F32;
    return Raw2{h[wide ? 2 * i : i], h[wide ? 2 * i + 1 : i]};
}

__device__ __forceinline__ float raw2_value(const Raw2& r, int dtype) {
    const float f32 = __uint_as_float((r.hi << 16) | (r.lo & 0xffffu));
    const float bf16 = __uint_as_float(r.lo << 16);
    const float f16 = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(r.lo)));
    return dtype == NQ_DTYPE_F32 ? f32 : (dtype == NQ_DTYPE_BF16 ? bf16 : f16);
}

}  // namespace
