// Products to f32 accuracy on the bf16 matrix cores for weights that are not
// whole 128-column int4 groups: the int8 format, the grouped products' plain
// f32 experts, and int4 matrices of any extents (their groups then run across
// rows).  Every weight is dequantised exactly as the per-element kernels do
// it, in f32, and both sides are split into bf16 terms (bf16split.hpp):
//     f32 rows x weights:  3 x 3 terms, the six products above 2^-27 kept
//     f16 rows:            2 x 3 terms (an f16 is two terms exactly), five
//     bf16 rows:           1 x 3 terms, three
// summed in f32 by v_mfma_f32_32x32x16_bf16, the small products first.  What
// is dropped (2^-26 of a product) is below the rounding of one f32 sum.
// bf16 ends where f32 does, at 2^-126, and a third term is 2^-17 of its value:
// so f32 values are split as 2^24 times themselves (exact), which puts even
// their last bit, 2^-149, among bf16's normal numbers, and the sums are scaled
// back (exact but for results that are subnormal).  Without it relative errors
// were 4e-5 at 2^-120 and 2e-3 at 2^-126.  It costs a multiplication an f32
// value, 1-2% and up to 6% where the narrow tile splits few rows (us without /
// with, one card): int8 512 x 4096 x 4096 92.7 / 94.0, 256 rows of 8 f32 experts
// of 2048 x 4096 71.9 / 73.0, int4 100 x 4100 x 4004 46.3 / 46.8, int8 33 x 4864
// x 352 29.9 / 31.5, 8 rows of 4 f32 experts of 156 x 2397 10.7 / 11.3.  Operands from 2^104 on (sums from 2^80 with f32 experts) leave
// the range and are computed again as below.
//
// Bound: the matrix cores, at three to six times the product's flops; for few
// rows the weight bytes.
//
// A workgroup of eight waves (sixteen for the narrow tile, 32 columns) computes
// a BM x BN tile, BN = 64 WN columns: wave (wn, g) owns 64 columns and the K group g of KG.  The weights need no LDS:
// a lane loads eight consecutive k of two adjacent columns, which after the
// split are exactly its operands of two n-tiles (MFMA column c of n-tile j is
// tile column 2 c + j).  The activations are shared by the waves of a K group
// and go through LDS, split once, as 16-byte chunks of eight k, the layout the
// A operands are read in.  Both are loaded a stage (32 k) ahead.  The K
// groups' sums meet in LDS in group order: a tile list too short for the chip
// still fills it, without a workspace, so products on different streams share
// nothing and a capture needs no earlier call.
//
// A product that overflowed, scaled or not, or met an infinity or a NaN (any
// of which the split turns into a non-finite sum) is computed again by the
// per-element loop, so such values read as they do there.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bf16split.hpp"
#include "internal.hpp"
#include "splitk.hpp"

namespace accel {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
// vectors at their elements' alignment: rows of any width start anywhere
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint16_t u16x8u __attribute__((ext_vector_type(8), aligned(2)));
typedef uint16_t u16u __attribute__((aligned(1)));

constexpr int KS = 32;   // k of a stage
constexpr float kUp = 0x1p24f, kDown = 0x1p-24f;   // f32 values in the split

// ---- activations ----------------------------------------------------------

struct ActF32 {
    static constexpr const char* kName = "ActF32";
    typedef float T;
    static constexpr int kTerms = 3;
    static constexpr float kScale = kUp, kUnscale = kDown;   // of the values split
    static __device__ __forceinline__ float value(T v) { return v; }
};
struct ActF16 {
    static constexpr const char* kName = "ActF16";
    typedef uint16_t T;
    static constexpr int kTerms = 2;
    static constexpr float kScale = 1.0f, kUnscale = 1.0f;
    static __device__ __forceinline__ float value(T v) { return half_bits_to_float(v); }
};
struct ActBf16 {
    static constexpr const char* kName = "ActBf16";
    typedef uint16_t T;
    static constexpr int kTerms = 1;   // itself: not split
    static constexpr float kUnscale = 1.0f;
    static __device__ __forceinline__ float value(T v) { return __uint_as_float((uint32_t)v << 16); }
};

// ---- weight sources ---------------------------------------------------------
//
// A lane's unit is eight rows of two columns.  load(r, i, F, d0, d1) fetches
// row i of a unit: F is the flat index of the (uniform) row and tile column,
// d0 and d1 the lane's distances to its two columns.  pair() gives row i's
// weights to split, 1 / kUnscale times what at() gives: dequantised as the
// per-element kernels do it.  FORM says how rows
// lie: kOdd, any N; kEven, N even, so a pair is adjacent and in one
// quantisation block, one load; kRows, N a multiple of the block, so a row's
// scales start at a whole block.  kOne is a lane of one column, any N: the
// narrow tile's.
// F and the row's base stay in scalar registers.
enum { kOdd, kEven, kRows, kOne };
constexpr bool paired(int form) { return form == kEven || form == kRows; }

// Plain f32 weights (the grouped products' experts, [K, N] each).
template <int FORM>
struct F32W {
    using One = F32W<kOne>;
    One one() const { return {w}; }
    static constexpr float kUnscale = kDown;
    static std::string name() { return tname("F32W", FORM); }   // as a kernel trace shows it
    const float* w;
    __device__ __forceinline__ F32W expert(int e, size_t per) const { return {w + e * per}; }
    struct Regs { float v[8][2]; };
    __device__ __forceinline__ void load(Regs& r, int i, uint64_t F, uint32_t d0,
                                         uint32_t d1) const {
        const float* p = w + F;
        if constexpr (paired(FORM)) {
            const f32x2u t =
                __builtin_nontemporal_load(reinterpret_cast<const f32x2u*>(p + d0));
            r.v[i][0] = t.x;
            r.v[i][1] = t.y;
        } else {
            r.v[i][0] = p[d0];
            if constexpr (FORM == kOdd) r.v[i][1] = p[d1];
        }
    }
    __device__ __forceinline__ void pair(Regs& r, int i, int, float& w0, float& w1) const {
        asm volatile("" : "+v"(r.v[i][0]));   // as in Int8W
        w0 = r.v[i][0] * kUp;
        if constexpr (FORM != kOne) {
            asm volatile("" : "+v"(r.v[i][1]));
            w1 = r.v[i][1] * kUp;
        }
    }
    __device__ __forceinline__ float at(uint64_t f) const { return w[f]; }
};

template <int FORM>
struct Int8W {
    using One = Int8W<kOne>;
    One one() const { return {q, s}; }
    static constexpr float kUnscale = 1.0f;   // a weight is 0 or at least 2^-24
    static std::string name() { return tname("Int8W", FORM); }
    const int8_t* q;
    const uint16_t* s;
    struct Regs { uint32_t q[8], s[8], q1[8], s1[8]; };   // q1, s1: odd N only
    __device__ __forceinline__ void load(Regs& r, int i, uint64_t F, uint32_t d0,
                                         uint32_t d1) const {
        const int8_t* qp = q + F;
        const uint16_t* sp = s + (F >> 5);
        const uint32_t fs = (uint32_t)F & 31u;
        if constexpr (paired(FORM)) {
            r.q[i] = *reinterpret_cast<const u16u*>(qp + d0);
            r.s[i] = FORM == kRows ? sp[d0 >> 5] : sp[(fs + d0) >> 5];
        } else {
            r.q[i] = (uint8_t)qp[d0];
            r.s[i] = sp[(fs + d0) >> 5];
            if constexpr (FORM == kOdd) {
                r.q1[i] = (uint8_t)qp[d1];
                r.s1[i] = sp[(fs + d1) >> 5];
            }
        }
    }
    __device__ __forceinline__ void pair(Regs& r, int i, int, float& w0, float& w1) const {
        // without the marks the compiler unpacks a word where it was loaded,
        // waiting for it there
        asm volatile("" : "+v"(r.q[i]), "+v"(r.s[i]));
        const float s0 = half_bits_to_float((uint16_t)r.s[i]);
        w0 = (float)(int8_t)r.q[i] * s0;
        if constexpr (paired(FORM)) {
            w1 = (float)(int8_t)(r.q[i] >> 8) * s0;
        } else if constexpr (FORM == kOdd) {
            asm volatile("" : "+v"(r.q1[i]), "+v"(r.s1[i]));
            w1 = (float)(int8_t)r.q1[i] * half_bits_to_float((uint16_t)r.s1[i]);
        }
    }
    __device__ __forceinline__ float at(uint64_t f) const {
        return (float)q[f] * half_bits_to_float(s[f >> 5]);
    }
};

// The int4 format with groups of 128 flat weights that may run across rows:
// (code - z) * s, or z where the scale is zero.
template <int FORM>
struct Int4W {
    using One = Int4W<kOne>;
    One one() const { return {c, s, z}; }
    static constexpr float kUnscale = 1.0f;   // a weight is 0 or at least 2^-48
    static std::string name() { return tname("Int4W", FORM); }
    const uint8_t* c;      // two codes a byte, low nibble first
    const uint16_t* s;
    const uint16_t* z;
    // an experts' stacked planes: whole groups each
    __device__ __forceinline__ Int4W expert(int e, size_t per) const {
        return {c + e * (per >> 1), s + e * (per >> 7), z + e * (per >> 7)};
    }
    struct Regs { uint32_t c[8], s[8], z[8], c1[8], s1[8], z1[8]; };   // the last three: odd N only
    __device__ __forceinline__ void load(Regs& r, int i, uint64_t F, uint32_t d0,
                                         uint32_t d1) const {
        const uint8_t* cp = c + (F >> 1);
        const uint16_t* sp = s + (F >> 7);
        const uint16_t* zp = z + (F >> 7);
        const uint32_t fg = FORM == kRows ? 0u : (uint32_t)F & 127u;
        if constexpr (paired(FORM)) {
            r.c[i] = cp[d0 >> 1];
            r.s[i] = sp[(fg + d0) >> 7];
            r.z[i] = zp[(fg + d0) >> 7];
        } else {
            const uint32_t fc = (uint32_t)F & 1u;
            r.c[i] = cp[(fc + d0) >> 1];
            r.s[i] = sp[(fg + d0) >> 7];
            r.z[i] = zp[(fg + d0) >> 7];
            if constexpr (FORM == kOdd) {
                r.c1[i] = cp[(fc + d1) >> 1];
                r.s1[i] = sp[(fg + d1) >> 7];
                r.z1[i] = zp[(fg + d1) >> 7];
            }
        }
    }
    static __device__ __forceinline__ float weight(uint32_t code, uint32_t sb, uint32_t zb) {
        const float sv = half_bits_to_float((uint16_t)sb), zv = half_bits_to_float((uint16_t)zb);
        // the selection is a row's, not a weight's: the product is zero there
        // (or NaN for an infinite zero point, and then computed again)
        return __builtin_fmaf((float)code - zv, sv, sv == 0.0f ? zv : 0.0f);
    }
    // flat: the first column's flat index, for which nibble is whose
    __device__ __forceinline__ void pair(Regs& r, int i, int flat, float& w0, float& w1) const {
        asm volatile("" : "+v"(r.c[i]), "+v"(r.s[i]), "+v"(r.z[i]));
        if constexpr (paired(FORM)) {
            w0 = weight(r.c[i] & 15u, r.s[i], r.z[i]);
            w1 = weight(r.c[i] >> 4, r.s[i], r.z[i]);
        } else {
            const int sh = 4 * (flat & 1);
            w0 = weight((r.c[i] >> sh) & 15u, r.s[i], r.z[i]);
            if constexpr (FORM == kOne) return;
            asm volatile("" : "+v"(r.c1[i]), "+v"(r.s1[i]), "+v"(r.z1[i]));
            w1 = weight((r.c1[i] >> (4 - sh)) & 15u, r.s1[i], r.z1[i]);
        }
    }
    __device__ __forceinline__ float at(uint64_t f) const {
        const float sv = half_bits_to_float(s[f >> 7]), zv = half_bits_to_float(z[f >> 7]);
        const uint32_t code = (c[f >> 1] >> (4 * (f & 1))) & 15u;
        return sv == 0.0f ? zv : ((float)code - zv) * sv;
    }
};

// ---- the tile -----------------------------------------------------------------

template <typename ACT, int TM, int WN, int KG>
struct Shape {
    static constexpr int TN = KG == 16 ? 1 : 2;        // columns a lane
    static constexpr int BM = 32 * TM, BN = 32 * TN * WN;
    static constexpr int TG = 64 * WN;                 // lanes of a K group
    static constexpr int NT = KG * TG;
    static constexpr int NA = ACT::kTerms;
    static constexpr int AU = BM * 4 / TG;             // A staging units a lane
    static_assert(BM * 4 % TG == 0, "whole units a lane");
    // a k octet's chunks, 16 bytes a row; the 64 spare bytes put a row's four
    // octets in different banks
    static constexpr int OCT = BM * 16 + 64;
    static constexpr int BUF = NA * 4 * OCT;
    // a one-wave group reads its own chunks only: no second buffer needed
    static constexpr int BUFS = WN == 1 ? 1 : 2;
    static constexpr int SUM_BYTES = KG * BM * BN * 4;
    static constexpr int LDS = KG * BUFS * BUF > SUM_BYTES ? KG * BUFS * BUF : SUM_BYTES;
};

// The per-element loop of one output (the arithmetic of the per-element
// kernels), for results the split could not represent.
template <typename W, typename ACT>
__device__ __attribute__((noinline)) float plain_dot(const typename ACT::T* a, W w, size_t arow,
                                                     int col, int K, int N) {
    float acc = 0.0f;
    for (int k = 0; k < K; k++)
        acc = __builtin_fmaf(ACT::value(a[arow + k]), w.at((uint64_t)k * N + col), acc);
    return acc;
}

// Rows [m0, min(m0 + BM, m_end)), columns [n0, min(n0 + BN, N)).
template <typename W, typename ACT, int TM, int WN, int KG>
__device__ __forceinline__ void split_tile(char* lds, const typename ACT::T* __restrict__ a,
                                           const W& w, void* __restrict__ out, int m0, int m_end,
                                           int n0, int K, int N, const Epilogue& ep) {
    using S = Shape<ACT, TM, WN, KG>;
    constexpr int NA = S::NA, BM = S::BM, BN = S::BN, TG = S::TG, TN = S::TN;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave / WN, wn = wave % WN;
    const int gt = tid - g * TG;
    const int lane = tid & 63;
    const int c32 = lane & 31, kg = lane >> 5;
    char* As = lds + g * S::BUFS * S::BUF;

    // K group g's whole stages [st0, st0 + mine); the last group takes the
    // ragged rest of K as one stage more
    const int full = K / KS;
    const int st0 = (int)((int64_t)full * g / KG);
    const int mine = (int)((int64_t)full * (g + 1) / KG) - st0;
    const int most = (full + KG - 1) / KG;   // the longest group's

    const int a_oct = gt & 3, a_row = gt >> 2;
    const typename ACT::T* ap[S::AU];
#pragma unroll
    for (int u = 0; u < S::AU; u++)
        ap[u] = a + (size_t)min(m0 + a_row + u * (TG / 4), m_end - 1) * K + 8 * a_oct;
    // the lane's columns as flat distances from the tile's first; columns past
    // the edge are clamped copies, never stored
    const int cp = TN * (32 * wn + c32);
    const uint32_t c0 = TN == 2 && N % 2 == 0 ? min(cp, N - 2 - n0) : min(cp, N - 1 - n0);
    const uint32_t c1 = min(cp + 1, N - 1 - n0);

    typename ACT::T ra[S::AU][8];
    typename W::Regs rb[2];
    bf16x8 bf[2][3][TN];     // [half stage][term][column]
    uint32_t ta[4][NA];      // a unit of A being split
    float wv[2][2];          // two rows of B being split: [row][column]

    auto load_a = [&](int u, int st) {
        const typename ACT::T* p = ap[u] + st * KS;
        if constexpr (sizeof(typename ACT::T) == 4) {
            const f32x4u x = *reinterpret_cast<const f32x4u*>(p);
            const f32x4u y = *reinterpret_cast<const f32x4u*>(p + 4);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                ra[u][j] = x[j];
                ra[u][4 + j] = y[j];
            }
        } else {
            const u16x8u x = *reinterpret_cast<const u16x8u*>(p);
#pragma unroll
            for (int j = 0; j < 8; j++) ra[u][j] = x[j];
        }
    };
    uint32_t d0 = (uint32_t)(8 * kg) * (uint32_t)N + c0;
    uint32_t d1 = (uint32_t)(8 * kg) * (uint32_t)N + c1;
    uint64_t half_row;   // flat index of the first row that load_b's calls share
    auto load_b = [&](int h, int i, int st) {   // row i of half h of stage st
        if (i == 0) half_row = (uint64_t)(st * KS + 16 * h) * N + n0;
        w.load(rb[h], i, half_row + (uint64_t)((uint32_t)i * (uint32_t)N), d0, d1);
    };
    auto split_a = [&](int u, int p) {   // pair p of unit u
        if constexpr (NA == 1)
            ta[p][0] = (uint32_t)ra[u][2 * p] | ((uint32_t)ra[u][2 * p + 1] << 16);
        else {
            // marked like the weights (Int8W::pair): scaled where they are split
            if constexpr (ACT::kScale != 1.0f)
                asm volatile("" : "+v"(ra[u][2 * p]), "+v"(ra[u][2 * p + 1]));
            split_terms<NA>(ACT::value(ra[u][2 * p]) * ACT::kScale,
                            ACT::value(ra[u][2 * p + 1]) * ACT::kScale, ta[p]);
        }
    };
    auto write_a = [&](int u, int buf) {
        const int row = a_row + u * (TG / 4);
        char* d = As + buf * S::BUF + a_oct * S::OCT + row * 16;
#pragma unroll
        for (int i = 0; i < NA; i++)
            *reinterpret_cast<u32x4*>(d + i * 4 * S::OCT) =
                (u32x4){ta[0][i], ta[1][i], ta[2][i], ta[3][i]};
    };
    auto dequant_b = [&](int h, int p, int st) {   // rows 2p, 2p + 1 of half h
#pragma unroll
        for (int i = 0; i < 2; i++)
            w.pair(rb[h], 2 * p + i,
                   n0 + (int)c0 + (st * KS + 16 * h + 8 * kg + 2 * p + i) * (N & 1), wv[i][0],
                   wv[i][1]);
    };
    auto split_b = [&](int h, int p, int c) {
        uint32_t t[3];
        split_terms<3>(wv[0][c], wv[1][c], t);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            u32x4 v = __builtin_bit_cast(u32x4, bf[h][i][c]);
            v[p] = t[i];
            bf[h][i][c] = __builtin_bit_cast(bf16x8, v);
        }
    };
    auto sync = [&] {
        if constexpr (WN == 1) {
            // the group is one wave: its LDS operations are in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][j][r] = 0.0f;

    // Half h of the stage in `buf`: its products, terms x + y <= 2 with the
    // smallest first, and between them `chunks` pieces of other work.
    constexpr int kSums = NA == 3 ? 6 : NA == 2 ? 5 : 3;   // kept term pairs
    constexpr int kMfma = kSums * TM * TN;
    auto multiply = [&](int buf, int h, auto chunks, auto&& other) {
        constexpr int C = decltype(chunks)::value;
        bf16x8 af[NA][TM];
#pragma unroll
        for (int i = NA - 1; i >= 0; i--)
#pragma unroll
            for (int t = 0; t < TM; t++)
                af[i][t] = *reinterpret_cast<const bf16x8*>(
                    As + buf * S::BUF + (i * 4 + 2 * h + kg) * S::OCT + (t * 32 + c32) * 16);
        int m = 0;
#pragma unroll
        for (int sum = 2; sum >= 0; sum--)
#pragma unroll
            for (int x = NA - 1; x >= 0; x--) {
                if (sum - x < 0 || sum - x > 2) continue;
#pragma unroll
                for (int t = 0; t < TM; t++)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            af[x][t], bf[h][sum - x][j], acc[t][j], 0, 0, 0);
                        if (C > 0) {
                            const int from = C * m / kMfma, to = C * (m + 1) / kMfma;
#pragma unroll
                            for (int c = from; c < to; c++) other(c);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        m++;
                    }
            }
    };
    // The pieces: splitting half `h` of B (stage `of`) and loading the rows of
    // the stage after it into the registers that frees: 12 + 8.
    auto b_piece = [&](int c, int h, int of, int load) {
        if (c < 12) {
            const int p = c / 3;
            if (c % 3 == 0) dequant_b(h, p, of);
            if (c % 3 == 1) split_b(h, p, 0);
            if (TN == 2 && c % 3 == 2) split_b(h, p, 1);
        } else {
            load_b(h, c - 12, load);
        }
    };
    // and splitting the units [u0, u1) of A into `buf` and loading theirs: 6 a unit
    auto a_piece = [&](int c, int u0, int buf, int load) {
        const int u = u0 + c / 6, p = c % 6;
        if (p < 4) split_a(u, p);
        if (p == 4) write_a(u, buf);
        if (p == 5) load_a(u, load);
    };
    const int last = st0 + mine - 1;
    using C0 = std::integral_constant<int, 0>;
    // units staged beside the first half; with one buffer all wait for the
    // second half's reads
    constexpr int U0 = S::BUFS == 1 ? 0 : (S::AU + 1) / 2;
    using CA = std::integral_constant<int, 20 + 6 * U0>;
    using CB = std::integral_constant<int, 20 + 6 * (S::AU - U0)>;
    if (mine > 0) {
#pragma unroll
        for (int u = 0; u < S::AU; u++) load_a(u, st0);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int i = 0; i < 8; i++) load_b(h, i, st0);
#pragma unroll
        for (int u = 0; u < S::AU; u++) {
#pragma unroll
            for (int p = 0; p < 4; p++) split_a(u, p);
            write_a(u, 0);
            load_a(u, min(st0 + 1, last));
        }
#pragma unroll
        for (int c = 0; c < 20; c++) b_piece(c, 0, st0, min(st0 + 1, last));
    }
    sync();
    for (int i = 0; i < most; i++) {
        if (i < mine) {
            const int st = st0 + i, n1 = min(st + 1, last), n2 = min(st + 2, last);
            // marked once a stage: widened to 64 bits outside the loop the
            // distances would cost an add at every load
            asm volatile("" : "+v"(d0), "+v"(d1));
            const int buf = S::BUFS == 2 ? i & 1 : 0, nbuf = S::BUFS == 2 ? buf ^ 1 : 0;
            multiply(buf, 0, CA{}, [&](int c) {
                if (c < 20) b_piece(c, 1, st, n1);
                else a_piece(c - 20, 0, nbuf, n2);
            });
            multiply(buf, 1, CB{}, [&](int c) {
                if (c < 20) b_piece(c, 0, n1, n2);
                else a_piece(c - 20, U0, nbuf, n2);
            });
        }
        sync();
    }
    // the ragged rest of K: activations past K are zero, weight rows clamped
    if (K % KS != 0) {
        const int k0 = full * KS;
        if (g == KG - 1) {
#pragma unroll
            for (int u = 0; u < S::AU; u++) {
#pragma unroll
                for (int j = 0; j < 8; j++)
                    ra[u][j] = k0 + 8 * a_oct + j < K ? ap[u][k0 + j] : (typename ACT::T)0;
#pragma unroll
                for (int p = 0; p < 4; p++) split_a(u, p);
                write_a(u, 0);
            }
        }
        sync();
        if (g == KG - 1) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const uint32_t r = (uint32_t)min(16 * h + 8 * kg + i, K - 1 - k0) * (uint32_t)N;
                    w.load(rb[h], i, (uint64_t)k0 * N + n0, r + c0, r + c1);
                }
#pragma unroll
                for (int c = 0; c < 12; c++) b_piece(c, h, full, 0);
                multiply(0, h, C0{}, [](int) {});
            }
        }
    }

    // out, through LDS in K group order
    constexpr float kBack = ACT::kUnscale * W::kUnscale;
    float odd = 0.0f;   // becomes NaN when a sum is not finite
    const int rows = min(BM, m_end - m0), cols = min(BN, N - n0);
    __syncthreads();   // every group has left its last stage
    float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int rl = t * 32 + 8 * (r >> 2) + 4 * kg + (r & 3);
            float* at = sums + (g * BM + rl) * BN + cp;
            if constexpr (TN == 2)
                *reinterpret_cast<f32x2*>(at) = (f32x2){acc[t][0][r], acc[t][TN - 1][r]};
            else
                *at = acc[t][0][r];
        }
    __syncthreads();
#pragma unroll 4
    for (int i = tid; i < BM * BN; i += S::NT) {
        const int rl = i / BN, cl = i % BN;
        float v = sums[i];
#pragma unroll
        for (int q = 1; q < KG; q++) v += sums[q * BM * BN + i];
        v *= kBack;
        if (rl < rows && cl < cols) {
            odd = __builtin_fmaf(v, 0.0f, odd);
            store_out(out, (size_t)(m0 + rl) * N + n0 + cl, n0 + cl, v, ep);
        }
    }
    if (__syncthreads_or(odd != 0.0f)) {
        for (int i = tid; i < BM * BN; i += S::NT) {
            const int rl = i / BN, cl = i % BN;
            if (rl >= rows || cl >= cols) continue;
            const size_t o = (size_t)(m0 + rl) * N + n0 + cl;
            const bool bad = ep.bf16 ? (static_cast<const uint16_t*>(out)[o] & 0x7f80) == 0x7f80
                                     : (__float_as_uint(static_cast<const float*>(out)[o]) &
                                        0x7f800000u) == 0x7f800000u;
            if (bad)
                store_out(out, o, n0 + cl,
                          plain_dot<W, ACT>(a, w, (size_t)(m0 + rl) * K, n0 + cl, K, N), ep);
        }
    }
}

template <typename W, typename ACT, int TM, int WN, int KG>
__global__ __launch_bounds__((Shape<ACT, TM, WN, KG>::NT), (KG == 16 ? 4 : 2)) void split_product_kernel(
    const typename ACT::T* __restrict__ a, W w, void* __restrict__ out, int M, int K, int N,
    Epilogue ep) {
    using S = Shape<ACT, TM, WN, KG>;
    __shared__ __attribute__((aligned(16))) char lds[S::LDS];
    const int tiles_m = (M + S::BM - 1) / S::BM;
    const int tiles = tiles_m * ((N + S::BN - 1) / S::BN);
    // The dispatcher deals workgroup b to XCD b % 8: each XCD takes an eighth
    // of the column tiles with all their row tiles, so a weight is fetched
    // into one L2.
    const int per_xcd = (tiles + 7) / 8;
    const int b = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || b >= tiles) return;
    split_tile<W, ACT, TM, WN, KG>(lds, a, w, out, (b % tiles_m) * S::BM, M,
                                   (b / tiles_m) * S::BN, K, N, ep);
}

// The grouped products (x [T, K] against `w`'s experts, off [E + 1]): a tile of
// one expert's rows, the tiles listed column by column so the blocks of an
// expert meet its weights in one L2.  Offsets in order put expert e's rows at
// [off[e], min(off[e + 1], T)); offsets that are not (their sum wrapped) give
// every workgroup a share of the outputs, one lane each, by the reference's
// e(t) = #{r : off[r + 1] <= t} (grouped.go:48-66).  The matvec form writes 0
// past the last segment; the matmul form writes only rows that
// [off[e], min(off[e + 1], T)) covers.
template <typename W, typename ACT, int TM, int WN, int KG>
__global__ __launch_bounds__((Shape<ACT, TM, WN, KG>::NT), (KG == 16 ? 4 : 2)) void split_grouped_kernel(
    const typename ACT::T* __restrict__ x, W w, const uint32_t* __restrict__ off,
    float* __restrict__ out, int E, int T, int K, int N, bool matvec) {
    using S = Shape<ACT, TM, WN, KG>;
    __shared__ __attribute__((aligned(16))) char lds[S::LDS];
    const size_t per = (size_t)K * N;
    const uint64_t lane0 = (uint64_t)blockIdx.x * S::NT + threadIdx.x;
    const uint64_t lanes = (uint64_t)gridDim.x * S::NT;
    auto rows_of = [&](int e) {
        const uint32_t first = off[e], last = min(off[e + 1], (uint32_t)T);
        return last > first ? (int)(last - first) : 0;
    };
    bool in_order = off[0] == 0;
    int blocks = 0;
    for (int e = 0; e < E; e++) {
        in_order = in_order && off[e + 1] >= off[e];
        blocks += (rows_of(e) + S::BM - 1) / S::BM;
    }
    if (!in_order) {
        for (uint64_t i = lane0; i < (uint64_t)T * N; i += lanes) {
            const uint32_t t = (uint32_t)(i / N);
            const int col = (int)(i % N);
            int e = 0;
            for (int r = 0; r < E; r++) e += off[r + 1] <= t ? 1 : 0;
            if (e >= E) {
                if (matvec) out[i] = 0.0f;
            } else if (matvec || (t >= off[e] && t < min(off[e + 1], (uint32_t)T))) {
                out[i] = plain_dot<W, ACT>(x, w.expert(e, per), (size_t)t * K, col, K, N);
            }
        }
        return;
    }
    if (matvec)
        for (uint64_t i = (uint64_t)min(off[E], (uint32_t)T) * N + lane0; i < (uint64_t)T * N;
             i += lanes)
            out[i] = 0.0f;
    const int tiles = blocks * ((N + S::BN - 1) / S::BN);
    const int per_xcd = (tiles + 7) / 8;
    const int b = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || b >= tiles) return;
    int block = b % blocks, e = 0;
    for (; e < E; e++) {
        const int n = (rows_of(e) + S::BM - 1) / S::BM;
        if (block < n) break;
        block -= n;
    }
    split_tile<W, ACT, TM, WN, KG>(lds, x, w.expert(e, per), out, (int)off[e] + block * S::BM,
                                   (int)min(off[e + 1], (uint32_t)T), (b / blocks) * S::BN, K, N,
                                   Epilogue{});
}

// Which tile: the tiles in rounds of the chip, times a K group's stages, times
// what a stage costs.  The stage costs are those of int8 weights and f32 rows
// (us, K = 4096, every CU busy): a wide tile splits its activations for more
// columns, a narrow one fills the chip with fewer rows and columns.  The other
// sources cost more or less a stage but keep the order.  Tiles of 64 x 256, 64 x
// 128, 64 x 64, 32 x 64 and 32 x 32 (us), the chosen one marked:
//   int8, f32 rows, K = N = 4096: 512 rows 137, 96*, 116, 154, 229; 128 rows 135,
//     77, 48, 38*, 56; 32 rows 134, 76, 47, 35, 27*; 33 x 4864 x 352 157, 88, 54,
//     40, 32*
//   int8, f16 rows, K = N = 4096: 512 rows 118, 79*, 93, 127, 191
//   int4, f32 rows, 4100 x 4004: 512 rows 170, 111*, 134, 186, 290; 256 rows 169,
//     98, 68*, 93, 142; 100 rows 169, 98, 60, 47*, 69; 32 rows 167, 97, 59, 46, 35*
//   int4, bf16 rows, 4100 x 4004: 512 rows 135, 75*, 89, 155, 225; 100 rows 134,
//     72, 43, 40*, 56; 32 rows 132, 70, 42, 40, 29*
//   8 f32 experts of 2048 x 4096: 256 rows 78, 73*, 82, 89, 115; 1024 rows 166,
//     159*, 184, 215, 308
// Few rows of many experts are where it misses, its row blocks being an estimate
// there: 60 rows of the same experts 76, 70, 79, 67, 79*; 16 rows of 4 of 1000 x
// 3000 43, 30, 24, 20, 25*.
enum class SplitTile { k64x256, k64x128, k64x64, k32x64, k32x32 };

SplitTile choose_tile(const Device* d, long long rows_blocks64, long long rows_blocks32, int K,
                      int N) {
    struct {
        SplitTile t;
        long long blocks;
        int cols, groups;
        double us;
    } const kTiles[] = {{SplitTile::k64x256, rows_blocks64, 256, 2, 2.6},
                        {SplitTile::k64x128, rows_blocks64, 128, 4, 2.85},
                        {SplitTile::k64x64, rows_blocks64, 64, 8, 3.5},
                        {SplitTile::k32x64, rows_blocks32, 64, 8, 2.4},
                        {SplitTile::k32x32, rows_blocks32, 32, 16, 3.1}};
    SplitTile best = SplitTile::k32x64;
    double best_us = 1e30;
    for (const auto& k : kTiles) {
        const long long tiles = k.blocks * ((N + k.cols - 1) / k.cols);
        const long long rounds = (tiles + d->cu_count - 1) / d->cu_count;
        const double us = (double)rounds * (((K + KS - 1) / KS + k.groups - 1) / k.groups) * k.us;
        if (us < best_us) {
            best_us = us;
            best = k.t;
        }
    }
    return best;
}

template <typename W, typename ACT, int TM, int WN, int KG>
hipError_t launch_split_tile(hipStream_t st, const typename ACT::T* a, W w, void* out, int M, int K,
                             int N, Epilogue ep) {
    using S = Shape<ACT, TM, WN, KG>;
    const long long tiles =
        (long long)((M + S::BM - 1) / S::BM) * ((N + S::BN - 1) / S::BN);
    ACCEL_LAUNCH(tname("split_product_kernel", W::name().c_str(), ACT::kName, TM, WN, KG) +
                     grid_note(tiles, 1),
                 (split_product_kernel<W, ACT, TM, WN, KG>),
                 dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(S::NT), 0, st, a, w, out, M, K, N, ep);
    return launch_status();
}

// Odd int4 widths load six words a row of a unit: with 64 rows' accumulators
// beside them a wave would spill, so they take the 32-row tile.
template <typename W> constexpr bool kNarrowOnly = false;
template <> constexpr bool kNarrowOnly<Int4W<kOdd>> = true;

template <typename W, typename ACT>
hipError_t launch_split(const Device* d, hipStream_t st, const typename ACT::T* a, W w, void* out,
                        int M, int K, int N, Epilogue ep) {
    const SplitTile tile = choose_tile(d, (M + 63) / 64, (M + 31) / 32, K, N);
    if constexpr (kNarrowOnly<W>)
        return tile == SplitTile::k32x32
                   ? launch_split_tile<typename W::One, ACT, 1, 1, 16>(st, a, w.one(), out, M, K, N, ep)
                   : launch_split_tile<W, ACT, 1, 1, 8>(st, a, w, out, M, K, N, ep);
    else switch (tile) {
        case SplitTile::k64x256: return launch_split_tile<W, ACT, 2, 4, 2>(st, a, w, out, M, K, N, ep);
        case SplitTile::k64x128: return launch_split_tile<W, ACT, 2, 2, 4>(st, a, w, out, M, K, N, ep);
        case SplitTile::k64x64: return launch_split_tile<W, ACT, 2, 1, 8>(st, a, w, out, M, K, N, ep);
        case SplitTile::k32x64: return launch_split_tile<W, ACT, 1, 1, 8>(st, a, w, out, M, K, N, ep);
        default:
            return launch_split_tile<typename W::One, ACT, 1, 1, 16>(st, a, w.one(), out, M, K, N, ep);
    }
}

// The most row blocks of BM rows that T rows of E experts make: each expert
// that has rows can end in a partial one.
long long most_blocks(int T, int E, int bm) { return (T + bm - 1) / bm + std::min(T, E); }

template <typename W, typename ACT, int TM, int WN, int KG>
hipError_t launch_grouped_tile(hipStream_t st, const typename ACT::T* x, W w, const uint32_t* off,
                               float* out, int E, int T, int K, int N, bool matvec) {
    using S = Shape<ACT, TM, WN, KG>;
    const long long wgs = most_blocks(T, E, S::BM) * ((N + S::BN - 1) / S::BN);
    ACCEL_LAUNCH(tname("split_grouped_kernel", W::name().c_str(), ACT::kName, TM, WN, KG),
                 (split_grouped_kernel<W, ACT, TM, WN, KG>),
                 dim3((unsigned)((wgs + 7) / 8 * 8)), dim3(S::NT), 0, st, x, w, off, out, E, T, K,
                 N, matvec);
    return launch_status();
}

// Where the rows are is known on the device only: the tile is chosen for rows
// spread over the experts, half a block left over in each.
template <typename W, typename ACT>
hipError_t launch_grouped(const Device* d, hipStream_t st, const typename ACT::T* x, W w,
                          const uint32_t* off, float* out, int E, int T, int K, int N,
                          bool matvec) {
    const int used = std::min(E, T);
    const SplitTile tile = choose_tile(d, T / 64 + (used + 1) / 2, T / 32 + (used + 1) / 2, K, N);
    if constexpr (kNarrowOnly<W>)
        return tile == SplitTile::k32x32
                   ? launch_grouped_tile<typename W::One, ACT, 1, 1, 16>(st, x, w.one(), off, out, E, T,
                                                                         K, N, matvec)
                   : launch_grouped_tile<W, ACT, 1, 1, 8>(st, x, w, off, out, E, T, K, N, matvec);
    else switch (tile) {
        case SplitTile::k64x256:
            return launch_grouped_tile<W, ACT, 2, 4, 2>(st, x, w, off, out, E, T, K, N, matvec);
        case SplitTile::k64x128:
            return launch_grouped_tile<W, ACT, 2, 2, 4>(st, x, w, off, out, E, T, K, N, matvec);
        case SplitTile::k64x64:
            return launch_grouped_tile<W, ACT, 2, 1, 8>(st, x, w, off, out, E, T, K, N, matvec);
        case SplitTile::k32x64:
            return launch_grouped_tile<W, ACT, 1, 1, 8>(st, x, w, off, out, E, T, K, N, matvec);
        default:
            return launch_grouped_tile<typename W::One, ACT, 1, 1, 16>(st, x, w.one(), off, out, E, T,
                                                                       K, N, matvec);
    }
}

template <typename ACT>
hipError_t launch_split_int8_act(const Device* d, hipStream_t st, const typename ACT::T* a,
                                 const int8_t* q, const uint16_t* s, float* out, int M, int K,
                                 int N) {
    if (N % 32 == 0)
        return launch_split<Int8W<kRows>, ACT>(d, st, a, {q, s}, out, M, K, N, Epilogue{});
    if (N % 2 == 0)
        return launch_split<Int8W<kEven>, ACT>(d, st, a, {q, s}, out, M, K, N, Epilogue{});
    return launch_split<Int8W<kOdd>, ACT>(d, st, a, {q, s}, out, M, K, N, Epilogue{});
}

}  // namespace

bool split_product_supported(int M, int K, int N) {
    // a lane's 32-bit distances span sixteen rows; the grid's 512-lane
    // or 1024-lane workgroups stay below 2^32 lanes at the smallest tile
    return N <= (1 << 24) &&
           (long long)((M + 31) / 32) * ((N + 31) / 32) <= (1ll << 21) && K < (1 << 30);
}

bool split_grouped_supported(int E, int T, int K, int N) {
    return N <= (1 << 24) && K < (1 << 30) &&
           most_blocks(T, E, 32) * ((N + 31) / 32) <= (1ll << 21);
}

hipError_t launch_split_grouped_f32(const Device* d, hipStream_t st, const float* x, const float* w,
                                    const uint32_t* off, float* out, int E, int T, int K, int N,
                                    bool matvec) {
    if (N % 2 == 0)
        return launch_grouped<F32W<kEven>, ActF32>(d, st, x, {w}, off, out, E, T, K, N, matvec);
    return launch_grouped<F32W<kOdd>, ActF32>(d, st, x, {w}, off, out, E, T, K, N, matvec);
}

hipError_t launch_split_int4(const Device* d, hipStream_t st, const void* a, bool bf16, Int4Planes w,
                             void* out, int M, int K, int N, Epilogue ep) {
    const uint8_t* c = reinterpret_cast<const uint8_t*>(w.codes);
    auto run = [&](auto act) {
        using ACT = decltype(act);
        const auto* x = static_cast<const typename ACT::T*>(a);
        if (N % 128 == 0)
            return launch_split<Int4W<kRows>, ACT>(d, st, x, {c, w.scales, w.zeros}, out, M, K, N, ep);
        if (N % 2 == 0)
            return launch_split<Int4W<kEven>, ACT>(d, st, x, {c, w.scales, w.zeros}, out, M, K, N, ep);
        return launch_split<Int4W<kOdd>, ACT>(d, st, x, {c, w.scales, w.zeros}, out, M, K, N, ep);
    };
    if (!bf16) return run(ActF32{});
    ep.bf16 = true;
    return run(ActBf16{});
}

hipError_t launch_split_grouped_int4(const Device* d, hipStream_t st, const float* x, Int4Planes w,
                                     const uint32_t* off, float* out, int E, int T, int K, int N,
                                     bool matvec) {
    const uint8_t* c = reinterpret_cast<const uint8_t*>(w.codes);
    if (N % 128 == 0)
        return launch_grouped<Int4W<kRows>, ActF32>(d, st, x, {c, w.scales, w.zeros}, off, out, E, T,
                                                    K, N, matvec);
    if (N % 2 == 0)
        return launch_grouped<Int4W<kEven>, ActF32>(d, st, x, {c, w.scales, w.zeros}, off, out, E, T,
                                                    K, N, matvec);
    return launch_grouped<Int4W<kOdd>, ActF32>(d, st, x, {c, w.scales, w.zeros}, off, out, E, T, K, N,
                                               matvec);
}

hipError_t launch_split_int8(const Device* d, hipStream_t st, const void* a, bool f16_act,
                             const int8_t* quants, const uint16_t* scales, float* out, int M,
                             int K, int N) {
    if (f16_act)
        return launch_split_int8_act<ActF16>(d, st, static_cast<const uint16_t*>(a), quants, scales,
                                             out, M, K, N);
    return launch_split_int8_act<ActF32>(d, st, static_cast<const float*>(a), quants, scales, out,
                                         M, K, N);
}

}  // namespace accel
