// Int4MatVec and Int4MatMul of up to four rows on matrices whose width is no
// multiple of a quantisation group, so groups and code words run across rows.
//
// Bound: one workgroup's instruction issue (about 60 a lane's word, 3 cycles
// each).  A strip walks all of K, so its time hardly depends on how many there
// are: 248 columns of 4096 rows take 38.5 us with 17 of them and 38.9 with 154,
// and the CUs past the strips' number are idle (126 of 256 at 32004 columns).
// Narrow strips over the whole chip meet L2 as well: a row's scale and zero are a
// 128-byte line each for two bytes.
//
// Row k's columns begin at nibble k N, so what a code word means for a column
// depends on k N mod 8 only.  A workgroup of 1024 lanes owns a strip of columns
// over all of K; lane (row phase p, l) takes rows p, p + RP, ... with RP a
// multiple of eight, so its words keep one alignment for the whole of K: word
// l of the strip, eight fixed columns and, since a word never straddles a
// group, one scale and zero per row.  No shifts, no second word; a zero scale is
// one selection a row.
// The windows of the phases differ by up to seven columns; a strip is eight
// columns narrower than its LPR words so that every phase covers all of it,
// and the sums meet by column in LDS, waves first (the phases of one lane are
// aligned alike in every wave), then the eight alignments, in fixed order.
// K is never split across workgroups: no workspace, no hand-off.
//
// A weight is (q - z) * s as in the per-element kernels, q - z in f32 and the
// scale folded into the activation; a zero scale reads as z.  The fold is with
// 2^24 s, which is at least 1: an activation times a small scale would go
// subnormal where its products do not (relative errors of 2e-4 to 2e-3 near
// 2^-124 with scales of 2^-14).  4096 x 32004 38.7 us without it, 38.9 with.  A
// sum that comes out infinite or NaN is computed again by the per-element loop.
//
// 4096 x 32004 (one row): 1305 us one lane per element, 39 us here (1.7 TB/s).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.hpp"
#include "splitk.hpp"

namespace accel {
namespace {

constexpr int kRagThreads = 1024;
constexpr int kRagBatch = 4;   // rows of a load batch, two batches out at a time
constexpr float kRagUp = 0x1p24f, kRagDown = 0x1p-24f;   // of the scales folded in

__device__ __forceinline__ float rag_act(float v) { return v; }
__device__ __forceinline__ float rag_act(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }

// The per-element kernels' loop for one output.
template <typename XT>
__device__ __attribute__((noinline)) float ragged_dot(const XT* x, const uint32_t* codes,
                                                      const uint16_t* scales,
                                                      const uint16_t* zeros, int col, int K,
                                                      int N) {
    float acc = 0.0f;
    for (int k = 0; k < K; k++) {
        const uint64_t f = (uint64_t)k * N + col;
        const uint32_t code = (codes[f >> 3] >> (4 * (f & 7))) & 15u;
        const float s = half_bits_to_float(scales[f >> 7]);
        const float z = half_bits_to_float(zeros[f >> 7]);
        acc = __builtin_fmaf(rag_act(x[k]), s == 0.0f ? z : ((float)code - z) * s, acc);
    }
    return acc;
}

// XT: f32 or bf16 bits.  M: rows computed (clamped copies past `rows`).
template <typename XT, int M, int LPR>
__global__ __launch_bounds__(kRagThreads) void ragged_rows_kernel(
    const XT* __restrict__ a, const uint32_t* __restrict__ codes,
    const uint16_t* __restrict__ scales, const uint16_t* __restrict__ zeros,
    void* __restrict__ out, int rows, int K, int N, Epilogue ep) {
    constexpr int STRIP = 8 * LPR - 8;
    constexpr int RP = kRagThreads / LPR;      // row phases
    constexpr int PW = 64 / LPR;               // of them in a wave
    constexpr int NW = kRagThreads / 64;
    static_assert(RP % 8 == 0, "a lane's rows share an alignment");
    // Where a wave holds fewer than eight phases, alignments repeat every
    // 8 / PW waves; each (alignment, window) column is summed over them.
    constexpr int WR = 8 / PW;                 // waves an alignment set spans
    __shared__ float red[NW][64 * 8];
    __shared__ float fin[8][8 * LPR + 8];

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int l = tid % LPR, p = tid / LPR;
    // neighbouring strips on one XCD: they share lines and groups
    const int strips = (N + STRIP - 1) / STRIP;
    const int per_xcd = (strips + 7) / 8;
    const int strip = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || strip >= strips) return;
    const int c0 = strip * STRIP;
    // first column of phase p's windows relative to c0, plus 8: 1 .. 8
    auto shift_of = [&](int phase) { return 8 - (int)(((uint32_t)phase * (uint32_t)(N & 7)) & 7u); };
    const int64_t f0 = (int64_t)p * N + c0 + shift_of(p) - 8 + 8 * l;
    const uint32_t w0 = f0 > 0 ? (uint32_t)(f0 >> 3) : 0u;
    // A row step is RP N nibbles, a batch of four a whole number of groups: the
    // lane's distances from a batch's (uniform) bases never change.
    const uint64_t step = (uint64_t)RP * (uint64_t)N >> 3;          // words
    const uint64_t step4 = (uint64_t)RP * (uint64_t)N >> 5;         // groups, four steps
    static_assert(RP % 32 == 0 && kRagBatch == 4, "four steps are whole groups");
    uint32_t dw = w0, dx = (uint32_t)p, dg[4];
#pragma unroll
    for (int u = 0; u < 4; u++) dg[u] = (uint32_t)((w0 + u * step) >> 4);

    float acc[M][8], bias[M];
#pragma unroll
    for (int m = 0; m < M; m++) {
        bias[m] = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) acc[m][j] = 0.0f;
    }
    struct Batch {
        uint32_t q[kRagBatch];
        uint16_t s[kRagBatch], z[kRagBatch];
        XT x[kRagBatch][M];
    };
    const XT* xp[M];
#pragma unroll
    for (int m = 0; m < M; m++) xp[m] = a + (size_t)min(m, rows - 1) * K;
    // The loads of the steps from i0.  Cached: neighbouring strips share the
    // 128-byte lines (non-temporal loads fetched them again: 81 against 60 us).
    auto load = [&](Batch& t, int i0) {
        const uint32_t* cp = codes + i0 * step;
        const uint16_t* sp = scales + (i0 >> 2) * step4;
        const uint16_t* zp = zeros + (i0 >> 2) * step4;
#pragma unroll
        for (int u = 0; u < kRagBatch; u++) {
            t.q[u] = (cp + u * step)[dw];
            t.s[u] = sp[dg[u]];
            t.z[u] = zp[dg[u]];
#pragma unroll
            for (int m = 0; m < M; m++) t.x[u][m] = (xp[m] + (i0 + u) * RP)[dx];
        }
    };
    // The same for the last steps: rows past the end count nothing, and row
    // K - 1's windows may run past the planes.
    auto load_end = [&](Batch& t, int i0) {
        const uint64_t last_word = ((uint64_t)K * (uint64_t)N + 7) / 8 - 1;
#pragma unroll
        for (int u = 0; u < kRagBatch; u++) {
            const int k = p + (i0 + u) * RP;
            const uint64_t w = k < K ? min(w0 + (i0 + u) * step, last_word) : 0;
            t.q[u] = codes[w];
            t.s[u] = k < K ? scales[w >> 4] : (uint16_t)0;
            t.z[u] = k < K ? zeros[w >> 4] : (uint16_t)0;
#pragma unroll
            for (int m = 0; m < M; m++) t.x[u][m] = k < K ? xp[m][k] : (XT)0;
        }
    };
    auto add = [&](const Batch& t) {
#pragma unroll
        for (int u = 0; u < kRagBatch; u++) {
            const float s = half_bits_to_float(t.s[u]) * kRagUp;
            const float z = half_bits_to_float(t.z[u]);
            // a nibble as an e4m3 byte is q 2^-9; the conversion's scale makes
            // it q, exactly
            const uint32_t even = t.q[u] & 0x0F0F0F0Fu, odd = (t.q[u] >> 4) & 0x0F0F0F0Fu;
            const f32x2 e01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(even, 512.0f, false);
            const f32x2 e23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(even, 512.0f, true);
            const f32x2 o01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(odd, 512.0f, false);
            const f32x2 o23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(odd, 512.0f, true);
            float x[M], xs[M];
#pragma unroll
            for (int m = 0; m < M; m++) {
                x[m] = rag_act(t.x[u][m]);
                xs[m] = x[m] * s;
            }
            // a zero scale's weights are z, and an infinite activation must not
            // meet the zero
            if (__builtin_amdgcn_ballot_w64(s == 0.0f)) {
#pragma unroll
                for (int m = 0; m < M; m++) {
                    const float xz = __builtin_fmaf(x[m], z, bias[m]);
                    bias[m] = s == 0.0f ? xz : bias[m];
                    xs[m] = s == 0.0f ? 0.0f : xs[m];
                }
            }
            const float d[8] = {e01.x - z, o01.x - z, e01.y - z, o01.y - z,
                                e23.x - z, o23.x - z, e23.y - z, o23.y - z};
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int j = 0; j < 8; j++) acc[m][j] = __builtin_fmaf(xs[m], d[j], acc[m][j]);
        }
    };
    // Batches of rows below K - 1, the next one's loads out while one is added
    // (without a branch between, or the waits drain them); then the rest.
    const int whole = (K - 1) / (RP * kRagBatch);
    if (whole > 0) {
        Batch b0, b1;
        load(b0, 0);
        for (int i = 0; i < whole; i += 2) {
            // marked here: widened to 64 bits outside the loop the distances
            // would cost an add at every load
            asm volatile(""
                         : "+v"(dw), "+v"(dx), "+v"(dg[0]), "+v"(dg[1]), "+v"(dg[2]), "+v"(dg[3]));
            load(b1, min(i + 1, whole - 1) * kRagBatch);
            add(b0);
            if (i + 1 >= whole) break;
            load(b0, min(i + 2, whole - 1) * kRagBatch);
            add(b1);
        }
    }
    for (int i0 = whole * kRagBatch; i0 * RP < K; i0 += kRagBatch) {
        Batch b;
        load_end(b, i0);
        add(b);
    }

#pragma unroll
    for (int m = 0; m < M; m++) {
        if (m >= rows) break;
        if (m) __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; j++)
            red[wave][lane * 8 + j] = __builtin_fmaf(acc[m][j], kRagDown, bias[m]);
        __syncthreads();
        // (set of WR waves, lane, j): the waves of the same place in their set
        for (int i = tid; i < WR * 512; i += kRagThreads) {
            const int first = i >> 9, at = i & 511;
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; w += WR) v += red[w + first][at];
            const int phase = first * PW + (at >> 3) / LPR;   // its alignment's first phase
            const int col = 8 * ((at >> 3) % LPR) + (at & 7) + shift_of(phase);   // + 8
            fin[phase][col] = v;
        }
        __syncthreads();
        const int cols = min(STRIP, N - c0);
        for (int c = tid; c < cols; c += kRagThreads) {
            float v = 0.0f;
#pragma unroll
            for (int ph = 0; ph < 8; ph++) v += fin[ph][c + 8];
            // an activation times its scale may overflow where its products
            // with the weights do not
            if ((__float_as_uint(v) & 0x7f800000u) == 0x7f800000u)
                v = ragged_dot(xp[m], codes, scales, zeros, c0 + c, K, N);
            store_out(out, (size_t)m * N + c0 + c, c0 + c, v, ep);
        }
    }
}

template <typename XT, int M, int LPR>
void launch_ragged(hipStream_t st, const XT* a, Int4Planes w, void* out, int rows, int K, int N,
                   Epilogue ep) {
    constexpr int STRIP = 8 * LPR - 8;
    const int strips = (N + STRIP - 1) / STRIP;
    ACCEL_LAUNCH(tname("ragged_rows_kernel", type_name<XT>(), M, LPR) + grid_note(strips, 1),
                 (ragged_rows_kernel<XT, M, LPR>), dim3((strips + 7) / 8 * 8), dim3(kRagThreads),
                 0, st, a, w.codes, w.scales, w.zeros, out, rows, K, N, ep);
}

// The strip: narrow strips end sooner (fewer row steps a lane), wide ones share
// their rows' scale and zero lines among more columns; the narrowest whose
// strips are one round of the chip, else the widest.  One row, 56 / 120 / 248
// columns (us): 4096 x 4004 15.6 / 21.3 / 38.5, 4096 x 16001 33.3 / 23.4 / 39.0,
// 4096 x 30001 49.0 / 25.0 / 38.8, 4096 x 32004 46.2 / 41.2 / 38.9.
template <typename XT, int M>
void launch_ragged_strip(const Device* d, hipStream_t st, const XT* a, Int4Planes w, void* out,
                         int rows, int K, int N, Epilogue ep) {
    if (N <= 56 * (long long)d->cu_count)
        launch_ragged<XT, M, 8>(st, a, w, out, rows, K, N, ep);
    else if (N <= 120 * (long long)d->cu_count)
        launch_ragged<XT, M, 16>(st, a, w, out, rows, K, N, ep);
    else
        launch_ragged<XT, M, 32>(st, a, w, out, rows, K, N, ep);
}

template <typename XT>
hipError_t launch_ragged_any(const Device* d, hipStream_t st, const XT* a, Int4Planes w, void* out,
                             int M, int K, int N, Epilogue ep) {
    if (M == 1)
        launch_ragged_strip<XT, 1>(d, st, a, w, out, M, K, N, ep);
    else if (M == 2)
        launch_ragged_strip<XT, 2>(d, st, a, w, out, M, K, N, ep);
    else
        launch_ragged_strip<XT, 4>(d, st, a, w, out, M, K, N, ep);
    return launch_status();
}

}  // namespace

bool int4_ragged_shape(const void* a, const void* codes, int K, int N) {
    return K >= (N % 128 ? 32 : 128) && N >= 64 &&
           ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(codes)) & 15) == 0;
}

bool int4_ragged_rows_supported(const void* a, const void* codes, int M, int K, int N) {
    // a lane's byte distances, over 64 rows, are 32-bit
    return M >= 1 && M <= 4 && N % 128 != 0 && int4_ragged_shape(a, codes, K, N) &&
           N < (1 << 26) && K < (1 << 30);
}

hipError_t launch_int4_ragged_rows(const Device* d, hipStream_t st, const void* a, bool bf16, Int4Planes w,
                                   void* out, int M, int K, int N, Epilogue ep) {
    if (bf16) {
        ep.bf16 = true;
        return launch_ragged_any(d, st, static_cast<const uint16_t*>(a), w, out, M, K, N, ep);
    }
    return launch_ragged_any(d, st, static_cast<const float*>(a), w, out, M, K, N, ep);
}

}  // namespace accel
