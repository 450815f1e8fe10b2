// Int4MatVec and Int4MatMul of up to four rows on matrices whose width is no
// multiple of a quantisation group, so groups and code words run across rows.
//
// Bound: HBM (the codes), then the VALU: about four instructions a weight.
//
// Row k's columns begin at nibble k N, so what a code word means for a column
// depends on k N mod 8 only.  A workgroup of 512 lanes owns a strip of columns
// over all of K; lane (row phase p, l) takes rows p, p + RP, ... with RP a
// multiple of eight, so its words keep one alignment for the whole of K: word
// l of the strip, eight fixed columns and, since a word never straddles a
// group, one scale and zero per row.  No shifts, no selections, no second word.
// The windows of the phases differ by up to seven columns; a strip is eight
// columns narrower than its LPR words so that every phase covers all of it,
// and the sums meet by column in LDS, waves first (the phases of one lane are
// aligned alike in every wave), then the eight alignments, in fixed order.
// K is never split across workgroups: no workspace, no hand-off.
//
// A weight is (q - z) * s as in the per-element kernels, q - z in f32 and the
// scale folded into the activation; a zero scale reads as z.
//
// 4096 x 32004 (one row): 1307 us one lane per element, 81 us here.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.hpp"
#include "splitk.hpp"

namespace accel {
namespace {

constexpr int kRagThreads = 512;
constexpr int kRagBatch = 8;   // rows a lane has in flight

__device__ __forceinline__ float rag_act(float v) { return v; }
__device__ __forceinline__ float rag_act(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }

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
    const uint32_t step = (uint32_t)((uint64_t)RP * (uint64_t)N >> 3);   // words a row step
    const uint32_t last_word = (uint32_t)(((uint64_t)K * (uint64_t)N + 7) / 8 - 1);

    float acc[M][8], bias[M];
#pragma unroll
    for (int m = 0; m < M; m++) {
        bias[m] = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) acc[m][j] = 0.0f;
    }
    const int steps = (K + RP - 1) / RP;
    for (int i0 = 0; i0 < steps; i0 += kRagBatch) {
        uint32_t q[kRagBatch];
        uint16_t sb[kRagBatch], zb[kRagBatch];
        XT xb[kRagBatch][M];
#pragma unroll
        for (int u = 0; u < kRagBatch; u++) {
            const int k = p + (i0 + u) * RP;
            // rows past the end load word 0's and count nothing
            const uint32_t w = k < K ? min(w0 + (uint32_t)(i0 + u) * step, last_word) : 0u;
            q[u] = __builtin_nontemporal_load(codes + w);
            sb[u] = scales[w >> 4];
            zb[u] = zeros[w >> 4];
#pragma unroll
            for (int m = 0; m < M; m++)
                xb[u][m] = a[(size_t)min(m, rows - 1) * K + min(k, K - 1)];
        }
#pragma unroll
        for (int u = 0; u < kRagBatch; u++) {
            const bool valid = p + (i0 + u) * RP < K;
            const float s = valid ? half_bits_to_float(sb[u]) : 0.0f;
            const float z = valid ? half_bits_to_float(zb[u]) : 0.0f;
            // nibbles as e4m3 bytes are q 2^-9, exactly
            const uint32_t even = q[u] & 0x0F0F0F0Fu, odd = (q[u] >> 4) & 0x0F0F0F0Fu;
            const f32x2 e01 = __builtin_amdgcn_cvt_pk_f32_fp8(even, false);
            const f32x2 e23 = __builtin_amdgcn_cvt_pk_f32_fp8(even, true);
            const f32x2 o01 = __builtin_amdgcn_cvt_pk_f32_fp8(odd, false);
            const f32x2 o23 = __builtin_amdgcn_cvt_pk_f32_fp8(odd, true);
            const float z9 = z * 0x1p-9f;
            const float d[8] = {e01.x - z9, o01.x - z9, e01.y - z9, o01.y - z9,
                                e23.x - z9, o23.x - z9, e23.y - z9, o23.y - z9};
            const float s9 = s * 512.0f;
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float x = valid ? rag_act(xb[u][m]) : 0.0f;
                // a zero scale's weights are z; neither side's product may meet
                // the other's infinite activation with its zero
                const float xs = s == 0.0f ? 0.0f : x * s9;
                const float xz = __builtin_fmaf(x, z, bias[m]);
                bias[m] = s == 0.0f ? xz : bias[m];
#pragma unroll
                for (int j = 0; j < 8; j++) acc[m][j] = __builtin_fmaf(xs, d[j], acc[m][j]);
            }
        }
    }

#pragma unroll
    for (int m = 0; m < M; m++) {
        if (m >= rows) break;
        if (m) __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; j++) red[wave][lane * 8 + j] = acc[m][j] + bias[m];
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

template <typename XT>
hipError_t launch_ragged_any(hipStream_t st, const XT* a, Int4Planes w, void* out, int M, int K,
                             int N, Epilogue ep) {
    if (M == 1)
        launch_ragged<XT, 1, 8>(st, a, w, out, M, K, N, ep);
    else if (M == 2)
        launch_ragged<XT, 2, 8>(st, a, w, out, M, K, N, ep);
    else
        launch_ragged<XT, 4, 8>(st, a, w, out, M, K, N, ep);
    return launch_status();
}

}  // namespace

bool int4_ragged_shape(const void* a, const void* codes, int K, int N) {
    return K >= 128 && N >= 64 &&
           ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(codes)) & 15) == 0;
}

bool int4_ragged_rows_supported(const void* a, const void* codes, int M, int K, int N) {
    // word indices are 32-bit, and a row step's words a 32-bit stride
    return M >= 1 && M <= 4 && N % 128 != 0 && int4_ragged_shape(a, codes, K, N) &&
           (uint64_t)K * (uint64_t)N < (1ull << 34) && N < (1 << 28) && K < (1 << 30);
}

hipError_t launch_int4_ragged_rows(hipStream_t st, const void* a, bool bf16, Int4Planes w,
                                   void* out, int M, int K, int N, Epilogue ep) {
    if (bf16) {
        ep.bf16 = true;
        return launch_ragged_any(st, static_cast<const uint16_t*>(a), w, out, M, K, N, ep);
    }
    return launch_ragged_any(st, static_cast<const float*>(a), w, out, M, K, N, ep);
}

}  // namespace accel
