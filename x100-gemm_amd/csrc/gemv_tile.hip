// Integer tile GEMV of the decode benchmarks (bench/q4_gemv.c, bench/moe_decode.c):
//   y[M][N] = W[N][K] . x[M][K]^T,  W int4 (two per byte) or int8,  x int8,  y int32 (exact).
//
// The weights stay in the reference's own packed layouts, so a matrix packed by its pack_w_int4 /
// pack_w_int8 (bench/q4_gemv.c:37-48, 55-62) is consumed as is:
//   int8:  [N/8][K/16][128]  byte n*16 + k of tile (nb, kb) = W[8nb + n][16kb + k];
//   int4:  [N/8][K/32][128]  byte n*16 + k of tile (nb, kp) holds W[8nb + n][32kp + k] in the
//                            low nibble and W[8nb + n][32kp + 16 + k] in the high nibble
//                            (two's-complement 4-bit values).
// k_gemv_tile: dot products, for one or two token rows; k_gemv_tile_mm: the matrix cores (tile_mm says
// which).  In k_gemv_tile one wave per 8-row N-block: lane l reads 16 bytes (row n = l % 8 of tile l / 8 of each 1 KiB
// chunk), so a wave load is 64 x 16 contiguous bytes; all chunk loads of the wave are issued
// before the first is used.  x rows sit in LDS with their 16-element sums.
//
// int4 values are handled as u ^ 8 (unsigned nibble u, so u ^ 8 = q + 8 in [0, 15]):
//   sum_k q_k x_k = sum_k (u_k ^ 8) x_k - 8 * sum_k x_k,
// with v_dot4_i32_i8 on the byte-wise (u ^ 8) values.
#include "x100_common.h"
#include "x100_internal.h"

namespace {

// x [M][K] int8 -> LDS (xs, 16-byte aligned) with per-16 sums xsum [M][K/16], 1024 vectors of 16
// bytes per pass: xload issues a pass's loads (bounds-checked buffer loads), xstore writes it.
X100_DEV void xload(rsrc_t xr, int v0, v4u (&t)[4])
{
#pragma unroll
    for (int i = 0; i < 4; i++)
        t[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, (v0 + (int)threadIdx.x + 256 * i) * 16, 0, 0);
}
// Vectors past the end go to the spare slot nv (no branch, so the loads are never sunk into one).
X100_DEV void xstore(const v4u (&t)[4], int v0, int nv, int8_t *xs, int *xsum)
{
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int v = min(v0 + (int)threadIdx.x + 256 * i, nv);
        *(v4u *)(xs + v * 16) = t[i];
        int s = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) s = dot4((int)t[i][j], 0x01010101, s);
        xsum[v] = s;
    }
}

// Sum over the 8 lanes l, l^8, l^16, ..., l^56 (same row n of the N-block).
X100_DEV int sum_stride8(int v)
{
    v += dpp_i<0x128>(0, v);         // row_ror:8 = lane (i + 8) mod 16 within a row: xor 8
    v += xor16_i(v);
    v += xor32_i(v);
    return v;
}

constexpr int CH = 4;   // 1 KiB chunks per load pass

// grid = ceil(N/8 * S / 4) blocks of 4 waves.  S waves share an N-block, each taking a contiguous
// share of its chunks (S = 2 or 4 when there are too few N-blocks to give every CU several waves);
// their int32 partial sums are added through LDS, which is exact in any order.
template <int MR, bool INT4, int S>
__global__ __launch_bounds__(256) void k_gemv_tile(int M, int N, int K, const uint8_t *__restrict__ W,
                                                   const int8_t *__restrict__ x, int32_t *__restrict__ y)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ int red[4][MR][8];                     // partial sums of the S waves of an N-block
    int8_t *xs = (int8_t *)smem;                      // [M][K] + one spare 16-byte slot
    int *xsum = (int *)(smem + (size_t)M * K + 16);   // [M][K/16] + one spare
    const int lane = threadIdx.x & 63, w = wave_id();
    const int Nb = N / 8;
    const int nbk = (int)blockIdx.x * (4 / S) + w / S;   // this wave's N-block
    const int ks = w % S;                                // its share of the N-block's chunks
    const int nb = min(nbk, Nb - 1);                     // clamped: the store below is skipped
    const int tiles = INT4 ? K / 32 : K / 16;            // 128-byte tiles per N-block
    const int nch = (tiles + 7) / 8;                     // 1 KiB chunks (8 tiles)
    const int cb = ks * nch / S, ce = (ks + 1) * nch / S;
    const rsrc_t wr = buf_rsrc(W + (size_t)nb * tiles * 128, (uint32_t)tiles * 128u);
    const int n = lane & 7;

    // x pass 0, then the first weight chunks, all in flight before x is stored.
    const int nv = M * K / 16;
    const rsrc_t xr = buf_rsrc(x, (uint32_t)M * K);
    v4u xt[4];
    xload(xr, 0, xt);
    // One token row: the x loads of every wave go out before any wave's weight loads (s_barrier, no
    // wait): int4 4864 x 896 3.03 -> 2.87 us; no change with int8 weights or several rows.
    if constexpr (MR == 1) __builtin_amdgcn_s_barrier();
    v4u wv[CH];
#pragma unroll
    for (int c = 0; c < CH; c++)
        wv[c] = __builtin_amdgcn_raw_buffer_load_b128(wr, ((cb + c) * 64 + lane) * 16, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    xstore(xt, 0, nv, xs, xsum);
    for (int v0 = 1024; v0 < nv; v0 += 1024) {
        xload(xr, v0, xt);
        xstore(xt, v0, nv, xs, xsum);
    }
    __syncthreads();

    int acc[MR];
#pragma unroll
    for (int m = 0; m < MR; m++) acc[m] = 0;
    for (int c0 = cb; c0 < ce; c0 += CH) {
        if (c0 > cb) {
#pragma unroll
            for (int c = 0; c < CH; c++)
                wv[c] = __builtin_amdgcn_raw_buffer_load_b128(wr, ((c0 + c) * 64 + lane) * 16, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int t = (c0 + c) * 8 + (lane >> 3);   // tile of this lane
            if (t < tiles && c0 + c < ce) {
                if (INT4) {
                    int lo[4], hi[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        lo[j] = (int)((wv[c][j] & 0x0F0F0F0Fu) ^ 0x08080808u);
                        hi[j] = (int)(((wv[c][j] >> 4) & 0x0F0F0F0Fu) ^ 0x08080808u);
                    }
#pragma unroll
                    for (int m = 0; m < MR; m++) {
                        if (m < M) {
                            const v4i xl = *(const v4i *)(xs + m * K + 32 * t);
                            const v4i xh = *(const v4i *)(xs + m * K + 32 * t + 16);
                            int s = acc[m];
#pragma unroll
                            for (int j = 0; j < 4; j++) {
                                s = dot4(lo[j], xl[j], s);
                                s = dot4(hi[j], xh[j], s);
                            }
                            acc[m] = s - 8 * (xsum[m * (K / 16) + 2 * t] + xsum[m * (K / 16) + 2 * t + 1]);
                        }
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < MR; m++) {
                        if (m < M) {
                            const v4i xv = *(const v4i *)(xs + m * K + 16 * t);
                            int s = acc[m];
#pragma unroll
                            for (int j = 0; j < 4; j++) s = dot4((int)wv[c][j], xv[j], s);
                            acc[m] = s;
                        }
                    }
                }
            }
        }
    }
    const bool store = nbk < Nb && lane < 8;
    if constexpr (S == 1) {
#pragma unroll
        for (int m = 0; m < MR; m++) {
            if (m < M) {
                const int v = sum_stride8(acc[m]);
                if (store) y[(size_t)m * N + nb * 8 + n] = v;
            }
        }
    } else {
#pragma unroll
        for (int m = 0; m < MR; m++) {
            const int v = sum_stride8(acc[m]);
            if (lane < 8) red[w][m][n] = v;
        }
        __syncthreads();
        if (ks == 0) {
#pragma unroll
            for (int m = 0; m < MR; m++) {
                if (m < M) {
                    int v = 0;
#pragma unroll
                    for (int k = 0; k < S; k++) v += red[w + k][m][n & 7];
                    if (store) y[(size_t)m * N + nb * 8 + n] = v;
                }
            }
        }
    }
}

// Several token rows on the matrix cores: v_mfma_i32_16x16x64_i8 with 16 weight rows (two N-blocks)
// against the token rows as columns (columns from M on: copies, not stored).  A step is four 128-byte
// tiles of each N-block, one 16-byte load per lane (lane l: row l % 8 of N-block l % 16 / 8, tile l / 16,
// 512 contiguous bytes per N-block), which is one A operand (int8) or two (int4: the low nibbles
// against the first 16 k of each tile, the high ones against the last 16, both as 16 q, so that the
// sums are 16 times the result: |sum| <= 2^14 K, below 2^31 for every K that the LDS takes).  S waves
// share the rows' steps.  x rows in LDS at a pitch of 16 mod 256 bytes: the 16 lanes of a read take 16
// different 16-byte columns of a bank line.
// U steps are loaded per pass, the first pass before x is waited for.  Bound by HBM on large matrices:
// int4 151936 x 2048 at M = 8 54.7 -> 29.3 us (5.5 TB/s), where the dot products and the nibble
// offsets of eight rows took longer than the weights.
template <bool INT4, int S, int U>
__global__ __launch_bounds__(256) void k_gemv_tile_mm(int M, int N, int K, int pitch, uint32_t mk16,
                                                      const uint8_t *__restrict__ W, const int8_t *__restrict__ x,
                                                      int32_t *__restrict__ y)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];   // x: [M][pitch] + a spare 16-byte slot
    __shared__ v4i red[S > 1 ? 4 : 1][64];
    const int lane = threadIdx.x & 63, w = wave_id(), g = lane >> 4, col = lane & 15;
    const int Nb = N / 8, tiles = INT4 ? K / 32 : K / 16, steps = (tiles + 3) / 4;
    const int rt = (int)blockIdx.x * (4 / S) + w / S, nb0 = 2 * rt;   // N-blocks nb0, nb0 + 1
    const int sb = w % S * steps / S, se = (w % S + 1) * steps / S;
    const rsrc_t wr = buf_rsrc(W + (size_t)min(nb0, Nb - 1) * tiles * 128, (uint32_t)(max(min(Nb - nb0, 2), 0) * tiles) * 128u);
    const uint32_t off = (uint32_t)((col >> 3) * tiles * 128 + (col & 7) * 16);
    auto load = [&](int s) __attribute__((always_inline)) {   // zeros past the steps, tiles or N-blocks
        const int t = 4 * s + g;
        return (v4i)__builtin_amdgcn_raw_buffer_load_b128(wr, (int)(s < se && t < tiles ? off + (uint32_t)t * 128u : ~0u), 0, 0);
    };

    const int vpr = K / 16, nv = M * vpr;
    const rsrc_t xr = buf_rsrc(x, (uint32_t)M * K);
    v4u xt[4];
    xload(xr, 0, xt);
    v4i wv[U];
#pragma unroll
    for (int u = 0; u < U; u++) wv[u] = load(sb + u);
    __builtin_amdgcn_sched_barrier(0);
    auto put = [&](int v0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int v = v0 + (int)threadIdx.x + 256 * i, r = (int)udiv16((uint32_t)min(v, nv), (uint32_t)vpr, mk16);
            *(v4u *)(smem + (v < nv ? r * pitch + 16 * (v - r * vpr) : M * pitch)) = xt[i];
        }
    };
    put(0);
    for (int v0 = 1024; v0 < nv; v0 += 1024) {
        xload(xr, v0, xt);
        put(v0);
    }
    __syncthreads();

    const uint8_t *xm = smem + min(col, M - 1) * pitch;
    v4i acc0 = {}, acc1 = {};
    for (int s0 = sb; s0 < se; s0 += U) {
        if (s0 > sb) {
#pragma unroll
            for (int u = 0; u < U; u++) wv[u] = load(s0 + u);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = 4 * min(s0 + u, steps - 1) + g;   // past the last step: zero weights
            if constexpr (INT4) {
                v4i lo, hi;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    lo[j] = (wv[u][j] << 4) & (int)0xF0F0F0F0;
                    hi[j] = wv[u][j] & (int)0xF0F0F0F0;
                }
                acc0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(lo, *(const v4i *)(xm + 32 * t), acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(hi, *(const v4i *)(xm + 32 * t + 16), acc1, 0, 0, 0);
            } else {
                v4i &a = u & 1 ? acc1 : acc0;
                a = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[u], *(const v4i *)(xm + 16 * t), a, 0, 0, 0);
            }
        }
    }
    v4i v = acc0 + acc1;
    if constexpr (S > 1) {
        red[w][lane] = v;
        __syncthreads();
        if (w % S) return;
#pragma unroll
        for (int k = 1; k < S; k++) v += red[w + k][lane];
    }
    if constexpr (INT4) v >>= 4;
    // rows 16 rt + 4 g + r of token row col
    typedef int v4i_a4 __attribute__((ext_vector_type(4), aligned(4)));
    if (col < M && nb0 + (g >> 1) < Nb) *(v4i_a4 *)(y + (size_t)col * N + 16 * rt + 4 * g) = v;
}

// Waves per N-block: enough to give the chip ~1024 waves when the matrix has few N-blocks, as long
// as every wave keeps at least 3 chunks.
inline int tile_split(int N, int nch)
{
    const int nblk = N / 8;
    const int by_waves = nblk >= 1024 ? 1 : nblk >= 512 ? 2 : 4;
    const int minch = 3;
    const int by_chunks = nch / 4 >= minch ? 4 : nch / 2 >= minch ? 2 : 1;
    return min(by_waves, by_chunks);
}

template <int MR, int S>
hipError_t launch_tile_s(bool int4, int M, int N, int K, const void *W, const int8_t *x, int32_t *y, hipStream_t s)
{
    const dim3 grid((N / 8 * S + 3) / 4);
    const size_t lds = (size_t)M * K + 16 + ((size_t)M * (K / 16) + 1) * 4;
    if (int4)
        hipLaunchKernelGGL((k_gemv_tile<MR, true, S>), grid, dim3(256), lds, s, M, N, K, (const uint8_t *)W, x, y);
    else if constexpr (MR == 1 || S != 2)
        hipLaunchKernelGGL((k_gemv_tile<MR, false, S>), grid, dim3(256), lds, s, M, N, K, (const uint8_t *)W, x, y);
    else   // two int8 rows come here with K <= 512 (S = 1) or above 2048 (S = 4)
        return hipErrorInvalidValue;
    return hipGetLastError();
}

template <int MR>
hipError_t launch_tile(bool int4, int M, int N, int K, const void *W, const int8_t *x, int32_t *y, hipStream_t s)
{
    const int tiles = int4 ? K / 32 : K / 16;
    switch (tile_split(N, (tiles + 7) / 8)) {
    case 1: return launch_tile_s<MR, 1>(int4, M, N, K, W, x, y, s);
    case 2: return launch_tile_s<MR, 2>(int4, M, N, K, W, x, y, s);
    default: return launch_tile_s<MR, 4>(int4, M, N, K, W, x, y, s);
    }
}

// k_gemv_tile_mm with S waves per 16 rows and U steps per pass: four waves on K (int8 from K = 1024 up with 8
// steps in flight per wave), fewer where the rows fill the chip and K is at most eight steps, which four waves
// cut to two or less each.  us, M = 2 and 8, dot products / S = 4 / 2 / 1: int8 131072x128 5.9, 8.5 / 8.0, 8.3 /
// 6.1, 6.6 / 3.7, 4.1; 40960x256 3.4, 5.0 / 4.1, 4.2 / 3.5, 3.6 / 3.5, 3.6; 65536x512 4.5, 8.1 / 5.2, 5.5 / 4.2,
// 4.4 / 4.2, 4.5; int4 65536x256 4.1, 6.7 / - / 4.9, 4.8 / 3.7, 3.6.  S = 4 takes 16 threads per row, which passes
// the 2^32 - 1 of one launch at N = 2^28.
hipError_t launch_tile_mm(bool int4, int M, int N, int K, const void *W, const int8_t *x, int32_t *y, hipStream_t s)
{
    const int steps = ((int4 ? K / 32 : K / 16) + 3) / 4, pitch = (K + 255) / 256 * 256 + 16;
    auto go = [&](auto k, int S) {
        hipLaunchKernelGGL(k, dim3(((N / 8 + 1) / 2 * S + 3) / 4), dim3(256), (size_t)M * pitch + 16, s, M, N, K, pitch,
                           udiv16_magic((uint32_t)(K / 16)), (const uint8_t *)W, x, y);
    };
    const bool rows = steps <= 8 || N >= 1 << 28;   // enough of them: fewer waves per 16
    if (int4) {
        if (rows && N >= 65536) go(k_gemv_tile_mm<true, 1, 2>, 1);
        else if (rows && N >= 16384) go(k_gemv_tile_mm<true, 2, 4>, 2);
        else if (steps <= 8) go(k_gemv_tile_mm<true, 4, 2>, 4);
        else go(k_gemv_tile_mm<true, 4, 4>, 4);
    } else {
        if (rows && N >= 65536) go(k_gemv_tile_mm<false, 1, 2>, 1);
        else if (rows && N >= 16384) go(k_gemv_tile_mm<false, 2, 4>, 2);
        else if (steps <= 8) go(k_gemv_tile_mm<false, 4, 2>, 4);
        else if (steps <= 16) go(k_gemv_tile_mm<false, 4, 4>, 4);
        else go(k_gemv_tile_mm<false, 4, 8>, 4);
    }
    return hipGetLastError();
}

// The matrix cores take three token rows and more; one row where the launch streams enough weights, two rows
// in between (us, dot products / matrix cores; int4, int8): 151936x2048 M = 1 27.6 / 25.6, 47.5 / 44.5, M = 8
// 54.7 / 29.3, 60.6 / 48.3; 4864x896 M = 1 2.8 / 2.8, 3.2 / 3.2, M = 8 5.0 / 2.9, 5.3 / 3.2.  With two rows the
// dot products keep a short K (30304x32 int4 3.4 / 3.7; 14536x160 int8 2.9 / 3.1) until 65536 rows, and a long K
// with too few 16-row tiles to split it over (1256x9216 int4 4.5 / 5.6).
inline bool tile_mm(int M, int N, int K)
{
    if (M > 2) return true;
    if (N >= 65536) return M == 2 || K >= 1024;
    if (M == 1) return false;
    return K <= 512 ? K > 128 && N < 4096 : K <= 2048 || N >= 4096;
}

}  // namespace

hipError_t x100_gemv_tile_launch(int int4, int M, int N, int K, const void *W, const int8_t *x, int32_t *y,
                                 hipStream_t s)
{
    if (M < 1 || M > 8 || N < 8 || N % 8 || K < 16 || K % (int4 ? 32 : 16)) return hipErrorInvalidValue;
    if ((size_t)M * K + 16 + ((size_t)M * (K / 16) + 1) * 4 > 64 * 1024) return hipErrorInvalidValue;
    if (tile_mm(M, N, K)) return launch_tile_mm(int4 != 0, M, N, K, W, x, y, s);
    if (M == 1) return launch_tile<1>(int4 != 0, M, N, K, W, x, y, s);
    return launch_tile<2>(int4 != 0, M, N, K, W, x, y, s);   // M = 2
}
