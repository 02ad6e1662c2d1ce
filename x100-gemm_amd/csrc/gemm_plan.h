// Which kernel an int8 product takes: sizes and alignment only, on the host.  Plain C++ without HIP, so
// that a test can evaluate it, with the kernels' 32-bit offsets, at sizes that no test multiplies.
#pragma once
#include <math.h>

#include <algorithm>
#include <stddef.h>
#include <stdint.h>

enum {
    X100_GEMM_AUTO = 0,
    X100_GEMM_TILE256 = 1,
    X100_GEMM_TILE128 = 2,
    X100_GEMM_SKINNY = 3,
    X100_GEMM_GENERIC = 4,
    X100_GEMM_TILE256_W4 = 5,   // 256x256 tile, 4 waves of 128x128
    X100_GEMM_TILE64 = 6,       // 64x64 tile, 2 x 2 waves of 32x32, two groups on K
    X100_GEMM_TILE32 = 7,       // 32x32 tile, four waves on K
};

// Tiles of k_gemm_tile.  T128 (one block per CU), T64 and T32x64 and T32 (several); the unaligned
// form takes 64x128 tiles of eight 32x32 waves in place of T128 (its staging registers).
enum Tile { T128, T64, T32x64, T32, NTILE };

// Estimated time (us) of a product on tile t: a start-up, C's traffic, and per 128-k stage the longer
// of one block's own step (latency: few tiles) and the device's rate for all tiles (operand delivery
// from L2, 12-16 TB/s: many tiles, which is why larger tiles win there).  Constants from graph
// replays over M, N, K = 1 .. 4096 (us measured, T128 / T64 / T32x64 / T32, C = A.B):
//   aligned   333x6144x2048  11.7 / 16.9 / 18.2 / 26.8    1024^3        7.7 / 5.6 / 6.2 / 8.3
//             2048^3         15.0 / 23.6 / 29.8 / 47.3    17x4096x4096  15.1 / 7.1 / 6.4 / 6.6
//             200x2048x2048   9.9 /  5.7 /  5.5 /  7.2    256^3         4.6 / 3.5 / 3.2 / 2.9
//   unaligned 1001x1503x999  10.3 / 11.2 / 12.0 / 16.6    2047x300x2040 10.9 / 9.0 / 10.6 / 12.8
//             33x2001x2001   13.5 / 10.1 /  8.3 /  7.3    37x41x257      5.4 / 4.3 / 4.1 / 3.6
inline double c_us(int M, int N, bool acc) { return (double)M * N * (acc ? 8 : 4) / 6.5e6; }
inline double tile_us(Tile t, bool aln, int M, int N, int K, bool acc)
{
    struct Cost {
        int bm, bn;
        double start, lat, thr;   // thr: a stage of 256 tiles
        int res;                  // blocks resident at once (LDS)
        double round;             // each further round of them (M > 16): their start and C are not hidden
    };
    static const Cost costs[2][NTILE] = {
        {{64, 128, 3.6, 0.60, 0.85, 256, 0}, {64, 64, 3.3, 0.38, 0.46, 256, 0}, {32, 64, 2.95, 0.33, 0.36, 256, 0}, {32, 32, 2.7, 0.25, 0.30, 256, 0}},
        {{128, 128, 3.9, 0.35, 0.60, 256, 1.5}, {64, 64, 3.1, 0.12, 0.245, 512, 0.8}, {32, 64, 2.95, 0.10, 0.172, 768, 0.3}, {32, 32, 2.65, 0.095, 0.155, 1280, 0}}};
    const Cost &c = costs[aln][t];
    const double tiles = (double)((M - 1) / c.bm + 1) * ((N - 1) / c.bn + 1), stages = (K - 1) / 128 + 1;
    double per;
    if (aln && t == T128) {   // one block per CU: whole rounds, and a last one that is at least a block's step
        const double full = (double)((long)tiles / 256), rem = tiles - 256 * full;
        per = full * c.thr + (rem > 0 ? fmax(c.lat, rem / 256 * c.thr) : 0.0);
    } else {
        per = fmax(c.lat, tiles / 256 * c.thr);
    }
    return c.start + c_us(M, N, acc) + per * stages + (M > 16 ? (ceil(tiles / c.res) - 1) * c.round : 0.0);
}
inline Tile best_tile(bool aln, int M, int N, int K, bool acc, double &us)
{
    Tile best = T128;
    us = tile_us(T128, aln, M, N, K, acc);
    for (int t = T64; t < NTILE; t++) {
        const double u = tile_us((Tile)t, aln, M, N, K, acc);
        if (u < us) us = u, best = (Tile)t;
    }
    return best;
}
// k_gemm_big: rounds of 256 tiles, a last round no shorter than a block alone (4096^3 69.5 against 86
// us on T128; 2048^2 x 4096, 64 tiles, 42 against 29).
inline double big_us(int M, int N, int K, bool acc)
{
    const long tiles = (long)(M / 256) * (N / 256), full = tiles / 256, rem = tiles % 256;
    return 3.0 + c_us(M, N, acc) + K / 128.0 * (full * 1.77 + (rem ? fmax(1.13, rem / 256.0 * 1.77) : 0.0));
}
// The split-K kernels for M <= 16 (C = A.B pays a clearing launch).  They stream B at up to 5 TB/s in
// 128- or 256-column rows; the tiles reach 3.6 TB/s on a B beyond the caches, and less on rows that
// are not whole cache lines (4x4112x4112: 7.0 us split-K, 9.4 on T32; 16x1280x1280: 7.7 and 3.7); few tiles of a
// long K wait for each stage (9x3072x9984: 10.7 split-K, 22.4 on T32; 10x3456x8768 11.1 and 16.9).
inline double skinny_us(int M, int N, int K, bool acc)
{
    const double kn = (double)K * N, clear = acc ? 0.0 : 1.6;
    if (N % 128 == 0 && K % 512 == 0) return clear + 2.9 + kn / 16e6;
    return clear + (M <= 8 ? 4.7 + kn / 7e6 : 7.3 + kn / 4.3e6);
}
inline double skinny_tile_us(Tile &t, int M, int N, int K, bool acc)
{
    double us;
    t = best_tile(true, M, N, K, acc, us);
    if (N % 128) us = 2.65 + 1.5 * (us - 2.65);
    if ((double)K * N > (N % 128 ? 14e6 : 20e6)) us = fmax(us, 2.65 + 0.205 * ((K - 1) / 128 + 1));   // stages of a B beyond the L2s
    return fmax(us, 2.65 + (double)K * N / 3.6e6);
}

// k_gemm_big adds 32-bit byte offsets to 64-bit bases: up to row 127 of A (63 with superstages, K / 64 a
// multiple of 8) and row 31 of B, and, where C is added, row 143 of C (4-byte elements).  Above these
// sizes the offsets would wrap (C from N = 7.5 million columns).
inline bool big_super(int K) { return K / 64 % 8 == 0; }
inline uint64_t big_a_reach(int K) { return (big_super(K) ? 63ull : 127ull) * (uint64_t)K + 128; }
inline uint64_t big_b_reach(int N) { return 31ull * (uint64_t)N + 256; }
inline uint64_t big_c_reach(int N) { return 4 * (143ull * (uint64_t)N + 256); }
inline bool big_fits(int M, int N, int K, bool acc)
{
    const uint64_t lim = (uint64_t)1 << 32;
    return M % 256 == 0 && N % 256 == 0 && K % 64 == 0 && K >= 512 && big_a_reach(K) <= lim && big_b_reach(N) <= lim &&
           (!acc || big_c_reach(N) <= lim);
}

// k_gemm_mfma's tile by output size.  1024^2 x 4096 took 27.3 us on 64x64 tiles and 39.9 on 128x128, 2048^2 x
// 4096 52.6 on 128x128; 256^3 3.5 on 32x32 and 5.7 on 128x128.  Up to 64 rows or columns a 128x128 tile is half
// empty, which a short K shows (27 x 521408 x 64 50 against 31).
inline bool tile_launches(Tile t, bool aln, int M, int N);
inline Tile mfma_tile(int M, int N, int K)
{
    const double mn = (double)M * N;
    if (std::min(M, N) <= 64 && K <= 128 && mn >= 1e6 && tile_launches(T64, true, M, N)) return T64;
    return mn >= 4.0 * 1024 * 1024 ? T128 : mn >= 1024.0 * 1024 ? T64 : T32;
}
// Where k_gemm_mfma is the faster one: many outputs of a short K.  C's bytes are most of the time there, and
// two to five of its blocks share a CU, so that one block's C, start and end run under the others' products;
// T128 of k_gemm_tile has the CU for itself and T64 half of it.  us, k_gemm_mfma / k_gemm_tile:
//   C = A.B    256x416544x16   85 / 119    4096x4096x64   14.2 / 17.6    1024^2 x 64    3.6 / 4.2
//              16384^2 x 256  225 / 318    4096x4096x256  17.9 / 19.4    768x2944x192   5.2 / 6.7
//              256x2^20x256   307 / 425    1299x30864x368 66 / 55        9476x11984x512 190 / 169
//   C += A.B   4096x4096x64    22 / 34     4096x4096x256  27.3 / 38.6    7168x4096x320  50 / 60
//              50769x64x64    6.0 / 8.1    35584x192x128  18.8 / 12.6    31x209280x128  28 / 15
// The line is fitted to 2146 seeded sizes with K up to 1024 timed on both, a size that k_gemm_mfma would slow
// down counting twice.  It lies furthest where M, N and K divide into whole tiles and stages (no guards); C +=
// A.B, whose C k_gemm_tile reads under its stages, leaves the guarded form less, and so do 64x64 tiles and up to
// 64 rows or columns, where A or B is most of the traffic.
inline bool mfma_better(int M, int N, int K, bool acc)
{
    const double mn = 1e-6 * M * N;   // million outputs
    if (M <= 16 || mn < 1.0 || K > 448) return false;
    const int b = mfma_tile(M, N, K) == T128 ? 128 : 64;
    if (std::min(M, N) <= 64) return K <= (acc ? 64.0 : std::min(192.0, 96 * pow(mn, 0.15)));
    if (M % b == 0 && N % b == 0 && K % 64 == 0) return K <= (b == 128 ? std::min(448.0, 176 * pow(mn, 0.45)) : std::min(320.0, 224 * pow(mn, 0.45)));
    if (b == 64) return mn >= 1.5 && K <= std::min(208.0, 160 * pow(mn, 0.30));
    return K <= (acc ? std::min(224.0, 64 * pow(mn, 0.30)) : std::min(448.0, 112 * pow(mn, 0.30)));
}
// Threads of a launch of k_gemm_tile: the runtime takes at most 2^32 - 1 (one column of tiles reaches that at
// M = 2^30, where k_gemm_mfma's 128x128 tiles, 256 threads each, and the generic kernel's grid do not).
inline bool tile_launches(Tile t, bool aln, int M, int N)
{
    const uint64_t bm = t == T128 ? (aln ? 128 : 64) : t == T64 ? 64 : 32, bn = t == T128 ? 128 : t == T32 ? 32 : 64;
    return (((uint64_t)M - 1) / bm + 1) * (((uint64_t)N - 1) / bn + 1) * (t == T128 ? 512 : 256) < ((uint64_t)1 << 32);
}

enum GemmKernel { GK_REFUSED, GK_BIG8, GK_BIG4, GK_TILE, GK_MFMA, GK_SKINNY, GK_GENERIC };
struct GemmPlan {
    GemmKernel kernel;
    Tile tile;      // GK_TILE, GK_MFMA (T128, T64 or T32)
    bool aligned;   // GK_TILE: the DMA form
};

// aligned: K, N multiples of 16 and A, B, C 16-byte aligned.  A forced variant other than the generic one
// takes aligned operands only, and a forced 256x256 tile that the shape does not divide 128x128.
inline GemmPlan gemm_plan(int M, int N, int K, bool aligned, bool acc, int variant)
{
    // k_gemm_tile: 32-bit offsets inside a tile and a stage, and a whole 16-byte chunk in each operand; past them
    // k_gemm_mfma takes aligned operands (33 x 2^24 x 400 2.4-3.5 ms, on the generic kernel 20.6-20.9)
    const bool tiled = N < (1 << 24) && K < (1 << 24) && (size_t)M * K >= 16 && (size_t)K * N >= 16;
    const bool whole = big_fits(M, N, K, acc);
    const bool skinny = M <= 16 && (size_t)K * N < ((size_t)1 << 32);   // B must fit one buffer resource
    auto on_tile = [&](Tile t) {
        return GemmPlan{tiled && tile_launches(t, aligned, M, N) ? GK_TILE : aligned ? GK_MFMA : GK_GENERIC, t, aligned};
    };
    if (variant != X100_GEMM_AUTO && variant != X100_GEMM_GENERIC && !aligned) return {GK_REFUSED, T128, false};
    switch (variant) {
    case X100_GEMM_AUTO: {
        Tile t = T128;
        double us = 0;
        if (aligned && skinny && (!tiled || skinny_us(M, N, K, acc) <= skinny_tile_us(t, M, N, K, acc)))
            return {GK_SKINNY, t, true};
        if (!tiled) return aligned && whole ? GemmPlan{GK_BIG8, t, true} : on_tile(mfma_tile(M, N, K));
        if (aligned && !whole && mfma_better(M, N, K, acc)) return {GK_MFMA, mfma_tile(M, N, K), true};
        t = best_tile(aligned, M, N, K, acc, us);
        if (aligned && whole && us >= big_us(M, N, K, acc)) return {GK_BIG8, t, true};
        return on_tile(tile_launches(t, aligned, M, N) ? t : mfma_tile(M, N, K));
    }
    case X100_GEMM_TILE256: return whole ? GemmPlan{GK_BIG8, T128, true} : on_tile(T128);
    case X100_GEMM_TILE256_W4: return whole ? GemmPlan{GK_BIG4, T128, true} : on_tile(T128);
    case X100_GEMM_TILE128: return on_tile(T128);
    case X100_GEMM_TILE64: return on_tile(T64);
    case X100_GEMM_TILE32: return on_tile(T32);
    case X100_GEMM_SKINNY: return {skinny ? GK_SKINNY : GK_REFUSED, T128, true};
    case X100_GEMM_GENERIC: return {GK_GENERIC, T128, aligned};
    }
    return {GK_REFUSED, T128, false};
}
