// Host check of the int8 GEMM's kernel selection (csrc/gemm_plan.h).  Reads lines "M N K aligned acc variant"
// and prints each plan as "kernel tile aligned fits": fits is 0 where an offset that the chosen kernel forms in
// 32 bits, or its launch, would not hold the size.  The offsets are those of gemm_i8.hip, lane by lane.
#include <stdio.h>

#include <algorithm>

#include "gemm_plan.h"

static bool same(uint32_t a, uint64_t b) { return a == b; }

// k_gemm_big<NW>: aoff, boff and coff of every wave and lane.
static bool big_offsets(int NW, int N, int K, bool acc)
{
    const int WN = NW / 2, FN = 8 / WN;
    for (int w = 0; w < NW; w++)
        for (int lane = 0; lane < 64; lane++) {
            const int ra = big_super(K) ? 8 * w + (lane >> 3) : 16 * w + (lane >> 2), rb = 4 * w + (lane >> 4);
            if (!same((uint32_t)ra * (uint32_t)K + 127, (uint64_t)ra * K + 127)) return false;
            if (!same((uint32_t)rb * (uint32_t)N + 255, (uint64_t)rb * N + 255)) return false;
            for (int t = 0; t < 2 && acc; t++) {
                const int row = (w / WN) * 128 + 8 * t + (lane >> 3), col = (w % WN) * FN * 32 + 31;
                if (!same(4u * ((uint32_t)row * (uint32_t)N + col), 4 * ((uint64_t)row * N + col))) return false;
            }
        }
    return true;
}

// k_gemm_tile: rows of A and C below 128, k-rows of B below 128, the tile's columns after them.
static bool tile_offsets(int N, int K)
{
    return same(127u * (uint32_t)K + 128, 127ull * K + 128) && same(127u * (uint32_t)N + 128, 127ull * N + 128);
}

// Threads of the launch, 256x256 and split-K kernels aside (their C or B cannot be large enough).
static bool launches(const GemmPlan &p, int M, int N)
{
    static const int bm[] = {128, 64, 32, 32}, bn[] = {128, 64, 64, 32};
    const bool mfma = p.kernel == GK_MFMA;
    const uint64_t rows = p.kernel == GK_TILE && p.tile == T128 && !p.aligned ? 64 : bm[p.tile];
    const uint64_t nt = mfma ? (p.tile == T32 ? 64 : 256) : p.tile == T128 ? 512 : 256;
    return ((M - 1) / rows + 1) * ((N - 1) / (uint64_t)bn[p.tile] + 1) * nt <= 0xffffffffu;
}

int main()
{
    static const char *const kernels[] = {"refused", "big8", "big4", "tile", "mfma", "skinny", "generic"};
    static const char *const tiles[] = {"128", "64", "32x64", "32"};
    int M, N, K, aligned, acc, variant;
    while (scanf("%d %d %d %d %d %d", &M, &N, &K, &aligned, &acc, &variant) == 6) {
        const GemmPlan p = gemm_plan(M, N, K, aligned, acc, variant);
        bool fits = true;
        if (p.kernel == GK_BIG8 || p.kernel == GK_BIG4) fits = big_offsets(p.kernel == GK_BIG8 ? 8 : 4, N, K, acc);
        if (p.kernel == GK_TILE) fits = tile_offsets(N, K) && launches(p, M, N);
        if (p.kernel == GK_MFMA) fits = launches(p, M, N);
        printf("%s %s %d %d\n", kernels[p.kernel], p.kernel == GK_TILE || p.kernel == GK_MFMA ? tiles[p.tile] : "-", p.aligned, fits);
    }
    return 0;
}
