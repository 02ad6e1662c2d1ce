// Host check of csrc/resident_cache.h: prints the occupancy queries of a verify loop and whether every answer
// was the key's own.
#include <stdio.h>

#include "resident_cache.h"

int main()
{
    ResidentCache c;
    int queries = 0, wrong = 0;
    auto run = [&](int kernel, int nt, size_t lds, int dev) {
        const int want = 1 + kernel + 64 * dev + (int)(lds % 1009) + nt;
        const int got = c.get({(const void *)(0x7f4a00001000ull + 0x340ull * kernel), nt, dev, lds}, [&] { queries++; return want; });
        wrong += got != want;
    };
    // 100 steps of 1 to 8 token rows over five weight shapes: K sets the kernel, K and the rows the LDS
    for (int step = 0; step < 100; step++)
        for (int m = 1; m <= 8; m++)
            for (int shape = 0; shape < 5; shape++) run(2 * shape + (m > 4), 512, (size_t)m * (2064 + 1024 * shape) + 16, 0);
    printf("%d ", queries);
    queries = 0;
    // far more keys than entries, block sizes and devices among them: still the key's own answers
    for (int i = 0; i < 20000; i++) run(i * 7 % 64, 256 << (i % 3), (size_t)(i * 31 % 977) * 16, i % 4);
    printf("%d %d\n", queries > 0, wrong);
    return 0;
}
