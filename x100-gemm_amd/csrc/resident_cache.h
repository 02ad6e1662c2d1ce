// Occupancy of persistent launches, remembered per calling thread.  Plain C++ without HIP, so that a test can
// count the queries.
#pragma once
#include <stddef.h>
#include <stdint.h>

struct ResidentKey {
    const void *k;   // kernel address: template instances with the same signature are distinct kernels
    int nt, dev;
    size_t lds;
};
// 16 sets of 16 entries, the oldest of a set replaced.  A kernel's LDS depends on its token rows and on K, so a
// program has a key for each combination that it runs: verify steps of 1 to 8 rows over five shapes are 40,
// which 16 entries replaced in turn would have queried again at every launch.
class ResidentCache {
public:
    template <class Query>
    int get(const ResidentKey &q, Query &&query)
    {
        uint64_t h = (uint64_t)(uintptr_t)q.k * 0x9E3779B97F4A7C15ull;
        h = (h ^ q.lds) * 0x9E3779B97F4A7C15ull;
        h = (h ^ ((uint64_t)(uint32_t)q.dev << 32 | (uint32_t)q.nt)) * 0x9E3779B97F4A7C15ull;
        const int n = (int)(h >> 60);
        Entry *set = e_[n];
        for (int i = 0; i < 16; i++)
            if (set[i].blocks && set[i].q.k == q.k && set[i].q.nt == q.nt && set[i].q.dev == q.dev && set[i].q.lds == q.lds)
                return set[i].blocks;
        Entry &e = set[next_[n]++ & 15];
        e = Entry{q, query()};
        return e.blocks;
    }

private:
    struct Entry {
        ResidentKey q;
        int blocks;   // 0: empty
    };
    Entry e_[16][16] = {};
    uint8_t next_[16] = {};
};
