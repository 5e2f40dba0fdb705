// Checks the range bookkeeping of the device pools (gpuvoxels_amd/csrc/vx3h_pool.h) against a
// plain list of ranges, with array growths that fail: prints "ok <failures>" when every range
// lies inside its pool's arrays, none overlap, and an error leaves everything as it was; else
// "bad <reason>".
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../gpuvoxels_amd/csrc/vx3h_pool.h"

using namespace vx3;

#define BAD(...) do { printf("bad "); printf(__VA_ARGS__); printf("\n"); exit(0); } while (0)

namespace {
struct Pool { RangeAlloc ra; int cap = 0; };
struct Held { int start[3], n[3]; };

void check(Pool* pools, const std::vector<Held>& held) {
    for (int k = 0; k < 3; k++) {
        std::vector<int> used(pools[k].cap, 0);
        for (const Held& h : held) {
            if (h.start[k] < 0 || h.start[k] + h.n[k] > pools[k].cap) BAD("range [%d, +%d) of pool %d past %d", h.start[k], h.n[k], k, pools[k].cap);
            for (int i = 0; i < h.n[k]; i++) if (used[h.start[k] + i]++) BAD("overlap in pool %d", k);
        }
        if (pools[k].ra.hi > pools[k].cap) BAD("pool %d counts elements past its arrays", k);
        for (const auto& f : pools[k].ra.freeRanges) {
            if (f.first + f.second > pools[k].ra.hi) BAD("free range past the end of pool %d", k);
            for (int i = 0; i < f.second; i++) if (used[f.first + i]) BAD("a held element of pool %d is free", k);
        }
    }
}
}  // namespace

int main(int argc, char** argv) {
    srand(argc > 1 ? atoi(argv[1]) : 1);
    Pool pools[3];
    std::vector<Held> held;
    int failures = 0;
    for (int step = 0; step < 4000; step++) {
        if (!held.empty() && rand() % 100 < 45) {
            const int i = rand() % (int)held.size();
            for (int k = 0; k < 3; k++) pools[k].ra.release(held[i].start[k], held[i].n[k]);
            held[i] = held.back();
            held.pop_back();
        } else {
            Held h;
            for (int k = 0; k < 3; k++) { h.start[k] = -1; h.n[k] = 1 + rand() % 20; }
            RangeAlloc before[3] = {pools[0].ra, pools[1].ra, pools[2].ra};
            bool failed = false;
            Pool* const p[3] = {&pools[0], &pools[1], &pools[2]};
            int* const at[3] = {&h.start[0], &h.start[1], &h.start[2]};
            const int st = takeRanges(p, h.n, at, [&](Pool& q) {
                if (rand() % 3 == 0) { failed = true; return 1; }
                q.cap = q.ra.hi + rand() % 8;
                return 0;
            });
            if ((st != 0) != failed) BAD("status");
            if (st) {
                failures++;
                for (int k = 0; k < 3; k++)
                    if (pools[k].ra.hi != before[k].hi || pools[k].ra.freeRanges != before[k].freeRanges) BAD("pool %d changed by a failure", k);
            } else held.push_back(h);
        }
        check(pools, held);
    }
    for (const Held& h : held) for (int k = 0; k < 3; k++) pools[k].ra.release(h.start[k], h.n[k]);
    for (const Pool& p : pools) if (p.ra.hi || !p.ra.freeRanges.empty()) BAD("not empty in the end");
    printf("ok %d\n", failures);
    return 0;
}
