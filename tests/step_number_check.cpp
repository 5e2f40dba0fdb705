// Checks the fused kernel's report numbers (TsNumbers in gpuvoxels_amd/csrc/vx3h_steptile.h)
// across the largest one, against report words as the kernel keeps them: a word that no step of
// the present call wrote never holds a number of that call.  Prints "ok <restarts>" or "bad".
#include <cstdio>
#include <vector>

#include "../gpuvoxels_amd/csrc/vx3h_steptile.h"

using namespace vx3;

int main() {
    const unsigned lengths[] = {1, 2, 5, 7, 33, 1000, 3, 4096};
    int restarts = 0;
    for (unsigned start = 1; start < 60; start++) {   // the first call's distance from the end
        TsNumbers numbers;
        numbers.next = UINT32_MAX - start + 1;
        unsigned never = 0, stale = UINT32_MAX - start - 3;   // a word never written; one of an earlier step
        for (unsigned round = 0; round < 12; round++) {
            const unsigned n = 1 + lengths[round % 8];
            bool restart;
            const unsigned first = numbers.take(n, &restart);
            if (restart) { never = stale = 0; restarts++; }
            for (unsigned k = 0; k < n; k++) {
                const unsigned seq = first + k;
                if (seq == never || seq == stale) { printf("bad: number %u of the call from %u\n", seq, first); return 0; }
            }
            stale = first + n - 1;   // the call's last step reports
        }
    }
    TsNumbers longest;
    longest.next = 0x90000000u;
    bool restart;
    if (longest.take(0x80000000u, &restart) != 1 || !restart || longest.next != 0x80000001u) { printf("bad: longest call\n"); return 0; }
    printf("ok %d\n", restarts);
    return 0;
}
