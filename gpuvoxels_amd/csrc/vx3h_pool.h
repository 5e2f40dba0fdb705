// vx3h_pool.h -- ranges of the device arrays' index spaces (host bookkeeping only).
#ifndef VX3H_POOL_H
#define VX3H_POOL_H
#include <cstddef>
#include <iterator>
#include <map>

namespace vx3 {

// First-fit ranges of an index space that is in use below `hi`.
struct RangeAlloc {
    std::map<int, int> freeRanges;   // start -> length
    int hi = 0;
    int alloc(int n, int cap, bool& grow) {
        grow = false;
        for (auto it = freeRanges.begin(); it != freeRanges.end(); ++it) {
            if (it->second >= n) {
                int s = it->first, len = it->second;
                freeRanges.erase(it);
                if (len > n) freeRanges[s + n] = len - n;
                return s;
            }
        }
        int s = hi;
        hi += n;
        if (hi > cap) grow = true;
        return s;
    }
    void release(int s, int n) {
        if (n <= 0) return;
        freeRanges[s] = n;
        auto it = freeRanges.find(s);
        auto nx = std::next(it);
        if (nx != freeRanges.end() && it->first + it->second == nx->first) { it->second += nx->second; freeRanges.erase(nx); }
        if (it != freeRanges.begin()) {
            auto pv = std::prev(it);
            if (pv->first + pv->second == it->first) { pv->second += it->second; freeRanges.erase(it); it = pv; }
        }
        if (it->first + it->second == hi) { hi = it->first; freeRanges.erase(it); }
    }
};

// A range of n elements of a pool (with members ra and cap) whose arrays grow(pool) enlarges to
// at least ra.hi elements; grow returns 0 or an error.  After an error the pool's ranges are as
// they were: none may lie past the end of its arrays, or a later one there would be taken for
// allocated.
template <typename Pool, typename Grow> auto takeRange(Pool& p, int n, int& start, Grow grow) -> decltype(grow(p)) {
    bool more = false;
    start = p.ra.alloc(n, p.cap, more);
    if (!more) return decltype(grow(p))(0);
    const auto st = grow(p);
    if (st) {
        p.ra.release(start, n);
        start = 0;
    }
    return st;
}

// One range in each of N pools: all of them, or after an error none.
template <size_t N, typename Pool, typename Grow>
auto takeRanges(Pool* const (&p)[N], const int (&n)[N], int* const (&start)[N], Grow grow) -> decltype(grow(*p[0])) {
    for (size_t i = 0; i < N; i++)
        if (const auto st = takeRange(*p[i], n[i], *start[i], grow)) {
            for (; i > 0; i--) p[i - 1]->ra.release(*start[i - 1], n[i - 1]);
            return st;
        }
    return decltype(grow(*p[0]))(0);
}

}  // namespace vx3
#endif
