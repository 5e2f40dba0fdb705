// vx3h_steptile.cpp -- cutting a simulation into tiles for the fused per-step kernel.
//
// A link is computed by the tile that owns its negative end, and again by the tile of its
// positive end when that is another one, so fewer faces between tiles mean less work: a
// body of up to a tile's voxels stays whole (no halo at all), a larger one is cut into
// compact blocks by recursive bisection across the longest lattice extent.  The blocks
// are of at most VX3_TS_CUT voxels, so that the workgroup's last wave has no voxel of its
// own and computes the links that come in across the block's faces.
#include "vx3h_steptile.h"

#include <algorithm>
#include <climits>
#include <cstring>
#include <cstdint>
#include <numeric>

namespace vx3 {
namespace {

struct Item { int v, c[3]; };   // a voxel and its lattice index

struct Cutter {
    const int *lneg, *lpos, *vlinks;
    std::vector<int> mark, count;
    std::vector<Item> aside;
    int epoch = 0;
    std::vector<std::vector<int>> parts;

    int other(int l, int v) const { return lneg[l] == v ? lpos[l] : lneg[l]; }
    // owned + halo slots of a block
    size_t slotsOf(const Item* part, size_t n) {
        const int own = ++epoch, halo = ++epoch;
        for (size_t i = 0; i < n; i++) mark[part[i].v] = own;
        size_t s = n;
        for (size_t i = 0; i < n; i++)
            for (int d = 0; d < 6; d++) {
                const int l = vlinks[6 * (size_t)part[i].v + d];
                if (l < 0) continue;
                const int u = other(l, part[i].v);
                if (mark[u] != own && mark[u] != halo) { mark[u] = halo; s++; }
            }
        return s;
    }
    // Splits part[0, n) across its longest extent at the quantile that leaves each side a whole
    // number of the k blocks meant: the m lowest first, in the order they come (a histogram of
    // the coordinate finds the cut, so a level costs two passes).
    void cut(Item* part, size_t n, int k) {
        if (k <= 1) {
            size_t s = 0;
            if (n <= VX3_TS_CUT && (s = slotsOf(part, n)) <= VX3_TS_SLOTS && s - n <= VX3_TS_OWN) {
                parts.emplace_back(n);
                for (size_t i = 0; i < n; i++) parts.back()[i] = part[i].v;
                return;
            }
            k = 2;   // a single voxel has at most seven slots, so this ends
        }
        int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
        for (size_t i = 0; i < n; i++)
            for (int a = 0; a < 3; a++) {
                lo[a] = std::min(lo[a], part[i].c[a]);
                hi[a] = std::max(hi[a], part[i].c[a]);
            }
        int ax = 0;
        for (int a = 1; a < 3; a++) if (hi[a] - lo[a] > hi[ax] - lo[ax]) ax = a;
        const int kl = k / 2;
        size_t m = (size_t)((double)n * kl / k + 0.5);
        m = std::max<size_t>(1, std::min(m, n - 1));
        count.assign(hi[ax] - lo[ax] + 1, 0);
        for (size_t i = 0; i < n; i++) count[part[i].c[ax] - lo[ax]]++;
        int at = 0;
        size_t below = 0;
        while (below + count[at] < m) below += count[at++];
        size_t ties = m - below, j = 0, r = 0;   // of the voxels at the cut, the first `ties` go below
        at += lo[ax];
        aside.resize(std::max(aside.size(), n));
        for (size_t i = 0; i < n; i++) {
            const int c = part[i].c[ax];
            if (c < at || (c == at && ties > 0)) {
                if (c == at) ties--;
                part[j++] = part[i];
            } else
                aside[r++] = part[i];
        }
        std::copy(aside.begin(), aside.begin() + r, part + j);
        cut(part, m, kl);
        cut(part + m, n - m, k - kl);
    }
};

uint64_t spread(uint64_t x) {   // 21 bits to every third bit
    x &= 0x1fffff;
    x = (x | x << 32) & 0x1f00000000ffffull;
    x = (x | x << 16) & 0x1f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}

}  // namespace

bool planStepTiles(int nv, const int* ijk, int nl, const int* lneg, const int* lpos, const int* vlinks,
                   const char* interior, StepTilePlan* out, long long beside) {
    *out = StepTilePlan();
    if (nv <= 0) return false;
    int low[3];
    for (int a = 0; a < 3; a++) {
        int lo = INT_MAX, hi = INT_MIN;
        for (int v = 0; v < nv; v++) { lo = std::min(lo, ijk[3 * (size_t)v + a]); hi = std::max(hi, ijk[3 * (size_t)v + a]); }
        if ((long long)hi - lo > 0xFFFF) return false;
        low[a] = lo;
    }
    Cutter c;
    c.lneg = lneg; c.lpos = lpos; c.vlinks = vlinks;
    c.mark.assign(nv, 0);
    // connected bodies, one after another in `queue`: body b is queue[first[b], first[b + 1])
    std::vector<char> seen(nv, 0);
    std::vector<int> queue, first;
    queue.reserve(nv);
    for (int v = 0; v < nv; v++) {
        if (seen[v]) continue;
        first.push_back((int)queue.size());
        queue.push_back(v);
        seen[v] = 1;
        for (size_t i = first.back(); i < queue.size(); i++)
            for (int d = 0; d < 6; d++) {
                const int l = vlinks[6 * (size_t)queue[i] + d];
                if (l < 0) continue;
                const int u = c.other(l, queue[i]);
                if (!seen[u]) { seen[u] = 1; queue.push_back(u); }
            }
    }
    first.push_back(nv);
    // small bodies in Morton order of their middle, so that those sharing a tile are close
    std::vector<std::pair<uint64_t, int>> small;
    std::vector<Item> items;
    for (size_t i = 0; i + 1 < first.size(); i++) {
        int* b = queue.data() + first[i];
        const size_t n = first[i + 1] - first[i];
        size_t surface = 0;
        if (n <= VX3_TS_OWN) for (size_t j = 0; j < n; j++) surface += !interior[b[j]];
        if (n > VX3_TS_OWN || surface > VX3_TS_BLOCK) {
            // ascending; a body's voxels mostly have all indices of their range
            int lo = INT_MAX, hi = 0;
            for (size_t j = 0; j < n; j++) { lo = std::min(lo, b[j]); hi = std::max(hi, b[j]); }
            if ((size_t)(hi - lo) < 4 * n) {
                for (size_t j = 0; j < n; j++) seen[b[j]] = 2;
                size_t j = 0;
                for (int v = lo; v <= hi; v++) if (seen[v] == 2) { b[j++] = v; seen[v] = 1; }
            } else std::sort(b, b + n);
            items.resize(n);
            for (size_t j = 0; j < n; j++) items[j] = {b[j], {ijk[3 * (size_t)b[j]], ijk[3 * (size_t)b[j] + 1], ijk[3 * (size_t)b[j] + 2]}};
            c.cut(items.data(), n, (int)((n + VX3_TS_CUT - 1) / VX3_TS_CUT));
            continue;
        }
        uint64_t key = 0;
        for (int a = 0; a < 3; a++) {
            long long s = 0;
            for (size_t j = 0; j < n; j++) s += ijk[3 * (size_t)b[j] + a] - low[a];
            key |= spread((uint64_t)(s / (long long)n)) << a;
        }
        small.push_back({key, (int)i});
    }
    std::sort(small.begin(), small.end());
    // Several of them share a tile while that leaves the chip's 256 compute units about three
    // tiles for two units, a wavefront's voxels at the least, and while they lie close together:
    // a list rebuild looks at everything near the bounds of each wavefront's voxels, and the last
    // tile's rebuild is what a step waits for.  Measured on MI355X, us per step over steps 400 to
    // 800 of balls in one simulation (rebuilt every 8 steps), FP64, radius 2 unless stated:
    //   balls                     670   1000   1500   1500, radius 3   2048, FP32
    //   filled to 256 voxels     63.6      -   80.8            150.2         86.1
    //   1/256 of them, close     25.0   28.1   30.0             51.7         30.6
    //   1/384                    21.5   26.1   28.9             51.8         29.2
    //   1/512                    21.5   37.6   42.3             51.9         41.5
    //   one ball                 21.5      -   43.2             56.5         56.4
    //   per-step kernels         58.8      -   66.7            132.2         64.8
    // close: the box around them, a margin of 2 included, has less than 2.25 times their boxes'
    // volume (1.3 and 1.7 times: up to half as slow again, 3 times: no faster).
    // Many simulations side by side share the units: a tile is also filled to 1/640 of all their
    // voxels.  us per step, by the simulation's own alone and by both, FP64 and FP32 (from 1/384 to
    // 1/512 of all, 20 of 60 cubes of 4^3 are 8 to 12% slower, else it is the same):
    //   60 simulations of 120 cubes of 3^3     169.3  127.0    128.9   96.2
    //   30 of 100 balls of radius 2             79.4   66.7     75.0   71.8
    //   30 of 300 balls of radius 3            306.9  256.1    266.7  200.0
    const long long share = std::max((nv + 383LL) / 384, (nv + beside + 639) / 640);
    const size_t fill = (size_t)std::max(64LL, std::min((long long)VX3_TS_BLOCK, share));
    std::vector<int> open, body(nv, 0);   // (body: of the small ones, in that order)
    long long volumes = 0;   // of the boxes of those in `open`, and the box around them
    int box[2][3] = {};
    auto volume = [](const int (*b)[3]) {
        long long p = 1;
        for (int a = 0; a < 3; a++) p *= b[1][a] - b[0][a] + 5;
        return p;
    };
    for (const auto& k : small) {
        const int *b = queue.data() + first[k.second], *e = queue.data() + first[k.second + 1];
        int own[2][3], both[2][3];
        for (int a = 0; a < 3; a++) {
            own[0][a] = own[1][a] = ijk[3 * (size_t)*b + a];
            for (const int* v = b; v < e; v++) {
                own[0][a] = std::min(own[0][a], ijk[3 * (size_t)*v + a]);
                own[1][a] = std::max(own[1][a], ijk[3 * (size_t)*v + a]);
            }
            both[0][a] = std::min(own[0][a], box[0][a]);
            both[1][a] = std::max(own[1][a], box[1][a]);
        }
        if (!open.empty() && (open.size() + (e - b) > fill || 4 * volume(both) > 9 * (volumes + volume(own)))) {
            c.parts.push_back(open);
            open.clear();
        }
        if (open.empty()) { volumes = 0; memcpy(both, own, sizeof(own)); }
        volumes += volume(own);
        memcpy(box, both, sizeof(box));
        open.insert(open.end(), b, e);
        for (const int* v = b; v < e; v++) body[*v] = (int)(&k - small.data());
    }
    if (!open.empty()) c.parts.push_back(open);

    const int T = (int)c.parts.size();
    if (T > (INT_MAX >> VX3_TS_SLOT_BITS)) return false;
    std::vector<int> place(nv), hslot(nv, -1), touched;
    std::vector<std::pair<uint64_t, int>> keys;
    for (int t = 0; t < T; t++) {
        std::vector<int>& p = c.parts[t];
        // the surface first, body by body: a list rebuild bounds each 64 of a tile's surface voxels
        keys.resize(p.size());
        for (size_t i = 0; i < p.size(); i++) keys[i] = {(uint64_t)(interior[p[i]] != 0) << 32 | (uint32_t)body[p[i]], p[i]};
        std::sort(keys.begin(), keys.end());
        for (size_t i = 0; i < p.size(); i++) p[i] = keys[i].second;
        for (size_t i = 0; i < p.size(); i++) place[p[i]] = t << VX3_TS_SLOT_BITS | (int)i;
    }
    auto tileOf = [&](int v) { return place[v] >> VX3_TS_SLOT_BITS; };
    auto slotOf = [&](int v) { return place[v] & ((1 << VX3_TS_SLOT_BITS) - 1); };
    out->stat.assign((size_t)T * TsStat::ST_END, 0);
    out->tiles.reserve(T);
    for (int t = 0; t < T; t++) {
        const std::vector<int>& p = c.parts[t];
        TsTile d{};
        d.tile = t;
        d.nTiles = T;
        d.nOwn = (int)p.size();
        touched.clear();
        auto haloOf = [&](int u) {
            if (hslot[u] < 0) {
                hslot[u] = d.nOwn + (int)touched.size();
                touched.push_back(u);
            }
            return hslot[u];
        };
        unsigned short* nbr = out->row<unsigned short>(t, TsStat::NBR);
        int* orig = out->row<int>(t, TsStat::ORIG);
        int* link = out->row<int>(t, TsStat::LINK);
        int* in = out->row<int>(t, TsStat::IN);
        unsigned* at = out->row<unsigned>(t, TsStat::IJK);
        std::fill(nbr, nbr + 3 * VX3_TS_OWN, (unsigned short)0xFFFF);
        std::fill(orig, orig + VX3_TS_OWN, -1);
        std::fill(link, link + 3 * VX3_TS_OWN, -1);
        for (int i = 0; i < d.nOwn; i++) {
            const int v = p[i];
            if (!interior[v]) d.nSurf++;
            orig[i] = v;
            const unsigned x = ijk[3 * (size_t)v] - low[0], y = ijk[3 * (size_t)v + 1] - low[1], z = ijk[3 * (size_t)v + 2] - low[2];
            at[2 * i] = x | y << 16;
            at[2 * i + 1] = z | (121 * x + 11 * y + z) << 16;
            for (int a = 0; a < 3; a++) {
                const int l = vlinks[6 * (size_t)v + 2 * a];
                if (l < 0) continue;
                const int u = lpos[l];
                link[a * VX3_TS_OWN + i] = l;
                nbr[a * VX3_TS_OWN + i] = (unsigned short)(tileOf(u) == t ? slotOf(u) : haloOf(u));
            }
        }
        int n = 0;
        for (int a = 0; a < 3; a++) {
            for (int i = 0; i < d.nOwn; i++) {
                const int l = vlinks[6 * (size_t)p[i] + 2 * a + 1];
                if (l < 0 || tileOf(lneg[l]) == t) continue;
                in[n++] = haloOf(lneg[l]) | (i << 16);
                d.nIn[a]++;
            }
        }
        d.nHalo = (int)touched.size();
        int* halo = out->row<int>(t, TsStat::HALO);
        for (int h = 0; h < d.nHalo; h++) { halo[h] = place[touched[h]]; hslot[touched[h]] = -1; }
        out->maxSlots = std::max(out->maxSlots, d.nOwn + d.nHalo);
        out->maxOwn = std::max(out->maxOwn, d.nOwn);
        out->tiles.push_back(d);
    }
    (void)nl;
    return true;
}

}  // namespace vx3
