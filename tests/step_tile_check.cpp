// Checks planStepTiles (gpuvoxels_amd/csrc/vx3h_steptile.cpp) on one simulation's topology
// read from stdin: "nv nl", nv lines "i j k", nl lines "neg pos axis".  Prints "ok <tiles>
// <halo> <incoming>" when every invariant that the fused per-step kernel's indexing relies on
// holds, else "bad <reason>".
#include <cstdio>
#include <vector>

#include "../gpuvoxels_amd/csrc/vx3h_steptile.h"

using namespace vx3;

#define BAD(...) do { printf("bad "); printf(__VA_ARGS__); printf("\n"); return 0; } while (0)

int main() {
    int nv, nl;
    if (scanf("%d %d", &nv, &nl) != 2) BAD("header");
    std::vector<int> ijk(3 * nv), ln(nl), lp(nl), ax(nl), vl(6 * (size_t)nv, -1);
    for (int v = 0; v < nv; v++) if (scanf("%d %d %d", &ijk[3 * v], &ijk[3 * v + 1], &ijk[3 * v + 2]) != 3) BAD("voxel");
    for (int l = 0; l < nl; l++) {
        if (scanf("%d %d %d", &ln[l], &lp[l], &ax[l]) != 3) BAD("link");
        vl[6 * (size_t)ln[l] + 2 * ax[l]] = l;
        vl[6 * (size_t)lp[l] + 2 * ax[l] + 1] = l;
    }
    std::vector<char> interior(nv, 1);
    for (int v = 0; v < nv; v++) for (int d = 0; d < 6; d++) if (vl[6 * (size_t)v + d] < 0) interior[v] = 0;
    StepTilePlan p;
    if (!planStepTiles(nv, ijk.data(), nl, ln.data(), lp.data(), vl.data(), interior.data(), &p)) { printf("none\n"); return 0; }
    const int T = (int)p.tiles.size(), N = VX3_TS_OWN, SLOT = (1 << VX3_TS_SLOT_BITS) - 1;
    if (p.stat.size() != (size_t)T * TsStat::ST_END) BAD("array sizes");
    std::vector<int> slotOf(nv, -1), tileOf(nv, -1), linkAt(nl, -1);
    for (int t = 0; t < T; t++) {
        const TsTile& d = p.tiles[t];
        if (d.tile != t || d.nTiles != T) BAD("tile %d numbering", t);
        if (d.nOwn < 1 || d.nOwn > VX3_TS_OWN || d.nSurf > VX3_TS_BLOCK) BAD("tile %d owns %d, surface %d", t, d.nOwn, d.nSurf);
        if (d.nHalo > VX3_TS_OWN || d.nOwn + d.nHalo > VX3_TS_SLOTS || d.nOwn + d.nHalo > p.maxSlots || d.nOwn > p.maxOwn)
            BAD("tile %d slots %d + %d", t, d.nOwn, d.nHalo);
        if (d.nHalo && d.nOwn > VX3_TS_BLOCK) BAD("tile %d has a halo and voxels past the threads' number", t);
        if (d.nIn[0] + d.nIn[1] + d.nIn[2] > 3 * N) BAD("incoming links of tile %d", t);
        for (int i = 0; i < N; i++) {
            const int v = p.row<int>(t, TsStat::ORIG)[i];
            if ((v >= 0) != (i < d.nOwn)) BAD("padding of tile %d", t);
            if (v < 0) continue;
            if (slotOf[v] >= 0) BAD("voxel %d owned twice", v);
            if ((i < d.nSurf) != !interior[v]) BAD("surface voxels of tile %d are not its first", t);
            slotOf[v] = i;
            tileOf[v] = t;
            const unsigned *w = p.row<unsigned>(t, TsStat::IJK) + 2 * i, *w0 = p.row<unsigned>(tileOf[0] < 0 ? t : tileOf[0], TsStat::IJK) +
                               2 * (tileOf[0] < 0 ? i : slotOf[0]);
            const int r = tileOf[0] < 0 ? v : 0;   // lattice index relative to another voxel's
            const int dx = (int)(w[0] & 0xFFFF) - (int)(w0[0] & 0xFFFF), dy = (int)(w[0] >> 16) - (int)(w0[0] >> 16),
                      dz = (int)(w[1] & 0xFFFF) - (int)(w0[1] & 0xFFFF);
            if (dx != ijk[3 * v] - ijk[3 * r] || dy != ijk[3 * v + 1] - ijk[3 * r + 1] || dz != ijk[3 * v + 2] - ijk[3 * r + 2]) BAD("lattice index");
            if ((((w[1] >> 16) - (w0[1] >> 16)) & 0xFFFF) != (unsigned)((121 * dx + 11 * dy + dz) & 0xFFFF)) BAD("linear code");
        }
    }
    for (int v = 0; v < nv; v++) if (slotOf[v] < 0) BAD("voxel %d owned by none", v);
    long long halo = 0, in = 0;
    for (int t = 0; t < T; t++) {
        const TsTile& d = p.tiles[t];
        auto place = [&](int q) { return p.row<int>(q >> VX3_TS_SLOT_BITS, TsStat::ORIG)[q & SLOT]; };
        auto voxel = [&](int s) {   // voxel of a tile slot
            if (s < d.nOwn) return p.row<int>(t, TsStat::ORIG)[s];
            return s < d.nOwn + d.nHalo ? place(p.row<int>(t, TsStat::HALO)[s - d.nOwn]) : -1;
        };
        for (int h = 0; h < d.nHalo; h++) {
            const int q = p.row<int>(t, TsStat::HALO)[h];
            if (q < 0 || (q >> VX3_TS_SLOT_BITS) >= T || (q >> VX3_TS_SLOT_BITS) == t || (q & SLOT) >= p.tiles[q >> VX3_TS_SLOT_BITS].nOwn) BAD("halo");
        }
        for (int i = 0; i < N; i++)
            for (int a = 0; a < 3; a++) {
                const int v = p.row<int>(t, TsStat::ORIG)[i], l = p.row<int>(t, TsStat::LINK)[a * N + i];
                const int want = v < 0 ? -1 : vl[6 * (size_t)v + 2 * a];
                if (l != want) BAD("link of slot %d axis %d is %d, not %d", i, a, l, want);
                const int nb = p.row<unsigned short>(t, TsStat::NBR)[a * N + i];
                if (l < 0) { if (nb != 0xFFFF) BAD("neighbour without a link"); continue; }
                if (voxel(nb) != lp[l]) BAD("neighbour of slot %d axis %d", i, a);
                linkAt[l] = t;
            }
        int e = 0;
        std::vector<char> seen(nl, 0);
        for (int a = 0; a < 3; a++)
            for (int k = 0; k < d.nIn[a]; k++, e++) {
                const int x = p.row<int>(t, TsStat::IN)[e], hs = x & 0xFFFF, os = x >> 16;
                if (hs < d.nOwn || hs >= d.nOwn + d.nHalo || os >= d.nOwn) BAD("incoming link's slots");
                const int l = vl[6 * (size_t)voxel(os) + 2 * a + 1];
                if (l < 0 || ln[l] != voxel(hs) || seen[l]) BAD("incoming link");
                // its state is in the negative end's record, at that slot and axis
                const int q = p.row<int>(t, TsStat::HALO)[hs - d.nOwn];
                if (p.row<int>(q >> VX3_TS_SLOT_BITS, TsStat::LINK)[a * N + (q & SLOT)] != l) BAD("incoming link's state");
                seen[l] = 1;
            }
        for (int i = 0; i < d.nOwn; i++)
            for (int a = 0; a < 3; a++) {
                const int l = vl[6 * (size_t)voxel(i) + 2 * a + 1];
                if (l >= 0 && tileOf[ln[l]] != t && !seen[l]) BAD("link %d missing from tile %d", l, t);
            }
        halo += d.nHalo;
        in += e;
    }
    for (int l = 0; l < nl; l++) if (linkAt[l] < 0) BAD("link %d kept by none", l);
    printf("ok %d %lld %lld\n", T, halo, in);
    return 0;
}
