// vx3_tilestep.inl -- the fused per-step kernel: one launch advances simulations of any
// size by one step.
//
// For simulations too large for the resident kernels (vx3_resident.inl) without topology
// changes or extra forces.  A workgroup owns a tile of a simulation (TsTile): it reads its
// voxels' poses and those of their link partners in other tiles into LDS, computes the
// links, sums the loads and integrates its voxels, all from one copy of the state, and
// writes the other copy; the kernel boundary is the only barrier between tiles.  Against
// the per-step kernels of vx3_kernels.inl this saves, per step,
//   - the round trip of the link end loads through memory (96 bytes per link written, 288
//     per voxel read): a link's negative-end loads stay in the registers of the thread that
//     owns that voxel, its positive-end loads cross LDS, axis by axis;
//   - the small-angle links' angle1v (zero) and what other link state the material does not
//     use, the link's four index words and the contact snapshot (the old copy is one);
//   - all launches but one: collision lists are rebuilt inside the step by the tiles
//     themselves, and the control step is done at the next step's start, by every tile for
//     itself (the same result in each), from what the step's tiles reported.
// A link whose ends two tiles own is computed by both from the same inputs, bit for bit, so
// no loads cross tiles; the tile of its negative end keeps its state.
//
// A step that cannot be taken (a collision table too small: TsReport::grow) or not as a whole
// (a diverged link: its voxels do not move) is only known once every tile has run: the
// control step then leaves the old copy current (SC_TSPARV, SC_TSPARL, SC_TSTOP), so nothing
// has happened, or only the link pass has.  A running simulation's current copies are always
// those of the launch's parity, so a tile reads its state without waiting for the control
// words.
//
// Two sets of partner lists take turns, one from the table's start on and one at its end; where
// both do not fit, the entries of the older set are lost (which shows only where the new one is
// not taken: see listsLost for a table that is too small).
//
// Collision lists (the pair rule of vx3_kernels.inl's k_col_list, the same lists): each tile
// keeps the bounding boxes of its surface voxels, of all and of each wave's 64, as of the last
// rebuild and how far one of them has moved since; at a rebuild a tile walks the simulation's
// boxes, stages the surface voxels of the 64s within reach that lie in reach of its own waves'
// voxels, and each wave tests those in its reach (see tsLists).
//
// Included by the per-precision kernel units after vx3_kernels.inl (VX_NS, real).

namespace vx3 {
namespace VX_NS {

#define VX3_TS_STAGE 320      // staged candidates of a list rebuild
#define VX3_TS_COL 36         // partners of a voxel, and
#define VX3_TS_MORE 512       // further partners of all voxels of a tile, and
#define VX3_TS_IDS 2048       // candidates of a tile, that one walk over the candidates can list
#define VX3_TS_PIECES 512     // pieces of the tiles in reach, of up to 64 surface voxels

typedef TsState<(int)sizeof(real)> TsS;
typedef TsStat TsA;

// LDS of a step: material tables; poses (7 reals, 4 floats, the static word) of S slots; one
// axis' positive-end loads (6 reals and the end strain) of N owned voxels; negative-end loads
// and sums (12 reals, 4 floats) of the owned voxels past the threads' number; halo places.  The
// strides are constants, so that an access is one address register and an offset.
template <int S, int N> struct TsShape {
    static constexpr int X = N > VX3_TS_BLOCK ? N - VX3_TS_BLOCK : 0;
    static constexpr size_t tables = VX3_TS_TAB;
    static_assert(VX3_TS_TAB == VX3_RES_VMATS * sizeof(VoxMatDev) + VX3_RES_LMATS * sizeof(LinkMatDev), "the tables' image");
    static constexpr size_t step = tables + (size_t)S * (7 * sizeof(real) + 20) + (size_t)N * (6 * sizeof(real) + 4) +
                                   (size_t)X * (12 * sizeof(real) + 16) + VX3_TS_OWN * 4;
    // a list rebuild (before the poses are read): nearby masks, the offset table, staged
    // candidates (position, lattice index), all candidates' voxels, partner columns, pieces of
    // tiles in reach
    static constexpr size_t list = (size_t)VX3_TS_BLOCK * VX3_NEAR_WORDS * 4 + 11 * 11 * 11 * 2 + 10 +
                                   (size_t)VX3_TS_STAGE * (3 * sizeof(real) + 8) + VX3_TS_IDS * 4 +
                                   (size_t)VX3_TS_COL * VX3_TS_BLOCK * 2 + (size_t)VX3_TS_PIECES * 4 + VX3_TS_MORE * 4 + VX3_TS_BLOCK / 64 * 128 * 2;
    static constexpr size_t bytes = step > list ? step : list;
};

// values that are the same in every lane, kept in scalar registers
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ unsigned uni(unsigned x) { return (unsigned)__builtin_amdgcn_readfirstlane((int)x); }
__device__ __forceinline__ float uni(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }
__device__ __forceinline__ double uni(double x) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)), __builtin_amdgcn_readfirstlane(__double2loint(x)));
}
// lane k's value, k the same in every lane
__device__ __forceinline__ unsigned lanes(unsigned x, int k) { return (unsigned)__builtin_amdgcn_readlane((int)x, k); }
__device__ __forceinline__ float lanes(float x, int k) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), k)); }
__device__ __forceinline__ double lanes(double x, int k) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), k), __builtin_amdgcn_readlane(__double2loint(x), k));
}
// the launch's tile, field by field in scalar registers
struct TsT {
    int sim, tile, nTiles, rec, nOwn, nSurf, nHalo, nIn0, nIn1, nIn2, ctl, ph0, nPh, o0;
    __device__ __forceinline__ explicit TsT(const TsTile& t)
        : sim(uni(t.sim)), tile(uni(t.tile)), nTiles(uni(t.nTiles)), rec(uni(t.rec)), nOwn(uni(t.nOwn)), nSurf(uni(t.nSurf)),
          nHalo(uni(t.nHalo)), nIn0(uni(t.nIn[0])), nIn1(uni(t.nIn[1])), nIn2(uni(t.nIn[2])), ctl(uni(t.ctl)), ph0(uni(t.ph0)),
          nPh(uni(t.nPh)), o0(uni(t.o0)) {}
};
__device__ __forceinline__ char* tsStat(const TsArgs& ts, int rec) { return ts.stat + (size_t)rec * TsA::BYTES; }
__device__ __forceinline__ char* tsState(const TsArgs& ts, int rec, int copy) { return ts.state + ((size_t)rec * 2 + copy) * TsS::BYTES; }
// row `off` of a record: element i
template <typename E> __device__ __forceinline__ E& row(char* rec, int off, unsigned i) { return *(E*)(rec + off + i * (unsigned)sizeof(E)); }
template <typename E> __device__ __forceinline__ E& lrow(char* rec, int off, unsigned byte) { return *(E*)(rec + off + byte); }

// reports are agent-scope stores: every tile that writes one writes the same value
__device__ __forceinline__ void tsSay(unsigned* word, unsigned seq) { __hip_atomic_store(word, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// A float no smaller than |x| of a displacement x^2 = d2; of a NaN none (such a voxel is nobody's
// partner, and must not make its tile's bounds NaN)
__device__ __forceinline__ float tsReach(real d2) { return d2 >= 0 ? sqrtf((float)d2 * (1.0f + 0x1p-20f)) * (1.0f + 0x1p-20f) : 0.0f; }

// Bounds of the workgroup's surface voxels (mine: this thread's is one) into hull and box of
// parity p, and each wave's into red; empty where there are none.  All widened by *widen (LDS;
// may be written just before).  Synchronizes.
__device__ __forceinline__ void tsBox(TsAux& aux, int p, bool mine, float x, float y, float z, float (*red)[6], const unsigned* widen) {
    constexpr int W = VX3_TS_BLOCK / 64;
    const float inf = __builtin_inff();
    float m[6] = {mine ? x : inf, mine ? y : inf, mine ? z : inf, mine ? -x : inf, mine ? -y : inf, mine ? -z : inf};
#pragma unroll
    for (int k = 0; k < 6; k++) {
        for (int o = 32; o > 0; o >>= 1) m[k] = fminf(m[k], __shfl_xor(m[k], o, 64));
        if (k >= 3) m[k] = -m[k];
    }
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < 6; k++) red[threadIdx.x >> 6][k] = m[k];
    __syncthreads();
    const int k = threadIdx.x % 6;
    auto wider = [&](float e) {
        if (!widen) return e;
        const float m = __uint_as_float(*widen) + fabsf(e) * 0x1p-20f;
        return k < 3 ? e - m : e + m;
    };
    if (threadIdx.x < W * 6) aux.box[p][threadIdx.x / 6][k] = wider(red[threadIdx.x / 6][k]);
    if (threadIdx.x < 6) {
        float r = red[0][k];
        for (int w = 1; w < W; w++) r = k < 3 ? fminf(r, red[w][k]) : fmaxf(r, red[w][k]);
        aux.hull[p][k < 3 ? k : k + 1] = wider(r);
    }
    if (threadIdx.x == 6) aux.hull[p][3] = 0;
}

// The control step after a step: c becomes the simulation's control state at the start of the
// next one.  Every thread of the workgroup; the same result in each thread and each tile.
__device__ __forceinline__ void tsAdvance(const DevBatch<real>& b, const TsArgs& ts, const TsT& td, const SimCtl& sc, TsCtl& c,
                                          const TsReport& r, double* sQ, int* sStop) {
    if (c.state != 0 || (c.flags & SC_COL_GROW)) return;
    const unsigned seq = c.seq++;
    const bool sampled = c.sampled != 0;
    c.sampled = 0;
    int f = c.flags;
    if (!(f & SC_TSLOADED)) {   // the load's report: the staleness rule before the call's first step
        f |= SC_TSLOADED;
        if (r.stale == seq || ((f & SC_COLLISIONS) && sc.colInterval > 0 && c.steps % sc.colInterval == 0)) f |= SC_REBUILD;
        c.flags = f;
        return;
    }
    if (r.grow == seq) {   // nothing of that step counts: it is taken again once the host has enlarged the table
        c.flags = f | SC_COL_GROW;
        return;
    }
    c.steps++;
    if ((f & SC_COLLISIONS) && (f & SC_REBUILD) && r.diverged != seq) {   // (its lists come after the links)
        c.rebuilds++;
        f ^= SC_TSTOP;
    }
    f &= ~SC_REBUILD;
    if ((f & SC_COLLISIONS) && (r.stale == seq || (sc.colInterval > 0 && c.steps % sc.colInterval == 0))) f |= SC_REBUILD;
    f ^= SC_TSPARL;
    if (r.diverged == seq) {   // doTimeStep returns before the voxel loop
        c.flags = f | SC_DIVERGED_PENDING;
        c.state = 2;
        return;
    }
    c.flags = f ^ SC_TSPARV;
    if (sampled) {   // the tiles' partial sums, in an order that every tile uses
        const TsAux* P = ts.aux + td.rec - td.tile;
        double tot[4];
        for (int k = 0; k < 4; k++) {
            double s = 0;
            for (int t = threadIdx.x & 63; t < td.nTiles; t += 64) s += P[t].part[1 - ts.par][k];
            for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
            tot[k] = s;
        }
        double com[3];
        for (int k = 0; k < 3; k++) com[k] = tot[3] == 0 ? 0.0 : (1.0 / tot[3]) * tot[k];
        comSampled(c, com);
    }
    c.t += (double)sc.dt;
    c.prevDt = sc.dt;
    if (sc.maxSteps > 0 && c.steps >= sc.maxSteps) c.state = 1;
    else if (sc.stopLen > 0) {
        if (threadIdx.x == 0)
            *sStop = mathTreeEval(b.tokens + sc.stopOff, sc.stopLen, c.com[0], c.com[1], c.com[2], (double)sc.hits, c.t, c.recentAngle,
                                  sc.closeness, sc.closePairs, sc.nv, sQ) > 0;
        __syncthreads();
        if (uni(*sStop)) c.state = 1;
    }
}

// Batch arrays -> tile arrays (copy 0), at the start of a call: every simulation of the
// fused kernel that will step.  The staleness rule for the call's first step is evaluated
// here (afterwards at the end of each step).
__global__ void __launch_bounds__(VX3_TS_BLOCK) k_ts_load(DevBatch<real> b, TsArgs ts) {
    const TsT td(ts.tiles[blockIdx.x]);
    const SimCtl& sc = b.sims[td.sim];
    const int flags = uni(sc.flags);
    const int tid = threadIdx.x;
    const bool runs = uni(sc.state) == 0 && !(flags & (SC_COL_GROW | SC_LINKS_DONE));
    if (td.tile == 0 && tid == 0) {
        TsCtl& c = ts.ctl[td.ctl];
        c.t = sc.t; c.recentAngle = sc.recentAngle;
        for (int k = 0; k < 3; k++) { c.com[k] = sc.com[k]; c.comH0[k] = sc.comH0[k]; c.comH1[k] = sc.comH1[k]; }
        c.state = runs ? 0 : -1;   // -1: not in the tile arrays, every step skips it
        c.steps = sc.steps; c.flags = flags & ~(SC_TSLOADED | SC_TSPARV | SC_TSPARL);
        c.angleSamples = sc.angleSamples; c.rebuilds = sc.rebuilds;
        c.prevDt = sc.prevDt;
        c.seq = ts.seq0;
        c.sampled = 0;
        ts.report[td.ctl].nbUsed = 0;   // the first step's; each step clears the next one's
    }
    if (!runs) return;
    __shared__ unsigned sMoved;
    if (tid == 0) sMoved = 0;
    __syncthreads();
    char *const A = tsStat(ts, td.rec), *const C = tsState(ts, td.rec, 0), *const Q = A + (flags & SC_TSTOP ? TsA::LISTS : 0);
    float x = 0, y = 0, z = 0;
    const bool surf = tid < td.nSurf, col = (flags & SC_COLLISIONS) != 0;
    for (int i = tid; i < td.nOwn; i += VX3_TS_BLOCK) {
        const int g = row<int>(A, TsA::ORIG, i);
        const real* src[13] = {b.px, b.py, b.pz, b.ow, b.ox, b.oy, b.oz, b.mx, b.my, b.mz, b.ax, b.ay, b.az};
#pragma unroll
        for (int k = 0; k < 13; k++) row<real>(C, TsS::VR + k * TsS::RR, i) = src[k][g];
        const float* srf[4] = {b.tfac, b.psx, b.psy, b.psz};
#pragma unroll
        for (int k = 0; k < 4; k++) row<float>(C, TsS::VF + k * TsS::R4, i) = srf[k][g];
        row<int>(C, TsS::VI, i) = b.vflags[g];
        if (!col || i >= td.nSurf) continue;   // (a tile has at most one surface voxel per thread)
        x = (float)b.px[g]; y = (float)b.py[g]; z = (float)b.pz[g];
        const float w[3] = {b.lastWatch[3 * g], b.lastWatch[3 * g + 1], b.lastWatch[3 * g + 2]};
#pragma unroll
        for (int k = 0; k < 3; k++) row<float>(Q, TsA::LW + k * TsA::R4, i) = w[k];
        row<int>(Q, TsA::NBC, i) = b.nbCount[g];
        row<int>(Q, TsA::NBS, i) = b.nbStart[g];
        if (flags & SC_REBUILD) continue;
        const real dx = b.px[g] - (real)w[0], dy = b.py[g] - (real)w[1], dz = b.pz[g] - (real)w[2];
        const real d2 = dx * dx + dy * dy + dz * dz;
        if (d2 > (real)sc.colRecalcSq) tsSay(&ts.report[ts.ctlCap + td.ctl].stale, ts.seq0);
        atomicMax(&sMoved, __float_as_uint(tsReach(d2)));
    }
    for (int i = tid; i < td.nOwn; i += VX3_TS_BLOCK) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const int g = row<int>(A, TsA::LINK + a * TsA::R4, i);
            if (g < 0) continue;
            const real* src[9] = {b.q2x, b.q2y, b.q2z, b.a2x, b.a2y, b.a2z, b.a1x, b.a1y, b.a1z};
#pragma unroll
            for (int k = 0; k < 9; k++) row<real>(C, TsS::LR + (9 * a + k) * TsS::RR, i) = src[k][g];
            row<float>(C, TsS::LF + 2 * a * TsS::R4, i) = b.maxStrain[g];
            row<float>(C, TsS::LF + (2 * a + 1) * TsS::R4, i) = b.strainOffset[g];
            row<unsigned char>(C, TsS::LB + a * VX3_TS_OWN, i) = (unsigned char)b.lflags[g];
            row<float>(C, TsS::LS + a * TsS::R4, i) = b.strain[g];
        }
    }
    if (col) {
        // the box of the present positions, widened by how far they are from those of the last
        // rebuild: later displacements are measured from there
        __shared__ float red[VX3_TS_BLOCK / 64][6];
        tsBox(ts.aux[td.rec], 0, surf, x, y, z, red, &sMoved);
    }
}

// Tile arrays -> batch arrays, at the end of a call (the simulations k_ts_load took), after
// the last step's control step.
__global__ void __launch_bounds__(VX3_TS_BLOCK) k_ts_store(DevBatch<real> b, TsArgs ts) {
    __shared__ double sQ[VX3_DEV_MT_MAX + 1];
    __shared__ int sStop;
    const TsT td(ts.tiles[blockIdx.x]);
    SimCtl& sc = b.sims[td.sim];
    TsCtl c = ts.ctl[ts.par * ts.ctlCap + td.ctl];
    if (c.state < 0) return;
    tsAdvance(b, ts, td, sc, c, ts.report[(1 - ts.par) * ts.ctlCap + td.ctl], sQ, &sStop);
    const int tid = threadIdx.x;
    char *const A = tsStat(ts, td.rec), *const V = tsState(ts, td.rec, (c.flags & SC_TSPARV) != 0),
         *const L = tsState(ts, td.rec, (c.flags & SC_TSPARL) != 0), *const Q = A + (c.flags & SC_TSTOP ? TsA::LISTS : 0);
    const bool col = (c.flags & SC_COLLISIONS) != 0;
    for (int i = tid; i < td.nOwn; i += VX3_TS_BLOCK) {
        const int g = row<int>(A, TsA::ORIG, i);
        real* dst[13] = {b.px, b.py, b.pz, b.ow, b.ox, b.oy, b.oz, b.mx, b.my, b.mz, b.ax, b.ay, b.az};
#pragma unroll
        for (int k = 0; k < 13; k++) dst[k][g] = row<real>(V, TsS::VR + k * TsS::RR, i);
        float* dsf[4] = {b.tfac, b.psx, b.psy, b.psz};
#pragma unroll
        for (int k = 0; k < 4; k++) dsf[k][g] = row<float>(V, TsS::VF + k * TsS::R4, i);
        b.vflags[g] = row<int>(V, TsS::VI, i);
        if (!col || i >= td.nSurf) continue;
#pragma unroll
        for (int k = 0; k < 3; k++) b.lastWatch[3 * g + k] = row<float>(Q, TsA::LW + k * TsA::R4, i);
        b.nbCount[g] = row<int>(Q, TsA::NBC, i);
        b.nbStart[g] = row<int>(Q, TsA::NBS, i);
    }
    for (int i = tid; i < td.nOwn; i += VX3_TS_BLOCK) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const int g = row<int>(A, TsA::LINK + a * TsA::R4, i);
            if (g < 0) continue;
            const int lb = row<unsigned char>(L, TsS::LB + a * VX3_TS_OWN, i);
            const bool small = (lb & LF_SMALL_ANGLE) != 0;   // angle1v is zero in the small-angle frame
            real* dst[9] = {b.q2x, b.q2y, b.q2z, b.a2x, b.a2y, b.a2z, b.a1x, b.a1y, b.a1z};
#pragma unroll
            for (int k = 0; k < 9; k++) dst[k][g] = k >= 6 && small ? (real)0 : row<real>(L, TsS::LR + (9 * a + k) * TsS::RR, i);
            b.maxStrain[g] = row<float>(L, TsS::LF + 2 * a * TsS::R4, i);
            if (!b.lmatTab[b.lmeta[g] >> 2].linear) b.strainOffset[g] = row<float>(L, TsS::LF + (2 * a + 1) * TsS::R4, i);
            b.lflags[g] = lb;
            b.strain[g] = row<float>(L, TsS::LS + a * TsS::R4, i);
        }
    }
    if (td.tile == 0 && tid == 0) {   // the other tiles read no field that changes here
        sc.t = c.t; sc.recentAngle = c.recentAngle;
        for (int k = 0; k < 3; k++) { sc.com[k] = c.com[k]; sc.comH0[k] = c.comH0[k]; sc.comH1[k] = c.comH1[k]; }
        sc.steps = c.steps; sc.angleSamples = c.angleSamples; sc.rebuilds = c.rebuilds;
        sc.prevDt = c.prevDt;
        sc.flags = c.flags & ~(SC_TSLOADED | SC_TSPARV | SC_TSPARL);
        sc.state = c.state;
    }
}

// contact force of one voxel from its partner list, from the old copy of the state
struct TsContacts {
    const DevBatch<real>* b;
    const TsArgs* ts;
    const VoxMatDev* vm;      // LDS table
    const int* o2p;           // of the simulation: place of each sim-local voxel
    int v, v0, start, count, mat;
    real x, y, z, mx, my, mz, nom;
    float tf;
    // Partners whose loads are in flight together, those apart left after their distance.  FP32,
    // 300 balls with 17,800 pairs: 33 us a step, 45 one at a time and every pair computed.  FP64:
    // either takes registers that spill outside this loop too (2,048 balls 147 us, 141 without).
    static constexpr int AT_ONCE = sizeof(real) == 8 ? 1 : 4;
    template <typename T> __device__ __forceinline__ void subtract(V3<T>& force) const {
#pragma unroll 1
        for (int k0 = 0; k0 < count; k0 += AT_ONCE) {   // (past the last: the last again, left out)
            int us[AT_ONCE], qs[AT_ONCE];
            real px[AT_ONCE], py[AT_ONCE], pz[AT_ONCE];
            float tfs[AT_ONCE];
#pragma unroll
            for (int i = 0; i < AT_ONCE; i++) us[i] = b->nbList[start + (k0 + i < count ? k0 + i : count - 1)];
#pragma unroll
            for (int i = 0; i < AT_ONCE; i++) qs[i] = o2p[us[i] - v0];
#pragma unroll
            for (int i = 0; i < AT_ONCE; i++) {
                char* C = tsState(*ts, qs[i] >> VX3_TS_SLOT_BITS, ts->par);
                const int s = qs[i] & ((1 << VX3_TS_SLOT_BITS) - 1);
                px[i] = row<real>(C, TsS::VR, s); py[i] = row<real>(C, TsS::VR + TsS::RR, s); pz[i] = row<real>(C, TsS::VR + 2 * TsS::RR, s);
                tfs[i] = row<float>(C, TsS::VF, s);
            }
#pragma unroll
            for (int i = 0; i < AT_ONCE; i++) {
                if (AT_ONCE > 1 && (k0 + i >= count || pairApart(x, y, z, px[i], py[i], pz[i], tf, tfs[i], nom))) continue;
                const int u = us[i], rec = qs[i] >> VX3_TS_SLOT_BITS, s = qs[i] & ((1 << VX3_TS_SLOT_BITS) - 1);
                char* C = tsState(*ts, rec, ts->par);
                const real ux = px[i], uy = py[i], uz = pz[i];
                const real nx = row<real>(C, TsS::VR + 7 * TsS::RR, s), ny = row<real>(C, TsS::VR + 8 * TsS::RR, s),
                           nz = row<real>(C, TsS::VR + 9 * TsS::RR, s);
                const float tu = tfs[i];
                const VoxMatDev& mu = vm[row<unsigned>(tsStat(*ts, rec), TsA::ST, s) & 15];
                const VoxMatDev& mv = vm[mat];
                float fx, fy, fz;
                if (v < u)
                    pairContact(mv, mu, x, y, z, ux, uy, uz, mx, my, mz, nx, ny, nz, tf, tu, nom, fx, fy, fz);
                else {
                    pairContact(mu, mv, ux, uy, uz, x, y, z, nx, ny, nz, mx, my, mz, tu, tf, nom, fx, fy, fz);
                    fx = -fx; fy = -fy; fz = -fz;
                }
                force.x -= (T)fx; force.y -= (T)fy; force.z -= (T)fz;
            }
        }
    }
};

// The partner lists of the tile's surface voxels, from the old copy of the state; the whole
// workgroup.  g: the thread's voxel (batch index), mine: it is on the surface.  Returns false
// when the simulation's table is too small (no list is written then).  top: these lists go to the
// table's end and the second rows.  Writes the tile's boxes
// into the new copy.
//
// Bound by instruction issue and LDS latency with one wave per SIMD (the last tile's rebuild
// is what the step waits for), so what is kept small is the number of candidates a wave looks
// at and the instructions for each.  Measured on MI355X, cycles of a tile's rebuild, 300 balls
// of 123 voxels in FP32: 125,000 with every staged candidate tested by every voxel in turn,
// distance and nearby set together; 57,000 with a wave's own reach and the two parts of match.
// Staged candidates sorted into cells and walked voxel by voxel: slower than the first.
__device__ __forceinline__ bool tsLists(const DevBatch<real>& b, const TsArgs& ts, const TsT& td, SimCtl& sc, int* nbUsed, bool top,
                                        bool mine, int g, unsigned char* smem, float (*sReach)[6]) {
    unsigned* sMask = (unsigned*)smem;                                     // [word][thread]
    short* sBit = (short*)(sMask + VX3_NEAR_WORDS * VX3_TS_BLOCK);
    real* sX = (real*)(sBit + 11 * 11 * 11 + 5);   // 16-byte aligned
    uint2* sI = (uint2*)(sX + 3 * VX3_TS_STAGE);                           // [STAGE] lattice index (TsStat::IJK)
    int* sId = (int*)(sI + VX3_TS_STAGE);                                  // [IDS] voxel (batch index) of each candidate so far
    int* sPiece = sId + VX3_TS_IDS;                                        // tile << 9 | piece << 7 | voxels
    unsigned* sMore = (unsigned*)(sPiece + VX3_TS_PIECES);                 // [MORE] thread | candidate << 8: past a thread's column
    unsigned short* sCol = (unsigned short*)(sMore + VX3_TS_MORE);         // [COL][thread] candidates
    unsigned short* sPass = sCol + VX3_TS_COL * VX3_TS_BLOCK + threadIdx.x / 64 * 128;   // [wave][128] staged candidates in its reach
    int* sTile = (int*)sX;                                                 // [PIECES] tiles in reach, while nothing is staged
    static_assert(VX3_TS_PIECES * 4 <= 3 * VX3_TS_STAGE * sizeof(real), "tiles in reach share the stage's place");
    __shared__ int sN, sCand, sNear, sOver, sScan[VX3_TS_BLOCK / 64], sBase;
    __shared__ float sWide[VX3_TS_BLOCK / 64][6];
    const int tid = threadIdx.x;
    const int hops = sc.colNearHops;
    const bool masks = (sc.flags & SC_NEARMASK) != 0;
    char* const A = tsStat(ts, td.rec);
    const TsAux* aux = ts.aux + td.rec - td.tile;   // the simulation's tiles
    real x = 0, y = 0, z = 0;
    uint2 at0 = make_uint2(0, 0);
    auto hopsOf = [&](uint2 w) {   // lattice L1 distance
        return __builtin_amdgcn_sad_u16(w.x, at0.x, __builtin_amdgcn_sad_u16(w.y & 0xFFFF, at0.y & 0xFFFF, 0u));
    };
    if (mine) {
        char* const C = tsState(ts, td.rec, ts.par);
        x = row<real>(C, TsS::VR, tid); y = row<real>(C, TsS::VR + TsS::RR, tid); z = row<real>(C, TsS::VR + 2 * TsS::RR, tid);
        at0 = row<uint2>(A, TsA::IJK, tid);
        if (masks)
            for (int k = 0; k < VX3_NEAR_WORDS; k++) sMask[k * VX3_TS_BLOCK + tid] = b.nearMask[(size_t)k * b.Vcap + g];
    }
    for (int i = tid; i < 11 * 11 * 11; i += VX3_TS_BLOCK) sBit[i] = kNearBits.bit[i];
    // reach of each wave's voxels and of the tile: their box now and the watch radius, widened by
    // more than the boxes' float rounding (2^-24 of each coordinate) can explain, so that no
    // watched pair is missed
    tsBox(ts.aux[td.rec], 1 - ts.par, mine, (float)x, (float)y, (float)z, sReach, nullptr);
    // inside a body: no lists (FP32 cube of 192^3, rebuilt every 8 steps: 2,207 -> 1,731 us a step)
    if (td.nSurf == 0) return true;
    if (tid < VX3_TS_BLOCK / 64 * 6) {
        const int w = tid / 6, a = tid % 3;
        const float r = sqrtf(sc.colThreshSq) * (1.0f + 0x1p-20f);
        const float l = sReach[w][a], h = sReach[w][3 + a];
        const float e = l <= h ? r + (fmaxf(fabsf(l), fabsf(h)) + r) * 0x1p-20f : 0.0f;
        sWide[w][tid % 6] = tid % 6 < 3 ? l - e : h + e;   // (of no voxels: stays empty, +inf and -inf)
    }
    __syncthreads();
    const int lane = tid & 63;
    float own[6], all6[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
        own[k] = uni(sWide[tid >> 6][k]);
        float m = sWide[0][k];
        for (int w = 1; w < VX3_TS_BLOCK / 64; w++) m = k < 3 ? fminf(m, sWide[w][k]) : fmaxf(m, sWide[w][k]);
        all6[k] = uni(m);
    }
    auto within = [](const float* o, float fx, float fy, float fz) {
        return (fx >= o[0]) & (fx <= o[3]) & (fy >= o[1]) & (fy <= o[4]) & (fz >= o[2]) & (fz <= o[5]);
    };
    const real thresh = (real)sc.colThreshSq;
    int n = 0, from = 0;
    int* out = nullptr;   // second walk: the list's place in the table
    int before = 0;       // candidates staged before the present stage
    // `have` candidates (stage entries in the wave's list) against the wave's voxels.  A lane
    // holds one candidate in registers and the others read it from there: first the near ones of
    // each voxel, then, four at a time, these without itself and its nearby ones, in the list's
    // order.  (One wave per SIMD: instructions count, so neither part branches within a voxel.)
    auto match = [&](int have, auto f) {
        const int c = lane < have ? sPass[lane] : 0;
        const real cx = sX[c], cy = sX[VX3_TS_STAGE + c], cz = sX[2 * VX3_TS_STAGE + c];
        const uint2 cw = sI[c];
        unsigned near[2] = {0, 0};   // the first in the highest bit
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const int left = have - 32 * half < 32 ? have - 32 * half : 32;
            if (left <= 0) continue;
            unsigned w = 0;
            int i = 0;
#pragma unroll 1
            for (; i < left; i += 4)   // (entries past the last: of the first one; dropped below)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int k = 32 * half + i + q;
                    const real dx = x - lanes(cx, k), dy = y - lanes(cy, k), dz = z - lanes(cz, k);
                    w = w + w + (unsigned)(dx * dx + dy * dy + dz * dz <= thresh);   // (a NaN is near nothing)
                }
            near[half] = mine ? (w << (32 - i)) & (0xFFFFFFFFu << (32 - left)) : 0u;
        }
#pragma unroll 1
        for (int half = 0; half < 2; half++) {
            unsigned n = half ? near[1] : near[0];
            while (__any(n != 0)) {   // (every lane stays: the others read its candidate)
                unsigned is[4], l1[4], code[4];
                int k[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int p = __clz((int)n) & 31;   // (of 0: any lane's)
                    is[q] = n != 0;
                    n &= ~(0x80000000u >> p);
                    k[q] = __shfl(c, 32 * half + p, 64);
                    const uint2 w = make_uint2(__shfl(cw.x, 32 * half + p, 64), __shfl(cw.y, 32 * half + p, 64));
                    l1[q] = hopsOf(w);
                    code[q] = w.y >> 16;
                }
                // the nearby ones are within the hop radius, so (with masks) within the table's
                // offsets, whose index is the difference of the linear codes
#pragma unroll
                for (int q = 0; q < 4; q++) is[q] &= (unsigned)(l1[q] != 0);
                if (masks) {
                    int bit[4];
#pragma unroll
                    for (int q = 0; q < 4; q++)   // (index 0, offset (-5, -5, -5): no bit)
                        bit[q] = sBit[l1[q] <= (unsigned)hops ? (code[q] - (at0.y >> 16) + 665u) & 0xFFFFu : 0u];
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const unsigned w = sMask[(bit[q] < 0 ? 0 : bit[q] >> 5) * VX3_TS_BLOCK + tid];
                        is[q] &= bit[q] < 0 ? 1u : ~(w >> (bit[q] & 31));
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (!(is[q] & 1u)) continue;
                    const int id = (before + k[q]) & (VX3_TS_IDS - 1), u = sId[id];   // (the present stage's are always there)
                    if (!masks && l1[q] <= (unsigned)hops && nearbyOf(b, sc, g, u)) continue;
                    f(id, u);
                }
            }
        }
    };
    // the m staged candidates: those within the wave's reach, 64 at a time
    auto test = [&](int m, auto f) {
        int have = 0;
        for (int c0 = 0; c0 < m; c0 += 64) {
            const int c = c0 + lane;   // (entries past m: of an older stage, or of none; not used)
            const bool in = c < m && within(own, (float)sX[c], (float)sX[VX3_TS_STAGE + c], (float)sX[2 * VX3_TS_STAGE + c]);
            const unsigned long long some = __ballot(in);
            if (in) sPass[have + __popcll(some & ((1ull << lane) - 1))] = (unsigned short)c;
            have += __popcll(some);
            __builtin_amdgcn_wave_barrier();   // (a wave's LDS accesses are done in order)
            while (have >= 64 || (have > 0 && c0 + 64 >= m)) {
                match(have < 64 ? have : 64, f);
                have -= 64;
                __builtin_amdgcn_wave_barrier();
                if (lane < have) sPass[lane] = sPass[64 + lane];
                __builtin_amdgcn_wave_barrier();
            }
        }
    };
    struct Cand { real x, y, z; uint2 ijk; int id; bool is; };
    // every watched partner of the thread's voxel: f(place in sId, partner).  The 64s in reach are
    // read one per wave and round, those of their voxels within a wave's reach are staged, and
    // full stages are tested.
    auto walk = [&](auto f) {
        if (tid == 0) sN = 0;
        before = 0;
        constexpr int W = VX3_TS_BLOCK / 64, AT_ONCE = 4;
        // another tile's bounds are of its last rebuild: widened by how far its voxels moved (of no
        // voxels, +inf and -inf: NaN, which meets nothing)
        auto wider = [](float* e, float m) {
#pragma unroll
            for (int k = 0; k < 6; k++) {
                const float s = m + fabsf(e[k]) * 0x1p-20f;
                e[k] += k < 3 ? -s : s;
            }
        };
        auto meets = [](const float* e, const float* o) {
            bool in = true;
#pragma unroll
            for (int k = 0; k < 3; k++) in &= (e[k] <= o[3 + k]) & (e[3 + k] >= o[k]);
            return in;
        };
        // the pieces in reach of tiles [tA, tB): up to 64 surface voxels each
        auto gather = [&](int tA, int tB) {
            __syncthreads();
            if (tid == 0) { sCand = 0; sNear = 0; }
            __syncthreads();
            for (int t0 = tA; t0 < tB; t0 += AT_ONCE * VX3_TS_BLOCK) {
                float4 h[AT_ONCE][2];
#pragma unroll
                for (int q = 0; q < AT_ONCE; q++) {
                    const int t = t0 + q * VX3_TS_BLOCK + tid;
                    if (t >= tB) continue;
                    const float4* o = (const float4*)aux[t].hull[ts.par];
                    h[q][0] = o[0]; h[q][1] = o[1];
                }
#pragma unroll
                for (int q = 0; q < AT_ONCE; q++) {
                    const int t = t0 + q * VX3_TS_BLOCK + tid;
                    if (t >= tB) continue;
                    float e[6] = {h[q][0].x, h[q][0].y, h[q][0].z, h[q][1].x, h[q][1].y, h[q][1].z};
                    wider(e, h[q][0].w);
                    if (!meets(e, all6)) continue;
                    const int at = atomicAdd(&sNear, 1);
                    if (at < VX3_TS_PIECES) sTile[at] = t;
                }
            }
            __syncthreads();
            const int tiles = sNear < VX3_TS_PIECES ? sNear : VX3_TS_PIECES;
            for (int i = tid; i < tiles * W; i += VX3_TS_BLOCK) {
                const int t = sTile[i / W], p = i % W, left = ts.tiles[blockIdx.x - td.tile + t].nSurf - p * 64;
                float e[6];
#pragma unroll
                for (int k = 0; k < 6; k++) e[k] = aux[t].box[ts.par][p][k];
                wider(e, aux[t].hull[ts.par][3]);
                bool in = false;
#pragma unroll
                for (int w = 0; w < W; w++) in |= meets(e, sWide[w]);
                if (!in || left <= 0) continue;
                const int at = atomicAdd(&sCand, 1);
                if (at < VX3_TS_PIECES) sPiece[at] = t << 9 | p << 7 | (left < 64 ? left : 64);
            }
            __syncthreads();
        };
        gather(0, td.nTiles);
        // all of them at once, or where they do not fit, those of a few tiles at a time
        const bool all = sNear <= VX3_TS_PIECES && sCand <= VX3_TS_PIECES;
        constexpr int some4 = VX3_TS_PIECES / W;
        for (int t0 = 0; t0 < td.nTiles; t0 += all ? td.nTiles : some4) {
            if (!all) gather(t0, t0 + some4 < td.nTiles ? t0 + some4 : td.nTiles);
            const int pieces = sCand;
            auto fetch = [&](int piece, Cand& c) {
                c.is = false;
                if (piece >= pieces) return;
                const int w = sPiece[piece], rec = td.rec - td.tile + (w >> 9), j = (w >> 7 & 3) * 64 + lane;
                if (lane >= (w & 127)) return;
                char *const C = tsState(ts, rec, ts.par), *const U = tsStat(ts, rec);
                c.x = row<real>(C, TsS::VR, j); c.y = row<real>(C, TsS::VR + TsS::RR, j); c.z = row<real>(C, TsS::VR + 2 * TsS::RR, j);
                c.ijk = row<uint2>(U, TsA::IJK, j);
                c.id = row<int>(U, TsA::ORIG, j);
                c.is = true;
            };
            Cand cur, next;
            fetch(tid >> 6, cur);
            for (int p0 = 0; p0 < pieces; p0 += W) {
                const float fx = (float)cur.x, fy = (float)cur.y, fz = (float)cur.z;
                bool in = false;
                if (cur.is && within(all6, fx, fy, fz))
#pragma unroll
                    for (int w = 0; w < W; w++) in |= within(sWide[w], fx, fy, fz);
                fetch(p0 + VX3_TS_BLOCK / 64 + (tid >> 6), next);
                const unsigned long long some = __ballot(in);
                int k = 0;
                if (lane == 0 && some) k = atomicAdd(&sN, __popcll(some));   // fits: the stage is emptied below before it could not
                k = uni(k) + __popcll(some & ((1ull << lane) - 1));
                if (in) {
                    sX[k] = cur.x; sX[VX3_TS_STAGE + k] = cur.y; sX[2 * VX3_TS_STAGE + k] = cur.z;
                    sI[k] = cur.ijk;
                    sId[(before + k) & (VX3_TS_IDS - 1)] = cur.id;
                }
                cur = next;
                __syncthreads();
                const int m = sN;
                __syncthreads();   // every thread has read the count: the next round may add to it
                // all of them, or another round's might not fit
                if (m > VX3_TS_STAGE - VX3_TS_BLOCK || p0 + W >= pieces) {
                    test(m, f);
                    __syncthreads();
                    if (tid == 0) sN = 0;
                    before += m;
                    __syncthreads();
                }
            }
        }
    };
    if (tid == 0) sOver = 0;   // (walk synchronizes before its first test)
    bool again = false;
    int m = 0;
    auto take = [&](int at, int u) {
        if (again) { out[m++] = u; return; }
        if (n < VX3_TS_COL) sCol[n * VX3_TS_BLOCK + tid] = (unsigned short)at;
        else {
            const int k = atomicAdd(&sOver, 1);
            if (k < VX3_TS_MORE) sMore[k] = (unsigned)tid | (unsigned)at << 8;
        }
        n++;
    };
    // (one loop, not two calls: the walk is most of the kernel's code)
    for (;;) {
        walk(take);
        if (again) break;
        int total;
        const int off = resBlockScan<VX3_TS_BLOCK>(n, sScan, &total);
        if (tid == 0) {
            int at = total ? atomicAdd(nbUsed, total) : 0;
            if (at + total > sc.nbCap) {
                atomicMax(&sc.nbNeed, at + total);
                at = -1;
            }
            sBase = at < 0 || !top ? at : sc.nbCap - at - total;
        }
        __syncthreads();
        if (sBase < 0) return false;
        from = sc.nb0 + sBase + off;
        out = b.nbList + from;
        const int more = sOver;
        again = before > VX3_TS_IDS || more > VX3_TS_MORE;
        if (again) {   // lists that one walk cannot hold: walked once more, straight into the table
            __syncthreads();
            continue;
        }
        if (mine) {   // ascending partner order
            const int kept = n < VX3_TS_COL ? n : VX3_TS_COL;
            for (int i = 1; i < kept; i++) {
                const unsigned short c = sCol[i * VX3_TS_BLOCK + tid];
                const int u = sId[c];
                int j = i - 1;
                while (j >= 0) {
                    const unsigned short d = sCol[j * VX3_TS_BLOCK + tid];
                    if (sId[d] <= u) break;
                    sCol[(j + 1) * VX3_TS_BLOCK + tid] = d;
                    j--;
                }
                sCol[(j + 1) * VX3_TS_BLOCK + tid] = c;
            }
            // those past the column come in between: the lowest that is not yet written, each time
            int last = -1;
            for (int i = 0, k = 0; k < n;) {
                int next = 0x7FFFFFFF;
                if (k - i < n - kept)
                    for (int q = 0; q < more; q++) {
                        const unsigned w = sMore[q];
                        if ((int)(w & 255) != tid) continue;
                        const int u = sId[w >> 8];
                        if (u > last && u < next) next = u;
                    }
                for (; i < kept; i++) {
                    const int u = sId[sCol[i * VX3_TS_BLOCK + tid]];
                    if (u > next) break;
                    out[k++] = u;
                }
                if (k < n) { out[k++] = next; last = next; }
            }
        }
        break;
    }
    if (mine) {
        char* const Q = A + (top ? TsA::LISTS : 0);
        row<int>(Q, TsA::NBC, tid) = n;
        row<int>(Q, TsA::NBS, tid) = from;
        row<float>(Q, TsA::LW, tid) = (float)x;
        row<float>(Q, TsA::LW + TsA::R4, tid) = (float)y;
        row<float>(Q, TsA::LW + 2 * TsA::R4, tid) = (float)z;
        if (again)
            for (int i = 1; i < n; i++) {
                const int c = out[i];
                int j = i - 1;
                while (j >= 0 && out[j] > c) { out[j + 1] = out[j]; j--; }
                out[j + 1] = c;
            }
    }
    return true;
}

// One step of every simulation in the tile records, one workgroup per tile.
//
// Bound by latency: a workgroup is one chain of dependent loads (tile, state, neighbours; about
// 850 cycles each) and per axis one link's chain of divisions and square roots, with three
// workgroups of four waves on a compute unit to overlap them (registers: 168 for FP64 state,
// and LDS below 53 KB).  Hence 256 threads for up to 288 voxels (five waves would be one
// workgroup per unit), blocks of VX3_TS_CUT = 192 voxels (the fourth wave computes the links
// that come in), strides fixed at compile time (runtime strides spilled scalar registers), and
// loads issued before the control words they do not depend on.  Measured on MI355X, us per step
// in one call of many, per-step kernels -> this kernel:
//   64x64x32 cuboid, FP64, collisions (131,072 voxels)     66 -> 42
//   61x47x7 plate, FP32, collisions                        30 -> 22
//   2,048 balls of 257 voxels, FP64, rebuilt every 8      337 -> 141
//   300 balls of 123 voxels, FP32, rebuilt every 8         62 -> 23
template <int S, int N>
__global__ void __launch_bounds__(VX3_TS_BLOCK) __attribute__((amdgpu_waves_per_eu(3))) k_ts_step(DevBatch<real> b, TsArgs ts) {
    constexpr int X = TsShape<S, N>::X;
    extern __shared__ __align__(16) unsigned char smem[];
    double* const sQ = (double*)smem;   // the stop condition's values: before anything else is in LDS
    __shared__ double sRed[4][VX3_TS_BLOCK / 64];
    __shared__ float sBoxRed[VX3_TS_BLOCK / 64][6];
    __shared__ float sPhT[VX3_RES_PHASES];
    __shared__ float sDm[VX3_RES_VMATS];
    __shared__ int sStop;
    __shared__ unsigned sMoved;
    const int tid = threadIdx.x, par = ts.par;
    const TsT td(ts.tiles[blockIdx.x]);
    const bool own = tid < td.nOwn, surf = tid < td.nSurf;
    char *const A = tsStat(ts, td.rec), *const C = tsState(ts, td.rec, par), *const D = tsState(ts, td.rec, 1 - par);
    // ---- everything whose place the tile alone tells is on its way before the control words
    // are known: the own voxel's pose and links, the halo's places, the tables
    int nb[3] = {0xFFFF, 0xFFFF, 0xFFFF};
    int mask = 0;   // the voxel's flags (its link mask does not change)
    real poseR[7];
    float poseF[4];
    unsigned poseW = 0;
    // the state of a link of axis a: slot i of the record with state T
    auto readLink = [&](char* T, int a, unsigned i, LinkState<real>& ls) {
        char* const R = T + a * (9 * TsS::RR);
        ls.pos2 = V3<real>(row<real>(R, TsS::LR, i), row<real>(R, TsS::LR + TsS::RR, i), row<real>(R, TsS::LR + 2 * TsS::RR, i));
        ls.a2v = V3<real>(row<real>(R, TsS::LR + 3 * TsS::RR, i), row<real>(R, TsS::LR + 4 * TsS::RR, i),
                          row<real>(R, TsS::LR + 5 * TsS::RR, i));
        ls.maxStrain = row<float>(T + a * (2 * TsS::R4), TsS::LF, i);
        ls.flags = row<unsigned char>(T + a * VX3_TS_OWN, TsS::LB, i);
    };
    auto readPose = [&](char* T, char* U, unsigned i) {   // slot i of the record with state T and static part U
#pragma unroll
        for (int k = 0; k < 7; k++) poseR[k] = row<real>(T, TsS::VR + k * TsS::RR, i);
#pragma unroll
        for (int k = 0; k < 4; k++) poseF[k] = row<float>(T, TsS::VF + k * TsS::R4, i);
        poseW = row<unsigned>(U, TsA::ST, i);
    };
    LinkState<real> pre;   // the link that the first round of the next axis starts from
    if (own) {
#pragma unroll
        for (int a = 0; a < 3; a++) nb[a] = row<unsigned short>(A, TsA::NBR + 2 * a * VX3_TS_OWN, tid);
        mask = row<int>(C, TsS::VI, tid);
        readPose(C, A, tid);
        readLink(C, 0, tid, pre);   // (of no link: not used)
    }
    int halo0 = 0;
    if (tid < td.nHalo) halo0 = row<int>(A, TsA::HALO, tid);
    constexpr int TABW = (int)(VX3_TS_TAB / 4), TABN = (TABW + VX3_TS_BLOCK - 1) / VX3_TS_BLOCK;
    const int* const tab = ts.tab + (size_t)td.ctl * TABW;
    int tabW[TABN];
#pragma unroll
    for (int k = 0; k < TABN; k++) tabW[k] = k * VX3_TS_BLOCK + tid < TABW ? tab[k * VX3_TS_BLOCK + tid] : 0;
    // ---- the step before's control step; the result for the next launch
    SimCtl& sc = b.sims[td.sim];
    TsReport* const report = ts.report + par * ts.ctlCap + td.ctl;   // this step's
    int flags;
    unsigned seq;
    double tn;
    float prevDt;
    bool sample;
    {
        TsCtl c = ts.ctl[par * ts.ctlCap + td.ctl];
        const TsReport r = ts.report[(1 - par) * ts.ctlCap + td.ctl];
        c.state = uni(c.state); c.steps = uni(c.steps); c.flags = uni(c.flags); c.seq = uni(c.seq);
        if (c.state >= 0) tsAdvance(b, ts, td, sc, c, r, sQ, &sStop);
        flags = uni(c.flags);
        const int cycleStep = uni(sc.cycleStep);
        const bool runs = c.state == 0 && !(flags & SC_COL_GROW);
        sample = runs && cycleStep > 0 && (c.steps + 1) % cycleStep == 0;
        if (td.tile == 0 && tid == 0) {
            c.sampled = sample;
            ts.ctl[(1 - par) * ts.ctlCap + td.ctl] = c;
            ts.report[(1 - par) * ts.ctlCap + td.ctl].nbUsed = 0;   // the next step's rebuild counts from zero
        }
        if (!runs) return;
        seq = c.seq;
        tn = uni(c.t) + (double)uni(sc.dt);
        prevDt = uni(c.prevDt);
    }
    VoxMatDev* sVM = (VoxMatDev*)smem;
    LinkMatDev* sLM = (LinkMatDev*)(smem + VX3_RES_VMATS * sizeof(VoxMatDev));
    real* sPose = (real*)(smem + TsShape<S, N>::tables);   // [7][S]
    real* sLoad = sPose + 7 * S;                     // [6][N] positive-end loads of one axis
    real* sXn = sLoad + 6 * N;                       // [6][X] negative-end loads, and
    real* sXs = sXn + 6 * X;                         // [6][X] sums, of the owned voxels past the threads' number
    float* sF = (float*)(sXs + 6 * X);               // [4][S] thermal factor, Poisson strain
    float* sEnd = sF + 4 * S;                        // [N] positive-end strain
    float* sXe = sEnd + N;                           // [4][X] negative-end strain, strain sums of the three axes
    unsigned* sSt = (unsigned*)(sXe + 4 * X);        // [S]
    int* sHalo = (int*)(sSt + S);                    // [VX3_TS_OWN] places of the halo voxels
    const bool col = (flags & SC_COLLISIONS) != 0, poisson = (flags & SC_POISSON) != 0, vary = (flags & SC_VARY) != 0;
    const real nom = (real)uni(sc.voxSize);
    const float size = (float)uni(sc.voxSize);
    const float dtf = uni(sc.dt);
    if (tid == 0) sMoved = 0;
    // the lists that this step uses: those at the table's end, or at its start
    const bool top = ((flags & SC_TSTOP) != 0) != (col && (flags & SC_REBUILD));
    if (col && (flags & SC_REBUILD)) {
        if (!tsLists(b, ts, td, sc, &report->nbUsed, top, surf, surf ? row<int>(A, TsA::ORIG, tid) : -1, smem, sBoxRed)) {
            if (tid == 0) tsSay(&report->grow, seq);
            return;   // no tile's step counts
        }
        __syncthreads();   // its LDS is the poses' from here on
    } else if (col && tid < 32) {
        TsAux& x = ts.aux[td.rec];
        if (tid < 24) (&x.box[1 - par][0][0])[tid] = (&x.box[par][0][0])[tid];
        else if (tid != 27) x.hull[1 - par][tid - 24] = x.hull[par][tid - 24];   // ([3]: at the end of the step)
    }
    // ---- poses and tables into LDS
    auto putPose = [&](int slot) {
#pragma unroll
        for (int k = 0; k < 7; k++) sPose[k * S + slot] = poseR[k];
#pragma unroll
        for (int k = 0; k < 4; k++) sF[k * S + slot] = poseF[k];
        sSt[slot] = poseW;
    };
    if (own) putPose(tid);
    for (int h = tid; h < td.nHalo; h += VX3_TS_BLOCK) {
        const int q = h == tid ? halo0 : row<int>(A, TsA::HALO, h), rec = q >> VX3_TS_SLOT_BITS;
        readPose(tsState(ts, rec, par), tsStat(ts, rec), q & ((1 << VX3_TS_SLOT_BITS) - 1));
        putPose(td.nOwn + h);
        sHalo[h] = q;
    }
    if (X > 0 && VX3_TS_BLOCK + tid < td.nOwn) {
        readPose(C, A, VX3_TS_BLOCK + tid);
        putPose(VX3_TS_BLOCK + tid);
    }
#pragma unroll
    for (int k = 0; k < TABN; k++)
        if (k * VX3_TS_BLOCK + tid < TABW) ((int*)smem)[k * VX3_TS_BLOCK + tid] = tabW[k];
    if (vary && tid < td.nPh) sPhT[tid] = actuationTemp(sc.tempAmp, sc.tempPeriod, ts.ph[td.ph0 + tid], tn, (flags & SC_EXPANSION) != 0);
    if (tid < VX3_RES_VMATS) {   // damping multipliers 2*sqrt(m)*zeta/previousDt (VX_Voxel.h:131)
        const VoxMatDev& m = ((const VoxMatDev*)tab)[tid];
        sDm[tid] = 2 * m.sqrtMass * m.zetaInternal / (m.fixed ? 0.0f : prevDt);
    }
    __syncthreads();
    // ---- links, axis by axis, in jobs of one link: the owned voxels' positive-side links (the
    // first VX3_TS_BLOCK each by the thread that owns the voxel), then the links that come in
    // from other tiles; jobs past the threads' number take further rounds, begun at another wave
    // for each axis.  Everything is in the link's frame: a permutation of the components with
    // one sign flip, done when reading LDS.
    V3<real> fs(0, 0, 0), ms(0, 0, 0);
    float st[3] = {0, 0, 0};
    V3<real> fN, mN;
    float eN;
    auto nbOf = [&](int a) { return a == 0 ? nb[0] : a == 1 ? nb[1] : nb[2]; };
    // sums of a voxel's two directions of axis a: negative end (own link), positive end
    auto gather = [&](int a) {
        if (own) {
            float sum = 0;
            if (nbOf(a) != 0xFFFF) {
                fs.add(toAxisOriginal(a, fN));
                ms.add(toAxisOriginal(a, mN));
                sum += eN;
            }
            if (mask & (1 << (VF_LINKMASK_SHIFT + 2 * a + 1))) {
                fs.add(V3<real>(sLoad[tid], sLoad[N + tid], sLoad[2 * N + tid]));
                ms.add(V3<real>(sLoad[3 * N + tid], sLoad[4 * N + tid], sLoad[5 * N + tid]));
                sum += sEnd[tid];
            }
            if (a == 0) st[0] = sum; else if (a == 1) st[1] = sum; else st[2] = sum;
        }
        if constexpr (X > 0) {
            const int v = VX3_TS_BLOCK + tid;
            if (v < td.nOwn) {   // the same for a voxel past the threads' number, sums in LDS
                const int m = row<int>(C, TsS::VI, v);
                float sum = 0;
                real s[6];
#pragma unroll
                for (int k = 0; k < 6; k++) s[k] = a == 0 ? (real)0 : sXs[k * X + tid];
                if (row<unsigned short>(A + 2 * a * VX3_TS_OWN, TsA::NBR, v) != 0xFFFF) {
#pragma unroll
                    for (int k = 0; k < 6; k++) s[k] += sXn[k * X + tid];
                    sum += sXe[tid];
                }
                if (m & (1 << (VF_LINKMASK_SHIFT + 2 * a + 1))) {
#pragma unroll
                    for (int k = 0; k < 6; k++) s[k] += sLoad[k * N + v];
                    sum += sEnd[v];
                }
#pragma unroll
                for (int k = 0; k < 6; k++) sXs[k * X + tid] = s[k];
                sXe[(1 + a) * X + tid] = sum;
            }
        }
    };
    int inAt = 0;
#pragma unroll 1
    for (int a = 0;; a++) {
        const int cy = a == 1 ? 0 : 1, cz = a == 2 ? 0 : 2;   // components read as the frame's y and z (x: a)
        const int t0 = a == 0 ? 1 : 0, t1 = a == 2 ? 1 : 2;   // the two transverse axes, in order
        const int nIn = a == 0 ? td.nIn0 : a == 1 ? td.nIn1 : td.nIn2;
        const int jobs = td.nOwn + nIn;
#pragma unroll 1
        for (int j0 = 0; j0 < jobs; j0 += VX3_TS_BLOCK) {
            const int j = j0 == 0 ? tid : j0 + ((tid - 64 * a) & (VX3_TS_BLOCK - 1));
            int vn = -1, vp = 0;
            bool mine = false;
            LinkState<real> ls;
            char* T = C;         // the record that keeps the link, and its slot there
            unsigned li = j;
            if (j < td.nOwn) {
                vp = j0 == 0 ? nbOf(a) : row<unsigned short>(A + 2 * a * VX3_TS_OWN, TsA::NBR, j);
                if (vp != 0xFFFF) { vn = j; mine = true; }
            } else if (j < jobs) {
                const int e = row<int>(A, TsA::IN, inAt + j - td.nOwn);
                vn = e & 0xFFFF;
                vp = e >> 16;
                const int q = sHalo[vn - td.nOwn];
                T = tsState(ts, q >> VX3_TS_SLOT_BITS, par);
                li = q & ((1 << VX3_TS_SLOT_BITS) - 1);
            }
            if (vn < 0) continue;
            if (j0 == 0 && mine) ls = pre;
            else readLink(T, a, li, ls);
            const unsigned sn = sSt[vn];
            const LinkMatDev& mat = sLM[(sn >> (12 + 4 * a)) & 15];
            const int in_ = sn & 15, ip_ = sSt[vp] & 15;
            const VoxMatDev& mn = sVM[in_];
            const VoxMatDev& mp = sVM[ip_];
            ls.strain = 0;
            ls.strainOffset = 0;
            if (!mat.linear) ls.strainOffset = row<float>(T + a * (2 * TsS::R4), TsS::LF + TsS::R4, li);
            ls.a1v = V3<real>(0, 0, 0);
            if (!(ls.flags & LF_SMALL_ANGLE)) {
                char* const R = T + a * (9 * TsS::RR);
                ls.a1v = V3<real>(row<real>(R, TsS::LR + 6 * TsS::RR, li), row<real>(R, TsS::LR + 7 * TsS::RR, li),
                                  row<real>(R, TsS::LR + 8 * TsS::RR, li));
            }
            V3<real> fn, mn_;
            float en = 0;
            if (mn.fixed && mp.fixed) {   // not computed: its loads are never read, its strain stays zero
                if (mine) ls.strain = row<float>(C + a * TsS::R4, TsS::LS, j);
                if (vp < td.nOwn) sEnd[vp] = 0;
            } else {
                const real restLength = (real)0.5 * (nom * (real)sF[vn] + nom * (real)sF[vp]);
                float area, tss;
                if (mat.nu != 0.0f) {
                    float an, sN, ap, sP;
                    // CVX_Voxel::transverseArea / transverseStrainSum (VX_Voxel.cpp:345-373)
                    auto tr = [&](int v, bool nuZero, float& ar, float& su) {
                        if (nuZero) { ar = size * size; su = 0.0f; return; }
                        const float s0 = sF[(1 + t0) * S + v], s1 = sF[(1 + t1) * S + v];
                        ar = (float)((real)(size * size) * ((real)1 + (real)s0) * ((real)1 + (real)s1));
                        su = s0 + s1;
                    };
                    tr(vn, mn.nu == 0.0f, an, sN);
                    tr(vp, mp.nu == 0.0f, ap, sP);
                    area = 0.5f * (an + ap);
                    tss = 0.5f * (sN + sP);
                } else {
                    area = 0.5f * (size * size + size * size);
                    tss = 0.0f;
                }
                // the frame's components: toAxisX as a choice of LDS arrays and a sign
                auto flip = [](real v, bool f) { return f ? -v : v; };
                const V3<real> d(sPose[a * S + vp] - sPose[a * S + vn],
                                 flip(sPose[cy * S + vp] - sPose[cy * S + vn], a == 1),
                                 flip(sPose[cz * S + vp] - sPose[cz * S + vn], a == 2));
                const Q4<real> oN(sPose[3 * S + vn], sPose[(4 + a) * S + vn], flip(sPose[(4 + cy) * S + vn], a == 1),
                                  flip(sPose[(4 + cz) * S + vn], a == 2));
                const Q4<real> oP(sPose[3 * S + vp], sPose[(4 + a) * S + vp], flip(sPose[(4 + cy) * S + vp], a == 1),
                                  flip(sPose[(4 + cz) * S + vp], a == 2));
                V3<real> fP, mP;
                linkForces<real>(mat, 0, V3<real>(0, 0, 0), oN, d, oP, restLength, area, tss, mat.nu != 0.0f, sDm[in_], sDm[ip_], ls,
                                 fn, mn_, fP, mP);
                // CVX_Link::axialStrain(positiveEnd) (VX_Link.cpp:115-118)
                const float r = mat.strainRatio;
                en = 2.0f * ls.strain / (1.0f + r);
                if (vp < td.nOwn) {   // toAxisOriginal, the same choice when writing
                    sLoad[a * N + vp] = fP.x; sLoad[cy * N + vp] = flip(fP.y, a == 1); sLoad[cz * N + vp] = flip(fP.z, a == 2);
                    sLoad[(3 + a) * N + vp] = mP.x; sLoad[(3 + cy) * N + vp] = flip(mP.y, a == 1);
                    sLoad[(3 + cz) * N + vp] = flip(mP.z, a == 2);
                    sEnd[vp] = 2.0f * ls.strain * r / (1.0f + r);
                }
                if (ls.strain > 100) tsSay(&report->diverged, seq);   // Voxelyze.cpp:265
            }
            if (mine) {
                if (X == 0 || j0 == 0) { fN = fn; mN = mn_; eN = en; }
                else {
                    const int i = j - VX3_TS_BLOCK;
                    const V3<real> f = toAxisOriginal(a, fn), m = toAxisOriginal(a, mn_);
                    sXn[i] = f.x; sXn[X + i] = f.y; sXn[2 * X + i] = f.z;
                    sXn[3 * X + i] = m.x; sXn[4 * X + i] = m.y; sXn[5 * X + i] = m.z;
                    sXe[i] = en;
                }
                char* const R = D + a * (9 * TsS::RR);
                row<real>(R, TsS::LR, j) = ls.pos2.x; row<real>(R, TsS::LR + TsS::RR, j) = ls.pos2.y;
                row<real>(R, TsS::LR + 2 * TsS::RR, j) = ls.pos2.z;
                row<real>(R, TsS::LR + 3 * TsS::RR, j) = ls.a2v.x; row<real>(R, TsS::LR + 4 * TsS::RR, j) = ls.a2v.y;
                row<real>(R, TsS::LR + 5 * TsS::RR, j) = ls.a2v.z;
                if (!(ls.flags & LF_SMALL_ANGLE)) {
                    row<real>(R, TsS::LR + 6 * TsS::RR, j) = ls.a1v.x; row<real>(R, TsS::LR + 7 * TsS::RR, j) = ls.a1v.y;
                    row<real>(R, TsS::LR + 8 * TsS::RR, j) = ls.a1v.z;
                }
                char* const F = D + a * (2 * TsS::R4);
                row<float>(F, TsS::LF, j) = ls.maxStrain;
                if (!mat.linear) row<float>(F, TsS::LF + TsS::R4, j) = ls.strainOffset;
                row<unsigned char>(D + a * VX3_TS_OWN, TsS::LB, j) = (unsigned char)ls.flags;
                row<float>(D + a * TsS::R4, TsS::LS, j) = ls.strain;
            }
        }
        if (a == 2) break;
        inAt += nIn;
        if (own && nbOf(a + 1) != 0xFFFF) readLink(C, a + 1, tid, pre);
        __syncthreads();
        gather(a);
        __syncthreads();   // the next axis overwrites the load buffer
    }
    // ---- voxels: what the links did not need is on its way while the last axis' loads arrive
    V3<real> lm, am;
    float lw[3] = {0, 0, 0};
    int nc = 0;
    auto readRest = [&](int i) {
        lm = V3<real>(row<real>(C, TsS::VR + 7 * TsS::RR, i), row<real>(C, TsS::VR + 8 * TsS::RR, i), row<real>(C, TsS::VR + 9 * TsS::RR, i));
        am = V3<real>(row<real>(C, TsS::VR + 10 * TsS::RR, i), row<real>(C, TsS::VR + 11 * TsS::RR, i),
                      row<real>(C, TsS::VR + 12 * TsS::RR, i));
        nc = 0;
        if (col && i < td.nSurf) {
            char* const Q = A + (top ? TsA::LISTS : 0);
            nc = row<int>(Q, TsA::NBC, i);
#pragma unroll
            for (int k = 0; k < 3; k++) lw[k] = row<float>(Q, TsA::LW + k * TsA::R4, i);
        }
    };
    if (own) readRest(tid);
    __syncthreads();
    gather(2);
    double psx = 0, psy = 0, psz = 0, psm = 0;
#pragma unroll 1
    for (int i = tid; i < td.nOwn; i += VX3_TS_BLOCK) {
        if (X > 0 && i >= VX3_TS_BLOCK) {   // a voxel past the threads' number: its sums are in LDS
            readRest(i);
            fs = V3<real>(sXs[tid], sXs[X + tid], sXs[2 * X + tid]);
            ms = V3<real>(sXs[3 * X + tid], sXs[4 * X + tid], sXs[5 * X + tid]);
#pragma unroll
            for (int a = 0; a < 3; a++) {
                st[a] = sXe[(1 + a) * X + tid];
                nb[a] = row<unsigned short>(A, TsA::NBR + 2 * a * VX3_TS_OWN, i);
            }
            mask = row<int>(C, TsS::VI, i);
        }
        int vf = mask;
        const unsigned w = sSt[i];
        const VoxMatDev& m = sVM[w & 15];
        V3<real> pos(sPose[i], sPose[S + i], sPose[2 * S + i]);
        Q4<real> o(sPose[3 * S + i], sPose[4 * S + i], sPose[5 * S + i], sPose[6 * S + i]);
        const float tf = sF[i];
        const ExtDev* ext = (w >> 10) & 1 ? &b.extTab[b.vext[row<int>(A, TsA::ORIG, i)]] : nullptr;
        if (!m.fixed) {
            int ix = 0, iy = 0, iz = 0;
            if (ext) { ix = ext->ix; iy = ext->iy; iz = ext->iz; }
            TsContacts con{&b, &ts, sVM, nullptr, 0, 0, 0, nc, (int)(w & 15), pos.x, pos.y, pos.z, lm.x, lm.y, lm.z, nom, tf};
            if (nc > 0) {
                con.o2p = ts.o2p + td.o0;
                con.v = row<int>(A, TsA::ORIG, i);
                con.v0 = sc.v0;
                con.start = row<int>(A + (top ? TsA::LISTS : 0), TsA::NBS, i);
            }
            voxelStep<real>(m, ext, dtf, nom, ix, iy, iz, tf, fs, ms, con, pos, lm, o, am, vf);
        }
        const real out[13] = {pos.x, pos.y, pos.z, o.w, o.x, o.y, o.z, lm.x, lm.y, lm.z, am.x, am.y, am.z};
#pragma unroll
        for (int k = 0; k < 13; k++) row<real>(D, TsS::VR + k * TsS::RR, i) = out[k];
        row<int>(D, TsS::VI, i) = vf;
        // VX3 updateTemperature at t + dt (VX3_VoxelyzeKernel.cu:625-650)
        row<float>(D, TsS::VF, i) = vary && !m.fixed && !(m.thermalOnAfter > tn) ? 1 + sPhT[(w >> 4) & 63] * m.alphaCTE : tf;
        float ps[3] = {sF[S + i], sF[2 * S + i], sF[3 * S + i]};
        if (poisson) {   // CVX_Voxel::strain(true) (VX_Voxel.cpp:299-333), see poissonStrain
            bool tension[3];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const int n = (nb[a] != 0xFFFF) + ((vf >> (VF_LINKMASK_SHIFT + 2 * a + 1)) & 1);
                if (n == 2) st[a] *= 0.5f;
                tension[a] = (n == 2) || (ext && (n == 1 && ((ext->dofFixed & (1 << a)) || ext->force[a] != 0)));
            }
            if (!(tension[0] && tension[1] && tension[2])) {
                float add = 0;
#pragma unroll
                for (int a = 0; a < 3; a++) if (tension[a]) add += st[a];
                const float value = poissonValue(1.0f + add, m.nu);
#pragma unroll
                for (int a = 0; a < 3; a++) if (!tension[a]) st[a] = value;
            }
#pragma unroll
            for (int a = 0; a < 3; a++) ps[a] = st[a];
        }
#pragma unroll
        for (int a = 0; a < 3; a++) row<float>(D, TsS::VF + (1 + a) * TsS::R4, i) = ps[a];
        if (col && i < td.nSurf) {   // CVoxelyze::updateCollisions' staleness rule, for the next step
            const real dx = pos.x - (real)lw[0], dy = pos.y - (real)lw[1], dz = pos.z - (real)lw[2];
            const real d2 = dx * dx + dy * dy + dz * dz;
            if (d2 > (real)sc.colRecalcSq) tsSay(&report->stale, seq);
            atomicMax(&sMoved, __float_as_uint(tsReach(d2)));
        }
        if (sample && m.isMeasured) {
            const double mass = m.mass;
            psx += (double)pos.x * mass; psy += (double)pos.y * mass; psz += (double)pos.z * mass;
            psm += mass;
        }
    }
    if (col) {
        __syncthreads();
        if (tid == 0) ts.aux[td.rec].hull[1 - par][3] = __uint_as_float(sMoved);
    }
    if (sample) {   // FP64 center of mass of the measured voxels (VX3_VoxelyzeKernel.cu:477-493)
        for (int o = 32; o > 0; o >>= 1) {
            psx += __shfl_xor(psx, o, 64); psy += __shfl_xor(psy, o, 64);
            psz += __shfl_xor(psz, o, 64); psm += __shfl_xor(psm, o, 64);
        }
        if ((tid & 63) == 0) { sRed[0][tid >> 6] = psx; sRed[1][tid >> 6] = psy; sRed[2][tid >> 6] = psz; sRed[3][tid >> 6] = psm; }
        __syncthreads();
        if (tid < 4) {
            double s = 0;
            for (int w = 0; w < VX3_TS_BLOCK / 64; w++) s += sRed[tid][w];
            ts.aux[td.rec].part[par][tid] = s;
        }
    }
}

}  // namespace VX_NS
}  // namespace vx3
