// vx3_resident_all.inl -- the one-workgroup kernel for simulations whose links' loads fit LDS
// all at once.
//
// k_resident (vx3_resident.inl) computes the links axis by axis, because the loads of one axis
// are what its load buffer holds: three link passes, three gathers and seven barriers a step,
// in each of which most of a small simulation's threads wait.  Here a link of any axis takes
// any slot, so a step is one link pass over all of them, one gather and the voxel update: two
// barriers, and LPT rounds of links instead of three.  A thread owns one voxel and LPT links
// and keeps their state in registers; the axis of a link is a lane's own, a choice of LDS rows
// and a sign flip when reading poses and writing loads.  The sums of a voxel are taken in the
// same order from the same values, so the results are k_resident's bit for bit.
//
// Tiled (TILED): the tiles of a simulation too large for one workgroup, exactly as k_resident
// runs them (barrier, exchange records, divergence and repair launch are described there), with
// smaller tiles.  A link between owned voxels takes a low slot, so that the wavefronts of the
// low slots compute while the others' tiles arrive, and the links with a halo end follow.
//
// Included by the per-precision kernel units after vx3_resident.inl (VX_NS, real).

namespace vx3 {
namespace VX_NS {

template <int BS, int LPT, int LMAX, bool TILED = false> struct ResidentAllShape {
    static constexpr size_t tables = VX3_RES_VMATS * sizeof(VoxMatDev) + VX3_RES_LMATS * sizeof(LinkMatDev);
    static constexpr size_t bytes = tables + (size_t)BS * (7 * sizeof(real) + 4 * sizeof(float))   // pose; thermal factor, Poisson strain
                                  + (size_t)LMAX * (12 * sizeof(real) + 2 * sizeof(float))         // loads, end strains
                                  + (TILED ? (size_t)BS * 4 : 0);                                  // exchange voxel per slot
    static_assert(LMAX <= BS * LPT, "a slot per thread and round");
    // setup tables alias the load buffer: voxel -> slot per direction, and slot -> link
    static_assert((size_t)BS * 6 * 2 + (size_t)LMAX * 2 <= (size_t)LMAX * 12 * sizeof(real), "setup alias");
};

// Bound by the latency of a step's chain (poses from LDS, one link's divisions and square roots,
// a barrier, six gathers, the voxel update, a barrier), with up to three waves a SIMD in FP64 and
// four in FP32 to overlap it; by instruction issue where those are all full.  A block as wide as
// the links, so that most bodies take one round of them (768 threads is what the 168 registers
// of the FP64 chain leave, 1,024 fit FP32 with some state in scratch); the slots of a second
// round are what LDS leaves.  Measured on MI355X, us per step, k_resident -> this kernel:
//                                   FP64            FP32
//   one cube of 3^3             8.1 -> 4.8      7.1 -> 4.9
//   one cube of 6^3             8.6 -> 6.6      7.5 -> 5.5
//   one cube of 7^3, 9^3       11.1 -> 8.0     11.4 -> 9.7     (two rounds)
//   200 robots on 8^3 grids    12.3 -> 6.1     10.4 -> 5.4
//   200 robots on 10^3 grids   13.5 -> 9.1     10.9 -> 6.8
//   512 robots on 12^3 grids         -         22.3 -> 17.3   (first 3,000 steps; over 8,000, with
//                                              24.7 -> 18.7    ever more links at large angles)
template <int BS, int LPT, int LMAX, bool TILED = false>
__global__ void __launch_bounds__(BS) k_resident_all(DevBatch<real> b, const int* simList, int nSteps, TileArgs ta) {
    typedef ResidentAllShape<BS, LPT, LMAX, TILED> Shape;
    extern __shared__ __align__(16) unsigned char smem[];
    VoxMatDev* sVM = (VoxMatDev*)smem;
    LinkMatDev* sLM = (LinkMatDev*)(smem + VX3_RES_VMATS * sizeof(VoxMatDev));
    real* sP = (real*)(smem + Shape::tables);   // [7][BS] position, orientation
    real* sF = sP + 7 * BS;                     // [12][LMAX] negative-end force, moment, positive-end
    float* sTf = (float*)(sF + 12 * LMAX);
    float* sPs = sTf + BS;                      // [3][BS]
    float* sEs = sPs + 3 * BS;                  // [2][LMAX]
    int* sXv = (int*)(sEs + 2 * LMAX);          // TILED: per slot its exchange record (as in k_resident)
    unsigned short* sVL = (unsigned short*)sF;  // [6][BS] slot of the link in direction d (setup only)
    unsigned short* sSL = sVL + 6 * BS;         // [LMAX] link of a slot (setup only)
    __shared__ int sRun, sDiv;
    __shared__ int sTile;                       // TILED: 1 = some tile diverged this step, 2 = a barrier timed out
    __shared__ double sQ[VX3_DEV_MT_MAX + 1];
    __shared__ double sRed[4][BS / 64];
    __shared__ double sCom[3], sComH0[3], sComH1[3], sAngle;   // center-of-mass history, owned by thread 0
    __shared__ double sPhase[VX3_RES_PHASES];   // distinct actuation phase offsets of the sim
    __shared__ float sPhT[VX3_RES_PHASES];      // their temperatures for the step being run
    __shared__ int sNph;
    __shared__ float sDm[VX3_RES_VMATS];        // CVX_Voxel::dampingMultiplier per voxel material (dt is fixed)
    __shared__ int sScan[BS / 64];

    TileDesc td{};
    if (TILED) td = ta.tiles[blockIdx.x];
    SimCtl& scg = b.sims[TILED ? td.sim : simList[blockIdx.x]];
    const int tid = threadIdx.x;
    int divAt = -1;      // TILED: the launch's step at which a link diverged (a repair launch stops there)
    unsigned gen = 0;    // TILED: barriers passed in this launch
    if (scg.state != 0 || (scg.flags & SC_COL_GROW)) return;
    if (TILED && ta.repair) {   // only simulations whose previous launch saw a divergence run again
        const int dw = ta.sync[td.cOff];
        if (!dw) return;
        divAt = dw - 1;
    }
    const int v0 = scg.v0, l0 = scg.l0;
    // the voxels this workgroup integrates, the LDS pose slots it fills, the links it computes
    const int nv = TILED ? td.nOwn : scg.nv, nvAll = TILED ? td.nOwn + td.nHalo : scg.nv, nl = TILED ? td.nLinks : scg.nl;
    auto gvox = [&](int slot) { return v0 + (TILED ? ta.vox[td.vOff + slot] & 0x7fffffff : slot); };
    auto glink = [&](int j) { return l0 + (TILED ? ta.link[td.lOff + j] & 0x7fffffff : j); };
    // vneg | vpos << 16, as slots
    auto endsOf = [&](int l) { return TILED ? ta.ends[td.lOff + l] : (b.lneg[l0 + l] - v0) | ((b.lpos[l0 + l] - v0) << 16); };
    const double dt = scg.dt;
    const float dtf = scg.dt;
    const real nom = (real)scg.voxSize;
    const float size = (float)scg.voxSize;
    const int flags0 = scg.flags;
    const bool poisson = (flags0 & SC_POISSON) != 0, vary = (flags0 & SC_VARY) != 0, expansion = (flags0 & SC_EXPANSION) != 0;
    const double tempAmp = scg.tempAmp, tempPeriod = scg.tempPeriod;
    const int cycleStep = scg.cycleStep, maxSteps = scg.maxSteps;
    const int stopLen = scg.stopLen, stopOff = scg.stopOff;
    const int mat0 = scg.mat0, nvm = scg.nvm, nlm = scg.nlm;
    const size_t VC = (size_t)b.Vcap;

    // ---- setup: material tables, link slots, voxel -> slot table
    for (int i = 0; i < nvm; i++)
        ldsCopyWords((int*)&sVM[i], (const int*)&b.vmatTab[b.simMats[mat0 + i]], sizeof(VoxMatDev) / 4, tid, BS);
    for (int i = 0; i < nlm; i++)
        ldsCopyWords((int*)&sLM[i], (const int*)&b.lmatTab[b.simMats[mat0 + nvm + i]], sizeof(LinkMatDev) / 4, tid, BS);
    for (int i = tid; i < 6 * BS; i += BS) sVL[i] = 0xFFFF;
    // the lowest slots: the links that took the expensive branches last step (see k_resident);
    // TILED, those between owned voxels, which do not wait for the other tiles.  The others after
    // them, each in link order.
    auto early = [&](int l) {
        if (TILED) {
            const int e = endsOf(l);
            return (e & 0xFFFF) < nv && (e >> 16) < nv;
        }
        const int g = l0 + l;
        const real x = b.a2x[g], y = b.a2y[g], z = b.a2z[g];
        return !(b.lflags[g] & LF_SMALL_ANGLE) || x * x + y * y + z * z > (real)0.009;
    };
    int mine = 0;
#pragma unroll
    for (int k = 0; k < LPT; k++) {
        const int l = tid * LPT + k;
        if (l < nl && early(l)) mine++;
    }
    int nEarly;
    int at = resBlockScan<BS>(mine, sScan, &nEarly);
#pragma unroll
    for (int k = 0; k < LPT; k++) {   // thread tid places links [tid * LPT, tid * LPT + LPT)
        const int l = tid * LPT + k;
        if (l >= nl) continue;
        const bool first = early(l);
        const int slot = first ? at : nEarly + l - at;   // at: the early ones before l
        at += first;
        const int ax = b.lmeta[glink(l)] & 3, e = endsOf(l);
        sSL[slot] = (unsigned short)l;
        sVL[(2 * ax) * BS + (e & 0xFFFF)] = (unsigned short)slot;
        sVL[(2 * ax + 1) * BS + (e >> 16)] = (unsigned short)slot;
    }
    // 2*sqrt(m)*zeta/previousDt (VX_Voxel.h:131): the first step's previousDt is the dt of the
    // simulation's last step (which a caller-given dt may have set), every later one the launch's dt
    const float prevDt0 = scg.prevDt > 0 ? scg.prevDt : dtf;
    __syncthreads();
    if (tid < nvm) sDm[tid] = 2 * sVM[tid].sqrtMass * sVM[tid].zetaInternal / (sVM[tid].fixed ? 0.0f : prevDt0);
    auto localVmat = [&](int gidx) {
        int r = 0;
        for (int i = 0; i < nvm; i++) if (b.simMats[mat0 + i] == gidx) r = i;
        return r;
    };
    auto localLmat = [&](int gidx) {
        int r = 0;
        for (int i = 0; i < nlm; i++) if (b.simMats[mat0 + nvm + i] == gidx) r = i;
        return r;
    };
    int lEnds[LPT];   // vneg | vpos << 16 (sim-local), -1 = no link
    int lMats[LPT];   // link mat | neg voxel mat << 8 | pos voxel mat << 16 (local) | axis << 24
    int lIdx[LPT];    // sim-local link index
    LinkState<real> ls[LPT];
#pragma unroll
    for (int k = 0; k < LPT; k++) {
        const int slot = tid + k * BS;
        lEnds[k] = -1;
        if (slot >= nl) continue;
        const int l = sSL[slot], g = glink(l);
        lIdx[k] = l;
        lEnds[k] = endsOf(l);
        lMats[k] = localLmat(b.lmeta[g] >> 2) | (localVmat(b.vmat[b.lneg[g]]) << 8) | (localVmat(b.vmat[b.lpos[g]]) << 16) |
                   ((b.lmeta[g] & 3) << 24);
        ls[k].pos2 = V3<real>(b.q2x[g], b.q2y[g], b.q2z[g]);
        ls[k].a1v = V3<real>(b.a1x[g], b.a1y[g], b.a1z[g]);
        ls[k].a2v = V3<real>(b.a2x[g], b.a2y[g], b.a2z[g]);
        ls[k].strain = b.strain[g];
        ls[k].maxStrain = b.maxStrain[g];
        ls[k].strainOffset = b.strainOffset[g];
        ls[k].flags = b.lflags[g];
    }
    // Actuation phases: the temperature depends on the voxel only through its phase
    // offset, and simulations use few distinct offsets.  Wave 0 collects them
    // (lane i keeps entry i), so each step evaluates sin once per distinct offset;
    // the values are those the per-voxel formula gives.
    if (tid < 64) {
        // compared as bit patterns: every value, NaN included, equals itself
        long long tab = 0;
        int n = 0;
        bool over = false;
        for (int base = 0; base < nv && !over; base += 64) {
            const int v = base + tid;
            const long long ph = v < nv ? __double_as_longlong(b.phase[gvox(v)]) : 0;
            bool pending = v < nv;
            while (!over && __any(pending)) {
                const int src = __ffsll((unsigned long long)__ballot(pending)) - 1;   // lowest pending lane
                const long long cand = __shfl(ph, src, 64);
                if (!__any(tid < n && tab == cand)) {
                    if (n == VX3_RES_PHASES) over = true;
                    else {
                        if (tid == n) tab = cand;
                        n++;
                    }
                }
                if (ph == cand) pending = false;   // clears at least lane src
            }
        }
        if (tid < n) sPhase[tid] = __longlong_as_double(tab);
        if (tid == 0) sNph = over ? -1 : n;
    }
    __syncthreads();
    const int nph = sNph;
    if (nph < 0) {
        if (tid == 0) scg.state = 4;   // failed
        return;
    }
    // the thread's voxel
    V3<real> vm, va;
    int vf = 0, vmat = -1, vext = -1, vpi = 0;
    int vl[3] = {-1, -1, -1};   // slots of directions (2i, 2i+1) packed lo | hi << 16, 0xFFFF = none
    int vpm = 0;                // CVX_Voxel::strain's per-axis case, fixed for the launch (see k_resident)
    if (tid < nv) {
        const int g = gvox(tid);
        vm = V3<real>(b.mx[g], b.my[g], b.mz[g]);
        va = V3<real>(b.ax[g], b.ay[g], b.az[g]);
        vf = b.vflags[g];
        vmat = localVmat(b.vmat[g]);
        vext = b.vext[g];
        const long long ph = __double_as_longlong(b.phase[g]);
        for (int i = 0; i < nph; i++)
            if (__double_as_longlong(sPhase[i]) == ph) vpi = i;
        const ExtDev* ext = vext >= 0 ? &b.extTab[vext] : nullptr;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            vl[i] = (int)sVL[(2 * i) * BS + tid] | ((int)sVL[(2 * i + 1) * BS + tid] << 16);
            const int n = ((vl[i] & 0xFFFF) != 0xFFFF) + (((vl[i] >> 16) & 0xFFFF) != 0xFFFF);
            const bool tension = (n == 2) || (ext && n == 1 && ((ext->dofFixed & (1 << i)) || ext->force[i] != 0));
            vpm |= (n == 2 ? 1 << i : 0) | (tension ? 8 << i : 0);
        }
    }
    if (TILED) sXv[tid] = tid < nvAll ? ta.xidx[td.vOff + tid] : -1;
    if (tid < nvAll) {
        const int g = gvox(tid);
        const real* src[7] = {b.px, b.py, b.pz, b.ow, b.ox, b.oy, b.oz};
#pragma unroll
        for (int q = 0; q < 7; q++) sP[q * BS + tid] = src[q][g];
        sTf[tid] = b.tfac[g];
        sPs[tid] = b.psx[g]; sPs[BS + tid] = b.psy[g]; sPs[2 * BS + tid] = b.psz[g];
    }
    if (poisson) {
#pragma unroll
        for (int k = 0; k < LPT; k++) {
            if (lEnds[k] < 0) continue;
            const int slot = tid + k * BS, ax = lMats[k] >> 24, g = glink(lIdx[k]);
            sEs[slot] = b.es[(2 * ax) * VC + b.lneg[g]];
            sEs[LMAX + slot] = b.es[(2 * ax + 1) * VC + b.lpos[g]];
        }
    }
    double t = scg.t;
    int steps = scg.steps;
    int angleSamples = scg.angleSamples;
    int state = 0;
    if (tid == 0) {
        sRun = 1; sDiv = 0;
        for (int q = 0; q < 3; q++) { sCom[q] = scg.com[q]; sComH0[q] = scg.comH0[q]; sComH1[q] = scg.comH1[q]; }
        sAngle = scg.recentAngle;
    }
    __syncthreads();   // setup tables alias the load buffer: done with them
    // TILED: the second half of the simulation's barrier `gen`, whose arrival is pending:
    // wait for every tile, then (sampleNow) the tiles' centre-of-mass partial sums in tile
    // order into sRed[.][0], then (loadHalo) the halo poses into LDS.  1: some tile saw a
    // link diverge (leave; the repair launch takes over), 2: a tile did not arrive (the
    // simulation fails).
    bool pend = false;
    auto finishBarrier = [&](bool loadHalo, bool sampleNow) -> int {
        if (tid < 64) {   // the first wave; tile 0 of the simulation is workgroup blockIdx.x - td.tile
            int flag = 0;
            if (!tileWait(ta.sync + ta.flag0 + (blockIdx.x - td.tile), td.nTiles, gen, ta.repair, ta.spin)) flag = 2;
            else if (divAt < 0 && xget(ta.sync + td.cOff)) flag = 1;
            if (tid == 0) sTile = flag;
        }
        const int par = gen & 1;
        gen++;
        pend = false;
        __syncthreads();
        if (sTile == 2) {   // state stays as it was
            if (tid == 0) scg.state = 4;
            return 2;
        }
        if (sTile == 1) return 1;   // state untouched: the repair launch runs it to that step's link pass
        if (sampleNow) {   // the partial sums read in parallel, added in tile order by one thread
            const double* P = ta.part + td.pOff + (size_t)par * td.nTiles * 4;
            double* sP = (double*)sF;   // the load buffer is free between the voxel and link passes
            for (int j = tid; j < td.nTiles; j += BS) {
                const double a0 = xget(P + 4 * j), a1 = xget(P + 4 * j + 1), a2 = xget(P + 4 * j + 2), a3 = xget(P + 4 * j + 3);
                sP[4 * j] = a0; sP[4 * j + 1] = a1; sP[4 * j + 2] = a2; sP[4 * j + 3] = a3;
            }
            __syncthreads();
            if (tid == 0) {   // the same totals in every tile
                for (int q = 0; q < 4; q++) sRed[q][0] = 0;
                for (int j = 0; j < td.nTiles; j++)
                    for (int q = 0; q < 4; q++) sRed[q][0] += sP[4 * j + q];
            }
        }
        if (loadHalo) {
            const real* X = (const real*)ta.xch + td.xOff + (size_t)par * td.xPar;
            if (tid >= nv && tid < nvAll) {
                // every load issued before the first LDS write: one memory latency, not eleven
                const real* r = X + (size_t)sXv[tid] * VX3_XCH_STRIDE;
                real q[VX3_XCH_STRIDE - 1];
#pragma unroll
                for (int f = 0; f < VX3_XCH_STRIDE - 1; f++) q[f] = xget(r + f);
#pragma unroll
                for (int f = 0; f < 7; f++) sP[f * BS + tid] = q[f];
                sTf[tid] = (float)q[7]; sPs[tid] = (float)q[8]; sPs[BS + tid] = (float)q[9]; sPs[2 * BS + tid] = (float)q[10];
            }
            __syncthreads();
        }
        return 0;
    };
    for (int it = 0; it < nSteps; it++) {
        // keep per-step LDS address arithmetic inside the loop (register pressure)
#pragma unroll
        for (int k = 0; k < LPT; k++) { asm volatile("" : "+v"(lEnds[k])); asm volatile("" : "+v"(lMats[k])); }
        asm volatile("" : "+v"(vl[0])); asm volatile("" : "+v"(vl[1])); asm volatile("" : "+v"(vl[2])); asm volatile("" : "+v"(vmat));
        // temperatures of this step's distinct phases (read in the voxel pass, after the link barrier)
        if (vary && tid < nph) sPhT[tid] = actuationTemp(tempAmp, tempPeriod, sPhase[tid], t + dt, expansion);
        // ---- links
        auto linkAt = [&](int k) {
            const int slot = tid + k * BS, vn = lEnds[k] & 0xFFFF, vq = lEnds[k] >> 16, a = lMats[k] >> 24;
            const LinkMatDev& mat = sLM[lMats[k] & 0xFF];
            const int in_ = (lMats[k] >> 8) & 0xFF, ip_ = (lMats[k] >> 16) & 0xFF;
            const VoxMatDev &mn = sVM[in_], &mp = sVM[ip_];
            if (mn.fixed && mp.fixed) return;   // its slots are never read: both ends are fixed
            const int cy = a == 1 ? 0 : 1, cz = a == 2 ? 0 : 2;   // components read as the frame's y and z (x: a)
            const real restLength = (real)0.5 * (nom * (real)sTf[vn] + nom * (real)sTf[vq]);
            float area, tss;
            if (mat.nu != 0.0f) {
                float an, sn, ap, sp;
                const int t0 = a == 0 ? 1 : 0, t1 = a == 2 ? 1 : 2;   // the two transverse axes, in order
                // CVX_Voxel::transverseArea / transverseStrainSum (VX_Voxel.cpp:345-373)
                auto tr = [&](int v, bool nuZero, float& ar, float& su) {
                    if (nuZero) { ar = size * size; su = 0.0f; return; }
                    const float s0 = sPs[t0 * BS + v], s1 = sPs[t1 * BS + v];
                    ar = (float)((real)(size * size) * ((real)1 + (real)s0) * ((real)1 + (real)s1));
                    su = s0 + s1;
                };
                tr(vn, mn.nu == 0.0f, an, sn);
                tr(vq, mp.nu == 0.0f, ap, sp);
                area = 0.5f * (an + ap);
                tss = 0.5f * (sn + sp);
            } else {
                area = 0.5f * (size * size + size * size);
                tss = 0.0f;
            }
            auto flip = [](real v, bool f) { return f ? -v : v; };
            const V3<real> d(sP[a * BS + vq] - sP[a * BS + vn], flip(sP[cy * BS + vq] - sP[cy * BS + vn], a == 1),
                             flip(sP[cz * BS + vq] - sP[cz * BS + vn], a == 2));
            const Q4<real> oN(sP[3 * BS + vn], sP[(4 + a) * BS + vn], flip(sP[(4 + cy) * BS + vn], a == 1),
                              flip(sP[(4 + cz) * BS + vn], a == 2));
            const Q4<real> oP(sP[3 * BS + vq], sP[(4 + a) * BS + vq], flip(sP[(4 + cy) * BS + vq], a == 1),
                              flip(sP[(4 + cz) * BS + vq], a == 2));
            V3<real> fN, mN, fP, mP;
            linkForces<real>(mat, 0, V3<real>(0, 0, 0), oN, d, oP, restLength, area, tss, mat.nu != 0.0f, sDm[in_], sDm[ip_], ls[k],
                             fN, mN, fP, mP);
            auto put = [&](int row, const V3<real>& f) {
                sF[(row + a) * LMAX + slot] = f.x;
                sF[(row + cy) * LMAX + slot] = flip(f.y, a == 1);
                sF[(row + cz) * LMAX + slot] = flip(f.z, a == 2);
            };
            put(0, fN); put(3, mN); put(6, fP); put(9, mP);
            if (poisson) {
                // CVX_Link::axialStrain(positiveEnd) (VX_Link.cpp:115-118)
                const float r = mat.strainRatio;
                sEs[slot] = 2.0f * ls[k].strain / (1.0f + r);
                sEs[LMAX + slot] = 2.0f * ls[k].strain * r / (1.0f + r);
            }
            if (ls[k].strain > 100) sDiv = 1;
        };
        if (TILED && pend) {
            // those between owned voxels, then the wait and the halo, then those with a halo end
#pragma unroll
            for (int k = 0; k < LPT; k++)
                if (tid + k * BS < nEarly) linkAt(k);
            if (finishBarrier(true, false)) return;
#pragma unroll
            for (int k = 0; k < LPT; k++)
                if (lEnds[k] >= 0 && tid + k * BS >= nEarly) linkAt(k);
        } else {
#pragma unroll
            for (int k = 0; k < LPT; k++)
                if (lEnds[k] >= 0) linkAt(k);
        }
        __syncthreads();
        // ---- voxels
        // (a tile learns of its simulation's divergence only at the step's barrier and stops at that
        // step on a second run)
        const bool diverged = TILED ? it == divAt : sDiv != 0;
        steps++;
        const bool sample = !diverged && cycleStep > 0 && steps % cycleStep == 0;
        double psx = 0, psy = 0, psz = 0, psm = 0;
        const double tn = t + dt;
        if (!diverged && vmat >= 0) {
            V3<real> fs(0, 0, 0), ms(0, 0, 0);
            float st[3] = {0, 0, 0};
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int slot = e ? ((vl[a] >> 16) & 0xFFFF) : (vl[a] & 0xFFFF);
                    if (slot == 0xFFFF) continue;
                    const int c = 6 * e;
                    fs.add(V3<real>(sF[(c + 0) * LMAX + slot], sF[(c + 1) * LMAX + slot], sF[(c + 2) * LMAX + slot]));
                    ms.add(V3<real>(sF[(c + 3) * LMAX + slot], sF[(c + 4) * LMAX + slot], sF[(c + 5) * LMAX + slot]));
                    if (poisson) st[a] += sEs[e * LMAX + slot];
                }
            const VoxMatDev& m = sVM[vmat];
            V3<real> vp(sP[tid], sP[BS + tid], sP[2 * BS + tid]);
            if (!m.fixed) {
                const ExtDev* ext = vext >= 0 ? &b.extTab[vext] : nullptr;
                int ix = 0, iy = 0, iz = 0;
                if (ext) { ix = ext->ix; iy = ext->iy; iz = ext->iz; }
                Q4<real> vo(sP[3 * BS + tid], sP[4 * BS + tid], sP[5 * BS + tid], sP[6 * BS + tid]);
                voxelStep<real>(m, ext, dtf, nom, ix, iy, iz, sTf[tid], fs, ms, NoContacts(), vp, vm, vo, va, vf);
                sP[tid] = vp.x; sP[BS + tid] = vp.y; sP[2 * BS + tid] = vp.z;
                sP[3 * BS + tid] = vo.w; sP[4 * BS + tid] = vo.x; sP[5 * BS + tid] = vo.y; sP[6 * BS + tid] = vo.z;
            }
            if (vary && !m.fixed && !(m.thermalOnAfter > tn)) sTf[tid] = 1 + sPhT[vpi] * m.alphaCTE;
            if (poisson) {   // CVX_Voxel::strain(true) for the next step from this step's end strains (see k_resident)
#pragma unroll
                for (int i = 0; i < 3; i++) if (vpm & (1 << i)) st[i] *= 0.5f;
                if ((vpm & 56) != 56) {
                    float add = 0;
#pragma unroll
                    for (int i = 0; i < 3; i++) if (vpm & (8 << i)) add += st[i];
                    const float value = poissonValue(1.0f + add, m.nu);
#pragma unroll
                    for (int i = 0; i < 3; i++) if (!(vpm & (8 << i))) st[i] = value;
                }
                sPs[tid] = st[0]; sPs[BS + tid] = st[1]; sPs[2 * BS + tid] = st[2];
            }
            if (sample && m.isMeasured) {
                const double mass = m.mass;
                psx = (double)vp.x * mass; psy = (double)vp.y * mass; psz = (double)vp.z * mass;
                psm = mass;
            }
            if (TILED && sXv[tid] >= 0) {   // a voxel another tile reads: its record out as soon as it is final
                real q[VX3_XCH_STRIDE - 1] = {sP[tid], sP[BS + tid], sP[2 * BS + tid], sP[3 * BS + tid], sP[4 * BS + tid], sP[5 * BS + tid],
                                              sP[6 * BS + tid], (real)sTf[tid], (real)sPs[tid], (real)sPs[BS + tid], (real)sPs[2 * BS + tid]};
                real* r = (real*)ta.xch + td.xOff + (size_t)(gen & 1) * td.xPar + (size_t)sXv[tid] * VX3_XCH_STRIDE;
#pragma unroll
                for (int f = 0; f < VX3_XCH_STRIDE - 1; f++) xput(r + f, q[f]);
            }
        }
        if (sample) {
            // FP64 center of mass of the measured voxels (VX3_VoxelyzeKernel.cu:477-493)
            for (int o = 32; o > 0; o >>= 1) {
                psx += __shfl_xor(psx, o, 64); psy += __shfl_xor(psy, o, 64);
                psz += __shfl_xor(psz, o, 64); psm += __shfl_xor(psm, o, 64);
            }
            if ((tid & 63) == 0) { sRed[0][tid >> 6] = psx; sRed[1][tid >> 6] = psy; sRed[2][tid >> 6] = psz; sRed[3][tid >> 6] = psm; }
        }
        if (TILED && !diverged) {
            // ---- arrival at the simulation's barrier (TILED): the records are out; the wait
            // comes in the next step's link pass, or now on a sampling step (the centre of
            // mass needs every tile's partial sum)
            __builtin_amdgcn_s_waitcnt(0);   // this thread's exchange stores are complete
            __syncthreads();
            if (tid == 0) {
                if (sample) {
                    double* P = ta.part + td.pOff + (size_t)(gen & 1) * td.nTiles * 4;
                    double tot[4] = {0, 0, 0, 0};
                    for (int w = 0; w < BS / 64; w++)
                        for (int q = 0; q < 4; q++) tot[q] += sRed[q][w];
                    for (int q = 0; q < 4; q++) xput(P + 4 * td.tile + q, tot[q]);
                }
                if (sDiv) __hip_atomic_fetch_max(ta.sync + td.cOff, it + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                tileArrive(ta.sync + ta.flag0 + blockIdx.x, gen, ta.repair);
            }
            pend = true;
            if (sample && finishBarrier(true, true)) return;
        } else if (sample) __syncthreads();
        if (sample) {
            angleSamples++;
            if (tid == 0) {
                double tot[4] = {0, 0, 0, 0};
                if (TILED) {
                    for (int q = 0; q < 4; q++) tot[q] = sRed[q][0];
                } else {
                    for (int w = 0; w < BS / 64; w++)
                        for (int q = 0; q < 4; q++) tot[q] += sRed[q][w];
                }
                double* A = sComH0; double* B = sComH1; double* C = sCom;
                for (int q = 0; q < 3; q++) { A[q] = B[q]; B[q] = C[q]; C[q] = tot[3] == 0 ? 0.0 : (1.0 / tot[3]) * tot[q]; }
                const bool bc = B[0] == C[0] && B[1] == C[1] && B[2] == C[2];
                const bool ab = A[0] == B[0] && A[1] == B[1] && A[2] == B[2];
                if (bc || ab || angleSamples < 3) sAngle = 0;
                else {
                    double d1[3] = {B[0] - A[0], B[1] - A[1], B[2] - A[2]}, d2[3] = {C[0] - B[0], C[1] - B[1], C[2] - B[2]};
                    double dot = d1[0] * d2[0] + d1[1] * d2[1] + d1[2] * d2[2];
                    double l1 = sqrt((A[0] - B[0]) * (A[0] - B[0]) + (A[1] - B[1]) * (A[1] - B[1]) + (A[2] - B[2]) * (A[2] - B[2]));
                    double l2 = sqrt((B[0] - C[0]) * (B[0] - C[0]) + (B[1] - C[1]) * (B[1] - C[1]) + (B[2] - C[2]) * (B[2] - C[2]));
                    sAngle = acos(dot / (l1 * l2));
                }
            }
        }
        // ---- per-simulation control (uniform across the workgroup)
        if (diverged) { state = 2; break; }
        t = tn;
        bool stop = maxSteps > 0 && steps >= maxSteps;
        if (!stop && stopLen > 0 && tid == 0) sRun = mathTreeEval(b.tokens + stopOff, stopLen, sCom[0], sCom[1], sCom[2], 0, t, sAngle, 0, 0, scg.nv, sQ) > 0 ? 0 : 1;
        if (it == 0 && prevDt0 != dtf && tid < nvm) sDm[tid] = 2 * sVM[tid].sqrtMass * sVM[tid].zetaInternal / (sVM[tid].fixed ? 0.0f : dtf);
        __syncthreads();   // next step's link pass reads the new poses
        if (stop || !sRun) {
            if (TILED && pend && finishBarrier(false, false)) return;
            state = 1;
            break;
        }
    }
    if (TILED && pend && finishBarrier(false, false)) return;   // the launch's last step

    // ---- write back in the stream layout
#pragma unroll
    for (int k = 0; k < LPT; k++) {
        if (lEnds[k] < 0) continue;
        if (TILED && !(ta.link[td.lOff + lIdx[k]] & 0x80000000)) continue;   // the other tile writes it
        const int g = glink(lIdx[k]);
        b.q2x[g] = ls[k].pos2.x; b.q2y[g] = ls[k].pos2.y; b.q2z[g] = ls[k].pos2.z;
        b.a1x[g] = ls[k].a1v.x; b.a1y[g] = ls[k].a1v.y; b.a1z[g] = ls[k].a1v.z;
        b.a2x[g] = ls[k].a2v.x; b.a2y[g] = ls[k].a2v.y; b.a2z[g] = ls[k].a2v.z;
        b.strain[g] = ls[k].strain;
        b.maxStrain[g] = ls[k].maxStrain;
        b.strainOffset[g] = ls[k].strainOffset;
        b.lflags[g] = ls[k].flags;
        if (poisson) {
            const int slot = tid + k * BS, ax = lMats[k] >> 24;
            b.es[(2 * ax) * VC + b.lneg[g]] = sEs[slot];
            b.es[(2 * ax + 1) * VC + b.lpos[g]] = sEs[LMAX + slot];
        }
    }
    if (tid < nv) {
        const int g = gvox(tid);
        real* dst[7] = {b.px, b.py, b.pz, b.ow, b.ox, b.oy, b.oz};
#pragma unroll
        for (int q = 0; q < 7; q++) dst[q][g] = sP[q * BS + tid];
        b.mx[g] = vm.x; b.my[g] = vm.y; b.mz[g] = vm.z;
        b.ax[g] = va.x; b.ay[g] = va.y; b.az[g] = va.z;
        b.vflags[g] = vf;
        b.tfac[g] = sTf[tid];
        b.psx[g] = sPs[tid]; b.psy[g] = sPs[BS + tid]; b.psz[g] = sPs[2 * BS + tid];
    }
    if (tid == 0 && (!TILED || td.tile == 0)) {   // every tile holds the same control values
        if (steps != scg.steps) scg.prevDt = dtf;
        scg.t = t;
        scg.steps = steps;
        scg.angleSamples = angleSamples;
        for (int q = 0; q < 3; q++) { scg.com[q] = sCom[q]; scg.comH0[q] = sComH0[q]; scg.comH1[q] = sComH1[q]; }
        scg.recentAngle = sAngle;
        scg.state = state;
    }
}

}  // namespace VX_NS
}  // namespace vx3
