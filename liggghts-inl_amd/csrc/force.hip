// force.hip -- contact force pass and velocity-Verlet integrator.
//
// k_force: a group of G lanes per particle gathers over the particle's full
// neighbour row (lane g takes entries g, g+G, ...), then the group sums its
// partial forces and torques with a fixed xor-butterfly of shuffles, so every
// force and torque is summed by its owner in a fixed order: no atomics, no
// scatter, results independent of scheduling.  Replaces, per step,
// Verlet::force_clear (verlet.cpp:406-430), PairGran::compute
// (pair_gran_base.h:187-503), FixWallGran::post_force_primitive
// (fix_wall_gran.cpp:988-1120), FixGravity::post_force
// (fix_gravity.cpp:301-352) and FixFreeze::post_force (fix_freeze.cpp:121-144).
// The list is full (both directions), so a pair is evaluated once from each
// side; in the reference the j-side gets -F of the i-side evaluation, which
// for these laws is the same value (the per-side arithmetic is sign
// symmetric), and periodic-image pairs are evaluated from both sides there
// too (neigh_gran.cpp:570-640).
//
// An entry whose contact flag is still clear has never touched, so its
// history is zero; it is neither read nor, unless it touches now, written.
//
// k_force_t: the same pass with one list entry per lane (every chain without
// a cohesion model, the default).  Both kernels end in one per-particle
// epilogue (planes, gravity, freeze, the force and torque written) that also
// integrates when nothing adds to the forces after the pass, writing the new
// state to the other state buffers.
//
// k_integrate: FixNVESphere::initial_integrate / final_integrate
// (fix_nve_sphere.cpp:134-243) with dtf = 0.5*dt, INERTIA = 0.4; mode 3 runs
// final(n) and initial(n+1) in one pass over the state.
#include "contact_law.h"
#include "kernels.h"

#include <stdlib.h>

#include <algorithm>

#include <type_traits>

namespace dem {

// Blocks are dealt to the 8 XCDs round robin; remap so each XCD walks a
// contiguous range of Morton-ordered particles and their neighbours stay in
// that XCD's L2.
__device__ inline int xcd_block(int b, int nb_padded)
{
    const int per = nb_padded >> 3;
    return (b & 7) * per + (b >> 3);
}

template <int G>
__device__ inline double group_sum(double v)
{
    for (int o = G >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, G);
    return v;
}

template <int G>
__device__ inline int group_sum_int(int v)
{
    for (int o = G >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, G);
    return v;
}

// Slots [0, lim) of one entry's history into h, zeros past lim (all zeros
// when !known).  vec: the entry starts 16-byte aligned and lim is even, so
// the slots move as 16-byte pairs and a lane's history reaches the L2 in
// half the requests (the entries a wave touches are scattered, so every
// lane's access is a request of its own).
template <int HN>
__device__ inline void hist_load(const double *hp, int lim, bool vec, bool known, double (&h)[HN])
{
    static_assert(HN % 2 == 0, "pairs");
    if (vec) {
        const double2 *h2 = reinterpret_cast<const double2 *>(hp);
#pragma unroll
        for (int q = 0; q < HN / 2; q++) {
            double2 v = make_double2(0.0, 0.0);
            if (known && 2 * q < lim) v = h2[q];
            h[2 * q] = v.x;
            h[2 * q + 1] = v.y;
        }
    } else {
#pragma unroll
        for (int q = 0; q < HN; q++) h[q] = (known && q < lim) ? hp[q] : 0.0;
    }
}

template <int HN>
__device__ inline void hist_store(double *hp, int lim, bool vec, const double (&h)[HN])
{
    static_assert(HN % 2 == 0, "pairs");
    if (vec) {
        double2 *h2 = reinterpret_cast<double2 *>(hp);
#pragma unroll
        for (int q = 0; q < HN / 2; q++)
            if (2 * q < lim) h2[q] = make_double2(h[2 * q], h[2 * q + 1]);
    } else {
#pragma unroll
        for (int q = 0; q < HN; q++)
            if (q < lim) hp[q] = h[q];
    }
}

// What the owner of particle i adds after its pair sum: the primitive
// planes in the order the fixes were defined, gravity, fix freeze; then the
// force, torque and optional per-atom outputs are written.
template <bool MIXED, int WN>
__device__ inline void particle_epilogue(const ForceArgs &a, int i, const double4 pi, const double4 vmi,
                                         const double4 wi, int itype, bool fzi, const double *mat, uint32_t wm,
                                         double F[3], double T[3], int nc)
{
    const Model &M = a.M;
    // primitive planes, in the order the fixes were defined
    double pw = 0.0;    // force of the observed plane along its axis
    if (a.P.n && wm) {
        const double cdmw = M.cdf - 1.0;
        for (int k = 0; k < a.P.n; k++) {
            if (!(wm & (1u << k))) continue;
            const int d = a.P.dim[k];
            const double p = a.P.pos[k];
            const double radi = pi.w;
            // a blend rather than an index, so the coordinate stays in
            // registers (x*1 + y*0 + z*0 is x exactly)
            const double pos = pi.x * (double)(d == 0) + pi.y * (double)(d == 1) + pi.z * (double)(d == 2);
            const double dd = p - pos;
            const double delta[3] = {d == 0 ? dd : 0.0, d == 1 ? dd : 0.0, d == 2 ? dd : 0.0};
            const double deltan = (pos > p) ? pos - p - radi : p - pos - radi;
            const int wdn = M.wdnum;
            double *hp = a.whist + ((size_t)i * a.P.n + k) * wdn;
            if (deltan > M.cutneighmax) continue;
            if (deltan <= 0 || deltan < cdmw * radi) {
                if (deltan <= 0) {
                    ContactIn cw;
                    cw.is_wall = true;
                    cw.itype = itype;
                    cw.jtype = a.P.wtype[k];
                    cw.radi = radi;
                    cw.radj = 0.0;
                    cw.deltan_in = -deltan;
                    cw.delta[0] = -delta[0]; cw.delta[1] = -delta[1]; cw.delta[2] = -delta[2];
                    cw.r = cw.radi - cw.deltan_in;
                    cw.rinv = 1.0 / cw.r;
                    cw.radsum = cw.radi;
                    cw.mi = vmi.w; cw.mj = 0.0; cw.meff = vmi.w;
                    cw.vi[0] = vmi.x; cw.vi[1] = vmi.y; cw.vi[2] = vmi.z;
                    cw.vj[0] = 0.0; cw.vj[1] = 0.0; cw.vj[2] = 0.0;
                    cw.wi[0] = wi.x; cw.wi[1] = wi.y; cw.wi[2] = wi.z;
                    cw.wj[0] = 0.0; cw.wj[1] = 0.0; cw.wj[2] = 0.0;
                    constexpr int WHN = chain_max_dnum(WN);
                    const bool vec = (wdn & 1) == 0;
                    double h[WHN];
                    hist_load(hp, wdn, vec, true, h);
                    double dF[3], dT[3];
                    if (MIXED && WN == NM_HERTZ) contact_mixed(M, mat, cw, h, a.shearupdate, dF, dT);
                    else contact_fp64<WN>(M, M.lw, mat, cw, h, a.shearupdate, dF, dT);
                    if (a.shearupdate || WN != NM_HERTZ) hist_store(hp, wdn, vec, h);
                    F[0] += dF[0]; F[1] += dF[1]; F[2] += dF[2];
                    T[0] += dT[0]; T[1] += dT[1]; T[2] += dT[2];
                    if (k == a.obs_plane) pw = d == 0 ? dF[0] : (d == 1 ? dF[1] : dF[2]);
                } else {
                    contact_close(M.lw, hp);
                }
            } else {
                for (int q = 0; q < wdn; q++) hp[q] = 0.0;
            }
        }
    }
    if (M.gravity_on) {
        const double massone = vmi.w;
        F[0] += massone * M.gacc[0];
        F[1] += massone * M.gacc[1];
        F[2] += massone * M.gacc[2];
    }
    if (M.freeze_on && fzi && !a.defer_freeze) {
        F[0] = F[1] = F[2] = 0.0;
        T[0] = T[1] = T[2] = 0.0;
    }
    // a pass that also runs the next step's initial_integrate is never the
    // last of a dem_step call, and nothing after it reads the force and
    // torque (the next pass recomputes them): they are written only by the
    // other passes
    if (a.fuse != 3) {
        a.f4[i] = make_double4(F[0], F[1], F[2], 0.0);
        a.t4[i] = make_double4(T[0], T[1], T[2], 0.0);
    }
    if (a.ncontact) a.ncontact[i] = nc;
    if (a.pwf) a.pwf[i] = pw;
}

// final_integrate(n) and, with fuse = 3, initial_integrate(n+1) of one
// particle from its state and its final force and torque: the operations of
// k_integrate, written to the other state buffers
__device__ inline void integrate_into(const ForceArgs &a, int i, double4 x, double4 v, double4 w, const double F[3],
                                      const double T[3])
{
    // dtfm = dtf / (rmass*(1.+CAddRhoFluid/density)), CAddRhoFluid = 0
    const double dtfm = a.dtf / (v.w * (1. + 0.0 / 1.0));
    const double dtirotate = a.dtfrotate / (x.w * x.w * v.w);
    if (a.fuse & 2) {
        v.x += dtfm * F[0]; v.y += dtfm * F[1]; v.z += dtfm * F[2];
        w.x += dtirotate * T[0]; w.y += dtirotate * T[1]; w.z += dtirotate * T[2];
    }
    if (a.fuse & 1) {
        v.x += dtfm * F[0]; v.y += dtfm * F[1]; v.z += dtfm * F[2];
        x.x += a.dtv * v.x; x.y += a.dtv * v.y; x.z += a.dtv * v.z;
        w.x += dtirotate * T[0]; w.y += dtirotate * T[1]; w.z += dtirotate * T[2];
    }
    a.xn[i] = x;
    a.vn[i] = v;
    a.wn[i] = w;
    if (a.ctl) {   // Neighbor::check_distance of the next step
        const double4 b = a.xhold[i];
        const double dx = x.x - b.x, dy = x.y - b.y, dz = x.z - b.z;
        const long long step = a.ctl[a.par];
        if (dx * dx + dy * dy + dz * dz > a.deltasq)
            atomicCAS((unsigned long long *)&a.ctl[2], 0ull, (unsigned long long)(step + 1));
        if (i == 0) a.ctl[a.par ^ 1] = step + 1;
    }
}

// Whether this step of a checked period still runs: not once the period
// halted at or before it.  A halt that the pass records itself names the next
// step, so blocks that start after it still run.  The counter advances either
// way (from the pass's first particle).
__device__ inline bool period_runs(const ForceArgs &a, bool first)
{
    if (!a.ctl) return !(a.halt && *a.halt);
    const long long step = a.ctl[a.par], h = a.ctl[2];
    if (h == 0 || h > step) return true;
    if (first) a.ctl[a.par ^ 1] = step + 1;
    return false;
}

template <bool MIXED, int G, int NM, int WN, bool CH = false>
__global__ void __launch_bounds__(kBlock) k_force(ForceArgs a)
{
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int tid = blk * blockDim.x + threadIdx.x;
    if (!period_runs(a, tid == 0)) return;
    const int g = threadIdx.x & (G - 1);
    const int i = tid / G;
    const bool live = i < a.n;      // dead groups still join the shuffles
    const int ii = live ? i : a.n - 1;
    const Model &M = a.M;
    const double4 pi = a.xr[ii];
    const double4 vmi = a.vm[ii];
    const double4 wi = a.wt[ii];
    const int metai = (int)wi.w;
    const int itype = meta_type(metai);
    const bool fzi = meta_frozen(metai);
    // material tables of the particle's instance (partners share it)
    const double *mat = a.mat + (size_t)meta_inst(metai) * kMatStride;
    double F[3] = {0.0, 0.0, 0.0}, T[3] = {0.0, 0.0, 0.0};
    const int dnum = M.dnum;
    // slots of the contact chain; the cohesion slots after them belong to
    // the bond pass
    const int hdn = (CH && M.lp.off_coh >= 0) ? M.lp.off_coh : dnum;
    const double cdm = M.cdf * M.cdf;
    int nc = 0;

    ContactIn c;
    c.is_wall = false;
    c.itype = itype;
    c.radi = pi.w;
    c.mi = vmi.w;
    c.vi[0] = vmi.x; c.vi[1] = vmi.y; c.vi[2] = vmi.z;
    c.wi[0] = wi.x; c.wi[1] = wi.y; c.wi[2] = wi.z;
    c.deltan_in = 0.0;

    Row row = {0, 0, 0, 0};
    if (live) row = list_row(a.nstart, a.n, i);
    for (int q = g; q < row.cnt; q += G) {
        const int e = row.entry(q);
        const uint32_t w = a.nj[e];
        const int j = (int)(w & kJMask);
        const int code = (int)((w >> 26) & 31u);
        const double4 pj = a.xr[j];
        double xj0 = pj.x, xj1 = pj.y, xj2 = pj.z;
        if (code != kNoShift) {
            const double3 im = image_of(pj, code, M.prd);
            xj0 = im.x; xj1 = im.y; xj2 = im.z;
        }
        const double delx = pi.x - xj0;
        const double dely = pi.y - xj1;
        const double delz = pi.z - xj2;
        const double rsq = delx * delx + dely * dely + delz * delz;
        const double radj = pj.w;
        const double radsum = pi.w + radj;
        // cohesion force of a bonded entry, computed by the bond pass
        bool bonded = false;
        double coh[6];
        if (CH && (w & kBondBit) && a.bvalid[e]) {
            bonded = true;
            const double *bo = a.bout + (size_t)e * 6;
            for (int q = 0; q < 6; q++) coh[q] = bo[q];
        }
        if (rsq < radsum * radsum) {
            const double r = sqrt(rsq);
            if (r < 1e-20) atomicOr(a.err, 1);
            const double rinv = 1.0 / r;
            const double4 vmj = a.vm[j];
            const double4 wj = a.wt[j];
            const int metaj = (int)wj.w;
            c.jtype = meta_type(metaj);
            c.radj = radj;
            c.mj = vmj.w;
            double meff = c.mi * c.mj / (c.mi + c.mj);
            if (M.freeze_on && fzi) meff = c.mj;
            if (M.freeze_on && meta_frozen(metaj)) meff = c.mi;
            c.meff = meff;
            c.delta[0] = delx; c.delta[1] = dely; c.delta[2] = delz;
            c.r = r; c.rinv = rinv; c.radsum = radsum;
            c.vj[0] = vmj.x; c.vj[1] = vmj.y; c.vj[2] = vmj.z;
            c.wj[0] = wj.x; c.wj[1] = wj.y; c.wj[2] = wj.z;
            constexpr int HN = chain_max_dnum(NM);
            double h[HN];
            double *hp = a.hist + (size_t)e * dnum;
            const bool known = (w & (CH ? (kFlagBit | kBondBit) : kFlagBit)) != 0;
            const bool vec = ((dnum | hdn) & 1) == 0;
            hist_load(hp, hdn, vec, known, h);
            double dF[3], dT[3];
            if (MIXED && NM == NM_HERTZ) contact_mixed(M, mat, c, h, a.shearupdate, dF, dT);
            else if (CH) contact_fp64<NM, true>(M, M.lp, mat, c, h, a.shearupdate, dF, dT, coh,
                                                bonded ? M.cohesion : CM_OFF);
            else contact_fp64<NM>(M, M.lp, mat, c, h, a.shearupdate, dF, dT);
            // the hysteretic models write their state even in set-up passes
            if (a.shearupdate || !known || NM != NM_HERTZ) hist_store(hp, hdn, vec, h);
            if (!(w & kFlagBit)) a.nj[e] = w | kFlagBit;
            F[0] += dF[0]; F[1] += dF[1]; F[2] += dF[2];
            T[0] += dT[0]; T[1] += dT[1]; T[2] += dT[2];
            nc++;
        } else if (rsq < cdm * radsum * radsum) {
            // surfacesClose: history reset; a hysteretic chain also clears
            // its contact flag, so the entry no longer carries at a rebuild
            double *hp = a.hist + (size_t)e * dnum;
            if (!contact_close(M.lp, hp)) a.nj[e] = w & ~kFlagBit;
            if (CH && bonded) {
                F[0] += coh[0]; F[1] += coh[1]; F[2] += coh[2];
                T[0] += coh[3]; T[1] += coh[4]; T[2] += coh[5];
            }
        }
    }
    if (G > 1) {
        for (int k = 0; k < 3; k++) {
            F[k] = group_sum<G>(F[k]);
            T[k] = group_sum<G>(T[k]);
        }
        nc = group_sum_int<G>(nc);
    }
    if (!live || g != 0) return;

    particle_epilogue<MIXED, WN>(a, i, pi, vmi, wi, itype, fzi, mat, a.P.n ? a.wmask[i] : 0u, F, T, nc);
    if (a.fuse) integrate_into(a, i, pi, vmi, wi, F, T);
}

// ---------------------------------------------------------------------------
// k_force_t: a wave owns a tile of P consecutive particles.  Their entries
// are two contiguous ranges of the list: the partners that touched at the
// build and the others (dem_device.h).  An entry of the first range is
// evaluated in place, one per lane: its partner's state and its history are
// asked for together, before the overlap is known, since nearly all of them
// still touch.  The second range is only tested, 128 entries at a time; the
// few that touch now go to a queue in LDS and fill the lanes that the first
// range's last batch leaves idle.  Results go to LDS, FP32 for the mixed law
// (whose results are FP32 values) and FP64 otherwise, and every particle
// adds its own in list order, the first range before the queue: no
// atomics, and a sum that does not depend on where the tiles begin.
//
// What bounds it: the latency of its chain of gathers at 4 (mixed) or 3
// (FP64) waves per SIMD, which the 128 / 142 registers of the law allow, with
// 48 % of the issue slots taken by VALU.  1M-sphere column: 276 -> 231 us mixed,
// 282 -> 242 FP64, where every entry of whole rows, one after the other, went
// through the test and a queue.  HBM traffic there (4.52 contacts and 7.58
// partners per particle, 652 B that the pass cannot do without) 836 -> 779 B per
// particle, of which 217 + 217 are histories.  Slower here: histories and state
// through LDS in whole lines (249 to 270 us), the first batch fetched ahead of
// the test (256, one wave per SIMD fewer), tiles trimmed so that their batches
// fill (236).
constexpr int kQueue = 192;   // 63 waiting and the 128 of one test

template <int P, typename OutT>
struct TileLds {
    double4 x[P], v[P], w[P];        // the tile's state
    OutT out[6][64];                 // a batch's forces and torques
    int rs[2][P + 1];                // row starts, first and second range
    int q[kQueue];                   // queued entries
    uint8_t qo[kQueue];              // and their particles
    uint8_t run[2][P];               // a particle's run of queued results in a batch
    uint8_t own[16 * P];             // particle of each entry, first range then second
};

__device__ inline void wave_sync()
{
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One entry's DN history slots, in the widest pieces their alignment allows
template <int DN, int HN>
__device__ inline void slots_load(const double *hp, double (&h)[HN])
{
    static_assert(HN >= DN, "room for the slots");
    if constexpr (DN % 2 == 0) {
#pragma unroll
        for (int q = 0; q < DN / 2; q++) {
            const double2 v = reinterpret_cast<const double2 *>(hp)[q];
            h[2 * q] = v.x;
            h[2 * q + 1] = v.y;
        }
    } else {
#pragma unroll
        for (int q = 0; q < DN; q++) h[q] = hp[q];
    }
}

template <int DN, int HN>
__device__ inline void slots_store(double *hp, const double (&h)[HN])
{
    if constexpr (DN % 2 == 0) {
#pragma unroll
        for (int q = 0; q < DN / 2; q++) reinterpret_cast<double2 *>(hp)[q] = make_double2(h[2 * q], h[2 * q + 1]);
    } else {
#pragma unroll
        for (int q = 0; q < DN; q++) hp[q] = h[q];
    }
}

// contact_close with the chain's layout known; true if the flag stays set
template <int NM, int DN>
__device__ inline bool slots_close(double *hp)
{
    constexpr int s0 = chain_off_shear(NM);
    if constexpr (NM != NM_HERTZ)
#pragma unroll
        for (int q = 0; q < 10; q++) hp[q] = 0.0;
#pragma unroll
    for (int q = s0; q < DN; q++) hp[q] = 0.0;
    return NM == NM_HERTZ;
}

// DN: history slots of the pair chain (its rolling history included or not)
template <bool MIXED, int NM, int WN, int DN, int P>
__global__ void __launch_bounds__(kBlock) k_force_t(ForceArgs a)
{
    static_assert(P == 8 || P == 16 || P == 32 || P == 64, "a tile fits one wave");
    static_assert(!MIXED || NM == NM_HERTZ, "the mixed law is Hertz's");
    using OutT = typename std::conditional<MIXED, float, double>::type;
    using Lds = TileLds<P, OutT>;
    extern __shared__ __align__(16) char s_raw[];
    // lanes that sum: P particles times kParts groups of kPer components
    constexpr int kParts = P == 8 ? 6 : (P == 16 ? 3 : (P == 32 ? 2 : 1));
    constexpr int kPer = 6 / kParts;
    constexpr int kOwn = 16 * P;
    constexpr int RH = DN > chain_off_shear(NM) + 3 ? 1 : 0;
    static_assert(DN == chain_off_shear(NM) + 3 + 3 * RH, "shear, then rolling");
    // the mixed law asks the model whether it rolls, so its slots always exist
    constexpr int HN = MIXED ? chain_max_dnum(NM) : DN;

    // the wave's number in the block is the same for its lanes: every address
    // of the tile stays in scalar registers
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int p0 = (blk * (int)(blockDim.x >> 6) + wv) * P;
    if (p0 >= a.n) return;   // uniform over the wave
    if (!period_runs(a, p0 == 0 && lane == 0)) return;
    Lds &L = reinterpret_cast<Lds *>(s_raw)[wv];
    const int np = min(P, a.n - p0);
    const Model &M = a.M;
    uint32_t wm = 0;
    if (lane < np) {
        L.x[lane] = a.xr[p0 + lane];
        L.v[lane] = a.vm[p0 + lane];
        L.w[lane] = a.wt[p0 + lane];
        if (a.P.n) wm = a.wmask[p0 + lane];
        L.rs[0][lane] = a.nstart[p0 + lane];
        L.rs[1][lane] = a.nstart[a.n + p0 + lane];
    }
    const int A0 = a.nstart[p0], nA = a.nstart[p0 + np] - A0;
    const int B0 = a.nstart[a.n + p0], nB = a.nstart[a.n + p0 + np] - B0;
    if (lane == 0) {   // the ends of the last rows
        L.rs[0][np] = A0 + nA;
        L.rs[1][np] = B0 + nB;
    }
    wave_sync();
    // particle of each entry, written row by row; past kOwn entries by search
    if (lane < np) {
        for (int t = L.rs[0][lane] - A0; t < min(L.rs[0][lane + 1] - A0, kOwn); t++) L.own[t] = (uint8_t)lane;
        for (int t = L.rs[1][lane] - B0 + nA; t < min(L.rs[1][lane + 1] - B0 + nA, kOwn); t++)
            L.own[t] = (uint8_t)lane;
    }
    wave_sync();
    auto owner = [&](int range, int t) {   // t: entry of the tile, first range then second
        if (t < kOwn) return (int)L.own[t];
        const int e = range ? B0 + (t - nA) : A0 + t;
        int lo = 0, hi = np - 1;   // the last row starting at or before e
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (L.rs[range][mid] <= e) lo = mid;
            else hi = mid - 1;
        }
        return lo;
    };
    const double cdm = M.cdf * M.cdf;
    double acc[kPer];
#pragma unroll
    for (int c = 0; c < kPer; c++) acc[c] = 0.0;
    int nc = 0;

    // evaluate one batch: m1 entries of the first range from its entry t0 on,
    // then mq of the queue's first entries
    auto batch = [&](int t0, int m1, int mq) {
        const bool act = lane < m1 + mq;
        bool touch = false;
        int k = 0;
#pragma unroll
        for (int c = 0; c < 6; c++) L.out[c][lane] = (OutT)0;
        int e = A0 + t0 + lane;
        if (act) {
            if (lane >= m1) e = L.q[lane - m1];
            k = lane < m1 ? owner(0, t0 + lane) : (int)L.qo[lane - m1];
            // the partner's state and the history are asked for together, before
            // the overlap is known
            const uint32_t bw = a.nj[e];
            double *hp = a.hist + (size_t)e * DN;
            double bh[HN];
            slots_load<DN>(hp, bh);   // allocated, whatever it holds
            const int j = (int)(bw & kJMask);
            const double4 bx = a.xr[j];
            double4 bv, bs;
            if (MIXED && a.rec) {
                const float4 r0 = a.rec[2 * (size_t)j], r1 = a.rec[2 * (size_t)j + 1];
                bv = make_double4(r0.x, r0.y, r0.z, r0.w);
                bs = make_double4(r1.x, r1.y, r1.z, (double)__float_as_int(r1.w));
            } else {
                bv = a.vm[j];
                bs = a.wt[j];
            }
            const double4 pi = L.x[k];
            const int code = (int)((bw >> 26) & 31u);
            double xj0 = bx.x, xj1 = bx.y, xj2 = bx.z;
            if (code != kNoShift) {
                const double3 im = image_of(bx, code, M.prd);
                xj0 = im.x; xj1 = im.y; xj2 = im.z;
            }
            ContactIn c;
            c.delta[0] = pi.x - xj0;
            c.delta[1] = pi.y - xj1;
            c.delta[2] = pi.z - xj2;
            const double rsq = c.delta[0] * c.delta[0] + c.delta[1] * c.delta[1] + c.delta[2] * c.delta[2];
            c.radsum = pi.w + bx.w;
            touch = rsq < c.radsum * c.radsum;
            if (touch) {
                const double4 vmi = L.v[k], wi = L.w[k];
                const int metai = (int)wi.w, metaj = (int)bs.w;
                const double *mat = a.mat + (size_t)meta_inst(metai) * kMatStride;
                c.is_wall = false;
                c.itype = meta_type(metai);
                c.jtype = meta_type(metaj);
                c.radi = pi.w;
                c.radj = bx.w;
                c.mi = vmi.w;
                c.mj = bv.w;
                c.vi[0] = vmi.x; c.vi[1] = vmi.y; c.vi[2] = vmi.z;
                c.wi[0] = wi.x; c.wi[1] = wi.y; c.wi[2] = wi.z;
                c.vj[0] = bv.x; c.vj[1] = bv.y; c.vj[2] = bv.z;
                c.wj[0] = bs.x; c.wj[1] = bs.y; c.wj[2] = bs.z;
                c.deltan_in = 0.0;
                const double r = sqrt(rsq);
                if (r < 1e-20) atomicOr(a.err, 1);
                double meff = c.mi * c.mj / (c.mi + c.mj);
                if (M.freeze_on && meta_frozen(metai)) meff = c.mj;
                if (M.freeze_on && meta_frozen(metaj)) meff = c.mi;
                c.meff = meff;
                c.r = r;
                c.rinv = 1.0 / r;
                // an unflagged entry has no history yet
                const bool known = (bw & kFlagBit) != 0;
                if (!known)
#pragma unroll
                    for (int q = 0; q < HN; q++) bh[q] = 0.0;
                double dF[3], dT[3];
                if constexpr (MIXED)
                    contact_mixed(M, mat, c, bh, a.shearupdate, dF, dT);
                else
                    contact_fp64<NM, false, RH>(M, M.lp, mat, c, bh, a.shearupdate, dF, dT);
                // the hysteretic models write their state even in set-up passes
                if (a.shearupdate || !known || NM != NM_HERTZ) slots_store<DN>(hp, bh);
                if (!known) a.nj[e] = bw | kFlagBit;
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    L.out[q][lane] = (OutT)dF[q];
                    L.out[3 + q][lane] = (OutT)dT[q];
                }
            } else if (rsq < cdm * c.radsum * c.radsum) {
                // surfacesClose: history reset; a hysteretic chain also clears
                // its contact flag, so the entry no longer carries at a rebuild
                if (!slots_close<NM, DN>(hp)) a.nj[e] = bw & ~kFlagBit;
            }
        }
        const uint64_t tm = __ballot(touch);
        if (tm == 0) return;
        if (mq) {
            if (lane < P) L.run[0][lane] = L.run[1][lane] = 0;
            wave_sync();
            if (act && lane >= m1) {
                if (lane == m1 || L.qo[lane - m1 - 1] != k) L.run[0][k] = (uint8_t)lane;
                if (lane == m1 + mq - 1 || L.qo[lane - m1 + 1] != k) L.run[1][k] = (uint8_t)(lane + 1);
            }
        }
        wave_sync();
        const int pl = lane & (P - 1), part = lane / P;
        const bool sums = pl < np && part < kParts;
        if (sums) {
            const int l0 = max(L.rs[0][pl] - A0 - t0, 0), l1 = min(L.rs[0][pl + 1] - A0 - t0, m1);
            for (int l = l0; l < l1; l++)
#pragma unroll
                for (int c = 0; c < kPer; c++) acc[c] += (double)L.out[part * kPer + c][l];
            if (a.ncontact && l1 > l0) nc += __popcll((tm >> l0) & (l1 - l0 == 64 ? ~0ull : (1ull << (l1 - l0)) - 1ull));
            if (mq) {
                const int q1 = L.run[1][pl];
                for (int l = L.run[0][pl]; l < q1; l++) {
#pragma unroll
                    for (int c = 0; c < kPer; c++) acc[c] += (double)L.out[part * kPer + c][l];
                    nc++;
                }
            }
        }
        wave_sync();
    };

    // test the second range's entries [base, base + 128), touching ones to the queue
    int qlen = 0;
    auto filter = [&](int base) {
        uint32_t w[2];
        double4 pj[2];
        bool in[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            in[u] = base + 64 * u + lane < nB;
            w[u] = in[u] ? a.nj[B0 + base + 64 * u + lane] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 2; u++)
            if (in[u]) pj[u] = a.xr[w[u] & kJMask];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (base + 64 * u >= nB) break;
            const int t = base + 64 * u + lane;
            bool touch = false;
            int k = 0;
            if (in[u]) {
                k = owner(1, nA + t);
                const double4 pi = L.x[k];
                const int code = (int)((w[u] >> 26) & 31u);
                double xj0 = pj[u].x, xj1 = pj[u].y, xj2 = pj[u].z;
                if (code != kNoShift) {
                    const double3 im = image_of(pj[u], code, M.prd);
                    xj0 = im.x; xj1 = im.y; xj2 = im.z;
                }
                const double dx = pi.x - xj0, dy = pi.y - xj1, dz = pi.z - xj2;
                const double rsq = dx * dx + dy * dy + dz * dz;
                const double radsum = pi.w + pj[u].w;
                touch = rsq < radsum * radsum;
                if (!touch && rsq < cdm * radsum * radsum) {   // as in the batch
                    const int e = B0 + t;
                    if (!slots_close<NM, DN>(a.hist + (size_t)e * DN)) a.nj[e] = w[u] & ~kFlagBit;
                }
            }
            const uint64_t bm = __ballot(touch);
            if (touch) {
                const int pos = qlen + __popcll(bm & ((1ull << lane) - 1ull));
                L.q[pos] = B0 + t;
                L.qo[pos] = (uint8_t)k;
            }
            qlen += __popcll(bm);
            wave_sync();
        }
    };
    // Test the second range while the queue has room, evaluate the first
    // range, with the queue's first entries in its last batch's idle lanes,
    // then what is left of the queue and of the second range: every
    // particle's results come in list order.
    for (int b = 0, t0 = 0;;) {
        if (b < nB && qlen < 64 && (t0 == 0 || t0 == nA)) {
            filter(b);
            b += 128;
            continue;
        }
        const int m1 = min(64, nA - t0);
        const int mq = t0 + m1 == nA ? min(qlen, 64 - m1) : 0;
        if (m1 + mq == 0) break;
        batch(t0, m1, mq);
        t0 += m1;
        qlen -= mq;
        if (mq && qlen) {   // the rest to the front
            int tq[3];
            uint8_t to[3];
#pragma unroll
            for (int u = 0; u < 3; u++)
                if (64 * u + lane < qlen) {
                    tq[u] = L.q[mq + 64 * u + lane];
                    to[u] = L.qo[mq + 64 * u + lane];
                }
            wave_sync();
#pragma unroll
            for (int u = 0; u < 3; u++)
                if (64 * u + lane < qlen) {
                    L.q[64 * u + lane] = tq[u];
                    L.qo[64 * u + lane] = to[u];
                }
            wave_sync();
        }
    }

    // a particle's components back to its own lane
    double F[3], T[3];
#pragma unroll
    for (int c = 0; c < 6; c++) {
        const double v = kParts == 1 ? acc[c % kPer] : __shfl(acc[c % kPer], (c / kPer) * P + (lane & (P - 1)), 64);
        (c < 3 ? F[c] : T[c - 3]) = v;
    }
    if (lane < np) {
        const int i = p0 + lane;
        const double4 pi = L.x[lane], vmi = L.v[lane], wi = L.w[lane];
        const int metai = (int)wi.w;
        const double *mat = a.mat + (size_t)meta_inst(metai) * kMatStride;
        particle_epilogue<MIXED, WN>(a, i, pi, vmi, wi, meta_type(metai), meta_frozen(metai), mat, wm, F, T, nc);
        if (a.fuse) integrate_into(a, i, pi, vmi, wi, F, T);
    }
}

static int padded_blocks(long long threads, int block = kBlock)
{
    long long nb = (threads + block - 1) / block;
    return (int)((nb + 7) & ~7LL);
}

// Waves of a chain's tile kernel that the chip holds at once: 256 CUs of four
// SIMDs, and of a SIMD's 512 registers the law leaves 4 waves (mixed, 128), 3
// (FP64 Hertz, 142; hysteretic/nonlinear1 in tiles of 8 and 16, 162 to 168) or
// 2 (hysteretic/nonlinear2, 198 and more).
static int tile_slots(int nm, int wn, bool mixed)
{
    constexpr int simds = 1024;
    if (nm == NM_HYST2 || wn == NM_HYST2) return 2 * simds;
    return (mixed && wn == NM_HERTZ ? 4 : 3) * simds;
}

// Shape of the pass: ForceArgs::lanes/block (set by the autotuner or by
// hand), else DEM_CONTACT_LANES, else by the particle count.  lanes > 0: lane
// groups of that width per particle (k_force); lanes < 0: tiles of -lanes
// particles per wave (k_force_t).
//
// By the count: a small tile is the shorter chain of batches, a large one
// has fewer half-empty batches and less per-wave work.  The smallest whose
// waves fit the slots is the fastest there, and a few waves past them wait
// for a whole round.  Column of n spheres, us per pass with tiles of
//              n:    8 /   16        n:    8 /   16        n:   16 /   32
//   mixed  28,000 14.6 / 14.8   40,000 19.2 / 16.2  100,000 26.0 / 23.5
//   FP64   24,000 14.2 / 14.9   28,000 18.2 / 15.3   60,000 22.3 / 19.8
//   nl1    24,000 17.6 / 18.2   28,000 21.3 / 18.5   60,000 27.6 / 25.6
//   nl2    16,000 15.3 / 15.7   18,000 20.4 / 15.7   40,000 23.9 / 22.5
// and 16 / 32 on the near side: mixed 60,000 18.4 / 18.9, FP64 48,000 17.8 /
// 18.5, nl1 48,000 22.6 / 23.6, nl2 32,000 19.7 / 20.5.  From there on 32, and
// in FP64 64 once both keep every slot busy for many rounds (32 / 64: Hertz
// 200,000 42.8 / 46.9, 400,000 71.0 / 72.0, 500,000 87.2 / 83.7; nl1 150,000
// 53.6 / 57.6, 200,000 68.3 / 67.1, 500,000 186 / 170; nl2 150,000 54.3 / 57.3,
// 200,000 69.4 / 67.4, 500,000 185 / 167; mixed 500,000 73.7 / 81.2).
static int tile_by_count(int n, int nm, int wn, bool mixed)
{
    const int slots = tile_slots(nm, wn, mixed);
    if (n <= 8 * slots) return -8;
    if (n <= 16 * slots) return -16;
    return !mixed && n > 400000 ? -64 : -32;
}

// Not every shape is compiled for every chain.  Cohesion models: 4 lanes per
// particle.  Lane groups: Hertz chains with Hertz walls.  Hysteretic walls, a
// rare choice: tiles of 8, 16 and 32 for Hertz pairs (on few particles a tile
// of 32 leaves most of the chip idle: nonlinear1 walls, FP64, 8 / 32: 500 11.3 /
// 15.2, 8000 12.2 / 15.7, 24,000 14.2 / 16.6), 32 for hysteretic ones.
int force_compiled_shape(int g, const Model &M)
{
    if (M.cohesion != CM_OFF) return 4;
    const bool hp = M.lp.normal == NM_HERTZ, hw = M.lw.normal == NM_HERTZ;
    if (g > 0) return hp && hw ? g : -32;
    if (hw || (hp && (g == -8 || g == -16))) return g;
    return -32;
}

static int contact_shape(const ForceArgs &a, bool mixed)
{
    if (a.lanes) return force_compiled_shape(a.lanes, a.M);
    static const int env = [] {
        const char *s = getenv("DEM_CONTACT_LANES");
        const int g = s ? atoi(s) : 0;
        for (int v : {1, 2, 4, 8, 16, -8, -16, -32, -64})
            if (g == v) return g;
        return 0;
    }();
    if (env) return force_compiled_shape(env, a.M);
    return force_compiled_shape(tile_by_count(a.n, a.M.lp.normal, a.M.lw.normal, mixed), a.M);
}

bool force_can_fuse(const ForceArgs &a) { return a.M.cohesion == CM_OFF; }

template <bool MIXED, int NM, int WN, int P>
static void launch_tile(const ForceArgs &a, int B, hipStream_t s)
{
    using OutT = typename std::conditional<MIXED, float, double>::type;
    constexpr int D0 = chain_off_shear(NM) + 3;
    const int nb = padded_blocks(((long long)a.n + P - 1) / P * 64, B);
    const size_t lds = (B / 64) * sizeof(TileLds<P, OutT>);
    if (a.M.dnum == D0) k_force_t<MIXED, NM, WN, D0, P><<<nb, B, lds, s>>>(a);
    else k_force_t<MIXED, NM, WN, D0 + 3, P><<<nb, B, lds, s>>>(a);
}

template <bool MIXED, int NM, int WN>
static void launch_nm(const ForceArgs &a, hipStream_t s)
{
    const int shape = contact_shape(a, MIXED);
    // a tile's wave shares nothing with the others of its block
    const int B = a.block ? a.block : (shape > 0 ? kBlock : 64);
    if constexpr (NM == NM_HERTZ && WN == NM_HERTZ) {
        const int nb = padded_blocks((long long)a.n * (shape > 0 ? shape : 1), B);
        switch (shape) {
        case 1: k_force<MIXED, 1, NM, WN><<<nb, B, 0, s>>>(a); return;
        case 2: k_force<MIXED, 2, NM, WN><<<nb, B, 0, s>>>(a); return;
        case 4: k_force<MIXED, 4, NM, WN><<<nb, B, 0, s>>>(a); return;
        case 8: k_force<MIXED, 8, NM, WN><<<nb, B, 0, s>>>(a); return;
        case 16: k_force<MIXED, 16, NM, WN><<<nb, B, 0, s>>>(a); return;
        default: break;
        }
    }
    if constexpr (NM == NM_HERTZ || WN == NM_HERTZ)
        switch (shape) {
        case -8: launch_tile<MIXED, NM, WN, 8>(a, B, s); return;
        case -16: launch_tile<MIXED, NM, WN, 16>(a, B, s); return;
        default: break;
        }
    if constexpr (WN == NM_HERTZ)
        if (shape == -64) return launch_tile<MIXED, NM, WN, 64>(a, B, s);
    launch_tile<MIXED, NM, WN, 32>(a, B, s);
}

// with a cohesion model: FP64, 4 lanes per particle
template <int NM, int WN>
static void launch_ch(const ForceArgs &a, hipStream_t s)
{
    const int nb = padded_blocks((long long)a.n * 4);
    k_force<false, 4, NM, WN, true><<<nb, kBlock, 0, s>>>(a);
}

template <int NM>
static void launch_ch_wn(const ForceArgs &a, hipStream_t s)
{
    switch (a.M.lw.normal) {
    case NM_HYST1: launch_ch<NM, NM_HYST1>(a, s); break;
    case NM_HYST2: launch_ch<NM, NM_HYST2>(a, s); break;
    default: launch_ch<NM, NM_HERTZ>(a, s); break;
    }
}

template <bool MIXED, int NM>
static void launch_wn(const ForceArgs &a, hipStream_t s)
{
    switch (a.M.lw.normal) {
    case NM_HYST1: launch_nm<MIXED, NM, NM_HYST1>(a, s); break;
    case NM_HYST2: launch_nm<MIXED, NM, NM_HYST2>(a, s); break;
    default: launch_nm<MIXED, NM, NM_HERTZ>(a, s); break;
    }
}

// The mixed form applies to Hertz chains with Hertz-family rolling
// (epsd*); hysteretic chains and cdtnonlinear2 rolling run in FP64.
template <bool MIXED>
static void launch_force(const ForceArgs &a, hipStream_t s)
{
    if (a.n == 0) return;
    if (a.M.cohesion != CM_OFF) {
        switch (a.M.lp.normal) {
        case NM_HYST1: launch_ch_wn<NM_HYST1>(a, s); break;
        case NM_HYST2: launch_ch_wn<NM_HYST2>(a, s); break;
        default: launch_ch_wn<NM_HERTZ>(a, s); break;
        }
        return;
    }
    switch (a.M.lp.normal) {
    case NM_HYST1: launch_wn<false, NM_HYST1>(a, s); break;
    case NM_HYST2: launch_wn<false, NM_HYST2>(a, s); break;
    default:
        if (MIXED && a.M.rolling != 4) launch_wn<true, NM_HERTZ>(a, s);
        else launch_wn<false, NM_HERTZ>(a, s);
        break;
    }
}

void launch_force_fp64(const ForceArgs &a, hipStream_t s) { launch_force<false>(a, s); }
void launch_force_mixed(const ForceArgs &a, hipStream_t s) { launch_force<true>(a, s); }

// ---------------------------------------------------------------------------

// FixMove::initial_integrate / final_integrate, style linear
// (fix_move.cpp:430-490, :900-940): prescribed components follow
// x = x_origin + v * (step - time_origin) * dt with v fixed; the others are
// integrated from the force like fix nve.  It runs before nve/sphere, as
// the fix that the INL scripts define first.
__device__ inline void move_final(const IntegArgs &a, double dtfm, const double4 &f, double4 &v)
{
    if (!(a.mv_style & 1)) v.x += dtfm * f.x;
    if (!(a.mv_style & 2)) v.y += dtfm * f.y;
    if (!(a.mv_style & 4)) v.z += dtfm * f.z;
}

__device__ inline void move_initial(const IntegArgs &a, int i, double dtfm, const double4 &f, double4 &x, double4 &v)
{
    const double4 xo = a.xo[i];
    if (a.mv_style & 1) { v.x = a.mv_val[0]; x.x = xo.x + a.mv_val[0] * a.mv_delta; }
    else { v.x += dtfm * f.x; x.x += a.dtv * v.x; }
    if (a.mv_style & 2) { v.y = a.mv_val[1]; x.y = xo.y + a.mv_val[1] * a.mv_delta; }
    else { v.y += dtfm * f.y; x.y += a.dtv * v.y; }
    if (a.mv_style & 4) { v.z = a.mv_val[2]; x.z = xo.z + a.mv_val[2] * a.mv_delta; }
    else { v.z += dtfm * f.z; x.z += a.dtv * v.z; }
}

template <int MODE>
__global__ void __launch_bounds__(kBlock) k_integrate(IntegArgs a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    long long step = 0;
    if (a.ctl) {
        // a checked period: nothing runs once it halted at or before this
        // step (a later halt is the one this pass may record itself)
        step = a.ctl[a.par];
        const long long h = a.ctl[2];
        if (h != 0 && h <= step) {
            // the counter still advances, so that a later recorded step
            // reads a number past the halt
            if (i == 0) a.ctl[a.par ^ 1] = step + 1;
            return;
        }
        for (int m = 0; m < a.nmove; m++)
            if (i < a.mntri[m]) move_tri(a.mtri[m][i], a.mdx[m][0], a.mdx[m][1], a.mdx[m][2]);
        if (i == 0) a.ctl[a.par ^ 1] = step + 1;
    } else if (a.halt && *a.halt) {
        return;
    }
    if (i >= a.n) return;
    double4 x = a.xr[i];
    double4 v = a.vm[i];
    double4 w = a.wt[i];
    const double4 f = a.f4[i];
    const double4 t = a.t4[i];
    // dtfm = dtf / (rmass*(1.+CAddRhoFluid/density)), CAddRhoFluid = 0
    const double dtfm = a.dtf / (v.w * (1. + 0.0 / 1.0));
    const double dtirotate = a.dtfrotate / (x.w * x.w * v.w);
    const int gm = a.gm ? a.gm[i] : 0;
    const bool moved = a.mv_bit >= 0 && ((gm >> a.mv_bit) & 1);
    const bool integ = a.integ_bit < 0 || ((gm >> a.integ_bit) & 1);
    if (MODE & 2) {  // final_integrate(n)
        if (moved) move_final(a, dtfm, f, v);
        if (integ) {
            v.x += dtfm * f.x; v.y += dtfm * f.y; v.z += dtfm * f.z;
            w.x += dtirotate * t.x; w.y += dtirotate * t.y; w.z += dtirotate * t.z;
        }
    }
    if (MODE & 1) {  // initial_integrate(n+1)
        if (moved) move_initial(a, i, dtfm, f, x, v);
        if (integ) {
            v.x += dtfm * f.x; v.y += dtfm * f.y; v.z += dtfm * f.z;
            x.x += a.dtv * v.x; x.y += a.dtv * v.y; x.z += a.dtv * v.z;
            w.x += dtirotate * t.x; w.y += dtirotate * t.y; w.z += dtirotate * t.z;
        }
        a.xr[i] = x;
        if (a.ctl) {   // Neighbor::check_distance of the next step
            const double4 b = a.xhold[i];
            const double dx = x.x - b.x, dy = x.y - b.y, dz = x.z - b.z;
            if (dx * dx + dy * dy + dz * dz > a.deltasq)
                atomicCAS((unsigned long long *)&a.ctl[2], 0ull, (unsigned long long)(step + 1));
        }
    }
    a.vm[i] = v;
    a.wt[i] = w;
}

__global__ void __launch_bounds__(kBlock) k_pack_rec(const double4 *vm, const double4 *wt, float4 *rec, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double4 v = vm[i], w = wt[i];
    rec[2 * (size_t)i] = make_float4((float)v.x, (float)v.y, (float)v.z, (float)v.w);
    rec[2 * (size_t)i + 1] = make_float4((float)w.x, (float)w.y, (float)w.z, __int_as_float((int)w.w));
}

void launch_pack_rec(const double4 *vm, const double4 *wt, float4 *rec, int n, hipStream_t s)
{
    if (n == 0) return;
    k_pack_rec<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(vm, wt, rec, n);
}

void launch_integrate(const IntegArgs &a, int mode, hipStream_t s)
{
    if (a.n == 0) return;
    int nt = a.n;
    for (int m = 0; m < a.nmove; m++) nt = nt > a.mntri[m] ? nt : a.mntri[m];
    const int nb = (nt + kBlock - 1) / kBlock;
    if (mode == 1) k_integrate<1><<<nb, kBlock, 0, s>>>(a);
    else if (mode == 2) k_integrate<2><<<nb, kBlock, 0, s>>>(a);
    else k_integrate<3><<<nb, kBlock, 0, s>>>(a);
}

__global__ void __launch_bounds__(kBlock) k_check_distance(const double4 *xr, const double4 *xhold, int n,
                                                          double deltasq, int *flag)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double4 a = xr[i], b = xhold[i];
    const double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
    const double rsq = dx * dx + dy * dy + dz * dz;
    if (rsq > deltasq) atomicOr(flag, 1);
}

__global__ void __launch_bounds__(kBlock) k_check_halt(const double4 *xr, const double4 *xhold, int n,
                                                      double deltasq, long long *ctl, int par)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long long *cc = ctl;
    if (cc[2]) return;
    const long long step = cc[par];
    if (i == 0) ctl[par ^ 1] = step + 1;
    const double4 a = xr[i], b = xhold[i];
    const double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
    const double rsq = dx * dx + dy * dy + dz * dz;
    if (rsq > deltasq) atomicCAS((unsigned long long *)&ctl[2], 0ull, (unsigned long long)step);
}

void launch_check_halt(const double4 *xr, const double4 *xhold, int n, double deltasq, long long *ctl, int par,
                       hipStream_t s)
{
    if (n == 0) return;
    k_check_halt<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(xr, xhold, n, deltasq, ctl, par);
}

void launch_check_distance(const double4 *xr, const double4 *xhold, int n, double deltasq, int *flag,
                           hipStream_t s)
{
    if (n == 0) return;
    k_check_distance<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(xr, xhold, n, deltasq, flag);
}


// ---------------------------------------------------------------------------
// fix setforce / fix aveforce.  k_group_sum: each thread walks particles i,
// i + stride, ... in order, a fixed tree sums the block, one partial per
// block; setforce sets its components in the same pass (each particle is read
// and written by one thread).  k_group_total: the partials in block order.
// k_group_apply (aveforce): the average plus the added value.

constexpr int kGroupThreads = 256;

__global__ void __launch_bounds__(kGroupThreads) k_group_sum(GroupForceArgs a)
{
    __shared__ double s_p[4][kGroupThreads];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    const unsigned bit = 1u << a.bit;
    for (int i = blockIdx.x * kGroupThreads + threadIdx.x; i < a.n; i += gridDim.x * kGroupThreads) {
        if (!((unsigned)a.gmask[i] & bit)) continue;
        double4 f = a.f4[i];
        acc[0] += f.x;
        acc[1] += f.y;
        acc[2] += f.z;
        acc[3] += 1.0;
        if (!a.aveforce) {
            if (a.style[0]) f.x = a.val[0];
            if (a.style[1]) f.y = a.val[1];
            if (a.style[2]) f.z = a.val[2];
            a.f4[i] = f;
        }
    }
    for (int c = 0; c < 4; c++) s_p[c][threadIdx.x] = acc[c];
    __syncthreads();
    for (int w = kGroupThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int c = 0; c < 4; c++) s_p[c][threadIdx.x] += s_p[c][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 4) a.part[blockIdx.x * 4 + threadIdx.x] = s_p[threadIdx.x][0];
}

__global__ void k_group_total(GroupForceArgs a, int nb)
{
    if (threadIdx.x >= 4) return;
    double t = 0.0;
    for (int b = 0; b < nb; b++) t += a.part[b * 4 + threadIdx.x];
    a.total[threadIdx.x] = t;
}

__global__ void __launch_bounds__(kBlock) k_group_apply(GroupForceArgs a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    if (!((unsigned)a.gmask[i] & (1u << a.bit))) return;
    const double cnt = a.total[3];
    if (cnt == 0.0) return;
    const int ncount = (int)cnt;
    double4 f = a.f4[i];
    if (a.style[0]) f.x = a.total[0] / ncount + a.val[0];
    if (a.style[1]) f.y = a.total[1] / ncount + a.val[1];
    if (a.style[2]) f.z = a.total[2] / ncount + a.val[2];
    a.f4[i] = f;
}

void launch_group_force(const GroupForceArgs &a, hipStream_t s)
{
    if (a.n == 0) return;
    const int nb = (int)std::min<long long>(kGroupBlocks, ((long long)a.n + kGroupThreads - 1) / kGroupThreads);
    k_group_sum<<<nb, kGroupThreads, 0, s>>>(a);
    k_group_total<<<1, 64, 0, s>>>(a, nb);
    if (a.aveforce) k_group_apply<<<(a.n + kBlock - 1) / kBlock, kBlock, 0, s>>>(a);
}

}  // namespace dem
