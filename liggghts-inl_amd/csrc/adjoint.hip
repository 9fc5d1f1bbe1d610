// adjoint.hip -- reverse-mode gradients of the timestep over a window with a
// fixed neighbour list.
//
// Forward (in the engine): the list built at set-up is kept for the whole
// window; where a rebuild would fall, k_adj_mask does to the contact history
// what the rebuild's carry-over does (keep it only for pairs that touch and
// carry a contact flag, neigh_gran.cpp:592-612), and the distance check
// proves every particle stayed within half the skin, so the list still holds
// every pair that can touch.  The physics is that of normal stepping; only
// the order in which a particle's contact forces are summed differs.
//
// Backward, one step n at a time, from the step's force-pass inputs kept on a
// tape (x_n, v'_n, omega'_n, pair and wall history, list flags):
//   v_n = v'_n + dt/2 f_n / m                 final_integrate
//   f_n = Force(x_n, v'_n, omega'_n, H_{n-1}) contact pass
//   x_n = x_{n-1} + dt v'_n, v'_n = v_{n-1} + dt/2 f_{n-1} / m
// k_adj_step gathers, per particle, the vector-Jacobian products of the
// contact law (contact_adj.h) of its own entries (seeded with its force and
// torque adjoints) and of the reverse entries (seeded with the partner's), so
// every adjoint is written by the thread that owns it: no atomics, the same
// order on every run.  The parameter adjoints (Yeff, Geff, betaeff, mu) are
// summed per particle over the window, then per instance.
#define DEM_HD __host__ __device__
#include "contact_adj.h"
#include "contact_law.h"
#include "kernels.h"

namespace dem {

__global__ void __launch_bounds__(kBlock) k_adj_mask(AdjMaskArgs a)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= a.n) return;
    const double4 pi = a.xr[i];
    const Row row = list_row(a.nstart, a.n, i);
    for (int q = 0; q < row.cnt; q++) {
        const int e = row.entry(q);
        const uint32_t w = a.nj[e];
        const int j = (int)(w & kJMask);
        const int code = (int)((w >> 26) & 31u);
        const double4 pj = a.xr[j];
        double xj0 = pj.x, xj1 = pj.y, xj2 = pj.z;
        if (code != kNoShift) {
            const double3 im = image_of(pj, code, a.prd);
            xj0 = im.x; xj1 = im.y; xj2 = im.z;
        }
        const double dx = pi.x - xj0, dy = pi.y - xj1, dz = pi.z - xj2;
        const double rsq = dx * dx + dy * dy + dz * dz;
        const double radsum = (pi.w + pj.w) * a.cdf;
        const bool keep = (w & kFlagBit) && rsq < radsum * radsum;
        if (!keep) {
            if (w & kFlagBit) a.nj[e] = w & ~kFlagBit;
            for (int k = 0; k < a.dnum; k++) a.hist[(size_t)e * a.dnum + k] = 0.0;
        }
    }
}

// rev[e] = the entry (j -> i) of an entry (i -> j); an image entry's reverse
// carries the opposite image code
__global__ void __launch_bounds__(kBlock) k_adj_rev(const int *nstart, const uint32_t *nj, int *rev, int n)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const Row row = list_row(nstart, n, i);
    for (int k = 0; k < row.cnt; k++) {
        const int e = row.entry(k);
        const uint32_t w = nj[e];
        const int j = (int)(w & kJMask);
        const int mirror = 26 - (int)((w >> 26) & 31u);
        int r = -1;
        const Row rj = list_row(nstart, n, j);
        for (int q = 0; q < rj.cnt; q++) {
            const int f = rj.entry(q);
            const uint32_t u = nj[f];
            if ((int)(u & kJMask) == i && (int)((u >> 26) & 31u) == mirror) {
                r = f;
                break;
            }
        }
        rev[e] = r;
    }
}

__device__ inline LawP law_params(const double *mat, int it, int jt)
{
    LawP p;
    p.Y = tbl(mat, M_YEFF, it, jt);
    p.G = tbl(mat, M_GEFF, it, jt);
    p.B = tbl(mat, M_BETA, it, jt);
    p.MU = tbl(mat, M_MU, it, jt);
    return p;
}

// kAdjLanes lanes per particle, a pair of them per list entry: the even one
// evaluates the particle's own entry, the odd one the reverse entry, and the
// first lanes of the group then add the results, one component each, in entry
// order, own before reverse, from LDS: the sums a single thread walking the
// row would form.  The particle's first lane goes on to the planes.
// One reverse sweep of the law is a chain of several hundred FP64 operations on
// 256 registers and two spilled ones: the chain and two waves per SIMD bound the
// pass.  With a
// thread per particle, 22,793 spheres filled 90 blocks and a pass lasted as
// long as the longest row's two sweeps per contact: 120 us, 60 us now (the
// whole gradient, 400 steps, 77.5 -> 51 ms).  8 lanes give the same there and
// 14.2 ms against 13.0 at 1,838 spheres; three waves per SIMD spill (67 ms).
constexpr int kAdjLanes = 16;
constexpr int kAdjSums = 13;   // d, v, omega (3 each), Yeff, Geff, betaeff, mu
constexpr int kAdjBlock = 128;

__global__ void __launch_bounds__(kAdjBlock, 2) k_adj_step(AdjArgs a)
{
    __shared__ double s_r[kAdjSums][kAdjBlock];
    const int i = (blockIdx.x * kAdjBlock + threadIdx.x) / kAdjLanes;
    if (i >= a.n) return;   // uniform over the group; the rest is within it
    const int g = threadIdx.x & (kAdjLanes - 1);
    const int g0 = threadIdx.x & ~(kAdjLanes - 1);      // the group's first slot
    const int gshift = g0 & 63;
    const bool own = (g & 1) == 0;
    const Model &M = a.M;
    const double4 pi = a.xr[i], vmi = a.vm[i], wti = a.wt[i];
    const int metai = (int)wti.w;
    const int it = meta_type(metai);
    const int inst = meta_inst(metai);
    const double *mat = a.mat + (size_t)inst * kMatStride;
    const double mi = vmi.w, radi = pi.w;
    const double4 lxi = a.lx[i], lvi = a.lv[i], lwi = a.lw[i];
    // force and torque adjoints of this particle (dtf = dt/2, I = 0.4 m r^2)
    const double cf = a.ckick / mi, ct = a.ckick / (0.4 * radi * radi * mi);
    const double gFi[3] = {cf * lvi.x, cf * lvi.y, cf * lvi.z};
    const double gTi[3] = {ct * lwi.x, ct * lwi.y, ct * lwi.z};
    const int dn = a.dnum;
    const Row row = list_row(a.nstart, a.n, i);
    double sum = 0.0;   // of component g, lanes g < kAdjSums
    for (int q0 = 0; q0 < row.cnt; q0 += kAdjLanes / 2) {
        const int q = q0 + (g >> 1);
        bool done = false;   // this lane has a result
        if (q < row.cnt) {
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
            double d[3] = {pi.x - xj0, pi.y - xj1, pi.z - xj2};
            const double rsq = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
            const double radj = pj.w;
            const double radsum = radi + radj;
            if (!(rsq < radsum * radsum)) {
                // no contact: the history passes through unchanged
                if (own) {
                    const bool keep = !a.mask_step || (w & kFlagBit);
                    for (int k = 0; k < dn; k++) {
                        const double h = a.lh[(size_t)e * dn + k];
                        a.lh1[(size_t)e * dn + k] = keep ? h : 0.0;
                    }
                }
            } else {
                // the side this lane evaluates: its entry, state and adjoints
                const int r = own ? e : a.rev[e];
                if (r >= 0) {
                    const double4 vmj = a.vm[j], wtj = a.wt[j];
                    const int jt = meta_type((int)wtj.w);
                    const double mj = vmj.w;
                    const double4 vs = own ? vmi : vmj, vo = own ? vmj : vmi;
                    const double4 ws = own ? wti : wtj, wo = own ? wtj : wti;
                    double gF[3], gT[3];
                    if (own) {
                        for (int k = 0; k < 3; k++) {
                            gF[k] = gFi[k];
                            gT[k] = gTi[k];
                        }
                    } else {
                        const double4 lvj = a.lv[j], lwj = a.lw[j];
                        const double cfj = a.ckick / mj, ctj = a.ckick / (0.4 * radj * radj * mj);
                        gF[0] = cfj * lvj.x; gF[1] = cfj * lvj.y; gF[2] = cfj * lvj.z;
                        gT[0] = ctj * lwj.x; gT[1] = ctj * lwj.y; gT[2] = ctj * lwj.z;
                    }
                    const bool known = ((own ? w : a.nj[r]) & kFlagBit) != 0;
                    const double *h = a.hist + (size_t)r * dn;
                    LawIn in;
                    in.vi[0] = vs.x; in.vi[1] = vs.y; in.vi[2] = vs.z;
                    in.vj[0] = vo.x; in.vj[1] = vo.y; in.vj[2] = vo.z;
                    in.wi[0] = ws.x; in.wi[1] = ws.y; in.wi[2] = ws.z;
                    in.wj[0] = wo.x; in.wj[1] = wo.y; in.wj[2] = wo.z;
                    for (int k = 0; k < 3; k++) {
                        in.d[k] = own ? d[k] : -d[k];
                        in.sh[k] = known ? h[k] : 0.0;
                    }
                    in.radi = own ? radi : radj;
                    in.radj = own ? radj : radi;
                    in.radsum = radsum;
                    in.reff = radi * radj / (radi + radj);
                    in.meff = mi * mj / (mi + mj);
                    in.wall = 0;
                    LawIn g1 = {};
                    LawP gq{0, 0, 0, 0};
                    const double *matS = own ? mat : a.mat + (size_t)meta_inst((int)wtj.w) * kMatStride;
                    law_vjp(in, law_params(matS, own ? it : jt, own ? jt : it), a.dt, a.update, gF, gT,
                            a.lh + (size_t)r * dn, g1, gq);
                    // an entry read as zero history (no flag) does not depend on the
                    // stored values; a rebuild's mask zeroes the unflagged ones
                    if (own)
                        for (int k = 0; k < dn; k++) a.lh1[(size_t)e * dn + k] = known ? g1.sh[k] : 0.0;
                    for (int k = 0; k < 3; k++) {
                        s_r[k][threadIdx.x] = own ? g1.d[k] : -g1.d[k];
                        s_r[3 + k][threadIdx.x] = own ? g1.vi[k] : g1.vj[k];
                        s_r[6 + k][threadIdx.x] = own ? g1.wi[k] : g1.wj[k];
                    }
                    // the parameters' adjoints come from the own side alone
                    s_r[9][threadIdx.x] = own ? gq.Y : 0.0;
                    s_r[10][threadIdx.x] = own ? gq.G : 0.0;
                    s_r[11][threadIdx.x] = own ? gq.B : 0.0;
                    s_r[12][threadIdx.x] = own ? gq.MU : 0.0;
                    done = true;
                }
            }
        }
        uint32_t m = (uint32_t)(__ballot(done) >> gshift) & ((1u << kAdjLanes) - 1u);
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (g < kAdjSums)
            for (; m; m &= m - 1) sum += s_r[g][g0 + __ffs(m) - 1];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (g < kAdjSums) s_r[g][g0] = sum;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // primitive planes (the contact pass's plane loop, backwards): a plane the
    // particle does not touch passes its history on, one lane per plane
    const uint32_t wm = a.P.n ? a.wmask[i] : 0u;
    // selects rather than indexes, so that the vectors stay in registers
    auto along = [&](int d) { return d == 0 ? pi.x : (d == 1 ? pi.y : pi.z); };
    for (int k = g; k < a.P.n; k += kAdjLanes) {
        const double *lhw = a.lhw + ((size_t)i * a.P.n + k) * 3;
        double *lhw1 = a.lhw1 + ((size_t)i * a.P.n + k) * 3;
        const double p = a.P.pos[k], pos = along(a.P.dim[k]);
        const double deltan = (pos > p) ? pos - p - radi : p - pos - radi;
        if (!(wm & (1u << k)) || deltan > M.cutneighmax) {
            for (int q = 0; q < 3; q++) lhw1[q] = lhw[q];
        } else if (deltan > 0.0) {   // history zeroed by the pass
            for (int q = 0; q < 3; q++) lhw1[q] = 0.0;
        }
    }
    if (g != 0) return;
    double ax[3], av[3], aw[3];
    for (int k = 0; k < 3; k++) {
        ax[k] = s_r[k][g0];
        av[k] = s_r[3 + k][g0];
        aw[k] = s_r[6 + k][g0];
    }
    LawP gq{s_r[9][g0], s_r[10][g0], s_r[11][g0], s_r[12][g0]};
    if (wm) {
        const double obs = (a.wseed && a.obs_plane >= 0) ? a.wseed[inst] : 0.0;
        for (int k = 0; k < a.P.n; k++) {
            if (!(wm & (1u << k))) continue;
            const double *lhw = a.lhw + ((size_t)i * a.P.n + k) * 3;
            double *lhw1 = a.lhw1 + ((size_t)i * a.P.n + k) * 3;
            const int d = a.P.dim[k];
            const double p = a.P.pos[k];
            const double pos = along(d);
            const double deltan = (pos > p) ? pos - p - radi : p - pos - radi;
            if (deltan > M.cutneighmax || deltan > 0.0) continue;
            LawIn in = {};
            in.vi[0] = vmi.x; in.vi[1] = vmi.y; in.vi[2] = vmi.z;
            in.wi[0] = wti.x; in.wi[1] = wti.y; in.wi[2] = wti.z;
            for (int q = 0; q < 3; q++) {
                in.d[q] = q == d ? pos - p : 0.0;
                in.sh[q] = a.whist[((size_t)i * a.P.n + k) * a.wdnum + q];
            }
            in.radi = radi;
            in.radj = 0.0;
            in.radsum = radi;
            in.reff = radi;
            in.meff = mi;
            in.wall = 1;
            double gF[3];
            for (int q = 0; q < 3; q++) gF[q] = k == a.obs_plane && q == d ? gFi[q] + obs : gFi[q];
            LawIn g1 = {};
            law_vjp(in, law_params(mat, it, a.P.wtype[k]), a.dt, a.update, gF, gTi, lhw, g1, gq);
            for (int q = 0; q < 3; q++) {
                if (q == d) ax[q] += g1.d[q];
                av[q] += g1.vi[q];
                aw[q] += g1.wi[q];
                // a set-up pass leaves the plane history as it was
                lhw1[q] = g1.sh[q];
            }
        }
    }

    const double lx1[3] = {lxi.x + ax[0], lxi.y + ax[1], lxi.z + ax[2]};
    a.lx1[i] = make_double4(lx1[0], lx1[1], lx1[2], 0.0);
    a.lv1[i] = make_double4(lvi.x + av[0] + a.dt * lx1[0], lvi.y + av[1] + a.dt * lx1[1],
                            lvi.z + av[2] + a.dt * lx1[2], 0.0);
    a.lw1[i] = make_double4(lwi.x + aw[0], lwi.y + aw[1], lwi.z + aw[2], 0.0);
    double *g4 = a.gp + (size_t)i * 4;
    g4[0] += gq.Y;
    g4[1] += gq.G;
    g4[2] += gq.B;
    g4[3] += gq.MU;
}

// seed: lambda_x = w_height[b] / n_b along z for the mean height of instance b
__global__ void __launch_bounds__(kBlock) k_adj_seed(const double4 *wt, const double *wh, const double *count,
                                                    double4 *lx, int n)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int b = meta_inst((int)wt[i].w);
    const double c = count[(size_t)b * 5];
    lx[i] = make_double4(0.0, 0.0, (wh && c > 0.0) ? wh[b] / c : 0.0, 0.0);
}

// per-instance sums of the per-particle parameter adjoints, one block per
// instance over its contiguous range, fixed order
constexpr int kRedThreads = 256;

__global__ void __launch_bounds__(kRedThreads) k_adj_reduce(const int *cstart, int nkl, const double *gp,
                                                           double *out)
{
    __shared__ double s_v[4][kRedThreads];
    const int b = blockIdx.x;
    const int p0 = cstart[(size_t)b * nkl], p1 = cstart[(size_t)(b + 1) * nkl];
    double acc[4] = {0, 0, 0, 0};
    for (int p = p0 + threadIdx.x; p < p1; p += kRedThreads)
        for (int k = 0; k < 4; k++) acc[k] += gp[(size_t)p * 4 + k];
    for (int k = 0; k < 4; k++) s_v[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (int h = kRedThreads / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
            for (int k = 0; k < 4; k++) s_v[k][threadIdx.x] += s_v[k][threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x < 4) out[(size_t)b * 4 + threadIdx.x] = s_v[threadIdx.x][0];
}

static int blocks(long long n) { return (int)((n + kBlock - 1) / kBlock); }

void launch_adj_mask(const AdjMaskArgs &a, hipStream_t s)
{
    if (a.n) k_adj_mask<<<blocks(a.n), kBlock, 0, s>>>(a);
}

void launch_adj_rev(const int *nstart, const uint32_t *nj, int *rev, int n, hipStream_t s)
{
    if (n) k_adj_rev<<<blocks(n), kBlock, 0, s>>>(nstart, nj, rev, n);
}

void launch_adj_step(const AdjArgs &a, hipStream_t s)
{
    constexpr int per = kAdjBlock / kAdjLanes;
    if (a.n) k_adj_step<<<(a.n + per - 1) / per, kAdjBlock, 0, s>>>(a);
}

void launch_adj_seed(const double4 *wt, const double *wh, const double *count, double4 *lx, int n, hipStream_t s)
{
    if (n) k_adj_seed<<<blocks(n), kBlock, 0, s>>>(wt, wh, count, lx, n);
}

void launch_adj_reduce(const int *cstart, int nkl, int ninst, const double *gp, double *out, hipStream_t s)
{
    if (ninst) k_adj_reduce<<<ninst, kRedThreads, 0, s>>>(cstart, nkl, gp, out);
}

}  // namespace dem
