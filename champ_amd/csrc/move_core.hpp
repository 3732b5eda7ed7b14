// move_core.hpp -- the Jastrow and AO part of a single-electron move, by
// wavefronts: distances(iel) (distances.f90:3-167), jastrow4e with iflag = 0
// (jastrow4e.f90:3-358) and the radial functions and AOs (basis_fns.f90:8-214).
//
// Lanes take partner electrons, 64 at a time, and each pair's sum over the centres
// is one chain on its lane; sums over partners are taken in their order.  So ln J and
// the AOs do not depend on how many wavefronts share a walker or on which kernel
// asks: a trajectory amplifies roundings (a proposal with a small determinant
// ratio by its inverse), and a sweep, psie and a forced move have to agree.  (Their
// orbitals agree too with the tile form of the contraction in FP64; a tuned split-K or
// FP32 contraction of psie rounds differently from the sweep, which has its own.)
#pragma once
#include "een_poly.hpp"
#include "engine_internal.hpp"

namespace champ {

// Centres whose partner distances are in flight.  A ring, each value loaded again as it
// is taken, waits for one load where a group of centres loaded together waited for all of
// them: 69.7 -> 57.3 ms of moves a sweep of 160 electrons x 4096 walkers, 55.6 -> 51.0 on
// the FP32 path (one centre ahead there), 9.8 -> 8.4 at 256 walkers.  Eight give 55.7,
// 50.7 and 8.8.
#ifndef CHAMP_MOVE_PF
#define CHAMP_MOVE_PF 4
#endif

// Barrier of the wavefronts that share a walker: the block, or one wavefront.
template <bool BLOCK>
__device__ __forceinline__ void team_sync()
{
    if constexpr (BLOCK) __syncthreads();
    else __syncwarp();
}

// LDS of a walker: r, rr, -kap (1 - kap rr) / r, rvec (3) per centre (double),
// then in the arithmetic type the centres' e-e-n tables (value and d/dx, na
// entries each); after the pairs R, R' of each radial instance in their place
template <int N, typename T>
struct MoveLds {
    double *r, *rr, *fm, *rv;
    T *tab, *rad;
    static __host__ __device__ size_t doubles(int NC, int NRI)
    {
        const size_t t = N > 1 ? (size_t)2 * een_naz<N>() * NC : 0, q = (size_t)2 * NRI;
        return 6 * (size_t)NC + ((t > q ? t : q) * sizeof(T) + 7) / 8;
    }
    __device__ MoveLds(double *lds, int NC)
    {
        r = lds; rr = r + NC; fm = rr + NC; rv = fm + NC;
        tab = rad = (T *)(lds + 6 * NC);
    }
};

struct MoveGeo {
    int NE, NUP, NC, iel;
    const double *cent;
    const int *iwctype;
    const JasParams *jas;
};

// Centres, one wavefront: distance of the moved electron at xn, the e-e-n tables
// (een_poly.hpp), and in en[] the e-n term and its gradient.  rnew / rrnew: the
// walker's new distances in memory.
template <int N, typename T>
__device__ __forceinline__ void move_centres(const MoveGeo &g, const MoveLds<N, T> &L, int lane, double xn0, double xn1,
                                             double xn2, double *rnew, double *rrnew, double en[4])
{
    const JasParams &jp = *g.jas;
    const double kap = jp.kap, asymp_r = jp.asymp_r;
    double fs_en = 0, ge0 = 0, ge1 = 0, ge2 = 0;
    for (int c = lane; c < g.NC; c += WAVE) {
        const double rv0 = xn0 - g.cent[3 * c], rv1 = xn1 - g.cent[3 * c + 1], rv2 = xn2 - g.cent[3 * c + 2];
        double r2 = 0;
        r2 = r2 + rv0 * rv0; r2 = r2 + rv1 * rv1; r2 = r2 + rv2 * rv2;
        const double r = sqrt(r2);
        const double rr = scale_r(kap, r);
        const double dd7 = 1.0 - kap * rr;
        L.r[c] = r; L.rr[c] = rr; L.fm[c] = -kap * dd7 / r;
        L.rv[3 * c] = rv0; L.rv[3 * c + 1] = rv1; L.rv[3 * c + 2] = rv2;
        rnew[c] = r;
        rrnew[c] = rr;
        if constexpr (N > 1) een_tables<N, 1, T, double>(jp.c[g.iwctype[c]], 1.0 - kap * rr, L.tab + (size_t)c * 2 * een_naz<N>());
        if (rr != asymp_r) {
            const int it = g.iwctype[c];
            const double *a4 = jp.a4[it];
            double top = a4[0] * rr, topi = a4[0];
            double bot = 1 + a4[1] * rr, boti = a4[1], bot2 = bot * bot;
            double fen = top / bot - jp.ja[it];
            double feni = topi / bot - boti * top / bot2;
            double rprev = rr;  // rri(iord-1)
            for (int iord = 2; iord <= jp.norda; iord++) {
                double rp = powi(rr, iord);
                fen = fen + a4[iord] * rp;
                feni = feni + a4[iord] * iord * rprev;
                rprev = rp;
            }
            feni = feni * dd7 / r;
            fs_en += fen;
            ge0 += feni * rv0; ge1 += feni * rv1; ge2 += feni * rv2;
        }
    }
    en[0] = wave_sum(fs_en); en[1] = wave_sum(ge0); en[2] = wave_sum(ge1); en[3] = wave_sum(ge2);
}

// The pair of the moved electron and electron j on this lane (off: a lane without
// one): value and the gradients on the moved (gi) and on the partner electron (gj).
// rw / rrw: the walker's e-n distances and scaled distances [NC][NE] (FP64), ew its
// pair table (x, gradient factor; FP32, 8 bytes per pair instead of the two).
// T: arithmetic type of the pair loop, the e-e-n tables and the AO values
// (double on the FP64 path, float on the mixed path); distances of the moved
// electron, the state and every sum across lanes stay double, and so does the e-e
// value of a pair: its Pade constants are the same for all pairs, so an FP32 rounding
// of one does not average out over the partners.  With them in FP32 the change of ln J
// of a move against hpsi's FP64 pair sums (60 electrons) was off by -2.0e-6 in the mean,
// 2.1e-6 rms; with the value and the tables (een_tables) formed in FP64 by 4e-10 and
// 6e-8, in the same time (moves of 160 electrons x 4096 walkers 48.2 ms).
template <int N, typename T>
__device__ __forceinline__ void move_pair(const MoveGeo &g, const MoveLds<N, T> &L, const double *xw, double xn0,
                                          double xn1, double xn2, const double *rw, const double *rrw, const float2 *ew,
                                          int j, bool on, double &f, double gi[3], double gj[3])
{
    constexpr int NA = een_naz<N>(), PF = CHAMP_MOVE_PF;
    constexpr bool F32 = sizeof(T) == sizeof(float);
    const int NE = g.NE, NC = g.NC, iel = g.iel;
    const JasParams &jp = *g.jas;
    const double kap = jp.kap, asymp_r = jp.asymp_r;
    const T tkap = (T)kap;
    const int jq = j < NE ? j : 0;
    T fs = 0, sfu = 0, gm[3] = {0, 0, 0}, go[3] = {0, 0, 0};
    const double xd0 = xw[jq], xd1 = xw[NE + jq], xd2 = xw[2 * NE + jq];
    const T xj[3] = {(T)xd0, (T)xd1, (T)xd2};
    T dd1, fuf;
    double fv = 0;  // FP32 path: the e-e value
    {
        const T rmo[3] = {(T)(xn0 - xd0), (T)(xn1 - xd1), (T)(xn2 - xd2)};
        T rij, u;
        double ud = 0;
        if constexpr (F32) {
            double r2 = 0;
            r2 = r2 + (xn0 - xd0) * (xn0 - xd0); r2 = r2 + (xn1 - xd1) * (xn1 - xd1); r2 = r2 + (xn2 - xd2) * (xn2 - xd2);
            const double r = sqrt_inner(r2), x = exp_neg(-kap * r);
            ud = (1.0 - x) * asymp_r;
            rij = (T)r; dd1 = (T)x; u = (T)ud;
        } else {
            T r2 = 0;
            r2 = r2 + rmo[0] * rmo[0]; r2 = r2 + rmo[1] * rmo[1]; r2 = r2 + rmo[2] * rmo[2];
            rij = sqrt(r2);
            u = scale_r<T>(tkap, rij);
            dd1 = switched_from(kap, u);
        }
        fuf = -tkap * dd1 / rij;
        // e-e term (jastrow4e.f90: psi_ee with its u-derivative)
        const int I = j > iel ? j : iel, J = j > iel ? iel : j;
        T sspinn = 1; int isb = 0, ipar = 0;
        if (I < g.NUP || J >= g.NUP) {
            if (jp.nspin2b == 2) isb = 1;
            else if (jp.nocuspb == 0) sspinn = T(0.5);
            ipar = 1;
        }
        if (on && (F32 || u != (T)asymp_r)) {
            const double *b = jp.b[isb];
            T top = sspinn * (T)b[0] * u, topu = sspinn * (T)b[0];
            T bot = 1 + (T)b[1] * u, botu = (T)b[1], bot2 = bot * bot;
            T feeu = topu / bot - botu * top / bot2;
            if constexpr (F32) {
                fv = div_inner(sspinn * b[0] * ud, 1.0 + b[1] * ud) - jp.jb[ipar];
                double upd = ud;
                T up = u;
                for (int iord = 2; iord <= jp.nordb; iord++) {
                    feeu = feeu + (T)b[iord] * (T)iord * up;
                    up = u * up;
                    upd = ud * upd;
                    fv = fv + b[iord] * upd;
                }
                feeu = feeu * dd1 / rij;
            } else {
                T fee = top / bot - (T)jp.jb[ipar];
                T up = u;
                for (int iord = 2; iord <= jp.nordb; iord++) {
                    T un = u * up;
                    fee = fee + (T)b[iord] * un;
                    feeu = feeu + (T)b[iord] * (T)iord * up;
                    up = un;
                }
                feeu = feeu * dd1 / rij;
                fs += fee;
            }
            for (int k = 0; k < 3; k++) { gm[k] += feeu * rmo[k]; go[k] -= feeu * rmo[k]; }
        }
    }
    if constexpr (N > 1) {
        // distances of the partners to the centres, loaded PF centres ahead into a ring
        // (lanes past NE read electron 0)
        double rn[PF], rrn[PF];
        float2 en[PF];
        auto load = [&](int p, int c) {
            if constexpr (F32) {
                en[p] = ew[(size_t)c * NE + jq];
            } else {
                rn[p] = rw[(size_t)c * NE + jq];
                rrn[p] = rrw[(size_t)c * NE + jq];
            }
        };
#pragma unroll
        for (int p = 0; p < PF; p++) load(p, p < NC ? p : 0);
        for (int c0 = 0; c0 < NC; c0 += PF) {
#pragma unroll
            for (int p = 0; p < PF; p++) {
                const int c = c0 + p;
                if (c >= NC) break;
                double rjc = 0, rrjc = 0;
                float2 ejc = make_float2(0.0f, 0.0f);
                if constexpr (F32) ejc = en[p];
                else { rjc = rn[p]; rrjc = rrn[p]; }
                if (c + PF < NC) load(p, c + PF);
                const T *tab = L.tab + (size_t)c * 2 * NA;
                const double rrm = L.rr[c];
                const T fmf = (T)L.fm[c];
                const T rvm0 = (T)L.rv[3 * c], rvm1 = (T)L.rv[3 * c + 1], rvm2 = (T)L.rv[3 * c + 2];
                const T cx = (T)g.cent[3 * c], cy = (T)g.cent[3 * c + 1], cz = (T)g.cent[3 * c + 2];
                if (!on) continue;
                T swj;
                if constexpr (F32) {
                    swj = ejc.x;
                    if (rrm == asymp_r && swj == 0.0f) continue;
                } else {
                    if (rrm == asymp_r && rrjc == asymp_r) continue;
                    swj = (T)(1.0 - kap * rrjc);
                }
                const EenOut<T> e = een_eval_tab<N, 1, T>(tab, dd1, swj);
                fs += e.f;
                sfu += e.fu;
                const T fmv = e.fx * fmf;
                T fot;
                if constexpr (F32) fot = e.fy * ejc.y;
                else fot = e.fy * (-tkap * swj) / (T)rjc;
                gm[0] += fmv * rvm0; gm[1] += fmv * rvm1; gm[2] += fmv * rvm2;
                go[0] += fot * (xj[0] - cx); go[1] += fot * (xj[1] - cy);
                go[2] += fot * (xj[2] - cz);
            }
        }
    }
    const T fu = sfu * fuf;
    const T rmo[3] = {(T)(xn0 - (double)xj[0]), (T)(xn1 - (double)xj[1]), (T)(xn2 - (double)xj[2])};
    for (int k = 0; k < 3; k++) { gi[k] = (double)(gm[k] + fu * rmo[k]); gj[k] = (double)(go[k] - fu * rmo[k]); }
    f = fv + (double)fs;
}

// R, R' of the radial instances tid, tid + nthr, ... at the moved electron
template <int N, typename T>
__device__ __forceinline__ void move_radial(const MoveLds<N, T> &L, int tid, int nthr, const SplineTab &tab, int NRI,
                                            const int *ri_cent, const int *ri_type, const int *ri_rad,
                                            const double *ri_rmax)
{
    for (int ri = tid; ri < NRI; ri += nthr) {
        const double r = L.r[ri_cent[ri]];
        T wfv[3] = {T(0), T(0), T(0)};
        if (r <= ri_rmax[ri]) splfit_jx<T>(tab, ri_type[ri], ri_rad[ri], (T)r, grid_jx(tab, r), wfv, 1);
        L.rad[2 * ri] = wfv[0]; L.rad[2 * ri + 1] = wfv[1];
    }
}

// AO m of the moved electron: value and gradient (basis_fns ider = 1)
template <int N, typename T>
__device__ __forceinline__ void move_ao(const MoveLds<N, T> &L, int c, int ri, int code, T out[5])
{
    const T wfv[3] = {L.rad[2 * ri], L.rad[2 * ri + 1], T(0)};
    out[0] = out[1] = out[2] = out[3] = T(0);
    if (wfv[0] != T(0) || wfv[1] != T(0))  // else beyond the cut radius: exactly zero
        ao_combine<T>(code, (T)L.rv[3 * c], (T)L.rv[3 * c + 1], (T)L.rv[3 * c + 2], (T)L.r[c], wfv, 1, out);
}

}  // namespace champ
