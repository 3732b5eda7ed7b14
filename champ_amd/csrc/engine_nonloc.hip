// engine_nonloc.hip -- ECP quadrature of hpsi over the active (electron,
// centre) pairs of the whole population: nonloc_pot.f90:3-108 and
// nonloc.f90:5-315 with nonlocd_quad (:462-506) and nonlocj_quad4
// (:656-899), single determinant.
//
// One 256-thread block per pair, quadrature points in blocks of QB.  Per
// point q of a pair (i, ic) the kernel needs
//   psi ratio   = sum_m phi_m(x_q) W[i][m],  W = slmi_i . coef (one GEMM per hpsi)
//   log J ratio = sum_{j!=i} [b(u_qj) + sum_c P(u_qj, R_qc, R_jc)]
//                 + sum_c a(R_qc) - sum_j F[i][j]
// with P the e-e-n polynomial.  For a fixed (q, c) the polynomial is written
// as P = sum_k u^k sum_n A_kn(R_qc) R_jc^n (een_poly.hpp), so a lane that owns
// one centre c keeps A in registers for QB points and streams over electrons
// j: about a dozen FMAs per (q, c, j).
//   phase A  lanes over (j, q): u_qj into LDS, e-e sums b(u_qj)
//   phase B  lanes over (c, j-group): e-e-n and e-n sums
//   phase C  lanes over AOs: the psi ratio
// Reductions go lane -> wave (shuffles) -> per-wave slots in LDS -> thread 0,
// in a fixed order, so results do not depend on timing.
#include "een_poly.hpp"
#include "hpsi_args.hpp"

#include <algorithm>
#include <cmath>

namespace champ {

// psianl (nonlpsi.f90:88-105): e-n term at scaled distance rr
__device__ __forceinline__ double en_term(const JasParams &jp, int it, double rr)
{
    if (rr == jp.asymp_r) return 0.0;
    double psi = jp.a4[it][0] * rr / (1.0 + jp.a4[it][1] * rr) - jp.ja[it];
    double rrip = rr;
    for (int o = 2; o <= jp.norda; o++) { rrip = rrip * rr; psi = psi + jp.a4[it][o] * rrip; }
    return psi;
}

// psibnl (nonlpsi.f90:107-133): e-e term of electrons (i, j) at scaled u
__device__ __forceinline__ double ee_term(const JasParams &jp, int nup, int i, int j, double u)
{
    if (u == jp.asymp_r) return 0.0;
    const int I = j > i ? j : i, J = j > i ? i : j;
    double sspinn = 1.0;
    int isb = 0, ipar = 0;
    if (I < nup || J >= nup) {
        if (jp.nspin2b == 2) isb = 1;
        else if (jp.nocuspb == 0) sspinn = 0.5;
        ipar = 1;
    }
    const double *b = jp.b[isb];
    const double fee = b[0] * u / (1.0 + b[1] * u);
    double psi = sspinn * fee - jp.jb[ipar];
    double up = u;
    for (int o = 2; o <= jp.nordb; o++) { up = u * up; psi = psi + b[o] * up; }
    return psi;
}

// lanes of a wave with equal (lane % QB) summed; the result is in lanes 0..QB-1
template <int QB>
__device__ __forceinline__ double strided_sum(double v)
{
#pragma unroll
    for (int off = WAVE / 2; off >= QB; off >>= 1) v += __shfl_xor(v, off, WAVE);
    return v;
}

// Tuning of k_nonloc: quadrature points per block at e-e-n order <= 4 and the
// minimum waves per SIMD asked of the register allocator.
#ifndef CHAMP_NL_QB
#define CHAMP_NL_QB 4
#endif
#ifndef CHAMP_NL_WPE
#define CHAMP_NL_WPE 1
#endif

constexpr int NL_THREADS = 256;
constexpr int NL_WAVES = NL_THREADS / WAVE;

// FP64 on both paths: it subtracts hpsi's pair sums (F, FP64 where a quadrature runs)
// from its own at the points; in FP32 these would round their parameters, which adds up
// over the partners (mixed path, 60 electrons, order 1: energies 6e-7 off their FP64
// values in the median, 1.2e-5 rms over 300 walkers).  160 electrons x 1024 walkers:
// 26.5 ms, in FP32 24.4; 60 electrons x 1000 walkers, order 1: 2.9 ms in either.
template <int NORDC, int QB>
__global__ void __launch_bounds__(NL_THREADS) CHAMP_WAVES_PER_EU(CHAMP_NL_WPE) k_nonloc(HArgs a)
{
    HIP_DYNAMIC_SHARED(double, lds)
    const int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE;
    const int NE = a.NE, NC = a.NC, NQ = a.NQ, NB = a.NB, NRI = a.NRI;
    const JasParams &jp = *a.jas;
    const double kap = jp.kap, asymp = jp.asymp_r;
    double *S = lds;                        // [3][QB][NL_WAVES] per-wave sums: e-e, e-e-n + e-n, psi ratio
    double *XQ = S + 3 * QB * NL_WAVES;     // [QB][3] quadrature points
    double *FI = XQ + 3 * QB;               // [NL_WAVES] partial sums of F[i][.]
    double *GEO = FI + NL_WAVES;            // [QB][NC][5] point - centre: x, y, z, r, grid interval
    double *RAD = GEO + (size_t)QB * NC * 5;  // [QB][NRI] radial functions at the points
    double *U = RAD + (size_t)QB * NRI;     // [NE][QB] switched scaled e-e distances u(q, j)

    // XCD-aware assignment: workgroups are dealt round-robin to the 8 XCDs,
    // so the blocks b = x, x + 8, ... run on XCD x, which takes one contiguous
    // eighth of the pair list; inside it the blocks stride by their count, so
    // the blocks resident at one time work on neighbouring pairs (the same
    // one or two walkers, whose tables stay in that XCD's L2).
    const int G = gridDim.x, b = blockIdx.x;
    const int nx = (G % 8 == 0) ? 8 : 1, gx = G / nx, xcd = b % nx, j0 = b / nx;
    const int total = a.pair_total[0];
    const int per_x = (total + nx - 1) / nx;
    const int x_lo = xcd * per_x, x_hi = min(total, x_lo + per_x);

    for (int t = x_lo + j0; t < x_hi; t += gx) {
        int lo = 0, hi = a.W - 1;
        while (lo < hi) {  // walker: largest w with off[w] <= t
            const int mid = (lo + hi + 1) / 2;
            if (a.pair_off[mid] <= t) lo = mid; else hi = mid - 1;
        }
        const int w = lo;
        const size_t slot = (size_t)w * a.cap + (t - a.pair_off[w]);
        const int i = a.pair_e[slot], ic = a.pair_c[slot];
        const int lp = a.ecp->lpot[a.iwctype[ic]];
        const double *xw = a.xT + (size_t)w * 3 * NE;
        const double *F = a.fso + ((size_t)w * NE + i) * NE;
        const double *Wm = a.wmat + ((size_t)w * NE + i) * NB;
        const double *rrt = a.rrT + (size_t)w * NE * NC;
        const double cx = a.cent[3 * ic], cy = a.cent[3 * ic + 1], cz = a.cent[3 * ic + 2];
        const double rv0 = xw[i] - cx, rv1 = xw[NE + i] - cy, rv2 = xw[2 * NE + i] - cz;
        const double ren = a.r_en[((size_t)w * NC + ic) * NE + i], ri = 1.0 / ren;
        const double *qx = a.xq + (size_t)w * NQ, *qy = a.yq + (size_t)w * NQ, *qz = a.zq + (size_t)w * NQ;

        // sum_j F[i][j]: the old e-e and e-n values of electron i (F symmetric)
        double fs = 0.0;
        for (int j = tid; j < NE; j += NL_THREADS) fs += F[j];
        fs = wave_sum(fs);
        __syncthreads();  // LDS of the previous pair is free
        if (lane == 0) FI[wv] = fs;

        double pair_sum = 0.0;  // meaningful on thread 0
        for (int q0 = 0; q0 < NQ; q0 += QB) {
            if (tid < 3 * QB) {
                const int qq = tid / 3, k = tid % 3, q = min(q0 + qq, NQ - 1);
                const double *qv = k == 0 ? qx : (k == 1 ? qy : qz);
                XQ[tid] = ren * qv[q] + a.cent[3 * ic + k];
            }
            __syncthreads();

            // ---- phase A: u(q, j) and the e-e sums (lane keeps q = tid % QB)
            {
                const int qq = tid % QB;
                const double px = XQ[3 * qq], py = XQ[3 * qq + 1], pz = XQ[3 * qq + 2];
                double see = 0.0;
                for (int j = tid / QB; j < NE; j += NL_THREADS / QB) {
                    const double d0 = xw[j] - px, d1 = xw[NE + j] - py, d2 = xw[2 * NE + j] - pz;
                    double r2 = 0;
                    r2 = r2 + d0 * d0; r2 = r2 + d1 * d1; r2 = r2 + d2 * d2;
                    const double rjq = sqrt(r2);
                    const double u = scale_r<double>(kap, rjq);
                    const double xs = switched_from(kap, u);
                    U[(size_t)j * QB + qq] = xs;
                    if (j != i) see += ee_term(jp, a.NUP, i, j, u);
                }
                const double sees = strided_sum<QB>(see);
                if (lane < QB) S[(0 * QB + lane) * NL_WAVES + wv] = sees;
            }
            __syncthreads();

            // ---- phase B: e-e-n (lanes own a centre, stream over electrons) and e-n
            double acc[QB];
#pragma unroll
            for (int qq = 0; qq < QB; qq++) acc[qq] = 0.0;
            {
                const int CT = NC < NL_THREADS ? NC : NL_THREADS, JG = NL_THREADS / CT;
                for (int c0 = 0; c0 < NC; c0 += CT) {
                    const int c = c0 + tid % CT, jg = tid / CT;
                    if (jg < JG && c < NC) {
                        const int it = a.iwctype[c];
                        const double ecx = a.cent[3 * c], ecy = a.cent[3 * c + 1], ecz = a.cent[3 * c + 2];
                        double A[QB][een_naz<NORDC>()];
                        bool any_asym = false;
                        bool asym[QB];
#pragma unroll
                        for (int qq = 0; qq < QB; qq++) {
                            const double e0 = XQ[3 * qq] - ecx, e1 = XQ[3 * qq + 1] - ecy, e2 = XQ[3 * qq + 2] - ecz;
                            double r2 = 0;
                            r2 = r2 + e0 * e0; r2 = r2 + e1 * e1; r2 = r2 + e2 * e2;
                            const double rq = c == ic ? ren : sqrt(r2);
                            if (jg == 0) {  // geometry of the point seen from centre c, for the AOs
                                double *g = GEO + ((size_t)qq * NC + c) * 5;
                                g[0] = e0; g[1] = e1; g[2] = e2; g[3] = rq;
                                g[4] = (double)grid_jx(a.tab, rq);
                            }
                            const double rr = scale_r<double>(kap, rq);
                            const double xq = switched_from(kap, rr);
                            asym[qq] = rr == asymp;
                            any_asym = any_asym || asym[qq];
                            if (jg == 0 && q0 + qq < NQ) acc[qq] += en_term(jp, it, rr);
                            if constexpr (NORDC > 1) een_tables<NORDC, 0>(jp.c[it], xq, A[qq]);
                        }
                        if constexpr (NORDC > 1) {
                            // one partner of lookahead on the scaled distance
                            double rr_next = jg < NE ? rrt[(size_t)jg * NC + c] : 0.0;
                            for (int j = jg; j < NE; j += JG) {
                                const double rrj = rr_next;
                                if (j + JG < NE) rr_next = rrt[(size_t)(j + JG) * NC + c];
                                if (j == i) continue;
                                const double rj = 1.0 - kap * rrj;
                                const double *uj = U + (size_t)j * QB;
                                double P[QB];
#pragma unroll
                                for (int qq = 0; qq < QB; qq++) P[qq] = een_eval_tab<NORDC, 0>(A[qq], uj[qq], rj).f;
                                if (any_asym && rrj == asymp) {  // psinl: both distances asymptotic -> 0
#pragma unroll
                                    for (int qq = 0; qq < QB; qq++)
                                        if (asym[qq]) P[qq] = 0.0;
                                }
#pragma unroll
                                for (int qq = 0; qq < QB; qq++) acc[qq] += P[qq];
                            }
                        }
                    }
                }
            }
#pragma unroll
            for (int qq = 0; qq < QB; qq++) {
                const double v = wave_sum(acc[qq]);
                if (lane == 0) S[(1 * QB + qq) * NL_WAVES + wv] = v;
            }

            // ---- phase C: psi ratio sum_m phi_m(x_q) W[i][m]; radial functions once
            // per (point, centre, shell), the angular factor per AO
            __syncthreads();  // GEO complete
            for (int tt = tid; tt < QB * NRI; tt += NL_THREADS) {
                const int qq = tt / NRI, ri = tt % NRI;
                const double *g = GEO + ((size_t)qq * NC + a.ri_cent[ri]) * 5;
                double wfv[3] = {0.0, 0.0, 0.0};
                if (g[3] <= a.ri_rmax[ri]) splfit_jx<double>(a.tab, a.ri_type[ri], a.ri_rad[ri], g[3], (int)g[4], wfv, 0);
                RAD[(size_t)qq * NRI + ri] = wfv[0];
            }
            __syncthreads();
            double dr[QB];
#pragma unroll
            for (int qq = 0; qq < QB; qq++) dr[qq] = 0.0;
            for (int m = tid; m < NB; m += NL_THREADS) {
                const int c = a.ao_cent[m], ri = a.ao_ri[m];
                const SlmMono mono = slm_decode(a.ao_slm[m]);  // once per AO, branch-free
                const double wm = Wm[m];
#pragma unroll
                for (int qq = 0; qq < QB; qq++) {
                    const double *g = GEO + ((size_t)qq * NC + c) * 5;
                    const double y = slm_value<double>(mono, g[0], g[1], g[2]);
                    dr[qq] += (y * RAD[(size_t)qq * NRI + ri]) * wm;
                }
            }
#pragma unroll
            for (int qq = 0; qq < QB; qq++) {
                const double v = wave_sum(dr[qq]);
                if (lane == 0) S[(2 * QB + qq) * NL_WAVES + wv] = v;
            }
            __syncthreads();

            // ---- the vpsp_det terms of these points (nonloc.f90:248-274)
            if (tid == 0) {
                double fi = 0.0;
                for (int k = 0; k < NL_WAVES; k++) fi += FI[k];
                for (int qq = 0; qq < QB && q0 + qq < NQ; qq++) {
                    const int q = q0 + qq;
                    double see = 0.0, sen = 0.0, drq = 0.0;
                    for (int k = 0; k < NL_WAVES; k++) {
                        see += S[(0 * QB + qq) * NL_WAVES + k];
                        sen += S[(1 * QB + qq) * NL_WAVES + k];
                        drq += S[(2 * QB + qq) * NL_WAVES + k];
                    }
                    const double fsumn = see + sen - fi;
                    double costh = rv0 * qx[q] + rv1 * qy[q] + rv2 * qz[q];
                    costh = costh * ri;
                    double term_radial = 0.0;
                    for (int l = 1; l <= lp - 1; l++)
                        term_radial = term_radial + yl0(l, costh) * a.pair_vps[slot * CHAMP_MPS_L + l - 1];
                    const double trj = term_radial * a.ecp->wq[q] * exp(fsumn);
                    pair_sum = pair_sum + trj * drq;
                    // t_vpsp of the point (nonloc.f90:297) for DMC's T-moves
                    if (a.tstore) a.pair_psi[slot * NQ + q] = trj * drq;
                }
            }
            __syncthreads();  // S, XQ, U, GEO and RAD are rewritten by the next point block
        }
        if (tid == 0) a.pair_val[slot] = pair_sum;
    }
}

// ------------------------------------------------------------------------
// Matrix-core form of the quadrature's e-e-n sum.  With the split of
// een_poly.hpp the sum of point q (electron i, switched distances x_qb) over
// its partners j is
//   sum_{j != i} sum_{k >= 1} u_qj^k (M_k[q][j] + X_k[q] + Y_k[j])
//     + sum_b sum_n x_qb^n (sum_j C_0n(y_jb) - C_0n(y_ib)),
//   M_k[q][j] = sum_{(b, n)} x_qb^n C_kn(y_jb).
// Only M_k is a product of matrices, a (points x centres*powers) by a
// (centres*powers x partners) one with nc entries per centre (3 at N = 4);
// X_k is formed once per point, Y_k and sum_j C_0n once per walker
// (k_hpsi_vps).  Against a product with all twelve entries of A_kn this runs a
// quarter of the matrix instructions.
// A block takes MMA_GP active pairs of one walker (MMA_GP * NQ <= 48 points:
// three 16-row tiles).  Items (16 partners x 16 points) are dealt to the four
// waves in contiguous runs; up to three items of one partner tile run
// together, so that a lane builds the partner's entries once for them.  An
// item walks the centres four at a time: the four K-slots of an MFMA are four
// centres at one entry (k, n) (lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16]; element r of the accumulator holds the row of Mma::row).
// The partner distances are read from rr_en, partners innermost, so the 16
// lanes of a slot load one line.  The epilogue forms u_qj and the e-e term of
// its 4 x 1 (point, partner) entries and adds to sums in registers, reduced
// over the lanes once per group.
// Bound: the epilogue (square root, exponential and Pade division per
// (point, partner)) on the vector pipe, with the matrix cores beside it (42% and 29%
// busy in FP64, 64% and 21% in FP32); three
// waves per SIMD (168 registers) hide more of both than two.  No form spills a
// register: the thread's number is formed anew for each group and the lane's for each
// item, and machine-level loop-invariant motion is off for this source (build.py);
// else the addresses and constants of every phase stay live through all of them
// (56 registers spilled in FP64 at order 4, 83 at order 5).
// Measured (160 electrons, 40 centres, 4096 walkers): after ten sweeps (about 1e7
// points) 40.7 ms with all entries in the product, 17.1 with the split; FP32 28.8 and
// 13.1.  At the starting positions 13.9 ms with the spills, 13.2 without; FP32 10.9 and
// 9.3.  97 electrons, order 5, 611 walkers: 1.18 and 1.02; FP32 0.83 and 0.67.
constexpr int MMA_GP = NL_GROUP, MMA_MT = 3, MMA_MP = 16 * MMA_MT, MMA_THREADS = 256, MMA_WAVES = MMA_THREADS / WAVE;
constexpr int MMA_TG = MMA_THREADS / MMA_MP;  // thread groups over (point, centre) in the point phase

// accumulator type and instruction per arithmetic type; row of accumulator
// element r in lane slot sl = l / 16 (measured on gfx950 with one-hot
// operands: f64 D[4 r + l / 16][l % 16], f32 D[4 (l / 16) + r][l % 16])
template <typename T> struct Mma;
template <> struct Mma<double> {
    typedef dbl4 acc;
    static __device__ __forceinline__ acc zero() { return dbl4{0.0, 0.0, 0.0, 0.0}; }
    static __device__ __forceinline__ acc op(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ int row(int r, int sl) { return 4 * r + sl; }
};
template <> struct Mma<float> {
    typedef flt4 acc;
    static __device__ __forceinline__ acc zero() { return flt4{0.0f, 0.0f, 0.0f, 0.0f}; }
    static __device__ __forceinline__ acc op(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ int row(int r, int sl) { return 4 * sl + r; }
};

// The e-e term minus its asymptote of the epilogue, per spin class (0 unlike,
// 1 like) in a block's LDS: psi = p0 u / (1 + p1 u) - p2 + u^2 (p3 + u (p4 + ...)),
// the coefficients past nordb zero.  The float form is (u - U)(p0 / (1 + p1 u)
// + p2 + u (p3 + ...)) with u - U = -exp(-kap r) / kap for the distance to the
// asymptote U = 1/kap and the powers of U multiplied out (all of one sign pattern
// with the coefficients): near the asymptote nothing cancels.
constexpr int EE_NP = CHAMP_NORDP + 1;
template <typename T>
__device__ __forceinline__ void ee_table(const JasParams &jp, T *tab)
{
    for (int t = threadIdx.x; t < 2 * EE_NP; t += MMA_THREADS) {
        const int like = t / EE_NP, o = t % EE_NP;
        const double *b = jp.b[(like && jp.nspin2b == 2) ? 1 : 0];
        const double s0 = (like && jp.nspin2b == 1 && jp.nocuspb == 0) ? 0.5 : 1.0, U = jp.asymp_r;
        double v;
        if constexpr (sizeof(T) == sizeof(float)) {
            if (o == 0) v = s0 * b[0] / (1.0 + b[1] * U);
            else if (o == 1) v = b[1];
            else {  // coefficient of u^(o - 2): sum over the orders q >= o of b_q U^(q - 1 - (o - 2))
                v = 0.0;
                for (int q = jp.nordb; q >= 2 && q >= o - 1; q--) v += b[q] * powi(U, q - o + 1);
            }
        } else {
            v = o == 0 ? s0 * b[0] : o == 1 ? b[1] : o == 2 ? jp.jb[like] : (o - 1 <= jp.nordb ? b[o - 1] : 0.0);
        }
        tab[t] = (T)v;
    }
}

template <typename T>
__device__ __forceinline__ T ee_from_table(const T *p, T rr, T u, double asymp_r)
{
    const T pade = div_inner(p[0], T(1) + p[1] * rr);
    if constexpr (sizeof(T) == sizeof(float)) {
        T g = p[EE_NP - 1];
#pragma unroll
        for (int o = EE_NP - 2; o >= 2; o--) g = g * rr + p[o];
        return (T)(-(double)u * asymp_r) * (pade + g);
    } else {
        T g = p[EE_NP - 1];
#pragma unroll
        for (int o = EE_NP - 2; o >= 3; o--) g = g * rr + p[o];
        return rr * pade - p[2] + g * (rr * rr);
    }
}

#ifndef CHAMP_MMA_ILP
#define CHAMP_MMA_ILP 1
#endif

// MTN row tiles from mt0 of the partner tile at j0, added to psum[row tile][r]
template <int N, typename T, int MTN>
__device__ __forceinline__ void mma_item(const HArgs &a, int w, int j0, int mt0, int npts, const double *XP, const T *XQ,
                                         const double *XK, const int *IPT, double (&psum)[MMA_MT][4],
                                         const JasParams &jp, const int *sT, const T *EE)
{
    constexpr EenSplit<N> ES{};
    constexpr int NE_ = ES.nc > 0 ? ES.nc : 1, KC = ES.kmax > 0 ? ES.kmax : 1, NP = een_nsep<N>();
    typedef typename Mma<T>::acc Acc;
    int lane = threadIdx.x % WAVE;
    FORM_AGAIN(lane);
    const int sl = lane / 16, ln = lane % 16;
    const int NC = a.NC, NE = a.NE;
    const double kap = jp.kap;
    const int j = j0 + ln;
    const bool jv = j < NE;
    const int jq = jv ? j : 0;
    Acc acc[MTN][KC];
#pragma unroll
    for (int mt = 0; mt < MTN; mt++)
#pragma unroll
        for (int k = 0; k < KC; k++) acc[mt][k] = Mma<T>::zero();
    if constexpr (ES.nc > 0) {
        const double *rrw = a.rr_en + (size_t)w * NC * NE + jq;
        // partner distances two centre steps ahead
        double ynext = rrw[(size_t)min(sl, NC - 1) * NE], ynext2 = rrw[(size_t)min(sl + 4, NC - 1) * NE];
        for (int b0 = 0; b0 < NC; b0 += 4) {
            const int b = b0 + sl;
            const bool bv = b < NC;
            const double rrb = ynext;
            ynext = ynext2;
            if (b0 + 8 < NC) ynext2 = rrw[(size_t)min(b + 8, NC - 1) * NE];
            // the partner's entries at centre b, used by every row tile; every
            // coupled entry holds a positive power of y, so y = 0 clears the
            // lanes past the partners or the centres (XQ is padded with zeros)
            T yp[N + 1], tab[NE_];
            een_powers<N, T>((bv && jv) ? (T)(1.0 - kap * rrb) : T(0), yp);
            const double *ct = jp.c[bv ? sT[b] : 0];
#pragma unroll
            for (int k = 1; k <= KC; k++)
#pragma unroll
                for (int n = 1; n <= ES.nmax; n++)
                    if (ES.idx[k][n] >= 0) tab[ES.idx[k][n]] = een_coupled<N, T>(ct, yp, k, n);
            T xp[MTN][N + 1];
#pragma unroll
            for (int mt = 0; mt < MTN; mt++) een_powers<N, T>(XQ[(size_t)b * MMA_MP + (mt0 + mt) * 16 + ln], xp[mt]);
            // consecutive MFMAs go to different accumulators (row tile, power of
            // u), so none waits for the previous one's result
#pragma unroll
            for (int n = 1; n <= ES.nmax; n++)
#pragma unroll
                for (int k = 1; k <= KC; k++) {
                    if (ES.idx[k][n] < 0) continue;
#pragma unroll
                    for (int mt = 0; mt < MTN; mt++)
                        acc[mt][k - 1] = Mma<T>::op(xp[mt][n], tab[ES.idx[k][n]], acc[mt][k - 1]);
                }
        }
    }
    const double *xw = a.xT + (size_t)w * 3 * NE;
    const double xj = xw[jq], yj = xw[NE + jq], zj = xw[2 * NE + jq];
    double ys[NP];
#pragma unroll
    for (int k = 0; k < NP; k++) ys[k] = a.een_ys[((size_t)w * NP + k) * NE + jq];
#pragma unroll
    for (int mt = 0; mt < MTN; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            // every lane runs the entry (a branch would keep the entries from
            // overlapping); the ones that do not count are dropped at the end
            const int pt = (mt0 + mt) * 16 + Mma<T>::row(r, sl);
            const int ipt = IPT[pt];  // -1 past the group's points
            const T d0 = (T)(xj - XP[3 * pt]), d1 = (T)(yj - XP[3 * pt + 1]), d2 = (T)(zj - XP[3 * pt + 2]);
            T r2 = 0;
            r2 = r2 + d0 * d0; r2 = r2 + d1 * d1; r2 = r2 + d2 * d2;
            // the switched distance u = exp(-kap r) and the scaled one (1 - u) / kap
            const T u = exp_neg((T)(-kap * (double)sqrt_inner(r2)));
            const T rr = (T(1) - u) * (T)jp.asymp_r;
            T pv = T(0);
#pragma unroll
            for (int k = NP; k >= 1; k--) {
                const T m = (T)(XK[(k - 1) * MMA_MP + pt] + ys[k - 1]);
                pv = pv * u + ((k <= ES.kmax) ? (T)(m + acc[mt][k <= KC ? k - 1 : 0][r]) : m);
            }
            const bool like = (ipt < a.NUP) == (jq < a.NUP);
            const double e = (double)(pv * u) + (double)ee_from_table<T>(EE + (like ? EE_NP : 0), rr, u, jp.asymp_r);
            const double v = (jv && ipt >= 0 && j != ipt) ? e : 0.0;
            if constexpr (MTN == MMA_MT) {
                psum[mt][r] += v;
            } else {
#pragma unroll
                for (int t = 0; t < MMA_MT; t++)
                    if (t == mt0 + mt) psum[t][r] += v;
            }
            // CHAMP_MMA_ILP entries overlap; more would cost a wave of occupancy in registers
            if (r % CHAMP_MMA_ILP == CHAMP_MMA_ILP - 1) __builtin_amdgcn_sched_barrier(0);
        }
}

// LDS of k_nonloc_mma in doubles: XP, SP (e-n and uncoupled sums, e-e and
// e-e-n), partials of the point phase, SW, FI, IPT/PI (as doubles), XK, the
// pairs' k = 0 weights and XQ (tsize bytes per entry, centres padded to four)
__host__ __device__ __forceinline__ size_t mma_lds_doubles(int NC, int nordc, int tsize)
{
    const int np = nordc > 1 ? nordc - 1 : 0, NC4 = (NC + 3) / 4 * 4;
    return 3 * MMA_MP + 2 * MMA_MP + (size_t)(1 + np) * MMA_TG * MMA_MP + MMA_WAVES * MMA_MP + MMA_GP + MMA_MP +
           2 * MMA_GP + (size_t)np * MMA_MP + (size_t)MMA_GP * np * NC + ((size_t)NC4 * MMA_MP * tsize + 7) / 8;
}

#ifndef CHAMP_MMA_WPE
#define CHAMP_MMA_WPE 3
#endif
// T: arithmetic type of the Jastrow terms and of the matrix cores (double on
// the FP64 path, float on the mixed path); the sums over points, centres and
// partners that the split takes out of the product are double.
template <int NORDC, typename T>
__global__ void __launch_bounds__(MMA_THREADS) CHAMP_WAVES_PER_EU(CHAMP_MMA_WPE) k_nonloc_mma(HArgs a)
{
    HIP_DYNAMIC_SHARED(double, lds)
    constexpr int NP = een_nsep<NORDC>();
    static_assert(MMA_GP * 12 <= MMA_MP, "group size");
    const int NE = a.NE, NC = a.NC, NQ = a.NQ, NC4 = (NC + 3) / 4 * 4;
    // the Jastrow parameters and the centres' types in LDS (read before use
    // behind the group loop's first barrier): every centre step of every item
    // reads a type's e-e-n coefficients, every epilogue entry the e-e ones
    __shared__ JasParams sJ;
    __shared__ int sT[128];
    static_assert(sizeof(JasParams) % 8 == 0, "JasParams copied as 8-byte words");
    for (int t = threadIdx.x; t < (int)(sizeof(JasParams) / 8); t += MMA_THREADS)
        reinterpret_cast<unsigned long long *>(&sJ)[t] = reinterpret_cast<const unsigned long long *>(a.jas)[t];
    for (int t = threadIdx.x; t < NC; t += MMA_THREADS) sT[t] = a.iwctype[t];
    __shared__ T sEE[2 * EE_NP];
    ee_table<T>(*a.jas, sEE);
    const JasParams &jp = sJ;
    const double kapd = a.jas->kap;  // read directly: sJ is complete only after a barrier
    double *XP = lds;                                          // [MP][3]
    double *SP = XP + 3 * MMA_MP;                              // [2][MP]: e-n and point sums, e-e and e-e-n
    double *TP = SP + 2 * MMA_MP;                              // [1 + NP][TG][MP] partial sums
    double *SW = TP + (size_t)(1 + NP) * MMA_TG * MMA_MP;      // [WAVES][MP]
    double *FI = SW + MMA_WAVES * MMA_MP;                      // [GP]
    int *IPT = (int *)(FI + MMA_GP);                           // [MP] electron of each point
    int *PI = IPT + 2 * MMA_MP;                                // [GP][4]: i, ic
    double *XK = FI + MMA_GP + MMA_MP + 2 * MMA_GP;            // [NP][MP] X_k of each point
    double *D0 = XK + NP * MMA_MP;                             // [GP][NP][NC] sum_j C_0n(y_jb) - C_0n(y_ib)
    T *XQ = (T *)(D0 + (size_t)MMA_GP * NP * NC);              // [NC4][MP] switched point-centre distances
    for (int t = NC * MMA_MP + threadIdx.x; t < NC4 * MMA_MP; t += MMA_THREADS) XQ[t] = T(0);

    const int G = gridDim.x, bk = blockIdx.x;
    const int nx = (G % 8 == 0) ? 8 : 1, gx = G / nx, xcd = bk % nx, g0 = bk / nx;
    const int total = a.pair_total[1];
    const int per_x = (total + nx - 1) / nx;
    const int x_lo = xcd * per_x, x_hi = min(total, x_lo + per_x);

    for (int gi = x_lo + g0; gi < x_hi; gi += gx) {
        int tid = threadIdx.x;
        FORM_AGAIN(tid);
        const int lane = tid % WAVE, wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
        int lo = 0, hi = a.W - 1;
        while (lo < hi) {  // walker: largest w with grp_off[w] <= gi
            const int mid = (lo + hi + 1) / 2;
            if (a.grp_off[mid] <= gi) lo = mid; else hi = mid - 1;
        }
        const int w = lo;
        const int p0 = MMA_GP * (gi - a.grp_off[w]);
        const int np = min(MMA_GP, a.pair_count[w] - p0), npts = np * NQ;
        const double *xw = a.xT + (size_t)w * 3 * NE;
        __syncthreads();  // LDS of the previous group is free
        if (tid < np) {
            const size_t slot = (size_t)w * a.cap + p0 + tid;
            PI[4 * tid] = a.pair_e[slot];
            PI[4 * tid + 1] = a.pair_c[slot];
        }
        __syncthreads();
        for (int t = tid; t < MMA_MP; t += MMA_THREADS) IPT[t] = t < npts ? PI[4 * (t / NQ)] : -1;
        for (int t = tid; t < 3 * MMA_MP; t += MMA_THREADS) {
            const int pt = t / 3, k = t % 3, p = pt / NQ, q = pt % NQ;
            double v = 0.0;
            if (pt < npts) {
                const int i = PI[4 * p], ic = PI[4 * p + 1];
                const double ren = a.r_en[((size_t)w * NC + ic) * NE + i];
                const double *qv = (k == 0 ? a.xq : (k == 1 ? a.yq : a.zq)) + (size_t)w * NQ;
                v = ren * qv[q] + a.cent[3 * ic + k];
            }
            XP[t] = v;
        }
        if (wv < np) {  // sum_j F[i][j] of each pair
            const double *F = a.fso + ((size_t)w * NE + PI[4 * wv]) * NE;
            double fs = 0.0;
            for (int j = lane; j < NE; j += WAVE) fs += F[j];
            fs = wave_sum(fs);
            if (lane == 0) FI[wv] = fs;
        }
        for (int t = tid; t < np * NC; t += MMA_THREADS) {  // the pairs' weights of x^n (k = 0)
            const int p = t / NC, b = t % NC;
            double yp[NORDC + 1];
            een_powers<NORDC>(1.0 - kapd * a.rr_en[((size_t)w * NC + b) * NE + PI[4 * p]], yp);
            const double *ct = jp.c[sT[b]];
#pragma unroll
            for (int n = 1; n <= NP; n++)
                D0[((size_t)p * NP + n - 1) * NC + b] =
                    a.een_t0[((size_t)w * NP + n - 1) * NC + b] - een_coupled<NORDC>(ct, yp, 0, n);
        }
        __syncthreads();

        // ---- points: x_qb, the e-n sums and the parts of the e-e-n sum that
        // hold one point-centre distance (X_k; the k = 0 terms), in FP64 on both
        // paths: they weigh a whole point, X_k times the sum of its u^k over the
        // partners (13.3 ms of 160 electrons x 4096 walkers in FP64, 12.8 in FP32)
        {
            const int pt = tid % MMA_MP, tg = tid / MMA_MP;
            double sen = 0.0, sx[NP];
#pragma unroll
            for (int k = 0; k < NP; k++) sx[k] = 0.0;
            if (tg < MMA_TG) {
                const bool live = pt < npts;
                const int p = live ? pt / NQ : 0;
                const int i = live ? PI[4 * p] : 0, ic = live ? PI[4 * p + 1] : 0;
                const double px = live ? XP[3 * pt] : 0.0, py = live ? XP[3 * pt + 1] : 0.0;
                const double pz = live ? XP[3 * pt + 2] : 0.0;
                for (int b = tg; b < NC; b += MMA_TG) {
                    double xq = 0.0;
                    if (live) {
                        const double e0 = px - a.cent[3 * b], e1 = py - a.cent[3 * b + 1], e2 = pz - a.cent[3 * b + 2];
                        double r2 = 0;
                        r2 = r2 + e0 * e0; r2 = r2 + e1 * e1; r2 = r2 + e2 * e2;
                        const double rq = b == ic ? a.r_en[((size_t)w * NC + ic) * NE + i] : sqrt_inner(r2);
                        xq = exp_neg(-kapd * rq);
                        const double rr = (1.0 - xq) * jp.asymp_r;
                        sen += en_term(jp, sT[b], rr);
                        double xp[NORDC + 1];
                        een_powers<NORDC>(xq, xp);
                        een_uncoupled<NORDC>(jp.c[sT[b]], xp, sx);
#pragma unroll
                        for (int n = 1; n <= NP; n++) sen += xp[n] * D0[((size_t)p * NP + n - 1) * NC + b];
                    }
                    XQ[(size_t)b * MMA_MP + pt] = (T)xq;
                }
                TP[tg * MMA_MP + pt] = sen;
#pragma unroll
                for (int k = 0; k < NP; k++) TP[((k + 1) * MMA_TG + tg) * MMA_MP + pt] = sx[k];
            }
        }
        __syncthreads();
        for (int t = tid; t < (1 + NP) * MMA_MP; t += MMA_THREADS) {
            const int k = t / MMA_MP, pt = t % MMA_MP;
            double v = 0.0;
            for (int tg = 0; tg < MMA_TG; tg++) v += TP[(k * MMA_TG + tg) * MMA_MP + pt];
            if (k == 0) SP[pt] = v;
            else XK[(k - 1) * MMA_MP + pt] = v;
        }
        __syncthreads();

        // ---- e-e and e-e-n: items (16 partners x 16 points) in contiguous runs of
        // equal length per wave; the wave's sums go to its own row of SW
        {
            double psum[MMA_MT][4];
#pragma unroll
            for (int mt = 0; mt < MMA_MT; mt++)
#pragma unroll
                for (int r = 0; r < 4; r++) psum[mt][r] = 0.0;
            const int NT = (NE + 15) / 16, RT = (npts + 15) / 16, items = NT * RT;
            const int per = (items + MMA_WAVES - 1) / MMA_WAVES, it_hi = min(items, (wv + 1) * per);
            for (int it = wv * per; it < it_hi;) {
                const int tile = it / RT, m0 = it - tile * RT, cnt = min(RT - m0, it_hi - it);
                if (cnt == 3)
                    mma_item<NORDC, T, 3>(a, w, tile * 16, 0, npts, XP, XQ, XK, IPT, psum, jp, sT, sEE);
                else if (cnt == 2)
                    mma_item<NORDC, T, 2>(a, w, tile * 16, m0, npts, XP, XQ, XK, IPT, psum, jp, sT, sEE);
                else
                    mma_item<NORDC, T, 1>(a, w, tile * 16, m0, npts, XP, XQ, XK, IPT, psum, jp, sT, sEE);
                it += cnt;
            }
            // over the 16 partners of a tile (lanes of equal l / 16)
#pragma unroll
            for (int mt = 0; mt < MMA_MT; mt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const double v = row16_sum(psum[mt][r]);
                    if (lane % 16 == 0) SW[wv * MMA_MP + mt * 16 + Mma<T>::row(r, lane / 16)] = v;
                }
        }
        __syncthreads();
        for (int pt = tid; pt < MMA_MP; pt += MMA_THREADS) {
            double v = 0.0;
            for (int k = 0; k < MMA_WAVES; k++) v += SW[k * MMA_MP + pt];
            SP[MMA_MP + pt] = v;
        }
        __syncthreads();

        // ---- the vpsp_det terms (nonloc.f90:248-274): a thread per point
        // forms its term, then a thread per pair sums its points in order
        double *TRJ = TP;  // [MP], free once the point sums are in SP
        if (tid < npts) {
            const int pt = tid, p = pt / NQ, q = pt % NQ, i = PI[4 * p], ic = PI[4 * p + 1];
            const size_t slot = (size_t)w * a.cap + p0 + p;
            const int lp = a.ecp->lpot[sT[ic]];
            const double cx = a.cent[3 * ic], cy = a.cent[3 * ic + 1], cz = a.cent[3 * ic + 2];
            const double rv0 = xw[i] - cx, rv1 = xw[NE + i] - cy, rv2 = xw[2 * NE + i] - cz;
            const double ri = 1.0 / a.r_en[((size_t)w * NC + ic) * NE + i];
            const double *qx = a.xq + (size_t)w * NQ, *qy = a.yq + (size_t)w * NQ, *qz = a.zq + (size_t)w * NQ;
            const double fsumn = SP[pt] + SP[MMA_MP + pt] - FI[p];
            double costh = rv0 * qx[q] + rv1 * qy[q] + rv2 * qz[q];
            costh = costh * ri;
            double term_radial = 0.0;
            for (int l = 1; l <= lp - 1; l++)
                term_radial = term_radial + yl0(l, costh) * a.pair_vps[slot * CHAMP_MPS_L + l - 1];
            const double trj = term_radial * a.ecp->wq[q] * exp(fsumn);
            TRJ[pt] = trj * a.pair_psi[slot * NQ + q];
            // t_vpsp of the point (nonloc.f90:297) for DMC's T-moves
            if (a.tstore) a.pair_psi[slot * NQ + q] = TRJ[pt];
        }
        __syncthreads();
        if (tid < np) {
            const int p = tid;
            double pair_sum = 0.0;
            for (int q = 0; q < NQ; q++) pair_sum = pair_sum + TRJ[p * NQ + q];
            a.pair_val[(size_t)w * a.cap + p0 + p] = pair_sum;
        }
    }
}

// ------------------------------------------------------------------------
// The psi ratio of every quadrature point on its own: sum_m phi_m(x_q) W[i][m]
// (the orbital part of nonloc.f90:224-247, contracted with the inverse row
// once per electron: wmat), for the groups of MMA_GP pairs of k_nonloc_mma.
// The (point, centre) pairs within the centre's largest cut radius (about half
// of them at 160 electrons) are listed per type in LDS, and a lane takes one
// pair: the distance's interval and spline weights once, then every shell of
// the centre, whose values at the node lie together (ShellTab), times its
// angular sum with the W row.  All lanes of a type run the same segments, so
// the angular code is straight.  A lane's result goes to the pair's own slot and
// the slots are added in a fixed order, so the order of the list does not matter.
// Bound: the gathers of the spline tables (16 bytes per shell, node and lane): its waves
// wait 77% of their cycles, vector pipe 36% busy.
// Measured (160 electrons, 40 centres, 4096 walkers): 19.0 ms with a lane
// per (point, radial instance), 11.6 ms now (12.2 at three waves per SIMD, 13.1
// at six: more waves do not help, the table lines are the limit).
constexpr int PSI_MP = MMA_MP, PSI_THREADS = MMA_THREADS;
constexpr int PSI_TG = PSI_THREADS / PSI_MP;

__host__ __device__ __forceinline__ size_t psi_lds_bytes(int NC, int nseg, int nao)
{
    return (3 * PSI_MP + (size_t)PSI_MP * NC + PSI_TG * PSI_MP + nseg) * 8 +
           (2 * MMA_GP + PSI_MP + (size_t)PSI_MP * (NC + NC % 2) + 4 * (size_t)nseg + nao) * 4;
}

// sum over the AOs of a segment of W times the Cartesian monomial; w: the W row
// at the centre's first AO, ao: the segment's AOs
__device__ __forceinline__ double psi_angular(int kind, int code, const int *ao, const double *w, double x, double y,
                                              double z)
{
    const double cs = 0.28209479177387814, cp = 0.48860251190291992;
    const double cd1 = 0.630783130505040, cd2 = 1.092548430592079;
    const double cf = 0.74635266518023078, cf2 = 1.66889529453113635, cf3 = 2.89061144264055405;
    switch (kind) {
    case 0: return cs * w[ao[0]];
    case 1: return cp * (w[ao[0]] * x + w[ao[1]] * y + w[ao[2]] * z);
    case 2:
        return cd1 * (w[ao[0]] * (x * x) + w[ao[3]] * (y * y) + w[ao[5]] * (z * z)) +
               cd2 * (w[ao[1]] * (x * y) + w[ao[2]] * (x * z) + w[ao[4]] * (y * z));
    case 3: {
        const double xx = x * x, yy = y * y, zz = z * z;
        return cf * (w[ao[0]] * (xx * x) + w[ao[6]] * (yy * y) + w[ao[9]] * (zz * z)) +
               cf2 * (xx * (w[ao[1]] * y + w[ao[2]] * z) + yy * (w[ao[3]] * x + w[ao[7]] * z) +
                      zz * (w[ao[5]] * x + w[ao[8]] * y)) + cf3 * (w[ao[4]] * (x * y * z));
    }
    default: return slm_value<double>(slm_decode(code), x, y, z) * w[ao[0]];
    }
}

#ifndef CHAMP_PSI_WPE
#define CHAMP_PSI_WPE 4
#endif
__global__ void __launch_bounds__(PSI_THREADS) CHAMP_WAVES_PER_EU(CHAMP_PSI_WPE) k_nonloc_psi(HArgs a)
{
    HIP_DYNAMIC_SHARED(double, lds)
    const int tid = threadIdx.x, lane = tid % WAVE;
    const int NE = a.NE, NC = a.NC, NQ = a.NQ, NB = a.NB;
    const ShellTab &sh = a.shl;
    const int nrb = a.tab.nrbas_max;
    double *XP = lds;                              // [MP][3]
    double *RES = XP + 3 * PSI_MP;                 // [NC][MP] distance, then the pair's sum
    double *PS = RES + (size_t)PSI_MP * NC;        // [TG][MP] partials
    int *PI = (int *)(PS + PSI_TG * PSI_MP);       // [GP][2]: i, ic
    int *IPT = PI + 2 * MMA_GP;                    // [MP] electron of each point
    int *LIST = IPT + PSI_MP;                      // [NC][MP] pairs in range, by type from tc_off
    __shared__ double sCent[3 * 128];              // nuclear positions (ncent <= 128)
    __shared__ int cnt[CHAMP_MAXCT];
    // the segments of all types, their cut radii and AOs
    double *SRM = (double *)(LIST + (size_t)PSI_MP * NC + (NC & 1) * PSI_MP);
    int *SEG = (int *)(SRM + sh.nseg), *SAO = SEG + 4 * sh.nseg;
    for (int it = 0; it < sh.nct; it++)
        for (int t = sh.seg_off[it] + tid; t < sh.seg_off[it + 1]; t += PSI_THREADS)
            SRM[t] = a.tab.rmaxwf[(size_t)it * nrb + sh.seg[4 * t]];
    for (int t = tid; t < 4 * sh.nseg; t += PSI_THREADS) SEG[t] = sh.seg[t];
    for (int t = tid; t < sh.nao; t += PSI_THREADS) SAO[t] = sh.seg_ao[t];
    for (int t = tid; t < 3 * NC; t += PSI_THREADS) sCent[t] = a.cent[t];
    const int G = gridDim.x, bk = blockIdx.x;
    const int nx = (G % 8 == 0) ? 8 : 1, gx = G / nx, xcd = bk % nx, g0 = bk / nx;
    const int total = a.pair_total[1];
    const int per_x = (total + nx - 1) / nx;
    const int x_lo = xcd * per_x, x_hi = min(total, x_lo + per_x);
    for (int gi = x_lo + g0; gi < x_hi; gi += gx) {
        int lo = 0, hi = a.W - 1;
        while (lo < hi) {  // walker: largest w with grp_off[w] <= gi
            const int mid = (lo + hi + 1) / 2;
            if (a.grp_off[mid] <= gi) lo = mid; else hi = mid - 1;
        }
        const int w = lo;
        const int p0 = MMA_GP * (gi - a.grp_off[w]);
        const int np = min(MMA_GP, a.pair_count[w] - p0), npts = np * NQ;
        __syncthreads();  // LDS of the previous group is free
        if (tid < np) {
            const size_t slot = (size_t)w * a.cap + p0 + tid;
            PI[2 * tid] = a.pair_e[slot];
            PI[2 * tid + 1] = a.pair_c[slot];
        }
        if (tid < CHAMP_MAXCT) cnt[tid] = 0;
        __syncthreads();
        for (int t = tid; t < npts; t += PSI_THREADS) IPT[t] = PI[2 * (t / NQ)];
        for (int t = tid; t < 3 * npts; t += PSI_THREADS) {
            const int pt = t / 3, k = t % 3, p = pt / NQ, q = pt % NQ;
            const int i = PI[2 * p], ic = PI[2 * p + 1];
            const double ren = a.r_en[((size_t)w * NC + ic) * NE + i];
            const double *qv = (k == 0 ? a.xq : (k == 1 ? a.yq : a.zq)) + (size_t)w * NQ;
            XP[t] = ren * qv[q] + sCent[3 * ic + k];
        }
        __syncthreads();
        // ---- the pairs in range; the others' sums are exactly zero
        for (int it = 0; it < sh.nct; it++) {
            const int c0 = sh.tc_off[it], n = (sh.tc_off[it + 1] - c0) * npts;
            const double rmax = sh.rmax[it];
            for (int t0 = 0; t0 < n; t0 += PSI_THREADS) {
                const int t = t0 + tid;
                bool act = false;
                int item = 0;
                if (t < n) {
                    const int c = sh.tc_cent[c0 + t / npts], q = t % npts, p = q / NQ;
                    const double *xp = XP + 3 * q;
                    const double e0 = xp[0] - sCent[3 * c], e1 = xp[1] - sCent[3 * c + 1], e2 = xp[2] - sCent[3 * c + 2];
                    double r2 = 0;
                    r2 = r2 + e0 * e0; r2 = r2 + e1 * e1; r2 = r2 + e2 * e2;
                    const double r = c == PI[2 * p + 1] ? a.r_en[((size_t)w * NC + c) * NE + PI[2 * p]] : sqrt(r2);
                    act = r <= rmax;
                    item = c * PSI_MP + q;
                    RES[item] = act ? r : 0.0;
                }
                const uint64_t m = __ballot(act);
                int base = 0;
                if (lane == 0) base = atomicAdd(&cnt[it], __popcll(m));
                base = __shfl(base, 0, WAVE);
                if (act) LIST[c0 * PSI_MP + base + __popcll(m & ((1ull << lane) - 1))] = item;
            }
        }
        __syncthreads();
        // ---- a lane per listed pair (lanes past the list repeat its last pair)
        for (int it = 0; it < sh.nct; it++) {
            const int n = cnt[it];
            const int *list = LIST + sh.tc_off[it] * PSI_MP;
            const int s0 = sh.seg_off[it], s1 = sh.seg_off[it + 1];
            for (int t0 = 0; t0 < n; t0 += PSI_THREADS) {
                const int t = t0 + tid, item = list[min(t, n - 1)];
                const int c = item / PSI_MP, q = item % PSI_MP;
                const double r = RES[item];
                const double x = XP[3 * q] - sCent[3 * c], y = XP[3 * q + 1] - sCent[3 * c + 1], z = XP[3 * q + 2] - sCent[3 * c + 2];
                const double *wr = a.wmat + ((size_t)w * NE + IPT[q]) * NB + sh.ao_first[c];
                const int jx = grid_jx(a.tab, r);
                const bool inside = jx >= 1 && jx < a.tab.nr;
                double sw[4];
                const int jq = inside ? jx : 1;
                spline_weights(a.tab, r, jq, sw);
                const double *node = sh.tab + ((size_t)it * a.tab.nr + jq - 1) * nrb * 2;
                double sum = 0.0;
                for (int sidx = s0; sidx < s1; sidx++) {
                    const int ir = __builtin_amdgcn_readfirstlane(SEG[4 * sidx]);
                    const int kind = __builtin_amdgcn_readfirstlane(SEG[4 * sidx + 1]);
                    const int first = __builtin_amdgcn_readfirstlane(SEG[4 * sidx + 2]);
                    const int code = __builtin_amdgcn_readfirstlane(SEG[4 * sidx + 3]);
                    if (!(r <= SRM[sidx])) continue;  // beyond the shell's cut radius: exactly zero
                    double R = sw[0] * node[2 * ir] + sw[1] * node[2 * (nrb + ir)] + sw[2] * node[2 * ir + 1] +
                               sw[3] * node[2 * (nrb + ir) + 1];
                    if (!inside) {  // below the grid or on the exponential tail
                        double wfv[3];
                        splfit_jx<double>(a.tab, it, ir, r, jx, wfv, 0);
                        R = wfv[0];
                    }
                    sum += psi_angular(kind, code, SAO + first, wr, x, y, z) * R;
                }
                // the last pair's distance may still be read by lanes past the list
                if (t0 + PSI_THREADS >= n) __syncthreads();
                if (t < n) RES[item] = sum;
            }
        }
        __syncthreads();
        {
            const int q = tid % PSI_MP, s = tid / PSI_MP;
            if (s < PSI_TG && q < npts) {
                double v = 0.0;
                for (int c = s; c < NC; c += PSI_TG) v += RES[c * PSI_MP + q];
                PS[s * PSI_MP + q] = v;
            }
        }
        __syncthreads();
        for (int q = tid; q < npts; q += PSI_THREADS) {
            double v = 0.0;
            for (int k = 0; k < PSI_TG; k++) v += PS[k * PSI_MP + q];
            a.pair_psi[((size_t)w * a.cap + p0 + q / NQ) * NQ + q % NQ] = v;
        }
    }
}

static int launch_psi(champ_ctx *c, const HArgs &a)
{
    const size_t lds = psi_lds_bytes(c->NC, c->shl.nseg, c->shl.nao);
    if (lds > 64 * 1024)
        HIPCHECK(hipFuncSetAttribute((const void *)k_nonloc_psi, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int dev = 0, ncu = 256, per_cu = 1;
    HIPCHECK(hipGetDevice(&dev));
    HIPCHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_nonloc_psi, PSI_THREADS, lds));
    per_cu = std::max(1, per_cu);
    hipLaunchKernelGGL(k_nonloc_psi, dim3(ncu * per_cu), dim3(PSI_THREADS), lds, c->stream, a);
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}

template <int NORDC, typename T>
static int launch_mma(champ_ctx *c, const HArgs &a)
{
    int slot;
    tbegin(c, K_HPSI_PSI, &slot);
    const int rc = launch_psi(c, a);
    tend(c, slot);
    if (rc) return rc;
    const size_t lds = mma_lds_doubles(c->NC, NORDC, (int)sizeof(T)) * sizeof(double);
    if (lds > 160 * 1024) {
        set_error("nonloc: the quadrature kernel's LDS tables exceed 160 KB for this system");
        return CHAMP_ERR_UNSUPPORTED;
    }
    if (lds > 64 * 1024)
        HIPCHECK(hipFuncSetAttribute((const void *)k_nonloc_mma<NORDC, T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int dev = 0, ncu = 256, per_cu = 1;
    HIPCHECK(hipGetDevice(&dev));
    HIPCHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_nonloc_mma<NORDC, T>, MMA_THREADS, lds));
    per_cu = std::max(1, per_cu);
    tbegin(c, K_HPSI_NONLOC, &slot);
    hipLaunchKernelGGL((k_nonloc_mma<NORDC, T>), dim3(ncu * per_cu), dim3(MMA_THREADS), lds, c->stream, a);
    tend(c, slot);
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}

template <int NORDC, int QB>
static int launch_k(champ_ctx *c, const HArgs &a)
{
    const size_t lds = (3 * QB * NL_WAVES + 3 * QB + NL_WAVES + (size_t)QB * c->NC * 5 + (size_t)QB * c->NRI +
                        (size_t)c->NE * QB) *
                       sizeof(double);
    if constexpr (QB > 2)  // fewer points at a time
        if (lds > 160 * 1024) return launch_k<NORDC, 2>(c, a);
    if (lds > 160 * 1024) {
        set_error("nonloc: the quadrature kernel's LDS tables exceed 160 KB for this system");
        return CHAMP_ERR_UNSUPPORTED;
    }
    if (lds > 64 * 1024)
        HIPCHECK(hipFuncSetAttribute((const void *)k_nonloc<NORDC, QB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    // one wave of blocks: as many as can be resident at once
    int dev = 0, ncu = 256, per_cu = 1;
    HIPCHECK(hipGetDevice(&dev));
    HIPCHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_nonloc<NORDC, QB>, NL_THREADS, lds));
    per_cu = std::max(1, per_cu);
    int slot;
    tbegin(c, K_HPSI_NONLOC, &slot);
    hipLaunchKernelGGL((k_nonloc<NORDC, QB>), dim3(ncu * per_cu), dim3(NL_THREADS), lds, c->stream, a);
    tend(c, slot);
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}

static int launch_vector(champ_ctx *c, const HArgs &a)
{
    switch (c->hjas.nordc) {
    case 0: return launch_k<0, CHAMP_NL_QB>(c, a);
    case 1: return launch_k<1, CHAMP_NL_QB>(c, a);
    case 2: return launch_k<2, CHAMP_NL_QB>(c, a);
    case 3: return launch_k<3, CHAMP_NL_QB>(c, a);
    case 4: return launch_k<4, CHAMP_NL_QB>(c, a);
    case 5: return launch_k<5, 2>(c, a);
    default:
        set_error("nonloc: e-e-n order above 5 is not supported");
        return CHAMP_ERR_UNSUPPORTED;
    }
}

#ifndef CHAMP_NL_MMA
#define CHAMP_NL_MMA 1
#endif

// the matrix-core form: up to 12 points per pair (48 points per group), an
// e-e-n polynomial, and the LDS of both its kernels within 160 KB beside the
// static arrays (JasParams and 128 types, nuclear positions)
bool nonloc_on_matrix_cores(const champ_ctx *c)
{
    const size_t most = 160 * 1024 - sizeof(JasParams) - 3 * 128 * sizeof(double) - 512;
    return CHAMP_NL_MMA && c->tune_nonloc != 1 && c->NQ <= 12 && c->hjas.nordc >= 2 && c->hjas.nordc <= 5 &&
           mma_lds_doubles(c->NC, c->hjas.nordc, c->prec == CHAMP_PREC_MIXED ? 4 : 8) * 8 <= most &&
           psi_lds_bytes(c->NC, c->shl.nseg, c->shl.nao) <= most;
}

int launch_nonloc(champ_ctx *c, const HArgs &a)
{
    const bool mixed = c->prec == CHAMP_PREC_MIXED, mma = nonloc_on_matrix_cores(c);
    if (mma && mixed) {
        switch (c->hjas.nordc) {
        case 2: return launch_mma<2, float>(c, a);
        case 3: return launch_mma<3, float>(c, a);
        case 4: return launch_mma<4, float>(c, a);
        default: return launch_mma<5, float>(c, a);
        }
    }
    if (mma) {
        switch (c->hjas.nordc) {
        case 2: return launch_mma<2, double>(c, a);
        case 3: return launch_mma<3, double>(c, a);
        case 4: return launch_mma<4, double>(c, a);
        default: return launch_mma<5, double>(c, a);
        }
    }
    return launch_vector(c, a);
}

}  // namespace champ
