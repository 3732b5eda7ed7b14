// engine_kernels.hip -- FP64 walker-population kernels of the per-move path.
//
// Layout (walker-major, lanes run over the innermost index):
//   xT[w][3][NE], r_en/rr_en[w][NC][NE], fso[w][NE][NE] (symmetric),
//   g1/g2[w][NE][3][NE] (pair gradients on the first/second electron),
//   vjT[w][3][NE], slmi[w][2][NM][NM] (row i = electron, CHAMP slmi(j+(i-1)n)),
//   dorb[w][NE][3][NO].
// These kernels serve psie, forced moves and the sweeps of multideterminant trial
// functions, whose AO->MO contractions are population-wide GEMMs; the sweeps of one
// determinant are engine_sweep.hip.
#include "engine_internal.hpp"
#include "move_args.hpp"
#include "move_core.hpp"

#include <algorithm>
#include <cmath>

namespace champ {

// ------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_drift_old(MoveArgs a)
{
    const int lane = threadIdx.x % WAVE;
    const int w = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (w >= a.W) return;
    double v[3];
    drift_old(a, w, a.iel, lane, v);
    if (lane == 0) for (int k = 0; k < 3; k++) a.vold[3 * w + k] = v[k];
}

// ------------------------------------------------------------------------
// Move kernel A, a wavefront per 64 partner electrons of a walker (at most four; BLOCK)
// or one wavefront per walker:
//   mode 0: proposal from the drift at the old position: metrop1 (3 gauss
//           draws; metrop_mov1_driftdif.f90:105-117) or metrop6 (local
//           spherical move about the nearest nucleus; metrop6.hpp);
//   mode 1: xnew given.
//   then distances(iel) (distances.f90:3-167), jastrow4e with iflag=0
//   (jastrow4e.f90:3-358) and basis_fns(iel, ider=1) (basis_fns.f90:8-214)
//   writing the AO block that the MO GEMM contracts (orbitalse).
// The sweeps of one determinant take k_sweep (engine_sweep.hip) instead.
// A wavefront per 64 partners instead of one per walker: 256 electrons x 384
// walkers 188 -> 73 us.  Up to 64 electrons a walker has one wavefront, without the
// block's barriers, and above 512 walkers four of them share a block (launch_move_a_n).
// Waves per SIMD asked of the register allocator: four at order 5 on the FP32 path, which
// misses them by five registers (97 electrons x 2048 walkers 49 us, with three 60).
#ifndef CHAMP_MOVE_WPE
#define CHAMP_MOVE_WPE (NORDC == 5 && sizeof(T) == sizeof(float) ? 4 : 1)
#endif

template <int NORDC, typename T, bool BLOCK>
__global__ void __launch_bounds__(256) CHAMP_WAVES_PER_EU(CHAMP_MOVE_WPE) k_move_a(MoveArgs a)
{
    HIP_DYNAMIC_SHARED(double, lds)
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wv = BLOCK ? wave : 0;
    const int nthr = BLOCK ? blockDim.x : WAVE, nwv = nthr / WAVE, tid = BLOCK ? threadIdx.x : lane;
    const int w = BLOCK ? blockIdx.x : blockIdx.x * (blockDim.x / WAVE) + wave;
    if (!BLOCK && w >= a.W) return;
    const int NE = a.NE, NC = a.NC, iel = a.iel;
    const size_t nlds = MoveLds<NORDC, T>::doubles(NC, a.NRI);
    const MoveLds<NORDC, T> L(BLOCK ? lds : lds + wave * nlds, NC);
    // per 64 partners and lane: changes of the moved electron's sums [slot][4][WAVE]
    double *Ldelta = lds + nlds;  // BLOCK
    __shared__ double s_move[3];  // the proposal
    const MoveGeo geo{NE, a.NUP, NC, iel, a.cent, a.iwctype, a.jas};
    const double *xw = a.xT + (size_t)w * 3 * NE;
    double xn0 = 0, xn1 = 0, xn2 = 0, en[4];
    if (wv == 0) {
        if (a.mode == 0) {
            propose<0>(a, w, iel, lane, xw, xn0, xn1, xn2);
            xn0 = __shfl(xn0, 0, WAVE); xn1 = __shfl(xn1, 0, WAVE); xn2 = __shfl(xn2, 0, WAVE);
        } else {
            xn0 = a.xnew[3 * w]; xn1 = a.xnew[3 * w + 1]; xn2 = a.xnew[3 * w + 2];
        }
        move_centres<NORDC, T>(geo, L, lane, xn0, xn1, xn2, a.rnew + (size_t)w * NC, a.rrnew + (size_t)w * NC, en);
        if (BLOCK && lane == 0) { s_move[0] = xn0; s_move[1] = xn1; s_move[2] = xn2; }
    }
    team_sync<BLOCK>();
    if (BLOCK) { xn0 = s_move[0]; xn1 = s_move[1]; xn2 = s_move[2]; }
    const double *fso_row = a.fso + ((size_t)w * NE + iel) * NE;
    const double *g1_row = a.g1 + ((size_t)w * NE + iel) * 3 * NE;
    const double *g2_row = a.g2 + ((size_t)w * NE + iel) * 3 * NE;
    const double *vj = a.vjT + (size_t)w * 3 * NE;
    double *vjn = a.vjnT + (size_t)w * 3 * NE;
    double *fsn = a.fsn_row + (size_t)w * NE;
    double *g1n = a.g1n + (size_t)w * 3 * NE, *g2n = a.g2n + (size_t)w * 3 * NE;
    double d[4] = {0, 0, 0, 0};  // change of the moved electron's sums: value, gradient
    if (wv == 0 && lane == 0) {  // its own entries: the e-n terms
        fsn[iel] = en[0];
        d[0] += en[0] - fso_row[iel];
        for (int k = 0; k < 3; k++) {
            g1n[k * NE + iel] = g2n[k * NE + iel] = en[1 + k];
            d[1 + k] += en[1 + k] - g1_row[k * NE + iel];
        }
    }
    for (int j0 = WAVE * wv; j0 < NE; j0 += WAVE * nwv) {
        const int j = j0 + lane;
        const bool on = j < NE && j != iel;
        double f, gi[3], gj[3], dj[4] = {0, 0, 0, 0};
        move_pair<NORDC, T>(geo, L, xw, xn0, xn1, xn2, a.r_en + (size_t)w * NC * NE, a.rr_en + (size_t)w * NC * NE,
                            a.enp ? a.enp + (size_t)w * NC * NE : nullptr, j, on, f, gi, gj);
        if (on) {
            fsn[j] = f;
            dj[0] = f - fso_row[j];
            for (int k = 0; k < 3; k++) {
                g1n[k * NE + j] = gi[k];
                g2n[k * NE + j] = gj[k];
                vjn[k * NE + j] = vj[k * NE + j] + gj[k] - g2_row[k * NE + j];
                dj[1 + k] = gi[k] - g1_row[k * NE + j];
            }
        }
        if (BLOCK)
            for (int k = 0; k < 4; k++) Ldelta[(size_t)(j0 / WAVE * 4 + k) * WAVE + lane] = dj[k];
        else
            for (int k = 0; k < 4; k++) d[k] += dj[k];
    }
    team_sync<BLOCK>();
    if (wv == 0) {
        if (BLOCK)
            for (int j0 = 0; j0 < NE; j0 += WAVE)  // in the order of the partners
                for (int k = 0; k < 4; k++) d[k] += Ldelta[(size_t)(j0 / WAVE * 4 + k) * WAVE + lane];
        for (int k = 0; k < 4; k++) d[k] = wave_sum(d[k]);
        if (lane == 0) {
            const double fsn_tot = a.fsumo[w] + d[0];
            a.fsumn[w] = fsn_tot;
            a.psijn[w] = fsn_tot;
            for (int k = 0; k < 3; k++) vjn[k * NE + iel] = vj[k * NE + iel] + d[1 + k];
        }
    }
    // ---- AOs of the moved electron (ider = 1) into the GEMM operand, as FP64, or
    // as FP32 for the FP32 contraction (a.ao32)
    move_radial<NORDC, T>(L, tid, nthr, a.tab, a.NRI, a.ri_cent, a.ri_type, a.ri_rad, a.ri_rmax);
    team_sync<BLOCK>();
    double *ao = a.aomove + (size_t)w * 4 * a.NB;
    float *ao32 = (float *)a.aomove + (size_t)w * 4 * a.NB;
    for (int m = tid; m < a.NB; m += nthr) {
        T out[5];
        move_ao(L, a.ao_cent[m], a.ao_ri[m], a.ao_slm[m], out);
        if (a.ao32) {
            for (int k = 0; k < 4; k++) ao32[(size_t)k * a.NB + m] = (float)out[k];
        } else {
            for (int k = 0; k < 4; k++) ao[(size_t)k * a.NB + m] = (double)out[k];
        }
    }
}

// Sherman-Morrison rows of one wave of a 4-wave block: rows wv + 4 r (r < MR,
// i != row), columns lane and lane + WAVE (nel <= 2 WAVE).  Same arithmetic
// as the row-by-row loop; all loads are issued before the reductions.
template <int MR>
__device__ __forceinline__ void sm_rows(double *S, int NM, int nel, int row, double rt, const double *s_row,
                                        const double *s_orb, int wv, int lane)
{
    const bool j0 = lane < nel, j1 = lane + WAVE < nel;
    double v0[MR], v1[MR];
#pragma unroll
    for (int r = 0; r < MR; r++) {
        const int i = wv + 4 * r;
        const bool ok = i < nel && i != row;
        v0[r] = (ok && j0) ? S[(size_t)i * NM + lane] : 0.0;
        v1[r] = (ok && j1) ? S[(size_t)i * NM + lane + WAVE] : 0.0;
    }
    const double o0 = j0 ? s_orb[lane] : 0.0, o1 = j1 ? s_orb[lane + WAVE] : 0.0;
    const double w0 = j0 ? s_row[lane] : 0.0, w1 = j1 ? s_row[lane + WAVE] : 0.0;
#pragma unroll
    for (int r = 0; r < MR; r++) {
        const int i = wv + 4 * r;
        if (i >= nel) break;  // uniform in the wave
        double sum = 0;
        sum += v0[r] * o0;
        sum += v1[r] * o1;
        sum = wave_sum(sum);
        sum = sum / rt;
        if (i == row) continue;
        if (j0) S[(size_t)i * NM + lane] = v0[r] - w0 * sum;
        if (j1) S[(size_t)i * NM + lane + WAVE] = v1[r] - w1 * sum;
    }
}

// ------------------------------------------------------------------------
// Move kernel B, one 256-thread block per walker: determinante ratio
// (determinante.f90:38-46), drift at the new position (iflag_move=0,
// :158-199), metropolis decision (metrop_mov1_driftdif.f90:166-205) and on
// acceptance jassav + detsav with the Sherman-Morrison update applied in
// place (determinante.f90:47-62 + detsav.f90:42-93).
//   mode 0: decide with the walker's stream; 1: compute only; 2: commit acc[w].
//   MR: rows of the inverse per wave held in registers during the update
//   (0: row-by-row loop for spin blocks above 2 WAVE electrons).
template <int MR>
__global__ void __launch_bounds__(256) k_move_b(MoveArgs a)
{
    HIP_DYNAMIC_SHARED(double, lds)
    const int w = blockIdx.x, tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, nwv = blockDim.x / WAVE;
    const int NE = a.NE, NO = a.NO, iel = a.iel;
    const int iab = iel < a.NUP ? 0 : 1, nel = iab ? NE - a.NUP : a.NUP, ish = iab ? a.NUP : 0, row = iel - ish;
    double *S = a.slmi + ((size_t)w * 2 + iab) * a.NM * a.NM;
    const double *ob = a.orbn + (size_t)w * 4 * NO;
    double *s_row = lds, *s_orb = lds + a.NM;
    __shared__ double s_ratio, s_detn;
    __shared__ int s_acc;

    if (wv == 0) {
        const double *srow = S + (size_t)row * a.NM;
        double rt = 0;
        for (int j = lane; j < nel; j += WAVE) rt += srow[j] * ob[a.iworbd[ish + j]];
        rt = wave_sum(rt);
        double v0 = 0, v1 = 0, v2 = 0;
        if (a.md) {
            const double *vc = a.md_vcoln + (size_t)w * NO;
            for (int o = lane; o < NO; o += WAVE) {
                const double sn = vc[o];
                v0 += sn * ob[NO + o]; v1 += sn * ob[2 * NO + o]; v2 += sn * ob[3 * NO + o];
            }
        } else {
            for (int j = lane; j < nel; j += WAVE) {
                const double sn = srow[j] / rt;
                const int jo = a.iworbd[ish + j];
                v0 += sn * ob[NO + jo]; v1 += sn * ob[2 * NO + jo]; v2 += sn * ob[3 * NO + jo];
            }
        }
        v0 = wave_sum(v0); v1 = wave_sum(v1); v2 = wave_sum(v2);
        if (lane == 0) {
            const double *vjn = a.vjnT + (size_t)w * 3 * NE;
            const double vn[3] = {0.0 + v0 + vjn[iel], 0.0 + v1 + vjn[NE + iel], 0.0 + v2 + vjn[2 * NE + iel]};
            double detn;
            const int accept = decide<0>(a, w, iel, rt, vn, a.psijn[w], detn);
            s_ratio = rt; s_detn = detn; s_acc = accept;
        }
    }
    __syncthreads();
    if (!s_acc) return;
    const double rt = s_ratio;
    for (int j = tid; j < nel; j += blockDim.x) {
        s_row[j] = S[(size_t)row * a.NM + j];
        s_orb[j] = ob[a.iworbd[ish + j]];
    }
    __syncthreads();
    // Sherman-Morrison: rows i != iel (all rows of a wave loaded before any
    // is reduced, so their loads are in flight together)
    if constexpr (MR > 0)
        sm_rows<MR>(S, a.NM, nel, row, rt, s_row, s_orb, wv, lane);
    else
        for (int i = wv; i < nel; i += nwv) {
            if (i == row) continue;
            double *Si = S + (size_t)i * a.NM;
            double sum = 0;
            for (int j = lane; j < nel; j += WAVE) sum += Si[j] * s_orb[j];
            sum = wave_sum(sum);
            sum = sum / rt;
            for (int j = lane; j < nel; j += WAVE) Si[j] = Si[j] - s_row[j] * sum;
        }
    for (int j = tid; j < nel; j += blockDim.x) S[(size_t)row * a.NM + j] = s_row[j] / rt;
    // detsav: orbital gradients of iel, spin determinant
    double *dor = a.dorb + ((size_t)w * NE + iel) * 3 * NO;
    for (int t = tid; t < 3 * NO; t += blockDim.x) dor[t] = ob[NO + t];
    if (tid == 0) a.detiab[2 * w + iab] = s_detn;
    // position and distances
    if (tid < 3) a.xT[((size_t)w * 3 + tid) * NE + iel] = a.xnew[3 * w + tid];
    for (int c = tid; c < a.NC; c += blockDim.x) {
        const double rn = a.rnew[(size_t)w * a.NC + c], rrn = a.rrnew[(size_t)w * a.NC + c];
        a.r_en[((size_t)w * a.NC + c) * NE + iel] = rn;
        a.rr_en[((size_t)w * a.NC + c) * NE + iel] = rrn;
        if (a.enp) a.enp[((size_t)w * a.NC + c) * NE + iel] = enp_pack(a.jas->kap, a.jas->asymp_r, rn, rrn);
    }
    // jassav (iflag = 0)
    const double *fsn = a.fsn_row + (size_t)w * NE;
    const double *g1n = a.g1n + (size_t)w * 3 * NE, *g2n = a.g2n + (size_t)w * 3 * NE;
    const double *vjn = a.vjnT + (size_t)w * 3 * NE;
    double *vj = a.vjT + (size_t)w * 3 * NE;
    double *F = a.fso + (size_t)w * NE * NE;
    double *G1 = a.g1 + (size_t)w * NE * 3 * NE, *G2 = a.g2 + (size_t)w * NE * 3 * NE;
    for (int j = tid; j < NE; j += blockDim.x) {
        const double v = fsn[j];
        F[(size_t)iel * NE + j] = v;
        F[(size_t)j * NE + iel] = v;
        for (int k = 0; k < 3; k++) {
            G1[((size_t)iel * 3 + k) * NE + j] = g1n[k * NE + j];
            G2[((size_t)iel * 3 + k) * NE + j] = g2n[k * NE + j];
            G1[((size_t)j * 3 + k) * NE + iel] = g2n[k * NE + j];
            G2[((size_t)j * 3 + k) * NE + iel] = g1n[k * NE + j];
            vj[k * NE + j] = vjn[k * NE + j];
        }
    }
    if (tid == 0) a.fsumo[w] = a.fsumn[w];
}

// ------------------------------------------------------------------------
// rotqua (rotqua.f90:357-430) per walker with its own stream.
__global__ void k_rotqua(int W, int nq, uint64_t *rng, const double *xq0, const double *yq0, const double *zq0,
                         double *xq, double *yq, double *zq)
{
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= W) return;
    uint64_t s[4];
    for (int k = 0; k < 4; k++) s[k] = rng[4 * (size_t)w + k];
    // rejection sampling as in rotqua; the trip cap (probability of reaching
    // it ~ 0.215^1000) only guarantees that every thread finishes
    double x1 = 0, x2 = 0, x3, xsum = 0, cfi, sfi, sthet;
    for (int tries = 0; tries < 1000; tries++) {
        x1 = 1.0 - 2.0 * xo_uniform(s);
        x2 = 1.0 - 2.0 * xo_uniform(s);
        xsum = x1 * x1 + x2 * x2;
        if (xsum < 1.0) break;
    }
    double xsum2 = 2.0 * sqrt(fabs(1.0 - xsum));
    x1 = x1 * xsum2; x2 = x2 * xsum2; x3 = 1.0 - 2.0 * xsum;
    double theta = acos(x3);
    sthet = sin(theta);
    if (sthet < 1.0e-05) { cfi = 1.0; sfi = 0.0; x1 = 0.0; x2 = 0.0; x3 = 1.0; sthet = 0.0; }
    else { cfi = x1 / sthet; sfi = x2 / sthet; }
    double yy1 = x3 * cfi, yy2 = x3 * sfi, yy3 = -sthet, zz1 = -sfi, zz2 = cfi, zz3 = 0.0;
    double u1 = 1, u2 = 0, usum = 1;
    for (int tries = 0; tries < 1000; tries++) {
        u1 = xo_uniform(s) * 2.0 - 1.0;
        u2 = xo_uniform(s) * 2.0 - 1.0;
        usum = u1 * u1 + u2 * u2;
        if (usum < 1.0) break;
    }
    double uu = sqrt(usum);
    u1 = u1 / uu; u2 = u2 / uu;
    double y1 = yy1 * u1 + zz1 * u2, y2 = yy2 * u1 + zz2 * u2, y3 = yy3 * u1 + zz3 * u2;
    double z1 = yy1 * u2 - zz1 * u1, z2 = yy2 * u2 - zz2 * u1, z3 = yy3 * u2 - zz3 * u1;
    for (int iq = 0; iq < nq; iq++) {
        xq[(size_t)w * nq + iq] = xq0[iq] * x1 + yq0[iq] * y1 + zq0[iq] * z1;
        yq[(size_t)w * nq + iq] = xq0[iq] * x2 + yq0[iq] * y2 + zq0[iq] * z2;
        zq[(size_t)w * nq + iq] = xq0[iq] * x3 + yq0[iq] * y3 + zq0[iq] * z3;
    }
    for (int k = 0; k < 4; k++) rng[4 * (size_t)w + k] = s[k];
}

// ------------------------------------------------------------------------
// launchers
static inline int nblocks(int n, int per) { return (n + per - 1) / per; }

// xnew of every walker = the current position of electron iel (a proposal of
// zero length; the autotuner times move steps on it)
__global__ void k_stay(int W, int NE, int iel, const double *xT, double *xnew)
{
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= W) return;
    for (int k = 0; k < 3; k++) xnew[3 * w + k] = xT[((size_t)w * 3 + k) * NE + iel];
}

int launch_stay(champ_ctx *c, int iel)
{
    hipLaunchKernelGGL(k_stay, dim3(nblocks(c->W, 256)), dim3(256), 0, c->stream, c->W, c->NE, iel, c->xT, c->xnew);
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}

int launch_drift_old(champ_ctx *c, int iel)
{
    MoveArgs a = move_args(c, iel, 1, c->tau);
    hipLaunchKernelGGL(k_drift_old, dim3(nblocks(c->W, 4)), dim3(256), 0, c->stream, a);
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}

#ifndef CHAMP_MOVE_PACK  // variant builds: walkers per block of single-wavefront walkers
#define CHAMP_MOVE_PACK 0
#endif
template <int N, typename T>
static int launch_move_a_n(champ_ctx *c, const MoveArgs &a)
{
    const int slots = nblocks(c->NE, WAVE), nwv = std::min(4, slots);
    const size_t tables = MoveLds<N, T>::doubles(c->NC, c->NRI) * sizeof(double);
    if (slots == 1) {
        // up to 512 walkers a block each, so that they spread over the CUs.  us of the
        // kernel with one / four walkers to a block: 60 electrons x 64 21.5 / 23.3, x 1024
        // 27.9 / 27.6; 22 electrons x 512 22.7 / 24.5, x 2000 31.0 / 31.1 (mixed 32.6 / 30.3)
        int wpb = CHAMP_MOVE_PACK ? CHAMP_MOVE_PACK : c->W <= 512 ? 1 : 4;
        while (wpb > 1 && wpb * tables > MOVE_LDS_MAX) wpb /= 2;
        const size_t lds = wpb * tables;
        if (const int rc = move_lds((const void *)k_move_a<N, T, false>, lds)) return rc;
        hipLaunchKernelGGL((k_move_a<N, T, false>), dim3(nblocks(c->W, wpb)), dim3(wpb * WAVE), lds, c->stream, a);
    } else {
        const size_t lds = tables + (size_t)slots * 4 * WAVE * sizeof(double);
        if (const int rc = move_lds((const void *)k_move_a<N, T, true>, lds)) return rc;
        hipLaunchKernelGGL((k_move_a<N, T, true>), dim3(c->W), dim3(nwv * WAVE), lds, c->stream, a);
    }
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}

template <typename T>
static int launch_move_a_t(champ_ctx *c, const MoveArgs &a)
{
    switch (c->hjas.nordc) {
    case 5: return launch_move_a_n<5, T>(c, a);
    case 4: return launch_move_a_n<4, T>(c, a);
    case 3: return launch_move_a_n<3, T>(c, a);
    case 2: return launch_move_a_n<2, T>(c, a);
    default: return launch_move_a_n<0, T>(c, a);
    }
}

int launch_move_a(champ_ctx *c, int iel, int mode)
{
    if (c->hjas.nordc > 5) {
        set_error("move: e-e-n order above 5 is not supported");
        return CHAMP_ERR_UNSUPPORTED;
    }
    int slot;
    tbegin(c, K_MOVE_A, &slot);
    const MoveArgs a = move_args(c, iel, mode, c->tau);
    const int rc = c->prec == CHAMP_PREC_MIXED ? launch_move_a_t<float>(c, a) : launch_move_a_t<double>(c, a);
    tend(c, slot);
    return rc;
}

int launch_move_gemm(champ_ctx *c)
{
    // orbn[w][comp][o] = sum_m aomove[w][comp][m] * coef[o][m]: FP64 matrix cores,
    // or (mixed path, when the autotuner finds it faster) FP32 operands and accumulation
    int slot;
    tbegin(c, K_MOVE_GEMM, &slot);
    int rc = (c->prec == CHAMP_PREC_MIXED && c->tune_gemm[0] == GEMM_F32)
                 ? launch_gemm_f32(c, 4 * c->W, c->NO, c->NB, (const float *)c->aomove, c->NB, c->coef32, c->NB,
                                   c->orbn, c->NO)
                 : launch_gemm(c, true, 4 * c->W, c->NO, c->NB, c->aomove, c->NB, 0, c->coef, c->NB, 0, c->orbn, c->NO,
                               0, 1, c->tune_gemm[0]);
    tend(c, slot);
    return rc;
}

int launch_move_b(champ_ctx *c, int iel, int mode)
{
    MoveArgs a = move_args(c, iel, mode, c->tau);
    size_t lds = (size_t)2 * c->NM * sizeof(double);
    int slot;
    tbegin(c, K_MOVE_B, &slot);
    // rows per wave for the larger spin block (4 waves per block)
    const int nmx = std::max(c->NUP, c->NDN), rpw = (nmx + 3) / 4;
    const dim3 grid(c->W), block(256);
    if (nmx > 2 * WAVE) hipLaunchKernelGGL(k_move_b<0>, grid, block, lds, c->stream, a);
    else if (rpw <= 4) hipLaunchKernelGGL(k_move_b<4>, grid, block, lds, c->stream, a);
    else if (rpw <= 8) hipLaunchKernelGGL(k_move_b<8>, grid, block, lds, c->stream, a);
    else if (rpw <= 12) hipLaunchKernelGGL(k_move_b<12>, grid, block, lds, c->stream, a);
    else if (rpw <= 16) hipLaunchKernelGGL(k_move_b<16>, grid, block, lds, c->stream, a);
    else if (rpw <= 20) hipLaunchKernelGGL(k_move_b<20>, grid, block, lds, c->stream, a);
    else if (rpw <= 24) hipLaunchKernelGGL(k_move_b<24>, grid, block, lds, c->stream, a);
    else hipLaunchKernelGGL(k_move_b<32>, grid, block, lds, c->stream, a);
    tend(c, slot);
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}

int launch_rotqua(champ_ctx *c)
{
    hipLaunchKernelGGL(k_rotqua, dim3(nblocks(c->W, 256)), dim3(256), 0, c->stream, c->W, c->NQ, c->rng, c->xq0,
                       c->yq0, c->zq0, c->xq, c->yq, c->zq);
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}


}  // namespace champ
