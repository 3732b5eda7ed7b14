// engine_sweep.hip -- the fused sweep of one-determinant trial functions.
//
// Compiled without the machine-level loop-invariant motion (build.py): it lifts
// every lane's addresses and the constants of exp, log and sqrt out of the
// electron loop, which is longer than the registers reach: 82.3 ms of moves a sweep
// of 160 electrons x 4096 walkers with it, 68.7 without.
#include "move_args.hpp"
#include "move_core.hpp"

#include <algorithm>
#include <cmath>

namespace champ {

constexpr int SW_BLOCK = 256;  // threads per block at most

#ifndef CHAMP_SWEEP_WPE
#define CHAMP_SWEEP_WPE 2
#endif

// The kernel's first argument through its segment pointer, which the compiler
// may not take for the one it has read before (the host emulation has no such
// segment and uses the argument).
#ifndef MOVE_ARGS_AGAIN
__device__ __forceinline__ const MoveArgs &move_args_again()
{
    auto p = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const MoveArgs *)p;
}
#define MOVE_ARGS_AGAIN(a) move_args_again()
#endif

// What every move of every walker reads, in the block's LDS: the Jastrow
// parameters, the centres and their types.
struct MoveConst {
    const JasParams *jas;
    const double *cent;
    const int *iwctype;
    static __host__ __device__ size_t doubles(int NC)
    {
        return (sizeof(JasParams) / 8 + 3 * (size_t)NC + (NC + 1) / 2 + 1) / 2 * 2;
    }
    __device__ MoveConst(double *lds, const JasParams *j, const double *c, const int *t, int NC)
    {
        static_assert(sizeof(JasParams) % 8 == 0, "JasParams copied as 8-byte words");
        constexpr int n = sizeof(JasParams) / 8;
        double *lc = lds + n;
        int *lt = (int *)(lc + 3 * NC);
        for (int k = threadIdx.x; k < n; k += blockDim.x) lds[k] = ((const double *)j)[k];
        for (int k = threadIdx.x; k < 3 * NC; k += blockDim.x) lc[k] = c[k];
        for (int k = threadIdx.x; k < NC; k += blockDim.x) lt[k] = t[k];
        jas = (const JasParams *)lds; cent = lc; iwctype = lt;
        __syncthreads();
    }
};

// LDS of a block of wpb walkers with NW wavefronts each, in doubles: MoveConst,
// the walkers' MoveLds, their orbitals [wpb][4][npad] and inverse rows [wpb][npad],
// and two chunks of 64 NW AOs [k][4 wpb + pad] (the pad puts the four k of an
// instruction's operand on different banks), before them the partners' changes
// of the moved electron's sums [NE / 64][4][64] (NW > 1)
template <int N, typename T, int NW>
struct SweepLds {
    static __host__ __device__ int npad(int NM) { return (NM + 15) / 16 * 16; }
    static __host__ __device__ int stride(int wpb) { return 4 * wpb + (wpb == 4 ? 4 : 1); }
    static __host__ __device__ size_t walker(int NC, int NRI) { return (MoveLds<N, T>::doubles(NC, NRI) + 1) / 2 * 2; }
    static __host__ __device__ size_t chunks(int NE, int wpb)
    {
        const size_t a = (size_t)2 * NW * WAVE * stride(wpb), b = NW > 1 ? (size_t)(NE + WAVE - 1) / WAVE * 4 * WAVE : 0;
        return a > b ? a : b;
    }
    static __host__ __device__ size_t doubles(int NC, int NRI, int NM, int NE, int wpb)
    {
        return MoveConst::doubles(NC) + wpb * (walker(NC, NRI) + 5 * (size_t)npad(NM)) + chunks(NE, wpb);
    }
};

// Sum over 64 columns of a row held by 16 lanes, column l + 16 m in p[m], in the
// order of wave_sum over 64 lanes: 32 apart, 16 apart (on the lane), then 8, 4, 2, 1.
__device__ __forceinline__ double row16_sum_as_wave(const double p[4])
{
    double v = (p[0] + p[2]) + (p[1] + p[3]);
    v += dpp_mov<0x128>(v);  // row_ror 8: the lane 8 apart
    v += dpp_mov<0x124>(v);  // row_ror 4: 4 apart, the lanes 8 apart being equal
    v += dpp_mov<0x122>(v);
    v += dpp_mov<0x121>(v);
    return v;
}

// Sherman-Morrison update of a spin's inverse S [nel][NM] but its row `row`:
// S[i] -= (S[i] . orb / rt) srow.  Sixteen lanes take a row, MC columns each
// (nel <= 16 MC), so four rows share a wave and a row's dot product needs four
// register moves; its terms are added in the order of sm_rows (engine_kernels.hip).
// MB groups of rows are loaded before the first is reduced.
template <int MC, int MB>
__device__ __forceinline__ void sm_update(double *S, int NM, int nel, int row, double rt, const double *srow,
                                          const double *orb, int tid, int nthr)
{
    const int l = tid % 16, q = tid / 16, nq = nthr / 16;
    double o[MC], r[MC];
#pragma unroll
    for (int m = 0; m < MC; m++) {
        const int j = l + 16 * m;
        o[m] = j < nel ? orb[j] : 0.0;
        r[m] = j < nel ? srow[j] : 0.0;
    }
    for (int i0 = 0; i0 < nel; i0 += nq * MB) {  // the same trips for all lanes of a wave
        double v[MB][MC];
#pragma unroll
        for (int b = 0; b < MB; b++) {
            const int i = i0 + nq * b + q;
            const bool ok = i < nel && i != row;
            const double *Si = S + (size_t)(i < nel ? i : 0) * NM;
#pragma unroll
            for (int m = 0; m < MC; m++) v[b][m] = (ok && l + 16 * m < nel) ? Si[l + 16 * m] : 0.0;
        }
#pragma unroll
        for (int b = 0; b < MB; b++) {
            const int i = i0 + nq * b + q;
            const bool ok = i < nel && i != row;
            double *Si = S + (size_t)(i < nel ? i : 0) * NM;
            double p[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int m = 0; m < MC; m++) p[m % 4] += v[b][m] * o[m];
            const double s = row16_sum_as_wave(p) / rt;
#pragma unroll
            for (int m = 0; m < MC; m++)
                if (ok && l + 16 * m < nel) Si[l + 16 * m] = v[b][m] - r[m] * s;
        }
    }
}

// Orbitals of the moved electrons' spin, value and gradient, into orb_b [walker][4]
// [npad]: the AOs a chunk of 64 NW at a time through LDS against the occupied
// coefficients ct [nel][NB], tiles of 16 orbitals dealt to the wavefronts.  Four
// walkers x four components fill the 16 rows of an instruction and share every
// coefficient read; a block of one walker runs on the 4 x 4 x 4 form, four blocks of
// it for 16 orbitals (17 cycles; on the 16-row form, a quarter of it used, 66: 11.1
// against 10.0 ms of moves a sweep of 160 electrons x 256 walkers).  Four walkers a
// wavefront each on the 4 x 4 x 4 form read the coefficients four times: 2.59 against
// 2.36 ms at 60 electrons x 768 walkers.  Both forms add the four products of a step in
// order, and steps pair them as k_gemm_mfma.  The coefficients of the next KS AOs
// are loaded while these run.
template <int NORDC, typename T, int NW>
__device__ __forceinline__ void sweep_orbitals(const MoveArgs &a, const MoveLds<NORDC, T> &L, bool live, const double *ct,
                                               int nel, int npad, int bt, int wpb, double *chunks, double *orb_b)
{
    constexpr int NT = NW * WAVE, KS = NW > 1 ? 64 : 32, TC = 2, SPC = NT / KS;  // TC tiles at a time
    const int NB = a.NB, nt = (nel + 15) / 16, stride = SweepLds<NORDC, T, NW>::stride(wpb);
    const int r = bt % 16, q = (bt % WAVE) / 16, wvb = bt / WAVE, nwb = blockDim.x / WAVE, wb = bt / NT, tid = bt % NT;
    const bool rows16 = NW == 1 && wpb == 4;
    for (int t0 = wvb; t0 - wvb < nt; t0 += TC * nwb) {
        dbl4 acc16[TC];
        double acc4[TC], b0[TC][KS / 4], b1[TC][KS / 4];
#pragma unroll
        for (int i = 0; i < TC; i++) { acc16[i] = dbl4{0.0, 0.0, 0.0, 0.0}; acc4[i] = 0.0; }
        auto load = [&](int k0, double (*b)[KS / 4]) {
#pragma unroll
            for (int i = 0; i < TC; i++) {
                const int t = t0 + i * nwb, col = 16 * t + r;
                if (t >= nt) continue;
                const double *cp = ct + (size_t)(col < nel ? col : 0) * NB + 4 * q;
                if (k0 + KS <= NB) {
#pragma unroll
                    for (int k = 0; k < KS / 4; k++) b[i][k] = cp[k0 + 16 * (k / 4) + k % 4];
                } else {
#pragma unroll
                    for (int k = 0; k < KS / 4; k++) {
                        const int kk = k0 + 16 * (k / 4) + k % 4;
                        b[i][k] = kk + 4 * q < NB ? cp[kk] : 0.0;
                    }
                }
            }
        };
        auto mma = [&](const double *A, const double (*b)[KS / 4]) {  // A: the chunk from the stage's first AO
            if (rows16) {
#pragma unroll
                for (int k = 0; k < KS / 4; k++) {
                    const double av = A[(size_t)(16 * (k / 4) + 4 * q + k % 4) * stride + r];
#pragma unroll
                    for (int i = 0; i < TC; i++)
                        if (t0 + i * nwb < nt) acc16[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, b[i][k], acc16[i], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int k = 0; k < KS / 4; k++) {
                    const double av = A[(size_t)(16 * (k / 4) + 4 * q + k % 4) * stride + 4 * wb + r % 4];
#pragma unroll
                    for (int i = 0; i < TC; i++)
                        if (t0 + i * nwb < nt) acc4[i] = __builtin_amdgcn_mfma_f64_4x4x4f64(av, b[i][k], acc4[i], 0, 0, 0);
                }
            }
        };
        load(0, b0);
        int buf = 0;
        for (int m0 = 0; m0 < NB; m0 += NT, buf ^= 1) {
            double *A = chunks + (size_t)buf * NT * stride;
            const int m = m0 + tid;
            T out[5] = {T(0), T(0), T(0), T(0), T(0)};
            if (live && m < NB) move_ao(L, a.ao_cent[m], a.ao_ri[m], a.ao_slm[m], out);
#pragma unroll
            for (int k = 0; k < 4; k++) A[(size_t)tid * stride + 4 * wb + k] = (double)out[k];
            if (nwb > 1) __syncthreads();  // the other buffer was read before the last one
            else __syncwarp();
#pragma unroll
            for (int st = 0; st < SPC; st += 2) {
                const int k0 = m0 + st * KS;
                if (k0 + KS < NB) load(k0 + KS, b1);
                if (k0 < NB) mma(A + (size_t)st * KS * stride, b0);
                if (k0 + 2 * KS < NB) load(k0 + 2 * KS, b0);
                if (k0 + KS < NB) mma(A + (size_t)(st + 1) * KS * stride, b1);
            }
        }
#pragma unroll
        for (int i = 0; i < TC; i++) {
            const int t = t0 + i * nwb;
            if (t >= nt) continue;
            if (rows16) {
#pragma unroll
                for (int v = 0; v < 4; v++)  // rows 4 v + q: component q of the block's walker v
                    orb_b[(size_t)(4 * v + q) * npad + 16 * t + r] = acc16[i][v];
            } else {
                orb_b[(size_t)(4 * wb + q) * npad + 16 * t + r] = acc4[i];
            }
        }
        if (nwb > 1) __syncthreads();  // the chunks are written again
        else __syncwarp();
    }
}

// ------------------------------------------------------------------------
// One determinant: the moves of electrons e0 .. e1 - 1 of every walker in one
// launch.  Walkers do not meet inside a sweep, so a block takes its walkers
// through proposal, distances, jastrow4e, orbitalse, ratio, drift, decision and
// commit of one electron after the other: the AO block, the orbitals and the
// proposal's sums never leave the CU for another launch to read, no launch waits
// for the slowest walker, and the serial head of a move (drift, proposal,
// decision) overlaps other walkers' sums.
//   NW = 1: a wavefront per walker, up to four walkers to a block; NW = 4: a block
//   per walker.
// Sums keep the order of the separate kernels (k_move_a, k_gemm_mfma, k_move_b), so a
// sweep gives their bits.
// ms of a sweep's moves, as three launches per electron (Jastrow and AOs, matrix
// product, decision and commit) and so: 160 electrons x 4096 walkers 90.3 -> 57.5
// (mixed 72.9 -> 51.0), x 256 27.2 -> 8.4; 60 x 768 5.0 -> 2.2; 22 x 256 1.15 -> 0.49;
// 10 x 4 0.41 -> 0.17.  Few walkers: the chains of one move (of 10 us at 10 electrons 4
// are the proposal's and 3 the decision's scalar code); many: memory latency, two waves
// per SIMD (227 registers at order 4) waiting 62% of their cycles, with the vector pipe
// 31% busy and 2.5 TB/s (16 bytes per pair and centre, and the commits) at 160 x 4096.
template <int NORDC, typename T, int NW, int MOVERS>
__global__ void __launch_bounds__(SW_BLOCK) CHAMP_WAVES_PER_EU(CHAMP_SWEEP_WPE) k_sweep(MoveArgs args, int e0, int e1)
{
    HIP_DYNAMIC_SHARED(double, lds)
    using SL = SweepLds<NORDC, T, NW>;
    constexpr int NT = NW * WAVE;
    constexpr bool BLOCK = NW > 1;
    __shared__ double s_xn[SW_BLOCK / NT][3], s_en[4], s_rt[SW_BLOCK / NT], s_detn[SW_BLOCK / NT], s_sum[4];
    __shared__ int s_acc[SW_BLOCK / NT];
    const MoveConst mc(lds, args.jas, args.cent, args.iwctype, args.NC);
    const int wpb = blockDim.x / NT;
    for (int iel = e0; iel < e1; iel++) {
        // the arguments are read anew for each electron: kept across the loop, they and
        // what follows from them would take more registers than there are
        const MoveArgs &a = MOVE_ARGS_AGAIN(args);
        int bt = threadIdx.x;
        FORM_AGAIN(bt);
        const int wb = bt / NT, tid = bt % NT, wv = tid / WAVE, lane = tid % WAVE, w = blockIdx.x * wpb + wb;
        const bool live = w < a.W;  // a wavefront past the last walker only shares the block's tiles
        const int NE = a.NE, NC = a.NC, NO = a.NO, NM = a.NM, npad = SL::npad(NM);
        double *lds_w = lds + MoveConst::doubles(NC);
        double *orb_b = lds_w + wpb * SL::walker(NC, a.NRI), *orb = orb_b + (size_t)wb * 4 * npad;
        double *row_s = orb_b + (size_t)(4 * wpb + wb) * npad, *chunks = orb_b + (size_t)5 * wpb * npad;
        const MoveLds<NORDC, T> L(lds_w + wb * SL::walker(NC, a.NRI), NC);
        double *xw = a.xT + (size_t)w * 3 * NE, *vj = a.vjT + (size_t)w * 3 * NE;
        double *rw = a.r_en + (size_t)w * NC * NE, *rrw = a.rr_en + (size_t)w * NC * NE;
        float2 *ew = a.enp ? a.enp + (size_t)w * NC * NE : nullptr;
        double *rnew = a.rnew + (size_t)w * NC, *rrnew = a.rrnew + (size_t)w * NC;
        double *fsn = a.fsn_row + (size_t)w * NE, *g1n = a.g1n + (size_t)w * 3 * NE, *g2n = a.g2n + (size_t)w * 3 * NE;
        double *F = a.fso + (size_t)w * NE * NE, *G1 = a.g1 + (size_t)w * NE * 3 * NE, *G2 = a.g2 + (size_t)w * NE * 3 * NE;
        const int iab = iel < a.NUP ? 0 : 1, nel = iab ? NE - a.NUP : a.NUP, ish = iab ? a.NUP : 0, row = iel - ish;
        double *S = a.slmi + ((size_t)w * 2 + iab) * NM * NM, *srow = S + (size_t)row * NM;
        double psijn = 0, vjn[3] = {0, 0, 0};
        if (live) {
            const MoveGeo geo{NE, a.NUP, NC, iel, mc.cent, mc.iwctype, mc.jas};
            double xn0 = 0, xn1 = 0, xn2 = 0, en[4];
            if (wv == 0) {
                propose<MOVERS>(a, w, iel, lane, xw, xn0, xn1, xn2);
                xn0 = __shfl(xn0, 0, WAVE); xn1 = __shfl(xn1, 0, WAVE); xn2 = __shfl(xn2, 0, WAVE);
                move_centres<NORDC, T>(geo, L, lane, xn0, xn1, xn2, rnew, rrnew, en);
                if (lane == 0) {
                    s_xn[wb][0] = xn0; s_xn[wb][1] = xn1; s_xn[wb][2] = xn2;
                    if (BLOCK) for (int k = 0; k < 4; k++) s_en[k] = en[k];
                }
            }
            team_sync<BLOCK>();
            if (BLOCK) {
                xn0 = s_xn[wb][0]; xn1 = s_xn[wb][1]; xn2 = s_xn[wb][2];
                for (int k = 0; k < 4; k++) en[k] = s_en[k];
            }
            // change of the moved electron's sums (value, gradient), its own entries first
            double d[4] = {0, 0, 0, 0};
            if (wv == 0 && lane == 0) {
                fsn[iel] = en[0];
                d[0] += en[0] - F[(size_t)iel * NE + iel];
                for (int k = 0; k < 3; k++) {
                    g1n[k * NE + iel] = g2n[k * NE + iel] = en[1 + k];
                    d[1 + k] += en[1 + k] - G1[((size_t)iel * 3 + k) * NE + iel];
                }
            }
            for (int j0 = WAVE * wv; j0 < NE; j0 += NT) {
                const int j = j0 + lane;
                const bool on = j < NE && j != iel;
                // the old row's loads are in flight during the pass
                const int jo = j < NE ? j : NE - 1;
                const double fo = F[(size_t)iel * NE + jo];
                double go[3];
                for (int k = 0; k < 3; k++) go[k] = G1[((size_t)iel * 3 + k) * NE + jo];
                double f, gi[3], gj[3], dj[4] = {0, 0, 0, 0};
                move_pair<NORDC, T>(geo, L, xw, xn0, xn1, xn2, rw, rrw, ew, j, on, f, gi, gj);
                if (on) {
                    fsn[j] = f;
                    dj[0] = f - fo;
                    for (int k = 0; k < 3; k++) {
                        g1n[k * NE + j] = gi[k];
                        g2n[k * NE + j] = gj[k];
                        dj[1 + k] = gi[k] - go[k];
                    }
                }
                if (BLOCK)
                    for (int k = 0; k < 4; k++) chunks[(size_t)(j0 / WAVE * 4 + k) * WAVE + lane] = dj[k];
                else
                    for (int k = 0; k < 4; k++) d[k] += dj[k];
            }
            team_sync<BLOCK>();
            if (wv == 0) {
                if (BLOCK)
                    for (int j0 = 0; j0 < NE; j0 += WAVE)  // in the order of the partners
                        for (int k = 0; k < 4; k++) d[k] += chunks[(size_t)(j0 / WAVE * 4 + k) * WAVE + lane];
#pragma unroll
                for (int k = 0; k < 4; k++) d[k] = wave_sum(d[k]);
                psijn = a.fsumo[w] + d[0];
                for (int k = 0; k < 3; k++) vjn[k] = vj[k * NE + iel] + d[1 + k];
                if (BLOCK && lane == 0) { s_sum[0] = psijn; for (int k = 0; k < 3; k++) s_sum[1 + k] = vjn[k]; }
            }
            move_radial<NORDC, T>(L, tid, NT, a.tab, a.NRI, a.ri_cent, a.ri_type, a.ri_rad, a.ri_rmax);
            team_sync<BLOCK>();
            if (BLOCK) { psijn = s_sum[0]; for (int k = 0; k < 3; k++) vjn[k] = s_sum[1 + k]; }
        }
        sweep_orbitals<NORDC, T, NW>(a, L, live, a.cocc[iab], nel, npad, bt, wpb, chunks, orb_b);
        if (!live) continue;
        // ---- determinant ratio, drift at the proposal, decision
        if (wv == 0) {
            double rt = 0, v0 = 0, v1 = 0, v2 = 0;
            for (int j = lane; j < nel; j += WAVE) {
                const double s = srow[j];
                row_s[j] = s;
                rt += s * orb[j];
            }
            rt = wave_sum(rt);
            for (int j = lane; j < nel; j += WAVE) {
                const double sn = row_s[j] / rt;
                v0 += sn * orb[npad + j]; v1 += sn * orb[2 * npad + j]; v2 += sn * orb[3 * npad + j];
            }
            v0 = wave_sum(v0); v1 = wave_sum(v1); v2 = wave_sum(v2);
            if (lane == 0) {
                const double vn[3] = {0.0 + v0 + vjn[0], 0.0 + v1 + vjn[1], 0.0 + v2 + vjn[2]};
                double detn;
                s_acc[wb] = decide<MOVERS>(a, w, iel, rt, vn, psijn, detn);
                s_rt[wb] = rt; s_detn[wb] = detn;
            }
        }
        team_sync<BLOCK>();
        if (s_acc[wb]) {
            // ---- commit: detsav and jassav (iflag = 0) with the Sherman-Morrison update
            const double rt = s_rt[wb];
            if (nel <= 16 * 2) sm_update<2, 8>(S, NM, nel, row, rt, row_s, orb, tid, NT);
            else if (nel <= 16 * 5) sm_update<5, 4>(S, NM, nel, row, rt, row_s, orb, tid, NT);
            else if (nel <= 16 * 10) sm_update<10, 2>(S, NM, nel, row, rt, row_s, orb, tid, NT);
            else
                for (int i = wv; i < nel; i += NW) {
                    if (i == row) continue;
                    double *Si = S + (size_t)i * NM, s = 0;
                    for (int j = lane; j < nel; j += WAVE) s += Si[j] * orb[j];
                    s = wave_sum(s);
                    s = s / rt;
                    for (int j = lane; j < nel; j += WAVE) Si[j] = Si[j] - row_s[j] * s;
                }
            for (int j = tid; j < nel; j += NT) srow[j] = row_s[j] / rt;
            double *dor = a.dorb + ((size_t)w * NE + iel) * 3 * NO;
            for (int j = tid; j < nel; j += NT) {
                const int jo = a.iworbd[ish + j];
                for (int k = 0; k < 3; k++) dor[k * NO + jo] = orb[(1 + k) * npad + j];
            }
            if (tid < 3) xw[tid * NE + iel] = s_xn[wb][tid];
            for (int c = tid; c < NC; c += NT) {
                const double rn = rnew[c], rrn = rrnew[c];
                rw[(size_t)c * NE + iel] = rn;
                rrw[(size_t)c * NE + iel] = rrn;
                if (sizeof(T) == sizeof(float)) ew[(size_t)c * NE + iel] = enp_pack(mc.jas->kap, mc.jas->asymp_r, rn, rrn);
            }
            for (int j = tid; j < NE; j += NT) {
                const double f = fsn[j];
                F[(size_t)iel * NE + j] = f;
                F[(size_t)j * NE + iel] = f;
                for (int k = 0; k < 3; k++) {
                    const double gi = g1n[k * NE + j], gj = g2n[k * NE + j];
                    const size_t r = ((size_t)iel * 3 + k) * NE + j, t = ((size_t)j * 3 + k) * NE + iel;
                    vj[k * NE + j] = j == iel ? vjn[k] : vj[k * NE + j] + gj - G2[r];
                    G1[r] = gi;
                    G2[r] = gj;
                    G1[t] = gj;
                    G2[t] = gi;
                }
            }
            if (tid == 0) {
                a.fsumo[w] = psijn;
                a.detiab[2 * w + iab] = s_detn[wb];
            }
        }
        team_sync<BLOCK>();
    }
}

static inline int nblocks(int n, int per) { return (n + per - 1) / per; }

#ifndef CHAMP_MOVE_NW  // variant builds: fixed wavefronts per walker
#define CHAMP_MOVE_NW 0
#endif
#ifndef CHAMP_SWEEP_BLOCK  // variant builds: threads per block of single-wavefront walkers
#define CHAMP_SWEEP_BLOCK 0
#endif

// Threads per block of single-wavefront walkers.  Up to 512 walkers a block each, so
// that they spread over the CUs; above, four share the coefficient reads and fill the
// matrix instruction.  ms of a sweep's moves in blocks of one / four walkers:
//   electrons 10, walkers 4     0.18 / 0.22    electrons 97, walkers 520  6.90 / 5.75
//   22, 256                     0.50 / 0.56    160, 520                   23.8 / 18.0
//   60, 256                     1.89 / 2.03    160, 1024                  28.5 / 19.3
//   60, 768                     2.19 / 2.24    160, 4096                  96.4 / 56.2
//   60, 1000                    2.54 / 2.30
static int one_wave_block(const champ_ctx *c)
{
    if (CHAMP_SWEEP_BLOCK) return CHAMP_SWEEP_BLOCK;
    return c->W <= 512 ? WAVE : SW_BLOCK;
}

// One wavefront per walker, or four: four while all the walkers' blocks of four are
// resident at once (two on a CU, 512) and a move has the work for them, and where the
// LDS of a block of single-wavefront walkers is too large; else one, which does
// without barriers.  ms of a sweep's moves with one / four:
//   electrons 10, walkers 4     0.18 / 0.18    electrons 97, walkers 520  5.75 / 6.80
//   22, 256                     0.50 / 0.49    160, 256                   17.8 / 8.4
//   60, 256                     1.89 / 1.62    160, 520                   18.0 / 17.4
//   60, 520                     2.16 / 3.31    160, 1024                  19.3 / 20.2
//   60, 768                     2.24 / 3.48    160, 4096                  56.2 / 79.1
template <int N, typename T>
static bool one_wave(const champ_ctx *c)
{
    if (SweepLds<N, T, 1>::doubles(c->NC, c->NRI, c->NM, c->NE, one_wave_block(c) / WAVE) * sizeof(double) > MOVE_LDS_MAX)
        return false;
    if (CHAMP_MOVE_NW) return CHAMP_MOVE_NW == 1;
    return c->NE <= 32 || c->W > 512;
}

template <int N, typename T, int NW, int MOVERS>
static int launch_m(champ_ctx *c, const MoveArgs &a, int e0, int e1)
{
    const int nthr = NW == 1 ? one_wave_block(c) : SW_BLOCK, wpb = nthr / (NW * WAVE);
    const size_t lds = SweepLds<N, T, NW>::doubles(c->NC, c->NRI, c->NM, c->NE, wpb) * sizeof(double);
    if (const int rc = move_lds((const void *)k_sweep<N, T, NW, MOVERS>, lds)) return rc;
    hipLaunchKernelGGL((k_sweep<N, T, NW, MOVERS>), dim3(nblocks(c->W, wpb)), dim3(nthr), lds, c->stream, a, e0, e1);
    HIPCHECK(hipGetLastError());
    return CHAMP_OK;
}

// MOVERS 1 leaves out the movers with long scalar code (propose)
template <int N, typename T>
static int launch_t(champ_ctx *c, const MoveArgs &a, int e0, int e1)
{
    const bool plain = a.imetro == 1 || (a.imetro == 2 && c->nloc > 0);
    if (one_wave<N, T>(c)) return plain ? launch_m<N, T, 1, 1>(c, a, e0, e1) : launch_m<N, T, 1, 0>(c, a, e0, e1);
    return plain ? launch_m<N, T, 4, 1>(c, a, e0, e1) : launch_m<N, T, 4, 0>(c, a, e0, e1);
}

template <typename T>
static int launch_nordc(champ_ctx *c, const MoveArgs &a, int e0, int e1)
{
    switch (c->hjas.nordc) {
    case 5: return launch_t<5, T>(c, a, e0, e1);
    case 4: return launch_t<4, T>(c, a, e0, e1);
    case 3: return launch_t<3, T>(c, a, e0, e1);
    case 2: return launch_t<2, T>(c, a, e0, e1);
    default: return launch_t<0, T>(c, a, e0, e1);
    }
}

int launch_sweep_moves(champ_ctx *c, int e0, int e1)
{
    if (c->hjas.nordc > 5) {
        set_error("move: e-e-n order above 5 is not supported");
        return CHAMP_ERR_UNSUPPORTED;
    }
    int slot;
    tbegin(c, K_SWEEP, &slot);
    const MoveArgs a = move_args(c, e0, 0, c->tau);
    const int rc = c->prec == CHAMP_PREC_MIXED ? launch_nordc<float>(c, a, e0, e1) : launch_nordc<double>(c, a, e0, e1);
    tend(c, slot);
    return rc;
}

}  // namespace champ
