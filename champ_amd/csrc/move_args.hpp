// move_args.hpp -- arguments of the move kernels, and the steps of a move that
// one wavefront takes for its walker: drift, proposal and decision.
#pragma once
#include "dmc_ae.hpp"
#include "engine_internal.hpp"
#include "metrop6.hpp"

#include <cmath>

namespace champ {

struct MoveArgs {
    int W, NE, NUP, NM, NC, NB, NO, iel, mode, pad;
    double tau, cdet0;
    const double *cent;
    const int *iwctype;
    SplineTab tab;
    const double *rmax_ao;
    const int *ao_cent, *ao_type, *ao_rad, *ao_slm, *iworbd;
    int NRI;
    const int *ri_cent, *ri_type, *ri_rad, *ao_ri;
    const double *ri_rmax;
    const JasParams *jas;
    double *xT, *r_en, *rr_en, *fso, *g1, *g2, *vjT, *fsumo, *dorb, *slmi, *detiab, *psido, *psijo, *psi2o;
    uint64_t *rng;
    double *xnew, *dfus2o, *rnew, *rrnew, *fsn_row, *g1n, *g2n, *vjnT, *fsumn, *aomove, *orbn;
    double *ratio, *psidn, *psijn, *vnew, *vold, *esum_dev;
    unsigned char *acc;
    int *status;
    int md;                            // multideterminant trial function
    const double *md_vcol, *md_vcoln;  // [W][NO] d ln psi_D / d phi_o(r_iel), current / proposed
    double *md_S, *md_Sn;              // [W] psi_D / (D_up,ref D_dn,ref), current / proposed
    int *md_cur;                       // [W][2] current buffer of the multideterminant state
    int ao32;                          // AO block stored as FP32 for the FP32 contraction
    int imetro;                        // mode-0 mover: 1 metrop1, 6 metrop6, 2 DMC (dmc_ps)
    M6Params m6p;
    double *dmc_acc;                   // [W][DMC_ACC] DMC move accumulators of the current step
    int *dmc_age;                      // [W] steps since the walker last moved
    double *m6rec;                     // [W][M6_REC]
    const EcpParams *ecp;              // znuc per type and nloc (metrop6's cusp and theta range)
    float2 *enp;                       // mixed path: [W][NC][NE] partner pair table (enp_pack), else null
    const double *cocc[2];             // [nel][NB] occupied coefficients per spin
};

static inline MoveArgs move_args(champ_ctx *c, int iel, int mode, double tau)
{
    MoveArgs a;
    a.W = c->W; a.NE = c->NE; a.NUP = c->NUP; a.NM = c->NM; a.NC = c->NC; a.NB = c->NB; a.NO = c->NO;
    a.iel = iel; a.mode = mode; a.pad = 0; a.tau = tau; a.cdet0 = c->cdet0;
    a.cent = c->cent; a.iwctype = c->iwctype; a.tab = c->tab; a.rmax_ao = c->rmax_ao;
    a.ao_cent = c->ao_cent; a.ao_type = c->ao_type; a.ao_rad = c->ao_rad; a.ao_slm = c->ao_slm;
    a.iworbd = c->iworbd; a.jas = c->jas;
    a.NRI = c->NRI; a.ri_cent = c->ri_cent; a.ri_type = c->ri_type; a.ri_rad = c->ri_rad; a.ao_ri = c->ao_ri;
    a.ri_rmax = c->ri_rmax;
    a.enp = c->enp;
    a.cocc[0] = c->cocc[0]; a.cocc[1] = c->cocc[1];
    a.xT = c->xT; a.r_en = c->r_en; a.rr_en = c->rr_en; a.fso = c->fso; a.g1 = c->g1; a.g2 = c->g2;
    a.vjT = c->vjT; a.fsumo = c->fsumo; a.dorb = c->dorb; a.slmi = c->slmi; a.detiab = c->detiab;
    a.psido = c->psido; a.psijo = c->psijo; a.psi2o = c->psi2o; a.rng = c->rng;
    a.xnew = c->xnew; a.dfus2o = c->dfus2o; a.rnew = c->rnew; a.rrnew = c->rrnew; a.fsn_row = c->fsn_row;
    a.g1n = c->g1n; a.g2n = c->g2n; a.vjnT = c->vjnT; a.fsumn = c->fsumn; a.aomove = c->aomove; a.orbn = c->orbn;
    a.ratio = c->ratio; a.psidn = c->psidn; a.psijn = c->psijn; a.vnew = c->vnew; a.vold = c->vold;
    a.esum_dev = c->esum_dev; a.acc = c->acc; a.status = c->status;
    a.md = c->md; a.md_vcol = c->md_vcol; a.md_vcoln = c->md_vcoln; a.md_S = c->md_S; a.md_Sn = c->md_Sn;
    a.md_cur = c->md_cur;
    a.ao32 = c->prec == CHAMP_PREC_MIXED && c->tune_gemm[0] == GEMM_F32;
    a.imetro = c->imetro;
    a.m6p = M6Params{c->m6_deltar, c->m6_deltat, c->m6_fbias};
    a.m6rec = c->m6rec;
    a.ecp = c->ecp;
    a.dmc_acc = c->dmc_acc;
    a.dmc_age = c->dmc_age;
    return a;
}

// ------------------------------------------------------------------------
// Drift at the current position of iel: compute_determinante_grad with
// iflag_move=1 (determinante.f90:127-157, determinante_ref_grad :285-328).
__device__ __forceinline__ void drift_old(const MoveArgs &a, int w, int iel, int lane, double v[3])
{
    const int iab = iel < a.NUP ? 0 : 1, nel = iab ? a.NE - a.NUP : a.NUP, ish = iab ? a.NUP : 0;
    const double *srow = a.slmi + ((size_t)w * 2 + iab) * a.NM * a.NM + (size_t)(iel - ish) * a.NM;
    const double *dor = a.dorb + ((size_t)w * a.NE + iel) * 3 * a.NO;
    double v0 = 0, v1 = 0, v2 = 0;
    if (a.md) {  // sum over every orbital of d ln psi_D / d phi_o grad phi_o
        const double *vc = a.md_vcol + (size_t)w * a.NO;
        for (int o = lane; o < a.NO; o += WAVE) {
            const double s = vc[o];
            v0 += s * dor[o]; v1 += s * dor[a.NO + o]; v2 += s * dor[2 * a.NO + o];
        }
    } else {
        for (int j = lane; j < nel; j += WAVE) {
            const double s = srow[j];
            const int jo = a.iworbd[ish + j];
            v0 += s * dor[jo];
            v1 += s * dor[a.NO + jo];
            v2 += s * dor[2 * a.NO + jo];
        }
    }
    v0 = wave_sum(v0); v1 = wave_sum(v1); v2 = wave_sum(v2);
    const double *vj = a.vjT + (size_t)w * 3 * a.NE;
    v[0] = 0.0 + v0 + vj[iel];
    v[1] = 0.0 + v1 + vj[a.NE + iel];
    v[2] = 0.0 + v2 + vj[2 * a.NE + iel];
}

// The proposal of electron iel on lane 0 of the wave, from the drift at its old
// position and the walker's stream.  Movers 0: any; 1: metrop1 and dmc_ps only
// (a kernel without the long scalar code of the others keeps its registers).
template <int MOVERS>
__device__ __forceinline__ void propose(const MoveArgs &a, int w, int iel, int lane, const double *xw, double &xn0,
                                        double &xn1, double &xn2)
{
    const int NE = a.NE, NC = a.NC;
    double vo[3];
    drift_old(a, w, iel, lane, vo);
    if (MOVERS == 0 && lane == 0 && a.imetro == 6) {
        uint64_t s[4];
        for (int k = 0; k < 4; k++) s[k] = a.rng[4 * (size_t)w + k];
        const double xo[3] = {xw[iel], xw[NE + iel], xw[2 * NE + iel]};
        double xn[3];
        m6_propose(a.cent, a.iwctype, a.ecp->znuc, a.ecp->nloc, NC, a.m6p, xo, vo, s, xn,
                   a.m6rec + (size_t)w * M6_REC);
        for (int k = 0; k < 4; k++) a.rng[4 * (size_t)w + k] = s[k];
        for (int k = 0; k < 3; k++) { a.xnew[3 * w + k] = xn[k]; a.vold[3 * w + k] = vo[k]; }
        xn0 = xn[0]; xn1 = xn[1]; xn2 = xn[2];
    } else if (MOVERS == 0 && lane == 0 && a.imetro == 2 && a.ecp->nloc == 0) {
        // dmc_ae proposal (dmc_ae_mov1.f90:226-353)
        uint64_t s[4];
        for (int k = 0; k < 4; k++) s[k] = a.rng[4 * (size_t)w + k];
        const double xo[3] = {xw[iel], xw[NE + iel], xw[2 * NE + iel]};
        double xn[3], dfus2o, fnormo;
        ae_propose(a.cent, a.iwctype, a.ecp->znuc, NC, a.tau, xo, vo, s, xn, dfus2o, fnormo);
        for (int k = 0; k < 4; k++) a.rng[4 * (size_t)w + k] = s[k];
        for (int k = 0; k < 3; k++) { a.xnew[3 * w + k] = xn[k]; a.vold[3 * w + k] = vo[k]; }
        a.dfus2o[w] = dfus2o;
        a.dmc_acc[(size_t)w * DMC_ACC + DMC_FNORMO] = fnormo;
        xn0 = xn[0]; xn1 = xn[1]; xn2 = xn[2];
    } else if (lane == 0 && a.imetro == 2) {
        // dmc_ps drift-diffusion proposal (dmc_ps_mov1.f90:291-303): the
        // drift is vavvt v, without metrop1's extra factor tau
        const double tau = a.tau, rttau = sqrt(tau), adrift = 0.5;
        uint64_t s[4];
        for (int k = 0; k < 4; k++) s[k] = a.rng[4 * (size_t)w + k];
        const double v2old = vo[0] * vo[0] + vo[1] * vo[1] + vo[2] * vo[2];
        const double vavvt = (sqrt(1.0 + 2.0 * adrift * v2old * tau) - 1.0) / (adrift * v2old);
        double dfus2o = 0.0, xn[3];
        for (int k = 0; k < 3; k++) {
            const double drift = vavvt * vo[k];
            const double dfus = xo_gauss(s) * rttau;
            const double dx = drift + dfus;
            dfus2o = dfus2o + dfus * dfus;
            xn[k] = xw[k * NE + iel] + dx;
        }
        for (int k = 0; k < 4; k++) a.rng[4 * (size_t)w + k] = s[k];
        for (int k = 0; k < 3; k++) { a.xnew[3 * w + k] = xn[k]; a.vold[3 * w + k] = vo[k]; }
        a.dfus2o[w] = dfus2o;
        xn0 = xn[0]; xn1 = xn[1]; xn2 = xn[2];
    } else if (lane == 0) {
        const double tau = a.tau, rttau = sqrt(tau), adrift = 0.5;
        uint64_t s[4];
        for (int k = 0; k < 4; k++) s[k] = a.rng[4 * (size_t)w + k];
        double v2old = vo[0] * vo[0] + vo[1] * vo[1] + vo[2] * vo[2];
        double vavvt = (sqrt(1.0 + 2.0 * adrift * v2old * tau) - 1.0) / (adrift * v2old);
        double dfus2o = 0.0, xn[3];
        for (int k = 0; k < 3; k++) {
            double drift = vavvt * vo[k] * tau;
            double dfus = xo_gauss(s) * rttau;
            double dx = drift + dfus;
            dfus2o = dfus2o + dfus * dfus;
            xn[k] = xw[k * NE + iel] + dx;
        }
        for (int k = 0; k < 4; k++) a.rng[4 * (size_t)w + k] = s[k];
        for (int k = 0; k < 3; k++) { a.xnew[3 * w + k] = xn[k]; a.vold[3 * w + k] = vo[k]; }
        a.dfus2o[w] = dfus2o;
        xn0 = xn[0]; xn1 = xn[1]; xn2 = xn[2];
    }
}

// The metropolis decision on lane 0 (determinante.f90:38-46,
// metrop_mov1_driftdif.f90:166-205, metrop6 and DMC): rt the determinant ratio,
// vn the drift at the proposal, psijn the proposed log Jastrow.  Sets the
// walker's psi on acceptance; returns it and the new spin determinant.
template <int MOVERS>
__device__ __forceinline__ int decide(const MoveArgs &a, int w, int iel, double rt, const double vn[3], double psijn,
                                      double &detn)
{
    const int NE = a.NE, iab = iel < a.NUP ? 0 : 1;
    detn = a.detiab[2 * w + iab] * rt;
    const double psidn = (rt == 0.0) ? 0.0
                                     : 0.0 + detn * a.detiab[2 * w + 1 - iab] * (a.md ? a.md_Sn[w] : a.cdet0);
    int accept = 0;
    if (MOVERS == 0 && a.mode == 0 && a.imetro == 6) {
        const double psi2n = 2 * (log(fabs(psidn)) + psijn);
        const double *xw = a.xT + (size_t)w * 3 * NE;
        const double xo[3] = {xw[iel], xw[NE + iel], xw[2 * NE + iel]};
        const double xn[3] = {a.xnew[3 * w], a.xnew[3 * w + 1], a.xnew[3 * w + 2]};
        const double *rec = a.m6rec + (size_t)w * M6_REC;
        const double p = m6_accept_prob(a.cent, a.iwctype, a.ecp->znuc, a.ecp->nloc, a.m6p, xo, xn, vn, psi2n,
                                        a.psi2o[w], psidn == 0.0, rec);
        uint64_t s[4];
        for (int k = 0; k < 4; k++) s[k] = a.rng[4 * (size_t)w + k];
        const double uacc = xo_uniform(s);
        for (int k = 0; k < 4; k++) a.rng[4 * (size_t)w + k] = s[k];
        accept = uacc < p;
        if (accept) {
            a.psi2o[w] = psi2n;
            atomicAdd(&a.esum_dev[0], 1.0);
        }
        // psi is evaluated at proposals that pass the geometric test only
        if (rt == 0.0 && rec[M6_LIVE] != 0.0) atomicOr(&a.status[w], CHAMP_WALKER_ZERO_RATIO);
    } else if (a.mode == 0 && a.imetro == 2) {
        // dmc_ps acceptance (dmc_ps_mov1.f90:325-399), ipq = 1, icross = 1,
        // iacc_rej = 1, node_cutoff = 0: node crossings are counted, not rejected
        const double tau = a.tau, adrift = 0.5;
        const double *xw = a.xT + (size_t)w * 3 * NE;
        double *ac = a.dmc_acc + (size_t)w * DMC_ACC;
        const double psido = a.psido[w];
        if (psidn * psido <= 0.0) ac[DMC_NODECR] += 1.0;
        double dfus2n = 0.0, fnorm_ratio = 1.0;
        if (MOVERS == 0 && a.ecp->nloc == 0) {
            // dmc_ae's reverse Green function (dmc_ae_mov1.f90:388-490)
            const double xo[3] = {xw[iel], xw[NE + iel], xw[2 * NE + iel]};
            const double xn[3] = {a.xnew[3 * w], a.xnew[3 * w + 1], a.xnew[3 * w + 2]};
            double fnormn;
            ae_reverse(a.cent, a.iwctype, a.ecp->znuc, a.NC, tau, xo, xn, vn, dfus2n, fnormn);
            fnorm_ratio = fnormn / ac[DMC_FNORMO];
        } else {
            const double v2new = vn[0] * vn[0] + vn[1] * vn[1] + vn[2] * vn[2];
            const double vavvt = (sqrt(1.0 + 2.0 * adrift * v2new * tau) - 1.0) / (adrift * v2new);
            for (int k = 0; k < 3; k++) {
                const double drift = vavvt * vn[k];
                const double xbac = a.xnew[3 * w + k] + drift;
                const double dfus = xbac - xw[k * NE + iel];
                dfus2n = dfus2n + dfus * dfus;
            }
        }
        const double dfus2o = a.dfus2o[w];
        const double rat = psidn / psido;
        double p = rat * rat * exp(2 * (psijn - a.psijo[w])) * exp((dfus2o - dfus2n) / (2.0 * tau)) * fnorm_ratio;
        const int age = a.dmc_age[w];
        if (age > 50) p = p * pow(1.1, (double)(age - 50));
        ac[DMC_PP] = ac[DMC_PP] * p;
        p = p < 1.0 ? p : (p >= 1.0 ? 1.0 : 0.0);  // dmin1(one, p); a NaN p never passes
        ac[DMC_PSUM] += p;
        ac[DMC_DFUS2AC] += p * dfus2o;
        ac[DMC_DFUS2UN] += dfus2o;
        uint64_t s[4];
        for (int k = 0; k < 4; k++) s[k] = a.rng[4 * (size_t)w + k];
        const double uacc = xo_uniform(s);
        for (int k = 0; k < 4; k++) a.rng[4 * (size_t)w + k] = s[k];
        accept = uacc < p;
        if (accept) {
            a.psi2o[w] = 2 * (log(fabs(psidn)) + psijn);
            atomicAdd(&a.esum_dev[0], 1.0);
            a.dmc_age[w] = 0;
            ac[DMC_IACCEPT] = 1.0;
        }
        if (rt == 0.0) atomicOr(&a.status[w], CHAMP_WALKER_ZERO_RATIO);
    } else if (a.mode == 0) {
        const double tau = a.tau, adrift = 0.5;
        const double psi2n = 2 * (log(fabs(psidn)) + psijn);
        const double v2new = vn[0] * vn[0] + vn[1] * vn[1] + vn[2] * vn[2];
        const double vavvt = (sqrt(1.0 + 2.0 * adrift * v2new * tau) - 1.0) / (adrift * v2new);
        const double *xw = a.xT + (size_t)w * 3 * NE;
        double dfus2n = 0.0;
        for (int k = 0; k < 3; k++) {
            double drift = vavvt * vn[k] * tau;
            double xbac = a.xnew[3 * w + k] + drift;
            double dfus = xbac - xw[k * NE + iel];
            dfus2n = dfus2n + dfus * dfus;
        }
        double p = exp(psi2n - a.psi2o[w]) * exp(-0.5 * (dfus2n - a.dfus2o[w]) / tau);
        if (psidn == 0.0) p = 0.0;
        p = p < 1.0 ? p : 1.0;
        uint64_t s[4];
        for (int k = 0; k < 4; k++) s[k] = a.rng[4 * (size_t)w + k];
        const double uacc = xo_uniform(s);
        for (int k = 0; k < 4; k++) a.rng[4 * (size_t)w + k] = s[k];
        accept = uacc < p;
        if (accept) {
            a.psi2o[w] = psi2n;
            atomicAdd(&a.esum_dev[0], 1.0);
        }
        if (rt == 0.0) atomicOr(&a.status[w], CHAMP_WALKER_ZERO_RATIO);
    } else if (a.mode == 2) {
        accept = a.acc[w] != 0;
        if (accept) a.psi2o[w] = 2 * (log(fabs(psidn)) + psijn);
    }
    a.ratio[w] = rt; a.psidn[w] = psidn;
    for (int k = 0; k < 3; k++) a.vnew[3 * w + k] = vn[k];
    if (accept) {
        a.psido[w] = psidn; a.psijo[w] = psijn;
        if (a.md) { a.md_S[w] = a.md_Sn[w]; a.md_cur[2 * w + iab] ^= 1; }
    }
    return accept;
}

constexpr size_t MOVE_LDS_MAX = 160 * 1024 - 512;  // beside the kernels' static LDS

static inline int move_lds(const void *fn, size_t lds)
{
    if (lds > MOVE_LDS_MAX) {
        set_error("move: the move kernel's LDS tables exceed 160 KB for this system");
        return CHAMP_ERR_UNSUPPORTED;
    }
    if (lds > 64 * 1024) HIPCHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    return CHAMP_OK;
}

}  // namespace champ
