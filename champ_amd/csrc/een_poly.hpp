// een_poly.hpp -- the electron-electron-nucleus part of the ijas=4 Jastrow
// (jastrow4.f90:203-262, nonlpsi.f90:4-86) as a polynomial with its structure
// fixed at compile time by the order nordc.
//
// With switched scaled distances u (electron-electron), x and y (the two
// electrons to one centre) the term sum is
//     P(u, x, y) = sum_t c_t u^k (x^l + y^l) (x y)^m
//                = sum_{k,n} A_kn(x) u^k y^n,
// where term t adds c_t x^(l+m) to A[k][m] and c_t x^m to A[k][l+m] (for l = 0
// both land on A[k][m], giving the factor 2 of ss(0) = 2).  For one electron
// and one centre the tables A, dA/dx and d2A/dx2 are built once; every partner
// electron then costs a Horner evaluation over the non-zero pattern.  All
// loop bounds and indices below are compile-time constants after unrolling.
#pragma once
#include "device_common.hpp"

namespace champ {

template <int N>
struct EenTable {
    int n;                    // number of terms (13 at N = 4)
    int k[40], l[40], m[40];  // (k, l, m) in the order of jastrow4.f90:203-213
    int idx[N + 1][N + 1];    // packed position of A[k][n], -1 where zero
    int naz;                  // number of non-zero A entries (12 at N = 4)
    int nmax[N + 1];          // highest non-zero power of y in row k, -1 if none
    int kmax;                 // highest power of u, -1 if no terms
    constexpr EenTable() : n(0), k{}, l{}, m{}, idx{}, naz(0), nmax{}, kmax(-1)
    {
        bool nz[N + 1][N + 1] = {};
        for (int nn = 2; nn <= N; nn++)
            for (int kk = nn - 1; kk >= 0; kk--) {
                const int lhi = kk == 0 ? nn - kk - 2 : nn - kk;
                for (int ll = lhi; ll >= 0; ll--) {
                    const int mm = (nn - kk - ll) / 2;
                    if (2 * mm == nn - kk - ll) {
                        k[n] = kk; l[n] = ll; m[n] = mm; n++;
                        nz[kk][mm] = true;
                        nz[kk][ll + mm] = true;
                    }
                }
            }
        for (int kk = 0; kk <= N; kk++) {
            nmax[kk] = -1;
            for (int nn = 0; nn <= N; nn++) {
                idx[kk][nn] = nz[kk][nn] ? naz++ : -1;
                if (nz[kk][nn]) nmax[kk] = nn;
            }
            if (nmax[kk] >= 0) kmax = kk;
        }
    }
};

// Switched scaled distance 1 - kap R(r) = exp(-kap r) of isc = 2
// (switch_scale2, scale_dist.f90:314-331) in the reference's form.  FP32 code takes
// exp(-kap r) itself: far from a centre (R -> 1/kap) the difference cancels.
__device__ __forceinline__ double switched_from(double kap, double R) { return 1.0 - kap * R; }

template <int N>
constexpr int een_naz() { return EenTable<N>{}.naz > 0 ? EenTable<N>{}.naz : 1; }

// Coefficient tables of one (electron, centre) at switched distance x:
// tab[d * naz + idx] = d^d A / dx^d for d = 0..D.  c = parameters of the
// centre's type in term order.  C: the type they are formed in; FP32 tables of
// pair sums are formed in FP64 and rounded once, since a rounded parameter would
// shift every pair the same way.
template <int N, int D, typename T = double, typename C = T>
__device__ __forceinline__ void een_tables(const double *c, C x, T *tab)
{
    constexpr EenTable<N> ET{};
    constexpr int NA = een_naz<N>();
    C xp[N + 1];
    xp[0] = C(1);
#pragma unroll
    for (int p = 1; p <= N; p++) xp[p] = p == 1 ? x : xp[1] * xp[p - 1];
    // one entry at a time: sum over the (term, half) pairs that land on it
#pragma unroll
    for (int d = 0; d <= D; d++)
#pragma unroll
        for (int e = 0; e < NA; e++) {
            C v = C(0);
#pragma unroll
            for (int t = 0; t < ET.n; t++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int n = h == 0 ? ET.m[t] : ET.l[t] + ET.m[t];
                    const int p = h == 0 ? ET.l[t] + ET.m[t] : ET.m[t];
                    if (ET.idx[ET.k[t]][n] != e || p < d) continue;
                    const C f = d == 0 ? C(1) : (d == 1 ? (C)p : (C)(p * (p - 1)));
                    v += (C)c[t] * f * xp[p - d];
                }
            tab[d * NA + e] = (T)v;
        }
}

// P and its derivatives at (u, y) from the tables of x:
//   D = 0: f;  D = 1: f, fu, fx, fy;  D = 2: also fuu, fxx, fyy, fux, fuy.
template <typename T = double>
struct EenOut {
    T f, fu, fx, fy, fuu, fxx, fyy, fux, fuy;
};

template <int N, int D, typename T = double>
__device__ __forceinline__ EenOut<T> een_eval_tab(const T *tab, T u, T y)
{
    constexpr EenTable<N> ET{};
    constexpr int NA = een_naz<N>();
    EenOut<T> o{0, 0, 0, 0, 0, 0, 0, 0, 0};
    // Horner in u over the row polynomials of y.  The derivative recurrences
    // (d2 = d2 y + d1, d1 = d1 y + p, p = p y + a) start from zero, so their
    // first updates are plain copies: the step counters are compile-time and
    // no multiply by a zero accumulator is emitted.  *2 names hold p''/2.
    T P = 0, Pu = 0, Puu2 = 0, Py = 0, Puy = 0, Pyy2 = 0, Px = 0, Pux = 0, Pxx = 0;
#pragma unroll
    for (int kk = N; kk >= 0; kk--) {
        if (kk > ET.kmax) continue;
        const int su = ET.kmax - kk;  // Horner step in u
        T q = 0, q1 = 0, q2 = 0, r = 0, s = 0;  // row k: value, d/dy, (d2/dy2)/2; dA/dx row; d2A/dx2 row
        const int nm = ET.nmax[kk];
        if (nm >= 0) {
            q = tab[ET.idx[kk][nm]];
            if (D >= 1) r = tab[NA + ET.idx[kk][nm]];
            if (D >= 2) s = tab[2 * NA + ET.idx[kk][nm]];
#pragma unroll
            for (int nn = N - 1; nn >= 0; nn--) {
                if (nn >= nm) continue;
                const int st = nm - 1 - nn;  // Horner step in y
                const int e = ET.idx[kk][nn];
                if (D >= 2 && st >= 1) q2 = st == 1 ? q1 : q2 * y + q1;
                if (D >= 1) q1 = st == 0 ? q : q1 * y + q;
                q = e >= 0 ? q * y + tab[e] : q * y;
                if (D >= 1) r = e >= 0 ? r * y + tab[NA + e] : r * y;
                if (D >= 2) s = e >= 0 ? s * y + tab[2 * NA + e] : s * y;
            }
        }
        if (su == 0) {
            P = q; Py = q1; Pyy2 = q2; Px = r; Pxx = s;
        } else {
            if (D >= 2 && su >= 2) Puu2 = su == 2 ? Pu : Puu2 * u + Pu;
            if (D >= 1) Pu = su == 1 ? P : Pu * u + P;
            P = P * u + q;
            if (D >= 2) Puy = su == 1 ? Py : Puy * u + Py;
            if (D >= 1) Py = Py * u + q1;
            if (D >= 2) Pyy2 = Pyy2 * u + q2;
            if (D >= 2) Pux = su == 1 ? Px : Pux * u + Px;
            if (D >= 1) Px = Px * u + r;
            if (D >= 2) Pxx = Pxx * u + s;
        }
    }
    o.f = P;
    if (D >= 1) { o.fu = Pu; o.fx = Px; o.fy = Py; }
    if (D >= 2) { o.fuu = T(2) * Puu2; o.fyy = T(2) * Pyy2; o.fxx = Pxx; o.fux = Pux; o.fuy = Puy; }
    return o;
}

// ------------------------------------------------------------------------
// The same polynomial split by what each part couples.  A term with m = 0 is
// c u^k (x^l + y^l): it depends on one electron-centre distance at a time, so
// summed over the centres it is u^k (X_k + Y_k) with one number per electron
// and power (k = 1 .. N - 1).  Only the terms with m >= 1 couple x and y:
//     sum_{k, n >= 1} C_kn(y) x^n u^k   (k = 0 .. N - 2),
// and those with k = 0 do not hold u, so that a sum over the partners needs
// sum_j C_0n(y_j) only.  At N = 4 three coupled entries (k >= 1) remain of
// the twelve of EenTable, at N = 5 six of eighteen.
template <int N>
struct EenSplit {
    int idx[N + 1][N + 1];  // packed position of C_kn, k >= 1, -1 where zero
    int nc;                 // number of them
    int kmax;               // highest coupled power of u (N - 2), 0 if none with k >= 1
    int nmax;               // highest power of x among them
    constexpr EenSplit() : idx{}, nc(0), kmax(0), nmax(0)
    {
        constexpr EenTable<N> ET{};
        bool nz[N + 1][N + 1] = {};
        for (int t = 0; t < ET.n; t++)
            if (ET.m[t] >= 1) {
                nz[ET.k[t]][ET.m[t]] = true;
                nz[ET.k[t]][ET.l[t] + ET.m[t]] = true;
            }
        for (int kk = 0; kk <= N; kk++)
            for (int nn = 0; nn <= N; nn++) {
                idx[kk][nn] = (kk >= 1 && nz[kk][nn]) ? nc++ : -1;
                if (idx[kk][nn] >= 0) {
                    if (kk > kmax) kmax = kk;
                    if (nn > nmax) nmax = nn;
                }
            }
    }
};
// numbers per electron of the uncoupled part, and of C_0n (both N - 1)
template <int N>
constexpr int een_nsep() { return N > 1 ? N - 1 : 0; }

// C_kn(y) of one (k, n); yp: the powers of y
template <int N, typename T>
__device__ __forceinline__ T een_coupled(const double *c, const T *yp, int k, int n)
{
    constexpr EenTable<N> ET{};
    T v = T(0);
#pragma unroll
    for (int t = 0; t < ET.n; t++) {
        if (ET.m[t] < 1 || ET.k[t] != k) continue;
        if (ET.m[t] == n) v += (T)c[t] * yp[ET.l[t] + ET.m[t]];
        if (ET.l[t] + ET.m[t] == n) v += (T)c[t] * yp[ET.m[t]];
    }
    return v;
}

template <int N, typename T>
__device__ __forceinline__ void een_powers(T y, T *yp)
{
    yp[0] = T(1);
#pragma unroll
    for (int p = 1; p <= N; p++) yp[p] = p == 1 ? y : y * yp[p - 1];
}

// s[k - 1] += sum over the uncoupled terms of power k of c_t y^l
template <int N, typename T>
__device__ __forceinline__ void een_uncoupled(const double *c, const T *yp, T *s)
{
    constexpr EenTable<N> ET{};
#pragma unroll
    for (int t = 0; t < ET.n; t++)
        if (ET.m[t] == 0) s[ET.k[t] - 1] += (T)c[t] * yp[ET.l[t]];
}

}  // namespace champ
