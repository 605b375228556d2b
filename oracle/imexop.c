/*
 * CPU oracle for the compressible implicit operator M + phi L and its
 * isothermal-wall treatment.
 *
 * TEST INFRASTRUCTURE ONLY.  Nothing in the product (the suzerain_amd
 * package, its HIP kernels or its C ABI) links, loads or calls this file.
 * Only tests/, __graft_entry__.smoke() and bench.py's cpu_baseline leg use
 * it, as the oracle or the timed CPU baseline.
 *
 * Restates, group of terms by group of terms:
 *   sz_or_imexop_accumulate   suzerain/rholut_imexop.c:43-531
 *                             (y <- (M + phi L) x + beta y, matrix free)
 *   sz_or_imexop_pack         suzerain/rholut_imexop.def:41-500
 *                             (P (M + phi L)^T P^T into band storage; packc
 *                             when ld = LD, packf when given LU + KL with
 *                             ld = LD + KL)
 *   sz_or_isothermal_op/rhs   apps/perfect/operator_hybrid_isothermal.cpp:
 *                             396-526 (IsothermalPATPTEnforcer)
 * The Giles non-reflecting upper-boundary matrices (a, b, c arguments of the
 * reference) are not restated: channel cases pass NULL for all three.
 *
 * Rounding convention (shared with the HIP kernels so both agree bit for
 * bit; contraction is off):
 *   kappa(km, kn) = ((k0 + k1 km^2) + k2 kn^2) + k3 km kn
 *                   + i (k4 km + k5 kn)                for each term's
 *                   scalar coefficient sans phi, with km^2 = km*km etc.
 *   alpha_t = phi * kappa_t                            (complex multiply
 *                   (fma(a.x,b.x,-a.y*b.y), fma(a.x,b.y,a.y*b.x)))
 *   W_g[r] = sum_t alpha_t ref_t[r] over a group g of terms sharing one
 *            derivative operator (first term a product, then fma)
 *   (D x)[r] = sum_c D[r][c] x[c] for c ascending over D's band, fma
 *   accumulate: acc[r] = sum over groups of W_g[r] (D_g x_j)[r] via
 *            acc + W t = (fma(-W.y,t.y,fma(W.x,t.x,acc.x)),
 *                         fma(W.y,t.x,fma(W.x,t.y,acc.y))),
 *            y[r] = ((beta y[r]) + acc[r]) + (M x_i)[r]  (mass last;
 *            beta == 0 never reads y)
 *   pack: A_ij[r][c] = sum over groups of W_g[r] D_g[r][c] (fma per
 *            component, skipping c outside D_g's own band), then + M[r][c]
 *            on diagonal blocks (mass last).
 * The reference evaluates the same sums in a different order (BLAS-like
 * loops, phi applied at pack time); it is matched to tolerance, not bits.
 *
 * Parity pins (tests/test_oracle_imexop.py): pack and accumulate agree as
 * matrices for every single nonzero reference profile and the wavenumber
 * set of tests/test_rholut_imexop.cpp:313-330; (M+phi L)^{-1}(M+phi L) = I
 * through the oracle's banded LU (tests/test_rholut_imexop.cpp:86-302);
 * at a uniform reference state at rest the operator equals the textbook
 * linearized compressible Navier-Stokes operator (acoustics, Stokes flow
 * with bulk viscosity, heat conduction) derived independently of the table.
 */
#include <complex.h>
#include <math.h>
#include <stddef.h>
#include <string.h>

typedef double complex zdouble;

static inline int imin(int a, int b) { return a < b ? a : b; }
static inline int imax(int a, int b) { return a > b ? a : b; }

/* Reference profile indices, in suzerain_rholut_imexop_ref member order
 * (suzerain/rholut_imexop.h:76-103). */
enum {
    ux, uy, uz, u2, uxux, uxuy, uxuz, uyuy, uyuz, uzuz,
    nu, nuux, nuuy, nuuz, nuu2, nuuxux, nuuxuy, nuuxuz, nuuyuy, nuuyuz,
    nuuzuz, ex_gradrho, ey_gradrho, ez_gradrho, e_divm, e_deltarho,
    NREF, ONE = -1
};
enum { M = 0, D1 = 1, D2 = 2 };

typedef struct { int ref; double k[6]; } term;

/* Everything one operator evaluation needs. */
typedef struct {
    zdouble phi;
    double km, kn;
    const double *const *ref;   /* NREF pointers */
    const int *refld;           /* NREF strides  */
    int n, ld, max_ku;          /* B-spline operators, transposed bands */
    const int *kl, *ku;         /* per-derivative bandwidths of D_T     */
    const double *dt;           /* derivative d at dt + d * dstride     */
    long dstride;
} ctx;

/* D_d[r][c] = D_T_d(c, r); nonzero for r - ku[d] <= c <= r + kl[d]. */
static inline double dget(const ctx *w, int d, int r, int c)
{
    return w->dt[d * w->dstride + (long)r * w->ld + w->max_ku + c - r];
}

static inline zdouble zmul(zdouble a, zdouble b)
{
    const double ax = creal(a), ay = cimag(a), bx = creal(b), by = cimag(b);
    const double yy = ay * by, yx = ay * bx;
    return CMPLX(fma(ax, bx, -yy), fma(ax, by, yx));
}

static inline zdouble zfma(zdouble a, zdouble b, zdouble c)
{
    const double bx = creal(b), by = cimag(b), cx = creal(c), cy = cimag(c);
    return CMPLX(fma(-by, cy, fma(bx, cx, creal(a))),
                 fma(by, cx, fma(bx, cy, cimag(a))));
}

static zdouble kappa(const double *k, double km, double kn)
{
    const double km2 = km * km, kn2 = kn * kn, kmkn = km * kn;
    double re = k[0] + k[1] * km2;
    re = re + k[2] * kn2;
    re = re + k[3] * kmkn;
    const double a = k[4] * km, b = k[5] * kn;
    return CMPLX(re, a + b);
}

static inline double refv(const ctx *w, int t, int r)
{
    return t == ONE ? 1.0 : w->ref[t][(long)r * w->refld[t]];
}

/* W_g[r] for one group of terms. */
static zdouble weight(const ctx *w, int nt, const term *t, const zdouble *al,
                      int r)
{
    const double v0 = refv(w, t[0].ref, r);
    double wx = creal(al[0]) * v0, wy = cimag(al[0]) * v0;
    for (int i = 1; i < nt; ++i) {
        const double v = refv(w, t[i].ref, r);
        wx = fma(creal(al[i]), v, wx);
        wy = fma(cimag(al[i]), v, wy);
    }
    return CMPLX(wx, wy);
}

static zdouble dapply(const ctx *w, int d, const zdouble *x, int r)
{
    double tx = 0, ty = 0;
    for (int c = imax(0, r - w->ku[d]); c <= imin(w->n - 1, r + w->kl[d]); ++c) {
        const double a = dget(w, d, r, c);
        tx = fma(a, creal(x[c]), tx);
        ty = fma(a, cimag(x[c]), ty);
    }
    return CMPLX(tx, ty);
}

/* acc += (sum_t alpha_t diag(ref_t)) D_d x, one call per group. */
static void group_acc(const ctx *w, int d, int nt, const term *t,
                      const zdouble *x, zdouble *acc)
{
    zdouble al[8];
    for (int i = 0; i < nt; ++i) al[i] = zmul(w->phi, kappa(t[i].k, w->km, w->kn));
    for (int r = 0; r < w->n; ++r)
        acc[r] = zfma(acc[r], weight(w, nt, t, al, r), dapply(w, d, x, r));
}

/* Dense-band element A_ij[r][c] contribution of one group, added in place. */
static void group_elem(const ctx *w, int d, int nt, const term *t,
                       const zdouble *al, int r, int c, double *ex, double *ey)
{
    if (c < r - w->ku[d] || c > r + w->kl[d]) return;
    const zdouble W = weight(w, nt, t, al, r);
    const double a = dget(w, d, r, c);
    *ex = fma(creal(W), a, *ex);
    *ey = fma(cimag(W), a, *ey);
}

/* ------------------------------------------------------------ term table
 * Each block (i, j) = (equation, input) of L, in E, u, v, w, rho order, is
 * a list of groups (derivative operator + terms).  Coefficients k0..k5 as in
 * kappa() above; the expressions follow rholut_imexop.c:121-502 with the
 * wavenumber polynomials expanded. */
#define MAXG 5
#define MAXT 5
typedef struct { int d, nt; term t[MAXT]; } group;
typedef struct { int ng; group g[MAXG]; } block;

#define K(r, a, b, c, dd, e, f) { r, { a, b, c, dd, e, f } }

static void build_table(const double *sc, block L[5][5])
{
    const double Re = sc[0], Pr = sc[1], Ma = sc[2], alpha = sc[3], gamma = sc[4];
    const double gm1 = gamma - 1, gm3 = gamma - 3;
    const double ap43 = alpha + 4.0 / 3.0, ap13 = alpha + 1.0 / 3.0;
    const double Ma2 = Ma * Ma, invRe = 1 / Re, invMa2 = 1 / Ma2;
    const double ginvPr = gamma / Pr, ginvRePr = gamma / (Re * Pr);
    const double MiR = Ma2 * invRe, MiRa = Ma2 * invRe * ap13;
    const double gRPg = ginvRePr / gm1, aiR = ap13 * invRe;
    memset(L, 0, sizeof(block) * 25);

    /* energy equation, rholut_imexop.c:121-222 */
    L[0][0] = (block){ 3, {
        { M, 3, { K(ux, 0, 0, 0, 0, -gamma, 0), K(uz, 0, 0, 0, 0, 0, -gamma),
                  K(nu, 0, -ginvRePr, -ginvRePr, 0, 0, 0) } },
        { D1, 1, { K(uy, -gamma, 0, 0, 0, 0, 0) } },
        { D2, 1, { K(nu, ginvRePr, 0, 0, 0, 0, 0) } } } };
    L[0][1] = (block){ 3, {
        { M, 3, { K(nuux, 0, MiR * (ginvPr - ap43), MiR * (ginvPr - 1), 0, 0, 0),
                  K(nuuz, 0, 0, 0, -MiRa, 0, 0), K(e_divm, 0, 0, 0, 0, -1, 0) } },
        { D1, 1, { K(nuuy, 0, 0, 0, 0, MiRa, 0) } },
        { D2, 1, { K(nuux, MiR * (1 - ginvPr), 0, 0, 0, 0, 0) } } } };
    L[0][2] = (block){ 3, {
        { M, 1, { K(nuuy, 0, MiR * (ginvPr - 1), MiR * (ginvPr - 1), 0, 0, 0) } },
        { D1, 3, { K(nuux, 0, 0, 0, 0, MiRa, 0), K(nuuz, 0, 0, 0, 0, 0, MiRa),
                   K(e_divm, -1, 0, 0, 0, 0, 0) } },
        { D2, 1, { K(nuuy, MiR * (ap43 - ginvPr), 0, 0, 0, 0, 0) } } } };
    L[0][3] = (block){ 3, {
        { M, 3, { K(nuux, 0, 0, 0, -MiRa, 0, 0),
                  K(nuuz, 0, MiR * (ginvPr - 1), MiR * (ginvPr - ap43), 0, 0, 0),
                  K(e_divm, 0, 0, 0, 0, 0, -1) } },
        { D1, 1, { K(nuuy, 0, 0, 0, 0, 0, MiRa) } },
        { D2, 1, { K(nuuz, MiR * (1 - ginvPr), 0, 0, 0, 0, 0) } } } };
    L[0][4] = (block){ 4, {
        { M, 4, { K(nuu2, 0, MiR, MiR, 0, 0, 0), K(nuuxux, 0, MiRa, 0, 0, 0, 0),
                  K(nuuxuz, 0, 0, 0, MiRa * 2, 0, 0),
                  K(nuuzuz, 0, 0, MiRa, 0, 0, 0) } },
        { M, 3, { K(ex_gradrho, 0, 0, 0, 0, -1, 0),
                  K(ez_gradrho, 0, 0, 0, 0, 0, -1),
                  K(e_deltarho, 0, -gRPg, -gRPg, 0, 0, 0) } },
        { D1, 3, { K(nuuxuy, 0, 0, 0, 0, -MiRa * 2, 0),
                   K(nuuyuz, 0, 0, 0, 0, 0, -MiRa * 2),
                   K(ey_gradrho, -1, 0, 0, 0, 0, 0) } },
        { D2, 3, { K(nuu2, -MiR, 0, 0, 0, 0, 0), K(nuuyuy, -MiRa, 0, 0, 0, 0, 0),
                   K(e_deltarho, gRPg, 0, 0, 0, 0, 0) } } } };

    /* streamwise momentum, rholut_imexop.c:236-313 */
    L[1][0] = (block){ 1, { { M, 1, { K(ONE, 0, 0, 0, 0, -gm1 * invMa2, 0) } } } };
    L[1][1] = (block){ 3, {
        { M, 3, { K(ux, 0, 0, 0, 0, gm3, 0), K(uz, 0, 0, 0, 0, 0, -1),
                  K(nu, 0, -invRe * ap43, -invRe, 0, 0, 0) } },
        { D1, 1, { K(uy, -1, 0, 0, 0, 0, 0) } },
        { D2, 1, { K(nu, invRe, 0, 0, 0, 0, 0) } } } };
    L[1][2] = (block){ 2, {
        { M, 1, { K(uy, 0, 0, 0, 0, gm1, 0) } },
        { D1, 2, { K(ux, -1, 0, 0, 0, 0, 0), K(nu, 0, 0, 0, 0, aiR, 0) } } } };
    L[1][3] = (block){ 1, {
        { M, 3, { K(ux, 0, 0, 0, 0, 0, -1), K(uz, 0, 0, 0, 0, gm1, 0),
                  K(nu, 0, 0, 0, -aiR, 0, 0) } } } };
    L[1][4] = (block){ 3, {
        { M, 5, { K(u2, 0, 0, 0, 0, -0.5 * gm1, 0), K(uxux, 0, 0, 0, 0, 1, 0),
                  K(uxuz, 0, 0, 0, 0, 0, 1),
                  K(nuux, 0, invRe * ap43, invRe, 0, 0, 0),
                  K(nuuz, 0, 0, 0, aiR, 0, 0) } },
        { D1, 2, { K(uxuy, 1, 0, 0, 0, 0, 0), K(nuuy, 0, 0, 0, 0, -aiR, 0) } },
        { D2, 1, { K(nuux, -invRe, 0, 0, 0, 0, 0) } } } };

    /* wall-normal momentum, rholut_imexop.c:315-387 */
    L[2][0] = (block){ 1, { { D1, 1, { K(ONE, -gm1 * invMa2, 0, 0, 0, 0, 0) } } } };
    L[2][1] = (block){ 2, {
        { M, 1, { K(uy, 0, 0, 0, 0, -1, 0) } },
        { D1, 2, { K(ux, gm1, 0, 0, 0, 0, 0), K(nu, 0, 0, 0, 0, aiR, 0) } } } };
    L[2][2] = (block){ 3, {
        { M, 3, { K(ux, 0, 0, 0, 0, -1, 0), K(uz, 0, 0, 0, 0, 0, -1),
                  K(nu, 0, -invRe, -invRe, 0, 0, 0) } },
        { D1, 1, { K(uy, gm3, 0, 0, 0, 0, 0) } },
        { D2, 1, { K(nu, ap43 * invRe, 0, 0, 0, 0, 0) } } } };
    L[2][3] = (block){ 2, {
        { M, 1, { K(uy, 0, 0, 0, 0, 0, -1) } },
        { D1, 2, { K(uz, gm1, 0, 0, 0, 0, 0), K(nu, 0, 0, 0, 0, 0, aiR) } } } };
    L[2][4] = (block){ 3, {
        { M, 3, { K(uxuy, 0, 0, 0, 0, 1, 0), K(uyuz, 0, 0, 0, 0, 0, 1),
                  K(nuuy, 0, invRe, invRe, 0, 0, 0) } },
        { D1, 4, { K(u2, -0.5 * gm1, 0, 0, 0, 0, 0), K(uyuy, 1, 0, 0, 0, 0, 0),
                   K(nuux, 0, 0, 0, 0, -aiR, 0), K(nuuz, 0, 0, 0, 0, 0, -aiR) } },
        { D2, 1, { K(nuuy, -ap43 * invRe, 0, 0, 0, 0, 0) } } } };

    /* spanwise momentum, rholut_imexop.c:389-459 */
    L[3][0] = (block){ 1, { { M, 1, { K(ONE, 0, 0, 0, 0, 0, -gm1 * invMa2) } } } };
    L[3][1] = (block){ 1, {
        { M, 3, { K(ux, 0, 0, 0, 0, 0, gm1), K(uz, 0, 0, 0, 0, -1, 0),
                  K(nu, 0, 0, 0, -aiR, 0, 0) } } } };
    L[3][2] = (block){ 2, {
        { M, 1, { K(uy, 0, 0, 0, 0, 0, gm1) } },
        { D1, 2, { K(uz, -1, 0, 0, 0, 0, 0), K(nu, 0, 0, 0, 0, 0, aiR) } } } };
    L[3][3] = (block){ 3, {
        { M, 3, { K(ux, 0, 0, 0, 0, -1, 0), K(uz, 0, 0, 0, 0, 0, gm3),
                  K(nu, 0, -invRe, -invRe * ap43, 0, 0, 0) } },
        { D1, 1, { K(uy, -1, 0, 0, 0, 0, 0) } },
        { D2, 1, { K(nu, invRe, 0, 0, 0, 0, 0) } } } };
    L[3][4] = (block){ 3, {
        { M, 5, { K(u2, 0, 0, 0, 0, 0, -0.5 * gm1), K(uxuz, 0, 0, 0, 0, 1, 0),
                  K(uzuz, 0, 0, 0, 0, 0, 1),
                  K(nuuz, 0, invRe, invRe * ap43, 0, 0, 0),
                  K(nuux, 0, 0, 0, aiR, 0, 0) } },
        { D1, 2, { K(uyuz, 1, 0, 0, 0, 0, 0), K(nuuy, 0, 0, 0, 0, 0, -aiR) } },
        { D2, 1, { K(nuuz, -invRe, 0, 0, 0, 0, 0) } } } };

    /* density, rholut_imexop.c:461-487 */
    L[4][1] = (block){ 1, { { M, 1, { K(ONE, 0, 0, 0, 0, -1, 0) } } } };
    L[4][2] = (block){ 1, { { D1, 1, { K(ONE, -1, 0, 0, 0, 0, 0) } } } };
    L[4][3] = (block){ 1, { { M, 1, { K(ONE, 0, 0, 0, 0, 0, -1) } } } };
}

/* Coefficients k0..k5 of every term, flattened in block, group, term
 * order, for tests that inspect the table (returns the term count). */
int sz_or_imexop_terms(const double *scenario, int *eq, int *in, int *op,
                       int *ref, double *k, int maxterms)
{
    block L[5][5];
    build_table(scenario, L);
    int cnt = 0;
    for (int i = 0; i < 5; ++i)
        for (int j = 0; j < 5; ++j)
            for (int g = 0; g < L[i][j].ng; ++g)
                for (int t = 0; t < L[i][j].g[g].nt; ++t) {
                    if (cnt < maxterms) {
                        eq[cnt] = i; in[cnt] = j; op[cnt] = L[i][j].g[g].d;
                        ref[cnt] = L[i][j].g[g].t[t].ref;
                        memcpy(k + 6 * cnt, L[i][j].g[g].t[t].k, 6 * sizeof(double));
                    }
                    ++cnt;
                }
    return cnt;
}

/* y_i <- (M + phi L) x restricted to present fields + beta y_i for each
 * output present.  in/out hold 5 pointers (E, u, v, w, rho order); a NULL
 * input omits that field (and its output).  Returns 0. */
int sz_or_imexop_accumulate(zdouble phi, double km, double kn,
                            const double *scenario,
                            const double *const *ref, const int *refld,
                            int n, const double *dt, int ld, long dstride,
                            int max_ku, const int *kl, const int *ku,
                            const zdouble *const *in, zdouble beta,
                            zdouble *const *out)
{
    block L[5][5];
    build_table(scenario, L);
    const ctx w = { phi, km, kn, ref, refld, n, ld, max_ku, kl, ku, dt, dstride };
    zdouble acc[n];
    for (int i = 0; i < 5; ++i) {
        if (!in[i]) continue;
        for (int r = 0; r < n; ++r) acc[r] = 0;
        for (int j = 0; j < 5; ++j) {
            if (!in[j]) continue;
            for (int g = 0; g < L[i][j].ng; ++g)
                group_acc(&w, L[i][j].g[g].d, L[i][j].g[g].nt, L[i][j].g[g].t,
                          in[j], acc);
        }
        for (int r = 0; r < n; ++r) {
            const zdouble by = beta == 0 ? 0 : zmul(beta, out[i][r]);
            const zdouble s = CMPLX(creal(by) + creal(acc[r]),
                                    cimag(by) + cimag(acc[r]));
            const zdouble m = dapply(&w, M, in[i], r);
            out[i][r] = CMPLX(creal(s) + creal(m), cimag(s) + cimag(m));
        }
    }
    return 0;
}

/* Geometry of suzerain_bsmbsm_construct, bsmbsm.h:130-149. */
static void geometry(int S, int n, int kl, int ku, int *KL, int *KU, int *LD)
{
    *KL = S * (kl + 1) - 1;
    *KU = S * (ku + 1) - 1;
    *LD = *KL + 1 + *KU;
}

/* P (M + phi L)^T P^T into band storage: element (R, C) of the permuted
 * transpose lands at papt[C * ldpapt + KU + R - C].  idx[5] gives the block
 * position of E, u, v, w, rho (negative omits that field); S is the count of
 * present fields.  Every band slot is written. */
int sz_or_imexop_pack(zdouble phi, double km, double kn, const double *scenario,
                      const double *const *ref, const int *refld,
                      int n, const double *dt, int ld, long dstride,
                      int max_kl, int max_ku, const int *kl, const int *ku,
                      const int *idx, zdouble *papt, int ldpapt)
{
    block L[5][5];
    build_table(scenario, L);
    const ctx w = { phi, km, kn, ref, refld, n, ld, max_ku, kl, ku, dt, dstride };
    int S = 0, field_of[5];
    for (int f = 0; f < 5; ++f) if (idx[f] >= 0) field_of[idx[f]] = f, ++S;
    int KL, KU, LD;
    geometry(S, n, max_kl, max_ku, &KL, &KU, &LD);
    const int N = S * n;
    /* per-block coefficients alpha_t = phi kappa_t */
    zdouble al[5][5][MAXG][MAXT];
    for (int i = 0; i < 5; ++i)
        for (int j = 0; j < 5; ++j)
            for (int g = 0; g < L[i][j].ng; ++g)
                for (int t = 0; t < L[i][j].g[g].nt; ++t)
                    al[i][j][g][t] = zmul(phi, kappa(L[i][j].g[g].t[t].k, km, kn));
    for (int C = 0; C < N; ++C) {
        for (int R = imax(0, C - KU); R <= imin(N - 1, C + KL); ++R) {
            /* (R, C) of P A^T P^T is (q(R), q(C)) of A^T, i.e. element
             * (q(C), q(R)) of A: equation block of q(C), input block of q(R) */
            const int qr = (R % S) * n + R / S, qc = (C % S) * n + C / S;
            const int bi = qc / n, r = qc % n;   /* A row:    equation, y */
            const int bj = qr / n, c = qr % n;   /* A column: input,    y */
            const int fi = field_of[bi], fj = field_of[bj];
            double ex = 0, ey = 0;
            if (c >= r - max_ku && c <= r + max_kl) {
                const block *b = &L[fi][fj];
                for (int g = 0; g < b->ng; ++g)
                    group_elem(&w, b->g[g].d, b->g[g].nt, b->g[g].t,
                               al[fi][fj][g], r, c, &ex, &ey);
                if (fi == fj && c >= r - ku[M] && c <= r + kl[M])
                    ex = ex + dget(&w, M, r, c);
            }
            papt[(long)C * ldpapt + KU + R - C] = CMPLX(ex, ey);
        }
    }
    return 0;
}

/* IsothermalPATPTEnforcer::op (operator_hybrid_isothermal.cpp:470-510) on
 * P A^T P^T band storage: at each enforced wall replace the energy and
 * momentum equations (columns of P A^T P^T) by
 *   d/dt rhoE - E_factor d/dt rho = 0,  d/dt m_k - vel_k d/dt rho = 0,
 * keeping the diagonal entry as the scaling (1 when it is zero).
 * walls[2] = {T, u, v, w} per wall; sc = scenario (Ma at [2], gamma at [4]). */
int sz_or_isothermal_op(int S, int n, int KL, int KU, zdouble *papt,
                        int ldpapt, const int *idx, const double *scenario,
                        const double *lower, const double *upper,
                        int enforce_lower, int enforce_upper)
{
    const double Ma = scenario[2], gamma = scenario[4];
    const double *spec[2] = { lower, upper };
    const int N = S * n;
    for (int wall = enforce_lower ? 0 : 1; wall < (enforce_upper ? 2 : 1); ++wall) {
        const double *p = spec[wall];
        const int y = wall ? n - 1 : 0;
        const double Ef = p[0] / (gamma * (gamma - 1))
                        + Ma * Ma / 2 * (p[1] * p[1] + p[2] * p[2] + p[3] * p[3]);
        const int ar = idx[4] * n + y;
        const int rho = (ar % n) * S + ar / n;           /* q^{-1} */
        const int eqs[4] = { idx[0], idx[1], idx[2], idx[3] };
        const double fac[4] = { Ef, p[1], p[2], p[3] };
        for (int k = 0; k < 4; ++k) {
            const int a = eqs[k] * n + y;
            const int col = (a % n) * S + a / n;   /* q^{-1} */
            zdouble *cp = papt + (long)col * ldpapt + KU - col;   /* cp[i]: (i,col) */
            zdouble scaling = cp[col];
            if (scaling == 0) scaling = 1;
            for (int i = imax(0, col - KU); i < imin(N, col + KL + 1); ++i) {
                cp[i] = i == col ? scaling
                      : i == rho ? CMPLX(-creal(scaling) * fac[k],
                                         -cimag(scaling) * fac[k])
                      : 0;
            }
        }
    }
    return 0;
}

/* IsothermalPATPTEnforcer::rhs (operator_hybrid_isothermal.cpp:513-524):
 * zero the permuted right hand side of the replaced equations. */
int sz_or_isothermal_rhs(int S, int n, zdouble *pb, const int *idx,
                         int enforce_lower, int enforce_upper)
{
    for (int wall = enforce_lower ? 0 : 1; wall < (enforce_upper ? 2 : 1); ++wall) {
        const int y = wall ? n - 1 : 0;
        for (int k = 0; k < 4; ++k) {
            const int a = idx[k] * n + y;
            pb[(a % n) * S + a / n] = 0;
        }
    }
    return 0;
}
