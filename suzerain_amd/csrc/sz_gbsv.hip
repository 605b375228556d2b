// Batched complex banded LU factorization and solve for gfx950.
//
// Semantics follow LAPACK ZGBTRF/ZGBTRS (and CGBTRF/CGBTRS for the single
// precision factor of the mixed-precision solver) as the reference calls
// them through suzerain_lapack_zgbtrf/zgbtrs (suzerain/blas_et_al/
// lapack.c:185-278) from bsmbsm_solver_zgbsv::solve_hook
// (suzerain/bsmbsm_solver.cpp:155-182):
//   * band storage, column major, leading dimension ldab >= 2*kl+ku+1, A(i,j)
//     at j*ldab + kl+ku + i-j on entry; U in rows 0..kl+ku and the
//     multipliers in rows kl+ku+1..2*kl+ku on exit (in place);
//   * partial pivoting with the pivot chosen by |Re|+|Im| (IZAMAX), first
//     maximum wins, ipiv 1-based;
//   * info = first 1-based column with an exactly zero pivot, else 0; the
//     factorization continues past a zero pivot without scaling or update.
//
// Two factorization kernels, both moving each element through HBM once: the
// active (kl+1) x (kl+ku+1) window of rows j..j+kl and columns j..j+kl+ku
// stays on chip, so an elimination step brings in one row (row j+kl+1) and
// sends out one row (U row j) and one column (the multipliers of column j).
//   * k_gbtrf_panel: one wavefront per system, one window column per lane,
//     the rows in registers, four columns at a time; no barriers.  Used for
//     the band shapes of the channel operators.
//   * k_gbtrf: one workgroup per system, the window in LDS as a circular
//     buffer in both directions; wave 0 does the pivot search, the swap and
//     the scaling, then all waves apply the rank-1 update.  Any band shape.
#include "sz_common.hpp"
#include "sz_row.hpp"

#include <cstdlib>
#include <type_traits>
#include <utility>

// the compiler's DPP move for 64-bit values (its builtin takes 32 bits only)
__device__ double sz_update_dpp(double, double, int, int, int, bool)
    __asm("llvm.amdgcn.update.dpp.f64");
__device__ int sz_writelane(int value, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

namespace {

using sz::cpx;

constexpr int TRS_NT = 64;
constexpr size_t LDS_MAX = 160 * 1024;

template <typename R>
__device__ inline void argmax_cabs1(R &best, int &bidx)
{
    for (int off = 32; off >= 1; off >>= 1) {
        const R ob = __shfl_xor(best, off);
        const int oi = __shfl_xor(bidx, off);
        if (ob > best || (ob == best && oi < bidx)) { best = ob; bidx = oi; }
    }
}

// Barrier ordering LDS only: global loads and stores in flight stay in
// flight (the factorization never communicates through global memory).
#define LDS_BARRIER()                                                         \
    do {                                                                      \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");       \
        __builtin_amdgcn_s_barrier();                                         \
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");       \
    } while (0)

template <int CTRL, typename R>
__device__ __forceinline__ R dpp_r(R v)
{
    if constexpr (sizeof(R) == 8) {
        const long long b = __builtin_bit_cast(long long, v);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, true);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF,
                                                   0xF, true);
        return __builtin_bit_cast(R, (long long)(((unsigned long long)(unsigned)hi << 32)
                                                 | (unsigned)lo));
    } else {
        return __builtin_bit_cast(
            R, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF,
                                           0xF, true));
    }
}

template <typename R>
__device__ __forceinline__ R readlane_r(R v, int lane)
{
    if constexpr (sizeof(R) == 8) {
        const long long b = __builtin_bit_cast(long long, v);
        const int lo = __builtin_amdgcn_readlane((int)b, lane);
        const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
        return __builtin_bit_cast(R, (long long)(((unsigned long long)(unsigned)hi << 32)
                                                 | (unsigned)lo));
    } else {
        return __builtin_bit_cast(R, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v),
                                                               lane));
    }
}

// Sum over the 64 lanes as the butterfly w[l] += w[l ^ off], off = 1, 2, 4,
// ..., 32, evaluated at lane 0 and returned to every lane.  After the
// offsets 1 and 2 a quad holds one value, so the half-row mirror (lane
// l ^ 7) delivers the l ^ 4 partner; after 4 the same holds for the row
// mirror (l ^ 15) and 8; rows then combine as (r0 + r1) + (r2 + r3).
template <typename R>
__device__ inline R wave_sum_asc(R v)
{
    v += dpp_r<0xB1>(v);                    // quad_perm [1,0,3,2]
    v += dpp_r<0x4E>(v);                    // quad_perm [2,3,0,1]
    v += dpp_r<0x141>(v);                   // row_half_mirror
    v += dpp_r<0x140>(v);                   // row_mirror
    return (readlane_r(v, 0) + readlane_r(v, 16)) +
           (readlane_r(v, 32) + readlane_r(v, 48));
}

template <typename R>
__device__ inline cpx<R> wave_csum(cpx<R> v)
{
    return cpx<R>{wave_sum_asc(v.x), wave_sum_asc(v.y)};
}

// The largest of the 64 lanes' values (no NaN among them).
template <typename R>
__device__ __forceinline__ R wave_max(R v)
{
    v = fmax(v, dpp_r<0xB1>(v));            // the stages of wave_sum_asc
    v = fmax(v, dpp_r<0x4E>(v));
    v = fmax(v, dpp_r<0x141>(v));
    v = fmax(v, dpp_r<0x140>(v));
    return fmax(fmax(readlane_r(v, 0), readlane_r(v, 16)),
                fmax(readlane_r(v, 32), readlane_r(v, 48)));
}

constexpr int TRF_PF = 8;   // incoming rows prefetched ahead of their step

template <typename R>
__device__ __forceinline__ cpx<R> ld_or_zero(const cpx<R> *p, bool ok)
{
    cpx<R> v;
    v.x = R(0);
    v.y = R(0);
    if (ok) {
        v.x = p->x;
        v.y = p->y;
    }
    return v;
}

template <typename R, int TRF_NT>
__global__ __launch_bounds__(TRF_NT)
void k_gbtrf(int n, int kl, int ku, cpx<R> *__restrict__ ab, int ldab,
             long long sab, int *__restrict__ ipiv, long long sipiv,
             int *__restrict__ info, const int *__restrict__ skip, int nsys)
{
    using T = cpx<R>;
    extern __shared__ __align__(16) unsigned char smem[];
    const int sys = blockIdx.x;
    if (sys >= nsys) return;
    if (skip && skip[sys] != 0) return;   // masked out by the caller
    ab += (size_t)sys * (size_t)sab;
    ipiv += (size_t)sys * (size_t)sipiv;
    const int tid = threadIdx.x;
    const int kv = kl + ku;
    const int WR = kl + 1, WC = kv + 1;
    T *W = reinterpret_cast<T *>(smem);   // W[rowslot*WC + colslot]
    T *Urow = W + WR * WC;                // pivot row after the swap
    T *Lcol = Urow + WC;                  // multipliers of column j
    __shared__ int s_ju, s_nz, s_info;

    for (int e = tid; e < WR * WC; e += TRF_NT) {
        const int r = e / WC, c = e - r * WC;
        const bool ok = r < n && c < n && r - c <= kl && c - r <= ku;
        W[e] = ld_or_zero(ab + (ok ? (size_t)c * ldab + kv + r - c : 0), ok);
    }
    if (tid == 0) { s_ju = 0; s_info = 0; }
    // Every thread issues the same global loads and stores at every step
    // (duplicates for tid >= WC hit the same addresses with the same values),
    // so the compiler can count outstanding memory operations exactly and
    // the prefetched rows below are waited for only when they are consumed.
    // Thread column cl brings in element cl of the row entering at each step:
    // row i = j + WR, column k = j + 1 + cl, i.e. band row kv + kl - cl.
    constexpr int NCL = TRF_NT >= 128 ? 1 : 2;   // entering-row columns per thread
    int cl[NCL], brow[NCL];
#pragma unroll
    for (int m = 0; m < NCL; ++m) {
        cl[m] = (tid + TRF_NT * m) % WC;
        brow[m] = kv + kl - cl[m];
    }
    const int rl = 1 + tid % (kl > 0 ? kl : 1);
    // q[u][m] holds the raw element (read from a clamped, always valid
    // address); rows or columns beyond n are zeroed when it is consumed.
    T q[TRF_PF][NCL];
#pragma unroll
    for (int u = 0; u < TRF_PF; ++u) {
#pragma unroll
        for (int m = 0; m < NCL; ++m) {
            const int i = u + WR, k = u + 1 + cl[m];
            const bool ok = i < n && k < n;
            q[u][m] = ab[ok ? (size_t)k * ldab + brow[m] : 0];
        }
    }
    __shared__ int s_p;
    LDS_BARRIER();

    int rs0 = 0, cs0 = 0;   // slots holding row j and column j
    for (int j0 = 0; j0 < n; j0 += TRF_PF) {
#pragma unroll
        for (int u = 0; u < TRF_PF; ++u) {
            const int j = j0 + u;
            if (j >= n) break;
            const int km = min(kl, n - 1 - j);
            if (tid < 64) {
                // ---- pivot search (IZAMAX: first maximum of |Re|+|Im|; a
                // NaN never beats a number, a NaN in the first slot wins)
                R best = R(-1);
                int bidx = 0x7fffffff;
                if (kl < 64) {
                    // a row a lane: the maximum by DPP, then its first lane.
                    // (Value and index through six lane exchanges, as for more
                    // rows: 600 systems n = 301, kl 17, ku 11 in 763 us, so
                    // 595.)
                    R a = R(-2);
                    if (tid <= km) {
                        int rs = rs0 + tid; if (rs >= WR) rs -= WR;
                        a = sz::cabs1(W[rs * WC + cs0]);
                        if (a != a) a = R(-1);
                    }
                    best = wave_max(a);
                    bidx = (int)__builtin_ctzll(__ballot(a == best));
                } else {
                    for (int r = tid; r <= km; r += 64) {
                        int rs = rs0 + r; if (rs >= WR) rs -= WR;
                        R a = sz::cabs1(W[rs * WC + cs0]);
                        if (a != a) a = R(-1);
                        if (a > best || (a == best && r < bidx)) { best = a; bidx = r; }
                    }
                    argmax_cabs1(best, bidx);
                }
                const T a0 = W[rs0 * WC + cs0];
                const R a0abs = sz::cabs1(a0);
                const int p = (a0abs != a0abs) ? 0 : bidx;
                int prs = rs0 + p; if (prs >= WR) prs -= WR;
                const T piv = W[prs * WC + cs0];
                const bool nz = sz::cnonzero(piv);
                int ju = s_ju;
                if (nz) ju = max(ju, min(j + ku + p, n - 1));
                const bool swap = nz && p != 0;
                // ---- row j after the swap -> Urow; old row j -> slot p
                for (int c = tid; c <= kv; c += 64) {
                    int cs = cs0 + c; if (cs >= WC) cs -= WC;
                    const T a = W[rs0 * WC + cs];
                    const T b = W[prs * WC + cs];
                    const bool sw = swap && c <= ju - j;
                    T uu;
                    uu.x = sw ? b.x : a.x;
                    uu.y = sw ? b.y : a.y;
                    if (sw) W[prs * WC + cs] = a;
                    Urow[c] = uu;
                }
                // ---- multipliers (row p now holds old row j's entry a0)
                T rcp;
                rcp.x = R(0);
                rcp.y = R(0);
                if (nz) rcp = sz::crcp(piv);
                for (int r = 1 + tid; r <= km; r += 64) {
                    int rs = rs0 + r; if (rs >= WR) rs -= WR;
                    const T w = W[rs * WC + cs0];
                    const bool use_a0 = swap && r == p;
                    T v;
                    v.x = use_a0 ? a0.x : w.x;
                    v.y = use_a0 ? a0.y : w.y;
                    const T l = sz::cmul(v, rcp);
                    T out;
                    out.x = nz ? l.x : v.x;
                    out.y = nz ? l.y : v.y;
                    Lcol[r] = out;
                }
                if (tid == 0) {
                    s_p = p;
                    s_ju = ju;
                    s_nz = nz ? 1 : 0;
                    if (!nz && s_info == 0) s_info = j + 1;
                }
            }
            LDS_BARRIER();

            const int ju = s_ju;
            const bool nz = s_nz != 0;
            // ---- rank-1 update of rows j+1..j+km, columns j+1..ju
            if (nz) {
                const int w = ju - j;
                const int lane = tid & 63;
                for (int c = 1 + lane; c <= w; c += 64) {
                    int cs = cs0 + c; if (cs >= WC) cs -= WC;
                    const T uu = Urow[c];
                    for (int r = 1 + (tid >> 6); r <= km; r += TRF_NT / 64) {
                        int rs = rs0 + r; if (rs >= WR) rs -= WR;
                        T *pa = W + rs * WC + cs;
                        *pa = sz::cfnms(*pa, Lcol[r], uu);
                    }
                }
            }
            // ---- U row j, multipliers of column j and the pivot index to
            // HBM: one unconditional store each per thread (redirected onto
            // U(j,j) when this thread has nothing of its own to write)
            {
                const int cmax = min(kv, n - 1 - j);
#pragma unroll
                for (int m = 0; m < NCL; ++m) {
                    const int ce = cl[m] <= cmax ? cl[m] : 0;
                    ab[(size_t)(j + ce) * ldab + kv - ce] = Urow[ce];
                }
                const int re = (kl > 0 && rl <= km) ? rl : 0;
                ab[(size_t)j * ldab + kv + re] = re ? Lcol[re] : Urow[0];
                ipiv[j] = j + s_p + 1;
            }
            // ---- column slot cs0 becomes column j+kv+1 (fill-in zeros) and
            // row slot rs0 becomes row j+kl+1 (prefetched PF steps ago)
            for (int r = tid; r < WR; r += TRF_NT)
                if (r != rs0) W[r * WC + cs0] = T{0, 0};
#pragma unroll
            for (int m = 0; m < NCL; ++m) {
                if (tid + TRF_NT * m < WC) {
                    const bool in = (j + WR < n) && (j + 1 + cl[m] < n);
                    int cs = cs0 + 1 + cl[m]; if (cs >= WC) cs -= WC;
                    T qv;
                    qv.x = in ? q[u][m].x : R(0);
                    qv.y = in ? q[u][m].y : R(0);
                    W[rs0 * WC + cs] = qv;
                }
                const int i = j + TRF_PF + WR, k = j + TRF_PF + 1 + cl[m];
                const bool ok = i < n && k < n;
                q[u][m] = ab[ok ? (size_t)k * ldab + brow[m] : 0];
            }
            LDS_BARRIER();
            if (++rs0 == WR) rs0 = 0;
            if (++cs0 == WC) cs0 = 0;
        }
    }
    if (tid == 0 && info) info[sys] = s_info;
}

constexpr int TRS_PRE = 18;

template <typename R>
__device__ __forceinline__ void chunk_load(R (&rx)[TRS_PRE], R (&ry)[TRS_PRE],
                                           const cpx<R> *__restrict__ ab,
                                           int ldab, int c0, int nc, int r0,
                                           int w)
{
    const int tot = nc * w;
#pragma unroll
    for (int m = 0; m < TRS_PRE; ++m) {
        const int e = threadIdx.x + TRS_NT * m;
        const bool ok = e < tot;
        const int jj = ok ? e / w : 0, rr = ok ? e - jj * w : 0;
        const cpx<R> v = ab[(size_t)(c0 + jj) * ldab + r0 + rr];
        rx[m] = v.x;
        ry[m] = v.y;
    }
}

template <typename R>
__device__ __forceinline__ void chunk_store(const R (&rx)[TRS_PRE],
                                            const R (&ry)[TRS_PRE], cpx<R> *st,
                                            int nc, int w)
{
    const int tot = nc * w;
#pragma unroll
    for (int m = 0; m < TRS_PRE; ++m) {
        const int e = threadIdx.x + TRS_NT * m;
        if (e < tot) st[e] = cpx<R>{rx[m], ry[m]};
    }
}


template <typename R>
__device__ inline cpx<R> cj_if(cpx<R> v, bool c)
{
    cpx<R> r;
    r.x = v.x;
    r.y = c ? -v.y : v.y;
    return r;
}

template <int... I, typename F>
__device__ __forceinline__ void unroll_impl(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int K, typename F>
__device__ __forceinline__ void unroll(F &&f)
{
    unroll_impl(f, std::make_integer_sequence<int, K>{});
}

// L^T x = y and the interchanges, the second half of a transposed solve, on x
// in LDS by one wavefront.
template <typename R>
__device__ __forceinline__ void lt_sweep(int n, int kl, int kv,
                                         const cpx<R> *__restrict__ ab, int ldab,
                                         const int *__restrict__ ipiv, bool cj, cpx<R> *x,
                                         int tid)
{
    using T = cpx<R>;
    // L^T x = y then undo the interchanges, descending.  Lane r
    // forms the terms r, r+64, ... of the dot product with the
    // multipliers of column j (one contiguous run, prefetched a few
    // steps ahead) and the butterfly combines them.
    if (kl > 0 && n > 1) {
        constexpr int QP = 4;
        auto laddr = [&](int jj, int r) -> size_t {   // L(jj+1+r, jj)
            const bool ok = jj >= 0 && r < min(kl, n - 1 - jj);
            return ok ? (size_t)jj * ldab + kv + 1 + r : 0;
        };
        T l1[QP], l2[QP];
        int qp[QP];
        // a zero the compiler takes for a lane's own: scalar loads would join
        // the counter that every wait for LDS drains
        int z = 0;
        asm volatile("" : "+v"(z));
#pragma unroll
        for (int u = 0; u < QP; ++u) {
            l1[u] = ab[laddr(n - 2 - u, tid)];
            l2[u] = ab[laddr(n - 2 - u, tid + TRS_NT)];
            qp[u] = ipiv[max(n - 2 - u, 0) + z];
            __builtin_amdgcn_sched_barrier(0);   // in order of use
        }
        for (int jb = n - 2; jb >= 0; jb -= QP) {
#pragma unroll
            for (int u = 0; u < QP; ++u) {
                const int j = jb - u;
                if (j < 0) break;
                const int lm = min(kl, n - 1 - j);
                T acc = {0, 0};
                if (tid < lm) acc = sz::cfma(acc, cj_if(l1[u], cj), x[j + 1 + tid]);
                if (tid + TRS_NT < lm)
                    acc = sz::cfma(acc, cj_if(l2[u], cj), x[j + 1 + tid + TRS_NT]);
                for (int r = tid + 2 * TRS_NT; r < lm; r += TRS_NT)
                    acc = sz::cfma(acc, cj_if(ab[laddr(j, r)], cj), x[j + 1 + r]);
                acc = wave_csum(acc);
                if (tid == 0) {
                    // component-wise (a struct copy here goes through
                    // scratch)
                    const T xo = x[j];
                    const R xjx = xo.x - acc.x, xjy = xo.y - acc.y;
                    int l = qp[u] - 1;
                    if (l < j || l >= n) l = j;
                    const R xlx = x[l].x, xly = x[l].y;
                    x[l].x = xjx;
                    x[l].y = xjy;
                    if (l != j) {
                        x[j].x = xlx;
                        x[j].y = xly;
                    }
                }
                l1[u] = ab[laddr(j - QP, tid)];
                l2[u] = ab[laddr(j - QP, tid + TRS_NT)];
                qp[u] = ipiv[max(j - QP, 0) + z];
                LDS_BARRIER();
            }
        }
    }
}

// trans: 0 = 'N', 1 = 'T', 2 = 'C'.  One 64-lane workgroup per system; the
// right-hand side lives in LDS, one barrier per elimination step.
// TR: transposed ('T'/'C').
template <typename R, bool TR>
__global__ __launch_bounds__(TRS_NT)
void k_gbtrs(int trans, int n, int kl, int ku, int nrhs,
             const cpx<R> *__restrict__ ab, int ldab, long long sab,
             const int *__restrict__ ipiv, long long sipiv,
             cpx<R> *__restrict__ b, int ldb, long long sb,
             const int *__restrict__ skip, int nsys)
{
    using T = cpx<R>;
    extern __shared__ __align__(16) unsigned char smem[];
    const int sys = blockIdx.x;
    if (sys >= nsys) return;
    if (skip && skip[sys] != 0) return;   // singular factor: leave b as is
    ab += (size_t)sys * (size_t)sab;
    ipiv += (size_t)sys * (size_t)sipiv;
    b += (size_t)sys * (size_t)sb;
    const int tid = threadIdx.x;
    const int kv = kl + ku;
    T *x = reinterpret_cast<T *>(smem);
    T *st = x + n;                                  // TRS_PRE*64 elements
    int *pv = reinterpret_cast<int *>(st + TRS_PRE * TRS_NT);
    const bool cj = (trans == 2);
    const int chL = kl > 0 ? min(64, (TRS_PRE * TRS_NT) / kl) : 1;
    const int chU = min(64, (TRS_PRE * TRS_NT) / (kv + 1));
    R rx[TRS_PRE], ry[TRS_PRE];   // next chunk of factor columns

    for (int s = 0; s < nrhs; ++s) {
        T *bs = b + (size_t)s * ldb;
        for (int i = tid; i < n; i += TRS_NT) x[i] = bs[i];
        LDS_BARRIER();
        if constexpr (!TR) {
            // L y = P b: multipliers are rows kv+1..kv+kl
            if (kl > 0 && n > 1) {
                chunk_load(rx, ry, ab, ldab, 0, min(chL, n - 1), kv + 1, kl);
                for (int j0 = 0; j0 < n - 1; j0 += chL) {
                    const int nc = min(chL, n - 1 - j0);
                    chunk_store(rx, ry, st, nc, kl);
                    for (int e = tid; e < nc; e += TRS_NT) pv[e] = ipiv[j0 + e];
                    if (j0 + chL < n - 1)
                        chunk_load(rx, ry, ab, ldab, j0 + chL, min(chL, n - 1 - j0 - chL),
                                kv + 1, kl);
                    LDS_BARRIER();
                    for (int jj = 0; jj < nc; ++jj) {
                        const int j = j0 + jj;
                        int l = pv[jj] - 1;
                        if (l < j || l >= n) l = j;
                        const T xl = x[l], xj = x[j];
                        const int lm = min(kl, n - 1 - j);
                        // after the interchange x[j] holds old x[l] and x[l]
                        // holds old x[j]; then x[j+1+r] -= m_r x[j]
                        for (int r = tid; r < lm; r += TRS_NT) {
                            const int i = j + 1 + r;
                            const T base = (i == l) ? xj : x[i];
                            x[i] = sz::cfnms(base, st[jj * kl + r], xl);
                        }
                        if (tid == 0) x[j] = xl;
                        LDS_BARRIER();
                    }
                }
            }
            // U x = y: column j of U is band rows kv-t (t = 0..kv)
            chunk_load(rx, ry, ab, ldab, n - min(chU, n), min(chU, n), 0, kv + 1);
            for (int j1 = n - 1; j1 >= 0; j1 -= chU) {
                const int nc = min(chU, j1 + 1);
                const int c0 = j1 - nc + 1;
                chunk_store(rx, ry, st, nc, kv + 1);
                if (c0 > 0) {
                    const int nn = min(chU, c0);
                    chunk_load(rx, ry, ab, ldab, c0 - nn, nn, 0, kv + 1);
                }
                LDS_BARRIER();
                for (int jj = nc - 1; jj >= 0; --jj) {
                    const int j = c0 + jj;
                    const T *u = st + jj * (kv + 1) + kv;   // u[-t] = U(j-t, j)
                    const T xo = x[j];
                    if (sz::cnonzero(xo)) {
                        const T xj = sz::cdiv(xo, u[0]);
                        const int tmax = min(kv, j);
                        for (int t = 1 + tid; t <= tmax; t += TRS_NT)
                            x[j - t] = sz::cfnms(x[j - t], u[-t], xj);
                        if (tid == 0) x[j] = xj;
                    }
                    LDS_BARRIER();
                }
            }
        } else {
            // U^T y = b, ascending and right-looking: once y_j is known,
            // lane t-1 subtracts U(j, j+t) y_j from the pending x[j+t], so
            // x[k] receives U(k-t, k) y_{k-t} for t = kv .. 1, the order of
            // the sequential LAPACK loop, and no step needs a reduction.
            // Lane 0 keeps x[j+1] (its own update) for the next division.
            {
                constexpr int QP = 4;                  // steps prefetched ahead
                const int t1 = tid + 1, t2 = tid + 1 + TRS_NT;
                auto uaddr = [&](int jj, int t) -> size_t {   // U(jj, jj+t)
                    const bool ok = t <= kv && jj + t < n;
                    return ok ? (size_t)(jj + t) * ldab + kv - t : 0;
                };
                T q1[QP], q2[QP], qd[QP];
                int z = 0;                             // (as in lt_sweep)
                asm volatile("" : "+v"(z));
#pragma unroll
                for (int u = 0; u < QP; ++u) {
                    q1[u] = ab[uaddr(u, t1)];
                    q2[u] = ab[uaddr(u, t2)];
                    qd[u] = ab[(size_t)min(u, n - 1) * ldab + kv + z];
                    __builtin_amdgcn_sched_barrier(0);   // in order of use
                }
                T xn = x[0];
                for (int jb = 0; jb < n; jb += QP) {
#pragma unroll
                    for (int u = 0; u < QP; ++u) {
                        const int j = jb + u;
                        if (j >= n) break;
                        T xj;
                        xj.x = readlane_r(xn.x, 0);
                        xj.y = readlane_r(xn.y, 0);
                        const T y = sz::cdiv(xj, cj_if(qd[u], cj));
                        if (tid == 0) x[j] = y;
                        if (t1 <= kv && j + t1 < n) {
                            const T v = sz::cfnms(x[j + t1], cj_if(q1[u], cj), y);
                            x[j + t1] = v;
                            if (tid == 0) xn = v;
                        }
                        if (t2 <= kv && j + t2 < n)
                            x[j + t2] = sz::cfnms(x[j + t2], cj_if(q2[u], cj), y);
                        for (int t = t2 + TRS_NT; t <= kv && j + t < n; t += TRS_NT)
                            x[j + t] = sz::cfnms(x[j + t], cj_if(ab[uaddr(j, t)], cj), y);
                        q1[u] = ab[uaddr(j + QP, t1)];
                        q2[u] = ab[uaddr(j + QP, t2)];
                        qd[u] = ab[(size_t)min(j + QP, n - 1) * ldab + kv + z];
                        LDS_BARRIER();
                        if (kv == 0 && tid == 0 && j + 1 < n) xn = x[j + 1];
                    }
                }
            }
            lt_sweep(n, kl, kv, ab, ldab, ipiv, cj, x, tid);
        }
        for (int i = tid; i < n; i += TRS_NT) bs[i] = x[i];
        LDS_BARRIER();
    }
}

// Orders LDS accesses of one wavefront (no s_barrier: a single wave).
#define WAVE_SYNC()                                                           \
    do {                                                                      \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                \
        __builtin_amdgcn_wave_barrier();                                      \
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");                \
    } while (0)

// ------------------------------------------------------- register solve
// The solves of k_gbtrs with the active part of the right hand side in
// registers, for the bands launch_gbtrs_reg admits: one wavefront per system,
// row i in lane i mod 64, NR registers deep.  A finished row's lane takes the
// row 64 NR further on from a prefetched register, so no value moves between
// lanes: a step broadcasts one element by readlane and every lane updates its
// own row, with the multiply-adds in the order of the LAPACK loops
// (bit-identical).
//   * SOLVE_N: L forward (multipliers of column j, interchanges by readlane and
//     writelane), then U backward (column j above the diagonal);
//   * SOLVE_T: U^T forward: lane = column, four rows of U (64 contiguous bytes
//     of the column) per load; then L^T backward, whose dot products are summed
//     as k_gbtrs sums them, by distance from the diagonal: there the window
//     itself moves by one lane a step;
//   * SOLVE_LT: the L^T half alone, after a factorization that solved U^T.
// The columns of the next PF steps are in flight: the barrier to the scheduler
// before each fetch keeps a load behind the last use of the registers it fills
// (else they are copied, and the copy waits for the load), and the first PF
// fetches in their order (else the first step of every PF waits for all).
// Bound by instruction issue of one wavefront (75 instructions a step; the
// division by U(j, j) has its reciprocal formed 64 at a time), for thousands of
// systems by issue of the SIMD; the factors' bytes take a third of the time.
// Measured, against x in LDS with a barrier a step: N of 576 systems n = 480,
// kl = ku = 34: 459 -> 294 us (455 MB); T of 600 systems n = 301, kl 17, ku 11,
// two right hand sides: 615 -> 253 us; L^T of 4560 systems n = 480, kl = 34:
// 483 -> 334 us; N in float, 300 systems n = 200, kl = ku = 24: 37 -> 19 us.
// What it loses: an element that is zero still costs N a step, where k_gbtrs left
// its column out (an all-zero right hand side, kl = 0, 1500 systems n = 480: 53
// -> 186 us).
template <typename R>
__device__ __forceinline__ R sel(bool c, R a, R b) { return c ? a : b; }

// v moved up by one lane, lane 0 taking first
template <typename R>
__device__ __forceinline__ R wave_shr(R v, R first)
{
    if constexpr (sizeof(R) == 8) {
        const long long b = __builtin_bit_cast(long long, v);
        const long long f = __builtin_bit_cast(long long, first);
        const int lo = __builtin_amdgcn_update_dpp((int)f, (int)b, 0x138, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp((int)(f >> 32), (int)(b >> 32), 0x138, 0xf,
                                                   0xf, false);
        return __builtin_bit_cast(R, (long long)(((unsigned long long)(unsigned)hi << 32)
                                                 | (unsigned)lo));
    } else {
        return __builtin_bit_cast(R, __builtin_amdgcn_update_dpp(
            __builtin_bit_cast(int, first), __builtin_bit_cast(int, v), 0x138, 0xf, 0xf,
            false));
    }
}

// a + b over the two rows of 16 lanes (16) or halves of the wave (32) that the
// gfx950 swaps exchange: [r0 + r1, r0 + r1, r2 + r3, r2 + r3] for 16
template <int W, typename R>
__device__ __forceinline__ R swap_add(R v)
{
    auto swap = [](unsigned a) __attribute__((always_inline)) {
        if constexpr (W == 16) return __builtin_amdgcn_permlane16_swap(a, a, false, false);
        else return __builtin_amdgcn_permlane32_swap(a, a, false, false);
    };
    if constexpr (sizeof(R) == 8) {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
        const auto lo = swap((unsigned)b), hi = swap((unsigned)(b >> 32));
        return __builtin_bit_cast(R, (unsigned long long)hi[0] << 32 | lo[0]) +
               __builtin_bit_cast(R, (unsigned long long)hi[1] << 32 | lo[1]);
    } else {
        const auto w = swap(__builtin_bit_cast(unsigned, v));
        return __builtin_bit_cast(R, (unsigned)w[0]) + __builtin_bit_cast(R, (unsigned)w[1]);
    }
}

// wave_csum's sums, re valid in lane 0 and im in lane 1: the first exchange
// sends one component and keeps the other, so the rest adds both at once.  An
// addend's order within a sum never matters, its grouping stays the butterfly's.
template <typename R>
__device__ __forceinline__ R wave_csum01(R re, R im, bool odd)
{
    R v = sel(odd, im, re) + dpp_r<0xB1>(sel(odd, re, im));   // l ^ 1
    v += dpp_r<0x4E>(v);                                      // l ^ 2
    v += dpp_r<0x104>(v);                                     // row_shl:4
    v += dpp_r<0x108>(v);                                     // row_shl:8
    return swap_add<32>(swap_add<16>(v));
}

// v's 32-bit words of lane l replaced by w's (both uniform)
template <typename R>
__device__ __forceinline__ R writelane_r(R v, R w, int l)
{
    if constexpr (sizeof(R) == 8) {
        const long long b = __builtin_bit_cast(long long, v);
        const long long f = __builtin_bit_cast(long long, w);
        const int lo = sz_writelane((int)f, l, (int)b);
        const int hi = sz_writelane((int)(f >> 32), l, (int)(b >> 32));
        return __builtin_bit_cast(R, (long long)(((unsigned long long)(unsigned)hi << 32)
                                                 | (unsigned)lo));
    } else {
        return __builtin_bit_cast(R, sz_writelane(
            __builtin_bit_cast(int, w), l, __builtin_bit_cast(int, v)));
    }
}

// Division by a diagonal, one a lane.  Smith's quotient is
// (x c1 + y c2, y c1 - x c2) / den with (c1, c2) = (1, ratio) or (ratio, 1).
// With rec = 1 / den rounded, q = n rec corrected twice by fma(n - q den, rec)
// is the rounded n / den (Markstein: the first correction leaves a neighbour
// of n / den, the second starts from an exact remainder), as long as nothing
// leaves the normal range: mid() keeps |n| and |den| far inside it, and any
// other value, zero included, takes the division itself.
template <typename R>
struct smith {
    R c1, c2, den, rec;
    unsigned long long mid;
};
template <typename R>
__device__ __forceinline__ bool mid(R a, R b)        // both of ordinary size
{
    constexpr int E = sizeof(R) == 8 ? 400 : 50;     // 2^-E <= |.| < 2^E
    constexpr int SH = sizeof(R) == 8 ? 21 : 24;     // exponent, sign shifted out
    constexpr unsigned BIAS = sizeof(R) == 8 ? 1023 : 127;
    auto key = [](R v) __attribute__((always_inline)) {
        unsigned h;
        if constexpr (sizeof(R) == 8)
            h = (unsigned)(__builtin_bit_cast(unsigned long long, v) >> 32);
        else
            h = __builtin_bit_cast(unsigned, v);
        return (h << 1) - ((BIAS - E) << SH);
    };
    return max(key(a), key(b)) < (2u * E << SH);
}
template <typename R>
__device__ __forceinline__ smith<R> smith_of(R zx, R zy)
{
    smith<R> d;
    const bool big = fabs(zx) >= fabs(zy);
    const R P = sel(big, zx, zy), Q = sel(big, zy, zx);
    const R ratio = Q / P;
    d.den = P + Q * ratio;
    d.rec = R(1) / d.den;
    d.c1 = sel(big, R(1), ratio);
    d.c2 = sel(big, ratio, R(1));
    d.mid = __ballot(mid(d.den, d.den));
    return d;
}

// x / z in lane jj (returned in q there) and its value v, uniform
template <typename R>
__device__ __forceinline__ void smith_div(const smith<R> &d, int jj, R x, R y, R &qx, R &qy,
                                          cpx<R> &v, bool &nz)
{
    const R n2 = x * d.c1 + y * d.c2, n3 = y * d.c1 - x * d.c2;
    R a = n2 * d.rec, b = n3 * d.rec;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        a = __builtin_fma(__builtin_fma(-d.den, a, n2), d.rec, a);
        b = __builtin_fma(__builtin_fma(-d.den, b, n3), d.rec, b);
    }
    nz = true;
    if (!((__ballot(mid(n2, n3)) & d.mid) >> jj & 1)) {
        nz = __ballot(sz::cnonzero(cpx<R>{x, y})) >> jj & 1;
        a = n2 / d.den;
        b = n3 / d.den;
    }
    qx = a;
    qy = b;
    v.x = readlane_r(a, jj);
    v.y = readlane_r(b, jj);
}

enum { SOLVE_N, SOLVE_T, SOLVE_LT };
template <typename R, int MODE, int NR>
__global__ __launch_bounds__(64)
void k_gbtrs_reg(int trans, int n, int kl, int ku, int nrhs, const cpx<R> *__restrict__ ab,
                 int ldab, long long sab, const int *__restrict__ ipiv, long long sipiv,
                 cpx<R> *__restrict__ b, int ldb, long long sb,
                 const int *__restrict__ skip, int nsys)
{
    using T = cpx<R>;
    constexpr int PF = 8;                    // columns requested ahead
    extern __shared__ __align__(16) unsigned char smem[];
    T *xs = reinterpret_cast<T *>(smem);     // n
    const int sys = blockIdx.x;
    if (sys >= nsys) return;
    if (skip && skip[sys] != 0) return;      // singular factor: leave b as is
    ab += (size_t)sys * (size_t)sab;
    ipiv += (size_t)sys * (size_t)sipiv;
    b += (size_t)sys * (size_t)sb;
    const int lane = threadIdx.x, kv = kl + ku;
    const bool cj = trans == 2;
    // xs[i], zero outside 0 .. n-1
    auto row = [&](int i, R &x, R &y) __attribute__((always_inline)) {
        const bool ok = i >= 0 && i < n;
        const R *v = reinterpret_cast<const R *>(xs + (ok ? i : 0));
        x = ok ? v[0] : R(0);
        y = ok ? v[1] : R(0);
    };
    // column j, or the nearest there is (its diagonal is loaded and unused)
    auto col = [&](int j) __attribute__((always_inline)) {
        return ab + (size_t)max(0, min(j, n - 1)) * ldab;
    };
    auto at = [&](const T *c, int i) __attribute__((always_inline)) {
        return sz::gload(reinterpret_cast<const T *>(reinterpret_cast<const char *>(c) +
                                                     (unsigned)i * (unsigned)sizeof(T)));
    };
    for (int s = 0; s < nrhs; ++s) {
        T *bs = b + (size_t)s * ldb;
        for (int i = lane; i < n; i += 64) xs[i] = sz::gload(bs + i);
        LDS_BARRIER();
        if constexpr (MODE == SOLVE_N) {
            // ---- L y = P b
            if (kl > 0) {
                R x, y, nx, ny, fx = R(0), fy = R(0), qx[PF], qy[PF];
                row(lane, x, y);
                row(64 + lane, nx, ny);
                // the interchange of step i (LAPACK's last row has none)
                auto pivot = [&](int i) __attribute__((always_inline)) {
                    const int c = min(i, n - 1), p = ipiv[c] - 1;
                    return p < c || p >= n || c == n - 1 ? c : p;
                };
                int pv = pivot(lane);
                // L(j + d, j), d = distance of this lane's row (0: none)
                auto fetch = [&](int j, R &vx, R &vy) __attribute__((always_inline)) {
                    const int d = (lane - j) & 63;
                    const T v = at(col(j), kv + (d <= min(kl, n - 1 - j) ? d : 0));
                    vx = v.x;
                    vy = v.y;
                };
                unroll<PF>([&](auto u_) __attribute__((always_inline)) {
                    fetch(decltype(u_)::value, qx[decltype(u_)::value], qy[decltype(u_)::value]);
                    __builtin_amdgcn_sched_barrier(0);
                });
                for (int j0 = 0; j0 < n; j0 += 64) {
                    for (int jj0 = 0; jj0 < 64 && j0 + jj0 < n; jj0 += PF) {
                        unroll<PF>([&](auto u_) __attribute__((always_inline)) {
                            constexpr int u = decltype(u_)::value;
                            const int jj = jj0 + u, j = j0 + jj;
                            const int pl = __builtin_amdgcn_readlane(pv, jj) & 63;
                            const R ax = readlane_r(x, pl), ay = readlane_r(y, pl);
                            // row p takes row j's value
                            const R jx = readlane_r(x, jj), jy = readlane_r(y, jj);
                            x = writelane_r(x, jx, pl);
                            y = writelane_r(y, jy, pl);
                            const int d = (lane - jj) & 63;
                            const bool in = d >= 1 && d <= min(kl, n - 1 - j);
                            const T v = sz::cfnms(T{x, y}, T{qx[u], qy[u]}, T{ax, ay});
                            x = sel(in, v.x, x);
                            y = sel(in, v.y, y);
                            fx = writelane_r(fx, ax, jj);
                            fy = writelane_r(fy, ay, jj);
                            x = sel(d == 0, nx, x);
                            y = sel(d == 0, ny, y);
                            __builtin_amdgcn_sched_barrier(0);
                            fetch(j + PF, qx[u], qy[u]);
                        });
                    }
                    if (j0 + lane < n) xs[j0 + lane] = T{fx, fy};
                    row(j0 + 128 + lane, nx, ny);
                    pv = pivot(j0 + 64 + lane);
                }
                LDS_BARRIER();
            }
            // ---- U x = y, descending; jt: the first column of a block of 64
            {
                R x[NR], y[NR], nx, ny, fx = R(0), fy = R(0), qx[PF][NR], qy[PF][NR];
                const int jl = (n - 1) & 63;
                const int back = (jl - lane) & 63;     // this lane: row jt - back
                unroll<NR>([&](auto m_) __attribute__((always_inline)) {
                    row(n - 1 - back - 64 * decltype(m_)::value, x[decltype(m_)::value],
                        y[decltype(m_)::value]);
                });
                row(n - 1 - back - 64 * NR, nx, ny);
                // U(j - t, j), t = distance of this lane's rows (t = 0: diagonal)
                auto fetch = [&](int j, R (&vx)[NR], R (&vy)[NR]) __attribute__((always_inline)) {
                    const int t0 = (j - lane) & 63;
                    const T *cp = col(j);
                    unroll<NR>([&](auto m_) __attribute__((always_inline)) {
                        constexpr int m = decltype(m_)::value;
                        const int t = t0 + 64 * m;
                        const T v = at(cp, kv - (t <= min(kv, j) ? t : 0));
                        vx[m] = v.x;
                        vy[m] = v.y;
                    });
                };
                unroll<PF>([&](auto u_) __attribute__((always_inline)) {
                    fetch(n - 1 - decltype(u_)::value, qx[decltype(u_)::value],
                          qy[decltype(u_)::value]);
                });
                for (int jt = n - 1; jt >= 0; jt -= 64) {
                    const int dc = max(jt - back, 0);
                    const T z = sz::gload(ab + (size_t)dc * ldab + kv);
                    const smith<R> dg = smith_of(z.x, z.y);
                    for (int k0 = 0; k0 < 64 && k0 <= jt; k0 += PF) {
                        unroll<PF>([&](auto u_) __attribute__((always_inline)) {
                            constexpr int u = decltype(u_)::value;
                            const int j = jt - k0 - u, jj = j & 63;
                            R wx, wy;
                            T v;
                            bool nz;
                            smith_div(dg, jj, x[0], y[0], wx, wy, v, nz);
                            const int t0 = (jj - lane) & 63, tl = nz ? min(kv, j) : 0;
                            unroll<NR>([&](auto m_) __attribute__((always_inline)) {
                                constexpr int m = decltype(m_)::value;
                                const int t = t0 + 64 * m;
                                const T w = sz::cfnms(T{x[m], y[m]}, T{qx[u][m], qy[u][m]}, v);
                                const bool in = t >= 1 && t <= tl;
                                x[m] = sel(in, w.x, x[m]);
                                y[m] = sel(in, w.y, y[m]);
                            });
                            const bool done = t0 == 0;   // (0 is left as it is)
                            fx = sel(done, nz ? wx : x[0], fx);
                            fy = sel(done, nz ? wy : y[0], fy);
                            unroll<NR>([&](auto m_) __attribute__((always_inline)) {
                                constexpr int m = decltype(m_)::value;
                                R ox = nx, oy = ny;
                                if constexpr (m + 1 < NR) {
                                    ox = x[m + 1];
                                    oy = y[m + 1];
                                }
                                x[m] = sel(done, ox, x[m]);
                                y[m] = sel(done, oy, y[m]);
                            });
                            __builtin_amdgcn_sched_barrier(0);
                            fetch(j - PF, qx[u], qy[u]);
                        });
                    }
                    if (jt - back >= 0) xs[jt - back] = T{fx, fy};
                    row(jt - 64 - back - 64 * NR, nx, ny);
                }
            }
            LDS_BARRIER();
        }
        if constexpr (MODE == SOLVE_T) {
            // ---- U^T y = b, ascending, four rows a block
            constexpr int NB = 4, RB = NR == 1 ? 4 : 2;      // RB blocks ahead
            R x[NR], y[NR], nx, ny, fx = R(0), fy = R(0);
            R ex[RB][NB][NR], ey[RB][NB][NR];
            const long long last = (long long)n * ldab - 1;
            unroll<NR>([&](auto m_) __attribute__((always_inline)) {
                row(lane + 64 * decltype(m_)::value, x[decltype(m_)::value],
                    y[decltype(m_)::value]);
            });
            row(lane + 64 * NR, nx, ny);
            // U(jb .. jb+3, c) of this lane's columns c = jb + d + 64 m
            auto fetch = [&](int jb, R (&vx)[NB][NR], R (&vy)[NB][NR]) __attribute__((always_inline)) {
                const int d = (lane - jb) & 63;
                unroll<NR>([&](auto m_) __attribute__((always_inline)) {
                    constexpr int m = decltype(m_)::value;
                    const int c = jb + d + 64 * m;
                    const long long at = (long long)c * ldab + kv - d - 64 * m;
                    const bool ok = c < n && kv >= d + 64 * m - (NB - 1);
                    unroll<NB>([&](auto i_) __attribute__((always_inline)) {
                        constexpr int i = decltype(i_)::value;
                        const long long k = ok ? at + i : 0;
                        const T v = sz::gload(ab + (k < 0 ? 0 : k > last ? last : k));
                        vx[i][m] = v.x;
                        vy[i][m] = v.y;
                    });
                });
            };
            unroll<RB>([&](auto h_) __attribute__((always_inline)) {
                constexpr int h = decltype(h_)::value;
                fetch(NB * h, ex[h], ey[h]);
            });
            for (int j0 = 0; j0 < n; j0 += 64) {
                const int dc = min(j0 + lane, n - 1);
                const T z = sz::gload(ab + (size_t)dc * ldab + kv);
                const smith<R> dg = smith_of(z.x, cj ? -z.y : z.y);
                for (int jj0 = 0; jj0 < 64 && j0 + jj0 < n; jj0 += RB * NB) {
                    unroll<RB>([&](auto h_) __attribute__((always_inline)) {
                        constexpr int h = decltype(h_)::value;
                        const int jb = j0 + jj0 + NB * h;
                        const int d = (lane - jb) & 63;
                        unroll<NB>([&](auto u_) __attribute__((always_inline)) {
                            constexpr int u = decltype(u_)::value;
                            const int jj = (jb + u) & 63;
                            R wx, wy;
                            T v;
                            bool nz;
                            smith_div(dg, jj, x[0], y[0], wx, wy, v, nz);
                            fx = sel(d == u, wx, fx);
                            fy = sel(d == u, wy, fy);
                            unroll<NR>([&](auto m_) __attribute__((always_inline)) {
                                constexpr int m = decltype(m_)::value;
                                const int t = d + 64 * m - u;
                                const T w = sz::cfnms(T{x[m], y[m]},
                                                      cj_if(T{ex[h][u][m], ey[h][u][m]}, cj),
                                                      v);
                                const bool in = t >= 1 && t <= kv;
                                x[m] = sel(in, w.x, x[m]);
                                y[m] = sel(in, w.y, y[m]);
                            });
                        });
                        // finished columns' lanes move on by 64
                        unroll<NR>([&](auto m_) __attribute__((always_inline)) {
                            constexpr int m = decltype(m_)::value;
                            R ox = nx, oy = ny;
                            if constexpr (m + 1 < NR) {
                                ox = x[m + 1];
                                oy = y[m + 1];
                            }
                            x[m] = sel(d < NB, ox, x[m]);
                            y[m] = sel(d < NB, oy, y[m]);
                        });
                        __builtin_amdgcn_sched_barrier(0);
                        fetch(jb + RB * NB, ex[h], ey[h]);
                    });
                }
                if (j0 + lane < n) xs[j0 + lane] = T{fx, fy};
                row(j0 + 64 + 64 * NR + lane, nx, ny);
            }
            LDS_BARRIER();
        }
        if constexpr (MODE != SOLVE_N) {
            // ---- L^T x = y and the interchanges, descending.  Lane r holds row
            // j + 1 + r and forms that row's term of the dot product with
            // column j's multipliers; the window then moves up by one lane.
            if (kl > 0 && n > 1) {
                R x, y, qx[PF], qy[PF];
                const int back = (n - 2 - lane) & 63;
                const bool odd = (lane & 1) != 0;
                row(n - 1 + lane, x, y);
                // the interchange of step i as the window's lane, -1 for none
                auto pivot = [&](int i) __attribute__((always_inline)) {
                    const int c = max(i, 0), p = ipiv[c] - 1;
                    return p <= c || p >= n || i < 0 ? -1 : p - c - 1;
                };
                int pv = pivot(n - 2 - back), npv = pivot(n - 2 - 64 - back);
                auto fetch = [&](int j, R &vx, R &vy) __attribute__((always_inline)) {
                    const T v = at(col(j), kv + (lane < min(kl, n - 1 - j) ? 1 + lane : 0));
                    vx = v.x;
                    vy = v.y;
                };
                unroll<PF>([&](auto u_) __attribute__((always_inline)) {
                    constexpr int u = decltype(u_)::value;
                    fetch(n - 2 - u, qx[u], qy[u]);
                    __builtin_amdgcn_sched_barrier(0);
                });
                int j = n - 2;
                for (int jt = n - 2; jt >= 0; jt -= 64) {
                    for (int k0 = 0; k0 < 64 && k0 <= jt; k0 += PF) {
                        // the lanes that PF steps move out of the window (kl <= 56:
                        // no interchange reaches them any more)
                        const int i = j + 1 + lane;
                        if (lane >= 64 - PF && i < n) xs[i] = T{x, y};
                        R ox[PF], oy[PF];
                        unroll<PF>([&](auto u_) __attribute__((always_inline)) {
                            constexpr int u = decltype(u_)::value;
                            const R *v = reinterpret_cast<const R *>(xs + max(j - u, 0));
                            ox[u] = v[0];
                            oy[u] = v[1];
                        });
                        unroll<PF>([&](auto u_) __attribute__((always_inline)) {
                            constexpr int u = decltype(u_)::value;
                            const bool in = lane < min(kl, n - 1 - j);
                            const T m = sz::cfma(T{R(0), R(0)}, cj_if(T{qx[u], qy[u]}, cj),
                                                 T{x, y});
                            const R acc = wave_csum01(sel(in, m.x, R(0)), sel(in, m.y, R(0)),
                                                      odd);
                            R vx = ox[u] - acc, vy = oy[u] - dpp_r<0x55>(acc);  // lane 0
                            const int p = __builtin_amdgcn_readlane(pv, j & 63);
                            if (p >= 0) {
                                const R px = readlane_r(x, p), py = readlane_r(y, p);
                                x = writelane_r(x, readlane_r(vx, 0), p);
                                y = writelane_r(y, readlane_r(vy, 0), p);
                                vx = px;
                                vy = py;
                            }
                            x = wave_shr(x, vx);
                            y = wave_shr(y, vy);
                            __builtin_amdgcn_sched_barrier(0);
                            fetch(j - PF, qx[u], qy[u]);
                            --j;
                        });
                    }
                    pv = npv;
                    npv = pivot(jt - 128 - back);
                }
                LDS_BARRIER();
                const int i = j + 1 + lane;
                if (i >= 0 && i < n) xs[i] = T{x, y};
            }
            LDS_BARRIER();
        }
        for (int i = lane; i < n; i += 64) sz::gstore(bs + i, xs[i]);
        LDS_BARRIER();
    }
}

// ------------------------------------------------------------ t16 solve
// A^T x = b (A^H x = b) from the factors, sixteen lanes per system and four
// systems per wavefront, for the band shapes of the channel operators.
//   * U^T y = b, ascending, in dot-product form: y_j = (b_j - sum_{t=1..kv}
//     U(j-t, j) y_{j-t}) / U(j, j).  Column j of U is one contiguous run of
//     the band storage, so every load reads whole cache lines.  Lane l of a
//     system owns the rows i = l (mod 16): during group g (columns 16g ..
//     16g+15) its register slot k holds y_{16(g-k)+l} (slot 0 fills during
//     the group), and slot k of column j is the run of band rows
//     kv - (j mod 16) - 16k + l, one load per slot.  No y moves between
//     lanes: a step shares only the 16-lane sum (four DPP stages).  Terms
//     outside the band are never loaded (zero), and the lane owning row j
//     finds the diagonal U(j, j) in its own slot 0, so it forms
//     y_j = (b_j - sum) / U(j, j) from its own registers.
//   * L^T x = y and the interchanges, descending, through LDS: lane l forms
//     the terms r = l (mod 16) of the dot product with the multipliers of
//     column j (one contiguous run), the 16-lane sum completes it and lane 0
//     of the system subtracts and swaps, as ZGBTRS does column by column.
// Factor columns are requested T16_PF steps before their use.  UT = false
// solves only the L^T half (U^T was solved during the factorization).  The
// sums run in a different order than ZGBTRS's; the solve is used where the
// result is refined or checked to a tolerance, not compared bit for bit.
constexpr int T16_PF = 8;

// Sum over the 16 lanes of a DPP row, delivered to all 16 (the first four
// stages of wave_sum_asc).
template <typename R>
__device__ __forceinline__ R rowsum16(R v)
{
    v += dpp_r<0xB1>(v);                    // quad_perm [1,0,3,2]
    v += dpp_r<0x4E>(v);                    // quad_perm [2,3,0,1]
    v += dpp_r<0x141>(v);                   // row_half_mirror
    v += dpp_r<0x140>(v);                   // row_mirror
    return v;
}

// Sum over LPS = 16 or 32 lanes delivered to all of them: the DPP row sum,
// then (32) the other row's sum by an LDS-free swizzle (xor 16 within 32).
template <int LPS, typename R>
__device__ __forceinline__ R lanesum(R v)
{
    v = rowsum16(v);
    if constexpr (LPS == 32) {
        static_assert(sizeof(R) == 4, "32-bit swizzle");
        const int o = __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F);
        v += __builtin_bit_cast(R, o);
    }
    return v;
}

// 1/z as conj(z)/|z|^2 after rescaling z by a power of two, so |z|^2
// neither overflows nor underflows; float uses the hardware reciprocal.
template <typename R>
__device__ __forceinline__ cpx<R> rcp_scaled(cpx<R> z)
{
    int e;
    (void)frexp(fmax(fabs(z.x), fabs(z.y)), &e);
    const R zx = ldexp(z.x, -e), zy = ldexp(z.y, -e);
    const R d = fma(zx, zx, zy * zy);
    R r;
    if constexpr (sizeof(R) == 4) r = __builtin_amdgcn_rcpf(d);
    else r = R(1) / d;
    return {ldexp(zx * r, -e), ldexp(-zy * r, -e)};
}

template <typename R, int KL, int KV, bool UT, bool CJ, int LPS = 16>
__global__ __launch_bounds__(64)
void k_gbtrs_t16(int n, const cpx<R> *__restrict__ ab, int ldab, long long sab,
                 const int *__restrict__ ipiv, long long sipiv,
                 cpx<R> *__restrict__ b, long long sb,
                 const int *__restrict__ skip, int nsys, int ldx,
                 const sz::gsys *__restrict__ gs)
{
    using T = cpx<R>;
    static_assert(LPS == 16 || LPS == 32, "lanes per system");
    constexpr int SPW = 64 / LPS;            // systems per wavefront
    constexpr int NS = (KV + LPS - 1) / LPS + 1;   // U^T register slots
    constexpr int NM = (KL + LPS - 1) / LPS;       // L^T terms per lane
    constexpr int PF = T16_PF;
    static_assert(LPS % PF == 0, "queue entries must repeat within a group");
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x, l = lane & (LPS - 1), grp = lane / LPS;
    const int sys = blockIdx.x * SPW + grp;
    // Every lane loads from the storage of its system (of system 0 past the
    // end of the batch), unconditionally and at clamped addresses, so the
    // loads in flight are the same on every path and the queue drains only
    // as far as each use needs; what a lane must not use is masked where
    // it is used.  nl: columns of the storage read (n >= 2); ns: columns
    // solved and stored (0 past the end and for skipped systems).
    const int s0 = sys < nsys ? sys : 0;
    const T *a;
    const int *pv;
    T *bs;
    int nl;
    // column strides of U and of the multipliers, and where the latter start
    int ldu = ldab, ldl = ldab;
    long long loff = KV + 1;
    if (gs) {
        const sz::gsys g = gs[s0];
        nl = g.n;
        a = reinterpret_cast<const T *>(g.ab);
        pv = reinterpret_cast<const int *>(g.ipiv);
        bs = reinterpret_cast<T *>(g.b);
        if (g.layout == 1) {
            ldu = KV + 1;
            ldl = KL;
            loff = (long long)nl * (KV + 1);
        }
    } else {
        nl = n;
        a = ab + (size_t)s0 * (size_t)sab;
        pv = ipiv + (size_t)s0 * (size_t)sipiv;
        bs = b + (size_t)s0 * (size_t)sb;
    }
    const int ns = (sys < nsys && !(skip && skip[sys] != 0)) ? nl : 0;
    const int nw = LPS == 16
        ? max(max(__builtin_amdgcn_readlane(ns, 0), __builtin_amdgcn_readlane(ns, 16)),
              max(__builtin_amdgcn_readlane(ns, 32), __builtin_amdgcn_readlane(ns, 48)))
        : max(__builtin_amdgcn_readlane(ns, 0), __builtin_amdgcn_readlane(ns, 32));
    if (nw == 0) return;
    T *x = reinterpret_cast<T *>(smem) + (size_t)grp * ldx;

    if constexpr (UT) {
        R yx[NS], yy[NS], qx[PF][NS], qy[PF][NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) yx[k] = yy[k] = R(0);
        // column c (wave-uniform, c mod LPS = u16) into one queue entry.
        // Lane l of slot k reads row KV - u16 - LPS k + l; lanes whose row
        // falls outside the U rows 0..KV of the column (masked at use in
        // any case) read the nearest U row instead, so the loads touch the
        // column's U lines only and stay inside the storage for every c.
        auto fetch = [&](int c, int u16, R (&fx)[NS], R (&fy)[NS]) {
            const T *col = a + (size_t)min(c, nl - 1) * ldu;
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const int r0 = KV - u16 - LPS * k;
                int row = r0 + l;
                if (r0 < 0) row = max(row, 0);
                if (r0 + LPS - 1 > KV) row = min(row, KV);
                const T v = sz::gload(col + row);
                fx[k] = v.x;
                fy[k] = v.y;
            }
        };
        T bn = sz::gload(bs + min(l, nl - 1));
        // the prologue issues the queue in order of use (no reordering
        // across entries), as every later step refills it
#pragma unroll
        for (int c = 0; c < PF; ++c) {
            fetch(c, c, qx[c], qy[c]);
            __builtin_amdgcn_sched_barrier(0);
        }
        // one group of LPS columns; HEAD: the first groups, where slot
        // k > g holds rows above row 0
        auto group = [&](int g, auto head) {
            constexpr bool HEAD = decltype(head)::value;
            const T bc = bn;
            bn = sz::gload(bs + min(LPS * g + LPS + l, nl - 1));
#pragma unroll
            for (int u = 0; u < LPS; ++u) {
                const int q = u % PF;
                // slots NS-1..1 in two independent chains, then slot 0 (the
                // newest y, the only term that waits on the last step)
                R ax2[2] = {R(0), R(0)}, ay2[2] = {R(0), R(0)};
                R sx = R(0), sy = R(0);
#pragma unroll
                for (int k = NS - 1; k >= 0; --k) {
                    // lanes with 1 <= u + LPS k - l <= KV hold a term
                    const int lo = u + LPS * k - KV, hi = u + LPS * k - 1;
                    if (hi < 0) continue;
                    R ax = qx[q][k], ay = CJ ? -qy[q][k] : qy[q][k];
                    if (lo > 0 || hi < LPS - 1 || (HEAD && k > 0)) {
                        const bool ok = l >= lo && l <= hi && (!HEAD || k == 0 || g >= k);
                        ax = ok ? ax : R(0);
                        ay = ok ? ay : R(0);
                    }
                    if (k > 0) {
                        ax2[k & 1] = fma(ax, yx[k], ax2[k & 1]);
                        ax2[k & 1] = fma(-ay, yy[k], ax2[k & 1]);
                        ay2[k & 1] = fma(ax, yy[k], ay2[k & 1]);
                        ay2[k & 1] = fma(ay, yx[k], ay2[k & 1]);
                    } else {
                        sx = ax2[0] + ax2[1];
                        sy = ay2[0] + ay2[1];
                        sx = fma(ax, yx[0], sx);
                        sx = fma(-ay, yy[0], sx);
                        sy = fma(ax, yy[0], sy);
                        sy = fma(ay, yx[0], sy);
                    }
                }
                if (u == 0) {                      // slot 0 holds no term yet
                    sx = ax2[0] + ax2[1];
                    sy = ay2[0] + ay2[1];
                }
                sx = lanesum<LPS>(sx);
                sy = lanesum<LPS>(sy);
                // lane u's slot 0 holds the diagonal U(j, j)
                const T dg = {qx[q][0], CJ ? -qy[q][0] : qy[q][0]};
                const T r = sz::cmul(T{bc.x - sx, bc.y - sy}, rcp_scaled(dg));
                if (l == u) {
                    yx[0] = r.x;
                    yy[0] = r.y;
                }
                fetch(LPS * g + u + PF, (u + PF) & (LPS - 1), qx[q], qy[q]);
            }
            if (LPS * g + l < ns) {
                x[LPS * g + l].x = yx[0];
                x[LPS * g + l].y = yy[0];
            }
#pragma unroll
            for (int k = NS - 1; k > 0; --k) {
                yx[k] = yx[k - 1];
                yy[k] = yy[k - 1];
            }
            yx[0] = yy[0] = R(0);
        };
        // two loops rather than a branch per group, so the queue registers
        // carry from group to group without copies
        const int ng = (nw + LPS - 1) / LPS, nh = min(ng, NS - 1);
        int g = 0;
        for (; g < nh; ++g) group(g, std::true_type{});
        for (; g < ng; ++g) group(g, std::false_type{});
        // the queue's last entries (columns past the end) are not used:
        // retire them here, so the L^T queue starts from an empty counter
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    } else {
        for (int i = l; i < ns; i += LPS) x[i] = sz::gload(bs + i);
    }
    WAVE_SYNC();

    if constexpr (KL > 0) {
        R lx[PF][NM], ly[PF][NM];
        int lp[PF];
        // step t: column j = ns - 2 - t, terms r < min(KL, t + 1); a lane
        // reads multiplier rows r = l + LPS m, the last run clamped to the
        // column, and the pivot of row j
        auto lfetch = [&](int t, R (&fx)[NM], R (&fy)[NM], int &p) {
            const int jl = max(nl - 2 - t, 0);
            const T *col = a + loff + (size_t)jl * ldl;
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const T v = sz::gload(col + min(l + LPS * m, KL - 1));
                fx[m] = v.x;
                fy[m] = v.y;
            }
            p = *sz::gmem(pv + jl);
        };
#pragma unroll
        for (int t = 0; t < PF; ++t) {
            lfetch(t, lx[t], ly[t], lp[t]);
            __builtin_amdgcn_sched_barrier(0);
        }
        // whole groups of 16 steps; steps past a system's last column
        // (j < 0) read and write nothing of it
        for (int t0 = 0; t0 < nw - 1; t0 += 16) {
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const int t = t0 + u;
                const int q = u % PF;
                const int j = ns - 2 - t;
                const int lm = min(KL, t + 1);
                R sx = R(0), sy = R(0);
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    const int r = l + LPS * m;
                    const bool ok = j >= 0 && r < lm;
                    const T xv = x[ok ? j + 1 + r : 0];
                    const R vx = ok ? xv.x : R(0), vy = ok ? xv.y : R(0);
                    const R ax = ok ? lx[q][m] : R(0);
                    const R ay = ok ? (CJ ? -ly[q][m] : ly[q][m]) : R(0);
                    sx = fma(ax, vx, sx);
                    sx = fma(-ay, vy, sx);
                    sy = fma(ax, vy, sy);
                    sy = fma(ay, vx, sy);
                }
                sx = lanesum<LPS>(sx);
                sy = lanesum<LPS>(sy);
                if (l == 0 && j >= 0) {
                    int p = lp[q] - 1;
                    if (p < j || p >= ns) p = j;
                    const R vx = x[j].x - sx, vy = x[j].y - sy;
                    const R px = x[p].x, py = x[p].y;
                    x[p].x = vx;
                    x[p].y = vy;
                    if (p != j) {
                        x[j].x = px;
                        x[j].y = py;
                    }
                }
                lfetch(t + PF, lx[q], ly[q], lp[q]);
                WAVE_SYNC();
            }
        }
    }
    WAVE_SYNC();
    for (int i = l; i < ns; i += LPS) sz::gstore(bs + i, x[i]);
}

// --------------------------------------------------------------- panel
// The factorization of the channel band shapes: one wavefront per system, no
// barriers, four columns at a time.  Lane l holds window column jb + d,
// d = (l - jb) mod 64, as PR = kl + 4 row slots in registers (slot s = row
// jb + s); columns jb+64 .. jb+kl+ku+3 (kl+ku >= 64) live in an LDS tail.  A
// block of four columns:
//   1. The panel columns go through LDS into row layout: slot 16m + i in
//      register m of the i-th lane of every 16-lane row, so each of the four
//      DPP rows holds the whole column.  Pivot search (maximum of the high
//      words by DPP, the low words on a tie only), interchange, multipliers
//      and the panel's own updates run there without leaving the row.  The
//      reciprocal's two quotients and the two of U^T's y are one division, a
//      numerator for each lane of a quad.
//   2. Every lane then applies the four interchanges and updates to its
//      column.  The multiplier of a slot is a row_newbcast operand of the
//      fused multiply-add itself: no readlane and no LDS read per multiplier
//      (two readlanes cost as much as a multiply-add: 13.8 against 6.0 cycles
//      for the pair, measured).
//   3. U rows leave and the next rows enter as 64 contiguous bytes per column,
//      the rows straight to LDS early in the block so that no wait for them
//      falls on the stores; the slots are renamed by four.  (One element at a
//      time moved 15.9 GB per 4560 systems fused, now 9.4 of 6.1 needed.  The
//      writes are what is needed, 3.8; 5.7 are read for 2.5: a miss brings a
//      128-byte line, whose other half is asked for four columns later, when it
//      has mostly left the L2.)
// Every updated element sees the fnms sequence of the unblocked loop.
//
// What bounds it: instruction issue and the pivot chain.  A column step of the
// fused kernel on the channel's operator is 440 vector instructions, 103 scalar
// and 35 of LDS (counters); 136 of them are the multiply-adds of step 2, which
// alone would take a quarter of the time: 13.4 TF/s of the 72.6 a large product
// reaches.  At two waves per SIMD (the window takes 152 of a lane's registers)
// the pivot chain of one wave runs beside the updates of the other and the
// vector unit is busy 70% of the time; of 4560 systems 464 are left for a third
// round of single waves.  N = 480, kl = ku = 34, diagonally dominant, alone and
// fused with U^T: 4560 systems 2.84 and 3.07 ms (an unblocked loop with readlane
// multipliers: 5.15 and 5.40), 2048 1.16 and 1.24, 1152 0.97 (1.50) and 1.10,
// one 0.66 and 0.75 (1.21); complex float 2.47 for 4560 (5.37).
//
// UT = true also solves U^T y = b on the way (the first half of ZGBTRS 'T'):
// lane l keeps the pending b of its column, y_j = b_j / U(j,j) is formed with
// the multipliers of column j and every lane with a column j+d, 1 <= d <=
// kl+ku, subtracts U(j, j+d) y_j -- x_k receives its terms for ascending
// rows, the sequential order of the LAPACK loop.  y overwrites b.
constexpr int PN_NB = 4;

// Waves per SIMD.  The window takes 152 (34 sub-diagonals) or 112 (24) of a
// lane's registers in double precision, so three waves fit only the narrower
// shape without U^T (fused they spill: 2.89 ms per 4560 systems of N = 365
// against 1.79).  Single precision would fit four, but runs faster with two
// (12,000 systems of N = 960: 11.7 ms against 13.1 with three and 13.5 with
// four; 4560 of N = 480: 2.49, 2.63, 2.72): a visit takes 32 bytes of a
// column's cache line, and more systems at once push the lines out of the L2
// between visits.
constexpr int panel_waves(size_t real, int wr, bool ut)
{
    return real == 8 && wr <= 25 && !ut ? 3 : 2;
}

// v of lane S of each 16-lane row, in every lane of that row
template <int S, typename R>
__device__ __forceinline__ R row_bcast(R v)
{
    if constexpr (sizeof(R) == 8)
        return sz_update_dpp(0.0, v, 0x150 + S, 0xF, 0xF, true);
    else
        return __builtin_bit_cast(
            R, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + S, 0xF,
                                           0xF, true));
}

// One element per lane from p (64 lanes) straight to LDS at dst, without
// passing through registers: complex doubles as they are, complex floats as
// a run of the real parts and a run of the imaginary ones (a transfer moves
// 4 or 16 bytes a lane).  take_lds reads a lane's own element back.
template <typename R>
__device__ __forceinline__ void load_lds(const cpx<R> *p, cpx<R> *dst)
{
    using G = const __attribute__((address_space(1))) unsigned;
    using L = __attribute__((address_space(3))) unsigned;
    if constexpr (sizeof(R) == 8) {
        __builtin_amdgcn_global_load_lds((G *)(p), (L *)(dst), 16, 0, 0);
    } else {
        __builtin_amdgcn_global_load_lds((G *)(p), (L *)(dst), 4, 0, 0);
        __builtin_amdgcn_global_load_lds((G *)(&p->y), (L *)(dst + 32), 4, 0, 0);
    }
}

template <typename R>
__device__ __forceinline__ void take_lds(const cpx<R> *src, int lane, R &x, R &y)
{
    const R *v = reinterpret_cast<const R *>(src);
    x = v[sizeof(R) == 8 ? 2 * lane : lane];
    y = v[sizeof(R) == 8 ? 2 * lane + 1 : 64 + lane];
}

// c ? a : b by value (a conditional between array elements is a choice of
// addresses, which can keep the arrays in scratch memory)
template <typename R>
__device__ __forceinline__ R pick(bool c, R a, R b) { return c ? a : b; }

template <typename R>
__device__ __forceinline__ R pick4(int k, R a, R b, R c, R e)
{
    return pick(k == 0, a, pick(k == 1, b, pick(k == 2, c, e)));
}

// slots S .. S1 of the window receive one update: four at a time from
// aligned slots, one at a time at the ends
template <int S, int S1, typename R, int PR, int NM>
__device__ __forceinline__ void panel_update(R (&ax)[PR], R (&ay)[PR], const R (&lx)[NM],
                                             const R (&ly)[NM], R ux, R uy)
{
    if constexpr (S <= S1) {
        if constexpr (S % 4 == 0 && S + 3 <= S1) {
            sz::fnms_row4<S % 16>(ax[S], ay[S], ax[S + 1], ay[S + 1], ax[S + 2], ay[S + 2],
                              ax[S + 3], ay[S + 3], lx[S / 16], ly[S / 16], ux, uy);
            panel_update<S + 4, S1>(ax, ay, lx, ly, ux, uy);
        } else {
            sz::fnms_row1<S % 16>(ax[S], ay[S], lx[S / 16], ly[S / 16], ux, uy);
            panel_update<S + 1, S1>(ax, ay, lx, ly, ux, uy);
        }
    }
}

// a[U] <-> a[sp] in the lanes of `in`; sp (uniform) in U+1 .. LAST.  The
// branch to the slot is inside the instructions: as branches of the source
// the exchanges are merged into one that indexes the window at run time, in
// scratch memory, or copy the window at every join.
#define PN_SWAP64(A, B)                                                         \
    "v_mov_b64 %[t], %[" A "]\n\tv_mov_b64 %[" A "], %[" B "]\n\t"              \
    "v_mov_b64 %[" B "], %[t]\n\t"
#define PN_SWAP32(A, B) "v_swap_b32 %[" A "], %[" B "]\n\t"
#define PN_ONE(SW, I)                                                           \
    "s_cmp_lg_u32 %[sp], %c[s" I "]\n\ts_cbranch_scc1 .Lpn" I "_%=\n\t"         \
    SW("ux", "x" I) SW("uy", "y" I) ".Lpn" I "_%=:\n\t"
#define PN_GROUP(SW)                                                            \
    "s_lshr_b32 %[g], %[sp], 2\n\ts_cmp_lg_u32 %[g], %c[grp]\n\t"               \
    "s_cbranch_scc1 .Lpn4_%=\n\ts_and_saveexec_b64 %[save], %[in]\n\t"          \
    PN_ONE(SW, "0") PN_ONE(SW, "1") PN_ONE(SW, "2") PN_ONE(SW, "3")             \
    "s_mov_b64 exec, %[save]\n\t.Lpn4_%=:"
template <int U, int S, int LAST, typename R, int PR>
__device__ __forceinline__ void slot_swap(R (&ax)[PR], R (&ay)[PR], int sp,
                                          unsigned long long in)
{
    if constexpr (S <= LAST) {
        // slots S .. S+3; in place of slot U itself or a slot past the window
        // (never sp) a spare register
        R nx[4], ny[4], t;
        unroll<4>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value, q = S + i;
            if constexpr (q > U && q < PR) {
                nx[i] = ax[q];
                ny[i] = ay[q];
            } else {
                nx[i] = ny[i] = R(0);
            }
        });
        unsigned g;
        unsigned long long save;
#define PN_OPERANDS                                                             \
        : [ux] "+v"(ax[U]), [uy] "+v"(ay[U]), [x0] "+v"(nx[0]), [y0] "+v"(ny[0]), \
          [x1] "+v"(nx[1]), [y1] "+v"(ny[1]), [x2] "+v"(nx[2]), [y2] "+v"(ny[2]), \
          [x3] "+v"(nx[3]), [y3] "+v"(ny[3]), [t] "=&v"(t), [g] "=&s"(g),        \
          [save] "=&s"(save)                                                    \
        : [sp] "s"(sp), [in] "s"(in), [grp] "n"(S / 4), [s0] "n"(S), [s1] "n"(S + 1), \
          [s2] "n"(S + 2), [s3] "n"(S + 3)                                      \
        : "scc"
        if constexpr (sizeof(R) == 8) asm volatile(PN_GROUP(PN_SWAP64) PN_OPERANDS);
        else asm volatile(PN_GROUP(PN_SWAP32) PN_OPERANDS);
#undef PN_OPERANDS
        unroll<4>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value, q = S + i;
            if constexpr (q > U && q < PR) {
                ax[q] = nx[i];
                ay[q] = ny[i];
            }
        });
        slot_swap<U, S + 4, LAST>(ax, ay, sp, in);
    }
}
#undef PN_GROUP
#undef PN_ONE
#undef PN_SWAP32
#undef PN_SWAP64

template <int CTRL>
__device__ __forceinline__ unsigned dpp_max(unsigned v)
{
    const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
    return v > o ? v : o;
}

// maximum over the 16 lanes of a row, in every lane of it
__device__ __forceinline__ unsigned row_max16(unsigned v)
{
    v = dpp_max<0xB1>(v);                    // quad_perm [1,0,3,2]
    v = dpp_max<0x4E>(v);                    // quad_perm [2,3,0,1]
    v = dpp_max<0x124>(v);                   // row_ror:4
    return dpp_max<0x128>(v);                // row_ror:8
}

// words of a nonnegative number, ordered as the number is: the high word
// (all of a float) and the low word
__device__ __forceinline__ unsigned key_hi(double v) { return (unsigned)__double2hiint(v); }
__device__ __forceinline__ unsigned key_lo(double v) { return (unsigned)__double2loint(v); }
__device__ __forceinline__ unsigned key_hi(float v) { return __builtin_bit_cast(unsigned, v); }
__device__ __forceinline__ unsigned key_lo(float) { return 0; }

template <typename R, int WR, int KV, bool UT, int WPE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void k_gbtrf_panel(int n, cpx<R> *__restrict__ ab, int ldab, long long sab,
                   int *__restrict__ ipiv, long long sipiv, int *__restrict__ info,
                   const int *__restrict__ skip, int nsys, cpx<R> *__restrict__ bv,
                   long long sb, const sz::gsys *__restrict__ gs)
{
    using T = cpx<R>;
    constexpr int NB = PN_NB, kl = WR - 1, ku = KV - kl;
    constexpr int PR = kl + NB;                    // rows of a block's window
    constexpr int NM = (PR + 15) / 16;             // registers of a panel column
    constexpr int NT = KV + NB > 64 ? KV + NB - 64 : 0;   // tail columns
    constexpr int PS = 16 * NM + 1;                // panel column stride in LDS
    constexpr unsigned INFW = sizeof(R) == 8 ? 0x7FF00000u : 0x7F800000u;
    static_assert(kl >= NB && ku >= NB, "interchanges reach every panel column");
    static_assert(NT == 0 || NT == 2 * NB, "tail");
    __shared__ T pbuf[NB * PS];
    __shared__ alignas(16) T qbuf[(NB + 2) * 64];  // what the next block needs
    __shared__ T tail[NT > 0 ? NT * PR : 1];
    __shared__ T tailb[NT > 0 ? NT : 1];

    const int sys = blockIdx.x;
    if (sys >= nsys) return;
    if (skip && skip[sys] != 0) return;
    if (gs) {                             // grouped: per-system order, storage
        const sz::gsys g = gs[sys];
        n = g.n;
        ab = reinterpret_cast<T *>(g.ab);
        ipiv = reinterpret_cast<int *>(g.ipiv);
        if constexpr (UT) bv = reinterpret_cast<T *>(g.b);
    } else {
        ab += (size_t)sys * (size_t)sab;
        ipiv += (size_t)sys * (size_t)sipiv;
        if constexpr (UT) bv += (size_t)sys * (size_t)sb;
    }
    int lane = threadIdx.x;

    auto band = [&](int i, int c) __attribute__((always_inline)) -> T {
        const bool ok = i < n && c < n && c - i <= ku && i - c <= kl;
        const T v = sz::gload(ab + (ok ? (size_t)c * ldab + KV + i - c : 0));
        return T{ok ? v.x : R(0), ok ? v.y : R(0)};
    };

    // component arrays throughout: arrays of structs go through scratch
    R ax[PR], ay[PR];
    unroll<PR>([&](auto s_) __attribute__((always_inline)) {
        constexpr int s = decltype(s_)::value;
        const T v = band(s, lane);
        ax[s] = v.x;
        ay[s] = v.y;
    });
    if constexpr (NT > 0) {
        for (int e = lane; e < NT * PR; e += 64) {
            const int t = e / PR;
            tail[e] = band(e - t * PR, 64 + t);
        }
    }
    for (int e = lane; e < NB * PS; e += 64) pbuf[e] = T{R(0), R(0)};
    R bx = R(0), by = R(0);
    if constexpr (UT) {
        const T v = sz::gload(bv + (lane < n ? lane : 0));
        bx = lane < n ? v.x : R(0);
        by = lane < n ? v.y : R(0);
        if (NT > 0 && lane < NT) {
            const int c = 64 + lane;
            const T w = sz::gload(bv + (c < n ? c : 0));
            tailb[lane] = T{c < n ? w.x : R(0), c < n ? w.y : R(0)};
        }
    }
    WAVE_SYNC();

    int first_zero = 0, ju = 0;
    for (int jb = 0; jb < n; jb += NB) {
        // what follows from the lane is recomputed in every block: held
        // through the loop it would not fit the registers
        asm volatile("" : "+v"(lane));
        const int l16 = lane & 15, lq = lane & 3;
        const int c0 = jb & 63;
        // ---- 1. panel columns (lanes with column jb + d, d < NB) to row layout
        if (((lane - c0) & 63) < NB) {
            T *dst = pbuf + ((lane - c0) & 63) * PS;
            unroll<PR>([&](auto s_) __attribute__((always_inline)) {
                constexpr int s = decltype(s_)::value;
                dst[s] = T{ax[s], ay[s]};
            });
        }
        // rows jb+PR .. jb+PR+3 of the next block's columns (of the tail's:
        // column lane/4, row lane%4) and the b of the columns it brings in,
        // straight to LDS: they arrive during the panel and the updates, and
        // registers to hold them are not to be had
        {
            const int cn = jb + NB + ((lane - c0 - NB) & 63);
            const T *src = ab + (cn < n ? (size_t)cn * ldab + KV + jb + PR - cn : 0);
            unroll<NB>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value;
                load_lds(cn < n && jb + PR + i < n ? src + i : ab, &qbuf[i * 64]);
            });
            if constexpr (NT > 0) {
                const int c = jb + NB + 64 + (lane >> 2), r = jb + PR + lq;
                load_lds(ab + (lane < NT * NB && c < n && r < n
                                   ? (size_t)c * ldab + KV + r - c : 0), &qbuf[NB * 64]);
            }
            if constexpr (UT) {
                const int c = jb + 64 + (NT > 0 ? NB + lane : (lane - c0) & 63);
                load_lds(bv + (c < n ? c : 0), &qbuf[(NB + 1) * 64]);
            }
        }
        WAVE_SYNC();
        R px[NB][NM], py[NB][NM];
        unroll<NB>([&](auto k_) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value;
            unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                constexpr int m = decltype(m_)::value;
                const T v = pbuf[k * PS + 16 * m + l16];
                px[k][m] = v.x;
                py[k][m] = v.y;
            });
        });
        R bkx[NB], bky[NB], yx[NB], yy[NB];
        if constexpr (UT) {
            unroll<NB>([&](auto k_) __attribute__((always_inline)) {
                constexpr int k = decltype(k_)::value;
                bkx[k] = readlane_r(bx, c0 + k);
                bky[k] = readlane_r(by, c0 + k);
            });
        }
        int jp[NB], jus[NB];
        unsigned nz = 0, odd = 0;                  // bit u: step u's
        unroll<NB>([&](auto uc_) __attribute__((always_inline)) {
            constexpr int u = decltype(uc_)::value;
            const int j = jb + u;
            const int km = min(kl, n - 1 - j);     // negative past the last column
            jp[u] = 0;
            yx[u] = yy[u] = R(0);
            if (j < n) {
                // the first row of the largest |Re|+|Im|; a NaN in row j wins,
                // any other NaN never does
                unsigned kh[NM], kw[NM], mx = 0, raw = 0;
                unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                    constexpr int m = decltype(m_)::value;
                    const int slot = 16 * m + l16;
                    const R m1 = fabs(px[u][m]) + fabs(py[u][m]);
                    unsigned h = key_hi(m1), w = key_lo(m1);
                    raw = max(raw, h);
                    const bool nan = m1 != m1;
                    bool ok = slot <= u + km && !(nan && slot != u);
                    if (m == 0) ok = ok && slot >= u;
                    h = nan ? INFW : h;
                    w = nan ? 0u : w;
                    kh[m] = ok ? h + 1 : 0u;
                    kw[m] = w;
                    mx = max(mx, kh[m]);
                });
                mx = row_max16(mx);
                auto first = [&](auto &&is) __attribute__((always_inline)) {
                    unsigned long long b = 0;
                    unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                        constexpr int m = decltype(m_)::value;
                        b |= (__ballot(is(m)) & 0xFFFFull) << (16 * m);
                    });
                    return b;
                };
                unsigned long long at = first([&](int m) { return kh[m] == mx; });
                if (sizeof(R) == 8 && (at & (at - 1)) != 0) {    // equal high words
                    unsigned ml = 0;
                    unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                        constexpr int m = decltype(m_)::value;
                        ml = max(ml, kh[m] == mx ? kw[m] : 0u);
                    });
                    ml = row_max16(ml);
                    at = first([&](int m) { return kh[m] == mx && kw[m] == ml; });
                }
                const int t = (int)__builtin_ctzll(at);
                jp[u] = t - u;
                if (jp[u] != 0) {                  // then the pivot is not zero
                    const int tm = t >> 4, tl = t & 15;
                    unroll<NB - u>([&](auto k_) __attribute__((always_inline)) {
                        constexpr int k = u + decltype(k_)::value;
                        R vx = px[k][0], vy = py[k][0];
                        const R jx = readlane_r(vx, u), jy = readlane_r(vy, u);
                        unroll<NM - 1>([&](auto m_) __attribute__((always_inline)) {
                            constexpr int m = 1 + decltype(m_)::value;
                            vx = pick(tm == m, px[k][m], vx);
                            vy = pick(tm == m, py[k][m], vy);
                        });
                        const R tx = readlane_r(vx, tl), ty = readlane_r(vy, tl);
                        unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                            constexpr int m = decltype(m_)::value;
                            const bool here = tm == m && l16 == tl;
                            px[k][m] = pick(here, jx, px[k][m]);
                            py[k][m] = pick(here, jy, py[k][m]);
                        });
                        px[k][0] = pick(l16 == u, tx, px[k][0]);
                        py[k][0] = pick(l16 == u, ty, py[k][0]);
                    });
                }
                T piv;
                piv.x = row_bcast<u>(px[u][0]);
                piv.y = row_bcast<u>(py[u][0]);
                const bool pz = __ballot(sz::cnonzero(piv)) != 0;
                nz |= pz ? 1u << u : 0u;
                if (pz) ju = max(ju, min(j + ku + jp[u], n - 1));
                else if (first_zero == 0) first_zero = j + 1;

                // sz::crcp of the pivot and y = sz::cdiv(b_j, pivot): Smith's
                // quotients have one denominator, so lane lq of a quad divides
                // the numerator of (1/z).x, (1/z).y, y.x or y.y
                const bool big = fabs(piv.x) >= fabs(piv.y);
                const R P = big ? piv.x : piv.y, Q = big ? piv.y : piv.x;
                const R r = Q / P, den = P + Q * r;
                R num = lq & 1 ? (big ? -r : R(-1)) : (big ? R(1) : r);
                if constexpr (UT) {
                    const R A = pick(big, bkx[u], bky[u]), B = pick(big, bky[u], bkx[u]);
                    const R n2 = A + B * r, n3 = B - A * r;
                    const R ny = lq & 1 ? (big ? n3 : -n3) : n2;
                    num = lq & 2 ? ny : num;
                }
                const R quo = num / den;
                const T rcp{dpp_r<0x00>(quo), dpp_r<0x55>(quo)};
                if constexpr (UT) {
                    yx[u] = readlane_r(quo, 2);
                    yy[u] = readlane_r(quo, 3);
                }
                if (pz) {
                    unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                        constexpr int m = decltype(m_)::value;
                        const T l = sz::cmul(T{px[u][m], py[u][m]}, rcp);
                        const bool below = m > 0 || l16 > u;
                        px[u][m] = pick(below, l.x, px[u][m]);
                        py[u][m] = pick(below, l.y, py[u][m]);
                    });
                    // a column with an infinity or NaN, or an overflowing
                    // reciprocal: its update spares the columns beyond ju
                    odd |= __ballot(raw >= INFW || key_hi(fabs(rcp.x)) >= INFW ||
                                    key_hi(fabs(rcp.y)) >= INFW) != 0 ? 1u << u : 0u;
                }
                // the panel's later columns, rows j+1 .. j+kl
                unroll<NB - (u + 1)>([&](auto k_) __attribute__((always_inline)) {
                    constexpr int k = u + 1 + decltype(k_)::value;
                    T uk;
                    uk.x = row_bcast<u>(px[k][0]);
                    uk.y = row_bcast<u>(py[k][0]);
                    if (pz) {
                        unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                            constexpr int m = decltype(m_)::value;
                            const T v = sz::cfnms(T{px[k][m], py[k][m]},
                                                  T{px[u][m], py[u][m]}, uk);
                            const bool in = (m > 0 || l16 > u) &&
                                            (16 * m + 15 <= u + kl || 16 * m + l16 <= u + kl);
                            px[k][m] = pick(in, v.x, px[k][m]);
                            py[k][m] = pick(in, v.y, py[k][m]);
                        });
                    }
                    if constexpr (UT) {
                        const T v = sz::cfnms(T{bkx[k], bky[k]}, uk, T{yx[u], yy[u]});
                        bkx[k] = v.x;
                        bky[k] = v.y;
                    }
                });
            }
            jus[u] = ju - jb;                      // last column of the update, as d
        });

        asm volatile("" : "+v"(lane));
        // the panel columns are final: back to LDS, where the updates below
        // read their multipliers, and 16-lane row k stores column jb + k
        // (rows jb .. jb+k+km) from there
        const int r16 = lane & 15, d = (lane - c0) & 63;
        if (lane < 16) {
            unroll<NB>([&](auto k_) __attribute__((always_inline)) {
                constexpr int k = decltype(k_)::value;
                unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                    constexpr int m = decltype(m_)::value;
                    pbuf[k * PS + 16 * m + r16] = T{px[k][m], py[k][m]};
                });
            });
        }
        WAVE_SYNC();
        {
            const int k = lane >> 4, j = jb + k;
            const int last = min(k + kl, n - 1 - jb);
            T *dst = ab + (size_t)min(j, n - 1) * ldab + KV - k;
            unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                constexpr int m = decltype(m_)::value;
                const R *x = reinterpret_cast<const R *>(pbuf + k * PS + 16 * m + r16);
                const T v{x[0], x[1]};
                if (j < n && 16 * m + r16 <= last) sz::gstore(dst + 16 * m + r16, v);
            });
            if (lane < NB && jb + lane < n) {
                const int q4 = pick4(lane, jp[0], jp[1], jp[2], jp[3]);
                *sz::gmem(ipiv + jb + lane) = jb + lane + q4 + 1;
                if constexpr (UT) {
                    T y;
                    y.x = pick4(lane, yx[0], yx[1], yx[2], yx[3]);
                    y.y = pick4(lane, yy[0], yy[1], yy[2], yy[3]);
                    sz::gstore(bv + jb + lane, y);
                }
            }
        }

        // ---- 2. the four interchanges and updates on every column
        unroll<NB>([&](auto uc_) __attribute__((always_inline)) {
            constexpr int u = decltype(uc_)::value;
            if (jp[u] != 0)
                slot_swap<u, u / 4 * 4, u + kl>(ax, ay, u + jp[u],
                                                __ballot(d >= u && d <= jus[u]));
            const R ux = ax[u], uy = ay[u];
            if constexpr (UT) {
                const T v = sz::cfnms(T{bx, by}, T{ux, uy}, T{yx[u], yy[u]});
                const bool in = jb + u < n && d > u && d - u <= KV;
                bx = pick(in, v.x, bx);
                by = pick(in, v.y, by);
            }
            if (nz >> u & 1) {
                R lx[NM], ly[NM];
                unroll<NM>([&](auto m_) __attribute__((always_inline)) {
                    constexpr int m = decltype(m_)::value;
                    const T v = pbuf[u * PS + 16 * m + r16];
                    lx[m] = v.x;
                    ly[m] = v.y;
                });
                panel_update<u + 1, u + kl>(ax, ay, lx, ly, ux, uy);
                // Columns beyond ju have U(j, c) = 0, which a finite
                // multiplier leaves alone but an infinite one or a NaN does
                // not: no step has reached them, so they are read again.
                if (odd >> u & 1) {
                    const int c = jb + d;
                    if (d > jus[u] && c < n) {
                        const T *col = ab + (size_t)c * ldab + KV - d;
                        unroll<PR>([&](auto s_) __attribute__((always_inline)) {
                            constexpr int s = decltype(s_)::value;
                            const T v = sz::gload(jb + s < n ? col + s : ab);
                            const bool ok = d - s <= ku && jb + s < n;
                            ax[s] = pick(ok, v.x, R(0));
                            ay[s] = pick(ok, v.y, R(0));
                        });
                    }
                }
            }
            if constexpr (NT > 0) {
                if (jus[u] >= 64 && (nz >> u & 1)) {       // a far pivot reached the tail
                    if (lane < NT && 64 + lane <= jus[u] && jp[u] != 0) {
                        R *x = reinterpret_cast<R *>(tail + lane * PR + u);
                        R *y = reinterpret_cast<R *>(tail + lane * PR + u + jp[u]);
                        const R x0 = x[0], x1 = x[1];
                        x[0] = y[0];
                        x[1] = y[1];
                        y[0] = x0;
                        y[1] = x1;
                    }
                    WAVE_SYNC();
                    const int t = lane >> 3;
                    if (64 + t <= jus[u]) {
                        const R *tu = reinterpret_cast<const R *>(tail + t * PR + u);
                        const T ut{tu[0], tu[1]};
                        for (int s = u + 1 + (lane & 7); s <= u + kl; s += 8) {
                            R *x = reinterpret_cast<R *>(tail + t * PR + s);
                            const R *lm = reinterpret_cast<const R *>(pbuf + u * PS + s);
                            const T v = sz::cfnms(T{x[0], x[1]}, T{lm[0], lm[1]}, ut);
                            x[0] = v.x;
                            x[1] = v.y;
                        }
                    }
                    WAVE_SYNC();
                }
            }
        });

        asm volatile("" : "+v"(lane));
        const bool leaving = ((lane - c0) & 63) < NB;    // a panel column's lane
        // what the loads brought, before this block's stores join their queue
        R qx[NB], qy[NB], qtx = R(0), qty = R(0), qbx = R(0), qby = R(0);
        {
            unroll<NB>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value;
                take_lds(&qbuf[i * 64], lane, qx[i], qy[i]);
            });
            if constexpr (NT > 0) take_lds(&qbuf[NB * 64], lane, qtx, qty);
            if constexpr (UT) take_lds(&qbuf[(NB + 1) * 64], lane, qbx, qby);
        }
        __builtin_amdgcn_sched_barrier(0);

        // ---- 3. U rows of the window's columns and of the tail's
        const int row = lane & 3;
        {
            const int d = (lane - c0) & 63, c = jb + d;
            if (!leaving && c < n) {
                T *dst = ab + (size_t)c * ldab + KV - d;
                unroll<NB>([&](auto i_) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_)::value;
                    if (d - i <= KV) sz::gstore(dst + i, T{ax[i], ay[i]});
                });
            }
            if constexpr (NT > 0) {
                const int t = lane >> 2, ct = jb + 64 + t;
                if (lane < NT * NB && ct < n && 64 + t - row <= KV) {
                    const R *x = reinterpret_cast<const R *>(tail + t * PR + row);
                    sz::gstore(ab + (size_t)ct * ldab + KV - 64 - t + row, T{x[0], x[1]});
                }
            }
        }

        // ---- the next block: slots renamed by NB, leaving lanes take the
        // columns after the window's last, the next rows enter
        // (as a loop this becomes a memmove, which keeps the arrays in scratch)
        unroll<PR - NB>([&](auto s_) __attribute__((always_inline)) {
            constexpr int s = decltype(s_)::value;
            ax[s] = ax[s + NB];
            ay[s] = ay[s + NB];
        });
        if constexpr (NT > 0) {
            if constexpr (UT) {
                T tb{R(0), R(0)};
                if (lane < NT) {
                    const R *x = reinterpret_cast<const R *>(tailb + lane);
                    tb = T{x[0], x[1]};
                    unroll<NB>([&](auto uc_) __attribute__((always_inline)) {
                        constexpr int u = decltype(uc_)::value;
                        const R *w = reinterpret_cast<const R *>(tail + lane * PR + u);
                        if (jb + u < n && 64 + lane - u <= KV && jb + 64 + lane < n)
                            tb = sz::cfnms(tb, T{w[0], w[1]}, T{yx[u], yy[u]});
                    });
                }
                WAVE_SYNC();
                if (lane < NT) tailb[lane] = tb;
                WAVE_SYNC();
                {
                    const R *x = reinterpret_cast<const R *>(tailb + (leaving ? (lane - c0) & 63 : 0));
                    bx = leaving ? x[0] : bx;
                    by = leaving ? x[1] : by;
                }
                const bool in = jb + NB + 64 + lane < n;
                const R *up = reinterpret_cast<const R *>(tailb + (lane < NB ? lane + NB : 0));
                const R nbx = lane < NB ? up[0] : in ? qbx : R(0);
                const R nby = lane < NB ? up[1] : in ? qby : R(0);
                WAVE_SYNC();
                if (lane < NT) tailb[lane] = T{nbx, nby};
            }
            if (leaving) {
                // (keeps the branch, whose reads land in place: speculated,
                // they would take a select each)
                asm volatile("; leaving");
                const T *col = tail + ((lane - c0) & 63) * PR + NB;
                unroll<PR - NB>([&](auto s_) __attribute__((always_inline)) {
                    constexpr int s = decltype(s_)::value;
                    const R *x = reinterpret_cast<const R *>(col + s);
                    ax[s] = x[0];
                    ay[s] = x[1];
                });
            }
            // the tail's later columns move up, its last four are new
            constexpr int MV = (NT - NB) * (PR - NB), MI = (MV + 63) / 64;
            R mvx[MI], mvy[MI];
            unroll<MI>([&](auto e_) __attribute__((always_inline)) {
                constexpr int e = decltype(e_)::value;
                const int x = min(lane + 64 * e, MV - 1), t = x / (PR - NB);
                const T v = tail[(t + NB) * PR + NB + x - t * (PR - NB)];
                mvx[e] = v.x;
                mvy[e] = v.y;
            });
            WAVE_SYNC();
            unroll<MI>([&](auto e_) __attribute__((always_inline)) {
                constexpr int e = decltype(e_)::value;
                const int x = lane + 64 * e, t = x / (PR - NB);
                if (x < MV) {
                    tail[t * PR + x - t * (PR - NB)] = T{mvx[e], mvy[e]};
                    R z = R(0);          // (a zero held through the loop gets spilled)
                    asm volatile("" : "+v"(z));
                    tail[(t + NB) * PR + x - t * (PR - NB)] = T{z, z};
                }
            });
            if (lane < NT * NB) {
                const int t = lane >> 2;
                const bool ok = jb + NB + 64 + t < n && jb + PR + row < n && t <= KV - 64 + row;
                tail[t * PR + PR - NB + row] = T{ok ? qtx : R(0), ok ? qty : R(0)};
            }
        } else {
            if (leaving) {
                asm volatile("; leaving");
                unroll<PR - NB>([&](auto s_) __attribute__((always_inline)) {
                    constexpr int s = decltype(s_)::value;
                    ax[s] = ay[s] = R(0);
                });
                if constexpr (UT) {
                    const bool in = jb + 64 + ((lane - c0) & 63) < n;
                    bx = in ? qbx : R(0);
                    by = in ? qby : R(0);
                }
            }
        }
        unroll<NB>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            const int dn = (lane - c0 - NB) & 63;
            const bool ok = jb + NB + dn < n && jb + PR + i < n && dn >= i && dn <= KV + i;
            ax[PR - NB + i] = pick(ok, qx[i], R(0));
            ay[PR - NB + i] = pick(ok, qy[i], R(0));
        });
        WAVE_SYNC();
    }
    if (lane == 0 && info) *sz::gmem(info + sys) = first_zero;
}

// Launches k_gbtrf_panel for the band shapes it is instantiated for -- kl =
// ku = 34 (five interleaved fields, k = 8 operators), kl = ku = 24 (k = 6)
// and kl = 34, ku = 20 -- and returns whether the call is one for it.  Its
// transfers to LDS move a complex double as 16 bytes, which are not documented
// for less than 16-byte alignment; an array aligned as C's double complex (8
// bytes) goes to the kernels whose loads the compiler chose.  (A grouped
// launch's arrays are the library's own.)
template <typename R, bool UT>
bool launch_panel(int n, int kl, int ku, void *ab, int ldab, long long sab, int *ipiv,
                  long long sipiv, int *info, const int *skip, int nsys, void *b,
                  long long sb, const sz::gsys *gs, hipStream_t stream)
{
    if (sizeof(R) == 8 && !gs &&
        (reinterpret_cast<uintptr_t>(ab) | reinterpret_cast<uintptr_t>(b)) % 16 != 0)
        return false;
#define SZ_PANEL(WR_, KV_)                                                      \
    hipLaunchKernelGGL((k_gbtrf_panel<R, WR_, KV_, UT, panel_waves(sizeof(R), WR_, UT)>), \
                       dim3(nsys), dim3(64), 0, stream, n,                      \
                       reinterpret_cast<cpx<R> *>(ab), ldab, sab, ipiv, sipiv, info, \
                       skip, nsys, reinterpret_cast<cpx<R> *>(b), sb, gs)
    if (kl == 34 && ku == 34) SZ_PANEL(35, 68);
    else if (kl == 24 && ku == 24) SZ_PANEL(25, 48);
    else if (kl == 34 && ku == 20) SZ_PANEL(35, 54);
    else return false;
#undef SZ_PANEL
    return true;
}

// Factorization kernels: k_gbtrf_panel for the channel band shapes and the
// LDS window kernel k_gbtrf for every other call.  SZ_GBTRF_KERNEL = "lds"
// (or "lds64"/"lds128", fewer threads) forces the LDS kernel.
template <typename R>
int launch_gbtrf(int n, int kl, int ku, void *ab, int ldab, long long sab,
                 int *ipiv, long long sipiv, int *info, const int *skip,
                 int nsys, hipStream_t stream)
{
    if (n < 0) return -1;
    if (kl < 0) return -2;
    if (ku < 0) return -3;
    if (ldab < 2 * kl + ku + 1) return -5;
    if (sab < (long long)ldab * n) return -6;
    if (sipiv < n) return -8;
    if (nsys < 0) return -10;
    if (nsys == 0 || n == 0) return 0;
    static const char *sel = getenv("SZ_GBTRF_KERNEL");
    if (!(sel && sel[0] == 'l') &&
        launch_panel<R, false>(n, kl, ku, ab, ldab, sab, ipiv, sipiv, info, skip, nsys,
                               nullptr, 0, nullptr, stream))
        return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
    const size_t lds = ((size_t)(kl + 1) * (kl + ku + 1) + (kl + ku + 1) + (kl + 1))
                       * sizeof(cpx<R>);
    if (lds > LDS_MAX) return SZ_ERR_LDS;
    int nt = (sel && sel[0] == 'l' && sel[3] == '6') ? 64
           : (sel && sel[0] == 'l' && sel[3] == '1') ? 128 : 256;
    // every column of the window and every multiplier needs a thread
    while (nt < 256 && (kl + ku + 1 > 2 * nt || kl > nt)) nt *= 2;
    if (kl + ku + 1 > 256 || kl > 256) return SZ_ERR_LDS;
    if (nt == 64)
        hipLaunchKernelGGL((k_gbtrf<R, 64>), dim3(nsys), dim3(64), lds, stream, n,
                           kl, ku, reinterpret_cast<cpx<R> *>(ab), ldab, sab,
                           ipiv, sipiv, info, skip, nsys);
    else if (nt == 128)
        hipLaunchKernelGGL((k_gbtrf<R, 128>), dim3(nsys), dim3(128), lds, stream, n,
                           kl, ku, reinterpret_cast<cpx<R> *>(ab), ldab, sab,
                           ipiv, sipiv, info, skip, nsys);
    else
        hipLaunchKernelGGL((k_gbtrf<R, 256>), dim3(nsys), dim3(256), lds, stream, n,
                           kl, ku, reinterpret_cast<cpx<R> *>(ab), ldab, sab,
                           ipiv, sipiv, info, skip, nsys);
    return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
}

// Factorization fused with the U^T half of a transposed solve of one right
// hand side per system (b, stride sb, overwritten by y); returns 1 when the
// band shape or the arrays' alignment has no fused kernel (the caller then
// factors and solves apart).
template <typename R>
int launch_gbtrf_ut(int n, int kl, int ku, void *ab, int ldab, long long sab,
                    int *ipiv, long long sipiv, int *info, void *b, long long sb,
                    int nsys, hipStream_t stream)
{
    if (n < 0) return -1;
    if (kl < 0) return -2;
    if (ku < 0) return -3;
    if (ldab < 2 * kl + ku + 1) return -5;
    if (sab < (long long)ldab * n) return -6;
    if (sipiv < n) return -8;
    if (sb < n) return -12;
    if (nsys < 0) return -10;
    if (nsys == 0 || n == 0) return 0;
    static const char *sel = getenv("SZ_GBTRF_KERNEL");
    if (sel && sel[0] == 'l') return 1;
    if (!launch_panel<R, true>(n, kl, ku, ab, ldab, sab, ipiv, sipiv, info, nullptr, nsys,
                               b, sb, nullptr, stream))
        return 1;
    return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
}

int trans_code(char t)
{
    switch (t) {
    case 'N': case 'n': return 0;
    case 'T': case 't': return 1;
    case 'C': case 'c': return 2;
    default: return -1;
    }
}

// Lanes per system of the transposed single precision solve: 16, or 32
// with SZ_T16_LANES=32.  Thirty-two lanes double the wavefronts in flight
// but add a swizzle stage to every step's sum and unroll 32 steps (247
// VGPRs instead of 200): measured on the precision form's 96^3 step 11.9 ms
// against 11.2 with 16 lanes, and within 1% at 192^3, so 16 stays the
// default.
int t16_lanes(int)
{
    static const int forced = [] {
        const char *e = std::getenv("SZ_T16_LANES");
        return e ? std::atoi(e) : 0;
    }();
    return forced == 32 ? 32 : 16;
}

// The sixteen-lane transposed solve for the channel band shapes in single
// precision (the refinement solves of the mixed precision solver); false
// when the shape or precision has no such kernel.  gs != nullptr: grouped,
// every system of order 2 or more (the kernel clamps its loads to the
// system's last column).
// Band shapes and right hand side lengths the single precision transposed
// solve takes (its LDS holds spw right hand sides of ldx elements).
bool t16_covers(int kl, int ku, int ldx, int lps)
{
    const size_t lds = (size_t)(64 / lps) * (size_t)ldx * sizeof(cpx<float>);
    return ldx > 0 && lds <= LDS_MAX &&
           ((kl == 34 && ku == 34) || (kl == 24 && ku == 24));
}

template <typename R>
bool launch_gbtrs_t16(int tc, int n, int kl, int ku, const void *ab, int ldab,
                      long long sab, const int *ipiv, long long sipiv, void *b,
                      long long sb, const int *skip, int nsys, int ldx,
                      const sz::gsys *gs, hipStream_t stream)
{
    if constexpr (sizeof(R) != 4) {
        return false;
    } else {
        if (tc == 0 || ldx <= 0 || (!gs && n < 2)) return false;
        const int lps = t16_lanes(nsys);
        const int spw = 64 / lps;
        const size_t lds = (size_t)spw * (size_t)ldx * sizeof(cpx<R>);
        if (!t16_covers(kl, ku, ldx, lps)) return false;
        const dim3 grid((nsys + spw - 1) / spw);
        const cpx<R> *a = reinterpret_cast<const cpx<R> *>(ab);
        cpx<R> *x = reinterpret_cast<cpx<R> *>(b);
#define SZ_T16(KL_, KV_, CJ_)                                                   \
        do {                                                                   \
            if (lps == 32)                                                     \
                hipLaunchKernelGGL((k_gbtrs_t16<R, KL_, KV_, true, CJ_, 32>), grid, \
                                   dim3(64), lds, stream, n, a, ldab, sab, ipiv, \
                                   sipiv, x, sb, skip, nsys, ldx, gs);         \
            else                                                               \
                hipLaunchKernelGGL((k_gbtrs_t16<R, KL_, KV_, true, CJ_, 16>), grid, \
                                   dim3(64), lds, stream, n, a, ldab, sab, ipiv, \
                                   sipiv, x, sb, skip, nsys, ldx, gs);         \
        } while (0)
        if (kl == 34 && ku == 34) {
            if (tc == 2) SZ_T16(34, 68, true);
            else SZ_T16(34, 68, false);
        } else if (kl == 24 && ku == 24) {
            if (tc == 2) SZ_T16(24, 48, true);
            else SZ_T16(24, 48, false);
        } else {
            return false;
        }
#undef SZ_T16
        return true;
    }
}

// The register solve where the band fits its lanes and the order is worth its
// fixed work (whole groups of 8 or 16 steps, two rounds of prefetches), else
// false: k_gbtrs takes any band its staging holds.  Measured as register / LDS
// time, both precisions, bands of 0 to 116 off-diagonals, one and three right
// hand sides, mean / worst:
//   N: order 1 1.0 to 2.0 / 2.5, order 2 0.9 to 1.2 / 1.5, order 3 0.8 to 1.1 /
//     1.3, order 8 0.55 to 0.8 / 1.0;
//   T, 600 systems: order 3 1.3 / 1.9, 5 1.05 / 1.3, 6 0.95 / 1.06, 8 0.8 / 1.0;
//   T, 2,400 to 20,000 systems: order 3 1.6 to 2.4 / 2.8, 6 1.3 / 1.6, 9 1.05 /
//     1.2, 11 1.05 / 1.3, 12 1.0 / 1.1, 16 0.75 / 0.9;
//   T without an L half (kl = 0): 600 systems: order 6 1.0 / 1.4, 9 1.0 / 1.1;
//     more: 12 1.1 / 1.3, 17 1.2 / 1.6, 24 0.95 / 1.2, 28 0.85 / 1.05, 33 1.0 / 1.2,
//     40 0.85 / 1.05.
template <typename R>
bool launch_gbtrs_reg(int tc, int n, int kl, int ku, int nrhs, const void *ab, int ldab,
                      long long sab, const int *ipiv, long long sipiv, void *b, int ldb,
                      long long sb, const int *skip, int nsys, hipStream_t stream,
                      bool lt_only = false)
{
    const int kv = kl + ku;
    // the transposed ones keep finished rows to the end of a block of four (U^T)
    // and of eight (L^T)
    if (tc == 0 ? kl > 63 || kv > 127 : kl > 56 || kv > 124) return false;
    const bool few = nsys <= 1024;           // at most one a SIMD: latency counts
    const int from = tc == 0 ? 3 : kl > 0 ? (few ? 6 : 12) : (few ? 9 : 24);
    if (n < from && !lt_only) return false;
    const size_t lds = (size_t)n * sizeof(cpx<R>);
#define SZ_REG(MODE_, NR_)                                                        \
    hipLaunchKernelGGL((k_gbtrs_reg<R, MODE_, NR_>), dim3(nsys), dim3(64), lds, stream, tc, \
                       n, kl, ku, nrhs, reinterpret_cast<const cpx<R> *>(ab), ldab, sab, \
                       ipiv, sipiv, reinterpret_cast<cpx<R> *>(b), ldb, sb, skip, nsys)
    if (lt_only) {                           // (the fused factorization is double)
        if constexpr (sizeof(R) == 8) SZ_REG(SOLVE_LT, 1);
        else return false;
    } else if (tc == 0) {
        if (kv <= 63) SZ_REG(SOLVE_N, 1);
        else SZ_REG(SOLVE_N, 2);
    } else {
        if (kv <= 60) SZ_REG(SOLVE_T, 1);
        else SZ_REG(SOLVE_T, 2);
    }
#undef SZ_REG
    return true;
}

template <typename R>
int launch_gbtrs(char trans, int n, int kl, int ku, int nrhs, const void *ab,
                 int ldab, long long sab, const int *ipiv, long long sipiv,
                 void *b, int ldb, long long sb, const int *skip, int nsys,
                 hipStream_t stream, bool lt_only = false)
{
    const int tc = trans_code(trans);
    if (tc < 0) return -1;
    if (n < 0) return -2;
    if (kl < 0) return -3;
    if (ku < 0) return -4;
    if (nrhs < 0) return -5;
    if (ldab < 2 * kl + ku + 1) return -7;
    if (sab < (long long)ldab * n) return -8;
    if (sipiv < n) return -10;
    if (ldb < (n > 1 ? n : 1)) return -12;
    if (sb < (long long)ldb * nrhs) return -13;
    if (nsys < 0) return -14;
    if (nsys == 0 || n == 0 || nrhs == 0) return 0;
    if (kl + ku + 1 > TRS_PRE * TRS_NT) return SZ_ERR_LDS;
    // the transposed solves keep only x in LDS; the forward one also stages
    // factor columns and pivots
    const size_t lds = tc == 0 ? ((size_t)n + (size_t)TRS_PRE * TRS_NT) * sizeof(cpx<R>)
                                     + 64 * sizeof(int)
                               : (size_t)n * sizeof(cpx<R>);
    if (lds > LDS_MAX) return SZ_ERR_LDS;
    if (nrhs == 1 && !lt_only &&
        launch_gbtrs_t16<R>(tc, n, kl, ku, ab, ldab, sab, ipiv, sipiv, b, sb, skip,
                            nsys, n, nullptr, stream))
        return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
    if (launch_gbtrs_reg<R>(tc, n, kl, ku, nrhs, ab, ldab, sab, ipiv, sipiv, b, ldb, sb,
                            skip, nsys, stream, lt_only))
        return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
    if (lt_only) return SZ_ERR_LDS;          // only after a fused factorization
    if (tc == 0)
        hipLaunchKernelGGL((k_gbtrs<R, false>), dim3(nsys), dim3(TRS_NT), lds, stream, tc, n,
                       kl, ku, nrhs, reinterpret_cast<const cpx<R> *>(ab), ldab,
                       sab, ipiv, sipiv, reinterpret_cast<cpx<R> *>(b), ldb, sb,
                       skip, nsys);
    else
        hipLaunchKernelGGL((k_gbtrs<R, true>), dim3(nsys), dim3(TRS_NT), lds, stream, tc, n,
                       kl, ku, nrhs, reinterpret_cast<const cpx<R> *>(ab), ldab,
                       sab, ipiv, sipiv, reinterpret_cast<cpx<R> *>(b), ldb, sb,
                       skip, nsys);
    return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
}

// Grouped launches: every system of gs (orders up to nmax, band storage at
// gs[s].ab with leading dimension ldab = 2 kl + ku + 1) in one launch.
// The precision solver's float factors, the only ones it groups: the panel
// kernel and the sixteen-lane solve take its band shapes at every order its
// sweep takes.
int launch_gbtrf_grouped(int kl, int ku, void *ab, int ldab, int *ipiv, int *info,
                         const int *skip, const sz::gsys *gs, int nsys,
                         hipStream_t stream)
{
    if (nsys <= 0) return nsys < 0 ? -10 : 0;
    if (ldab != 2 * kl + ku + 1) return -5;
    if (!((kl == 34 && ku == 34) || (kl == 24 && ku == 24))) return SZ_ERR_LDS;
    if (!launch_panel<float, false>(0, kl, ku, ab, ldab, 0, ipiv, 0, info, skip, nsys,
                                    nullptr, 0, gs, stream))
        return SZ_ERR_LDS;
    return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
}

// In place, for the listed systems of a grouped launch (global indices
// list[0 .. *count); those in [s0, s0 + ns) are taken, system s described by
// gs[s - s0]): factors in LAPACK band storage -> the split layout of gsys
// (layout 1).  Per system: the multipliers into temp, the U columns
// compacted in ascending chunks through LDS (a chunk's new place ends no
// later than its old one, so it never overwrites a column not yet read),
// then the multipliers after them.
constexpr int SPLIT_NT = 256, SPLIT_CH = 64;
template <typename T>
__global__ __launch_bounds__(SPLIT_NT)
void k_band_split(int kl, int ku, const sz::gsys *__restrict__ gs, int s0, int ns,
                  const int *__restrict__ list, const int *__restrict__ count,
                  T *__restrict__ temp, long long tstride)
{
    extern __shared__ __align__(16) unsigned char smem[];
    T *stage = reinterpret_cast<T *>(smem);      // SPLIT_CH x (kl + ku + 1)
    const int U = kl + ku + 1, LD = 2 * kl + ku + 1;
    T *tb = temp + (size_t)blockIdx.x * (size_t)tstride;
    const int cnt = *count;
    for (int j = blockIdx.x; j < cnt; j += gridDim.x) {
        const int s = list[j];
        if (s < s0 || s >= s0 + ns) continue;           // uniform
        const sz::gsys g = gs[s - s0];
        T *a = reinterpret_cast<T *>(g.ab);
        const int N = g.n;
        const long long nL = (long long)N * kl;
        for (long long e = threadIdx.x; e < nL; e += SPLIT_NT) {
            const long long c = e / kl;
            tb[e] = a[c * LD + U + (e - c * kl)];
        }
        for (int c0 = 0; c0 < N; c0 += SPLIT_CH) {
            const int m = min(SPLIT_CH, N - c0) * U;
            for (int e = threadIdx.x; e < m; e += SPLIT_NT) {
                const int c = e / U;
                stage[e] = a[(long long)(c0 + c) * LD + (e - c * U)];
            }
            __syncthreads();        // (also orders the multipliers' reads)
            for (int e = threadIdx.x; e < m; e += SPLIT_NT)
                a[(long long)c0 * U + e] = stage[e];
            __syncthreads();
        }
        for (long long e = threadIdx.x; e < nL; e += SPLIT_NT)
            a[(long long)N * U + e] = tb[e];
        __syncthreads();            // temp and LDS are the next system's
    }
}

int launch_gbtrs_grouped(char trans, int kl, int ku, const void *ab, int ldab,
                         const int *ipiv, void *b, const int *skip,
                         const sz::gsys *gs, int nsys, int nmax,
                         hipStream_t stream)
{
    const int tc = trans_code(trans);
    if (tc <= 0) return -1;              // the transposed solves only
    if (nsys <= 0) return nsys < 0 ? -10 : 0;
    if (!launch_gbtrs_t16<float>(tc, 0, kl, ku, ab, ldab, 0LL, ipiv, 0LL, b, 0LL, skip,
                                 nsys, nmax, gs, stream))
        return SZ_ERR_LDS;
    return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int sz_internal_gbtrf_grouped(int single, int kl, int ku, void *ab, int ldab,
                              int *ipiv, int *info, const int *skip,
                              const void *gs, int nsys, void *stream)
{
    if (!single) return SZ_ERR_LDS;
    return launch_gbtrf_grouped(kl, ku, ab, ldab, ipiv, info, skip,
                                static_cast<const sz::gsys *>(gs), nsys,
                                (hipStream_t)stream);
}

// 1 when the single precision grouped transposed solve of this band shape
// and largest order reads the split layout (gsys layout 1), else 0.
int sz_internal_gbtrs_split_ok(int kl, int ku, int nmax)
{
    return t16_covers(kl, ku, nmax, t16_lanes(0)) ? 1 : 0;
}

// Factors of the listed systems (see k_band_split) from LAPACK band storage
// to the split layout, single precision; temp holds grid * nmax * kl complex
// floats.
int sz_internal_band_split_grouped(int kl, int ku, const void *gs, int s0, int ns,
                                   int nmax, const int *list, const int *count,
                                   void *temp, int grid, void *stream)
{
    if (ns <= 0 || grid <= 0) return 0;
    const size_t lds = (size_t)SPLIT_CH * (size_t)(kl + ku + 1) * sizeof(cpx<float>);
    if (lds > LDS_MAX) return SZ_ERR_LDS;
    hipLaunchKernelGGL(k_band_split<cpx<float>>, dim3(grid), dim3(SPLIT_NT), lds,
                       (hipStream_t)stream, kl, ku, static_cast<const sz::gsys *>(gs),
                       s0, ns, list, count, static_cast<cpx<float> *>(temp),
                       (long long)nmax * kl);
    return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
}

int sz_internal_gbtrs_grouped(int single, char trans, int kl, int ku,
                              const void *ab, int ldab, const int *ipiv, void *b,
                              const int *skip, const void *gs, int nsys, int nmax,
                              void *stream)
{
    if (!single) return SZ_ERR_LDS;
    return launch_gbtrs_grouped(trans, kl, ku, ab, ldab, ipiv, b, skip,
                                static_cast<const sz::gsys *>(gs), nsys, nmax,
                                (hipStream_t)stream);
}

int sz_zgbtrf_batched(int n, int kl, int ku, void *ab, int ldab,
                      long long strideab, int *ipiv, long long strideipiv,
                      int *info, int nbatch, void *stream)
{
    return launch_gbtrf<double>(n, kl, ku, ab, ldab, strideab, ipiv, strideipiv,
                                info, nullptr, nbatch, (hipStream_t)stream);
}

int sz_cgbtrf_batched(int n, int kl, int ku, void *ab, int ldab,
                      long long strideab, int *ipiv, long long strideipiv,
                      int *info, int nbatch, void *stream)
{
    return launch_gbtrf<float>(n, kl, ku, ab, ldab, strideab, ipiv, strideipiv,
                               info, nullptr, nbatch, (hipStream_t)stream);
}

int sz_zgbtrs_batched(char trans, int n, int kl, int ku, int nrhs,
                      const void *ab, int ldab, long long strideab,
                      const int *ipiv, long long strideipiv, void *b, int ldb,
                      long long strideb, int nbatch, void *stream)
{
    return launch_gbtrs<double>(trans, n, kl, ku, nrhs, ab, ldab, strideab, ipiv,
                                strideipiv, b, ldb, strideb, nullptr, nbatch,
                                (hipStream_t)stream);
}

int sz_cgbtrs_batched(char trans, int n, int kl, int ku, int nrhs,
                      const void *ab, int ldab, long long strideab,
                      const int *ipiv, long long strideipiv, void *b, int ldb,
                      long long strideb, int nbatch, void *stream)
{
    return launch_gbtrs<float>(trans, n, kl, ku, nrhs, ab, ldab, strideab, ipiv,
                               strideipiv, b, ldb, strideb, nullptr, nbatch,
                               (hipStream_t)stream);
}

// Factor and solve U^T y = b in one pass (see launch_gbtrf_ut); 1 when the
// band shape has no fused kernel.
int sz_internal_zgbtrf_ut(int n, int kl, int ku, void *ab, int ldab,
                          long long strideab, int *ipiv, long long strideipiv,
                          int *info, void *b, long long strideb, int nbatch,
                          void *stream)
{
    return launch_gbtrf_ut<double>(n, kl, ku, ab, ldab, strideab, ipiv, strideipiv,
                                   info, b, strideb, nbatch, (hipStream_t)stream);
}

// The rest of ZGBTRS 'T' after sz_internal_zgbtrf_ut: L^T x = y and the
// interchanges; systems with skip[s] != 0 (a zero pivot) are left alone.
int sz_internal_zgbtrs_lt(int n, int kl, int ku, const void *ab, int ldab,
                          long long strideab, const int *ipiv,
                          long long strideipiv, void *b, long long strideb,
                          const int *skip, int nbatch, void *stream)
{
    return launch_gbtrs<double>('T', n, kl, ku, 1, ab, ldab, strideab, ipiv,
                                strideipiv, b, n, strideb, skip, nbatch,
                                (hipStream_t)stream, true);
}

int sz_internal_gbtrf_masked(int single, int n, int kl, int ku, void *ab,
                             int ldab, long long strideab, int *ipiv,
                             long long strideipiv, int *info, const int *skip,
                             int nbatch, void *stream)
{
    if (single)
        return launch_gbtrf<float>(n, kl, ku, ab, ldab, strideab, ipiv,
                                   strideipiv, info, skip, nbatch,
                                   (hipStream_t)stream);
    return launch_gbtrf<double>(n, kl, ku, ab, ldab, strideab, ipiv, strideipiv,
                                info, skip, nbatch, (hipStream_t)stream);
}

int sz_internal_gbtrs_masked(int single, char trans, int n, int kl, int ku,
                             int nrhs, const void *ab, int ldab,
                             long long strideab, const int *ipiv,
                             long long strideipiv, void *b, int ldb,
                             long long strideb, const int *skip, int nbatch,
                             void *stream)
{
    if (single)
        return launch_gbtrs<float>(trans, n, kl, ku, nrhs, ab, ldab, strideab,
                                   ipiv, strideipiv, b, ldb, strideb, skip,
                                   nbatch, (hipStream_t)stream);
    return launch_gbtrs<double>(trans, n, kl, ku, nrhs, ab, ldab, strideab, ipiv,
                                strideipiv, b, ldb, strideb, skip, nbatch,
                                (hipStream_t)stream);
}

int sz_zgbsv_batched(char trans, int n, int kl, int ku, int nrhs, void *ab,
                     int ldab, long long strideab, int *ipiv,
                     long long strideipiv, void *b, int ldb, long long strideb,
                     int *info, int nbatch, void *stream)
{
    int rc = sz_zgbtrf_batched(n, kl, ku, ab, ldab, strideab, ipiv, strideipiv,
                               info, nbatch, stream);
    if (rc) return rc;
    // Systems whose factorization hit an exact zero pivot keep their right
    // hand side untouched, as ZGBSV skips ZGBTRS when info > 0.
    return launch_gbtrs<double>(trans, n, kl, ku, nrhs, ab, ldab, strideab, ipiv,
                                strideipiv, b, ldb, strideb, info, nbatch,
                                (hipStream_t)stream);
}

}  // extern "C"
