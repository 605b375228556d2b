// Dealiased x/z transforms between the wave-space and physical-space layouts,
// the single-GPU replacement of pencil_grid::transform_wave_to_physical /
// transform_physical_to_wave (suzerain/pencil_grid.hpp:200-221, P3DFFT
// btran_c2r / ftran_r2c with the wall-normal transform disabled).
//
// Layouts (one field):
//   wave      complex, column major (Y, X, Z): element (y, kx, kz) at
//             y + Ny*(kx + Xw*kz), Xw = dNx/2 + 1, kz in [0, dNz)
//   physical  real, (X, Z, Y) with X fastest: (x, z, y) at x + dNx*(z + dNz*y)
// Both directions are unnormalized (FFTW conventions): wave -> physical uses
// exp(+2 pi i k x / N) (c2c along z, then c2r along x, the imaginary parts of
// the kx = 0 and Nyquist inputs ignored); physical -> wave uses
// exp(-2 pi i k x / N) (r2c along x, then c2c along z).  The factor
// chi = 1/(dNx dNz) is the caller's (the time stepper applies it).
//
// Dealiasing: only the modes a length-N transform retains are carried,
// kx in [0, (Nx-1)/2] and |kz| <= (Nz-1)/2 (Nyquist dropped, exactly the
// modes suzerain_diffwave_apply(0, 0, ...) keeps).  wave -> physical treats
// every other input mode as zero (as after zero_dealiasing_modes);
// physical -> wave writes zeros there, fusing the reference's forward
// transform and its zero_dealiasing_modes call (navier_stokes.hpp:953-976).
//
// Each direction is two kernels through an intermediate "mixed" array holding
// (y, kx, z) for the retained kx: element at y + Ny*(kx + xkeep*z).  The real
// x transforms pack two y lines into one complex transform.  Lengths N = N1 N2
// of the usual grids run as two passes of register transforms with one LDS
// exchange between them (k_fft_z2, k_fft_c2r2, k_fft_r2c2); any other 2^a 3^b
// length stages a tile of y lines in LDS and runs Stockham autosort passes of
// radices 4, 2, 3 there.
#include "sz_common.hpp"

#include <cmath>
#include <cstdlib>
#include <new>
#include <utility>
#include <vector>

namespace {

using sz::zd;
constexpr int NT = 256;
constexpr int MAXF = 16;
// LDS per block of the run-time-size kernels: two blocks per CU.  Their tiles
// (two buffers and the twiddles) are halved until they fit: 16 z lines up to
// length 155, 8 up to 301.
constexpr size_t FFT_LDS = 80 * 1024;

struct radix_plan {
    int n, nf;
    int f[MAXF];
};

bool make_plan(int n, radix_plan &p)
{
    p.n = n;
    p.nf = 0;
    int m = n;
    while (m % 4 == 0 && p.nf < MAXF) { p.f[p.nf++] = 4; m /= 4; }
    while (m % 2 == 0 && p.nf < MAXF) { p.f[p.nf++] = 2; m /= 2; }
    while (m % 3 == 0 && p.nf < MAXF) { p.f[p.nf++] = 3; m /= 3; }
    return m == 1;
}

// sign = +1 or -1; w = tw[m] = exp(+2 pi i m / n)
__device__ inline zd twiddle(const zd *tw, int m, int sign)
{
    const zd w = tw[m];
    return zd{w.x, sign > 0 ? w.y : -w.y};
}

__device__ inline void dft_small(int r, int sign, zd *x)
{
    if (r == 2) {
        const zd a = x[0], b = x[1];
        x[0] = sz::cadd(a, b);
        x[1] = sz::csub(a, b);
    } else if (r == 3) {
        const double s3 = 0.86602540378443864676372317075293618;  // sqrt(3)/2
        const zd a = x[0], b = x[1], c = x[2];
        const zd bc = sz::cadd(b, c), bmc = sz::csub(b, c);
        const zd t = {a.x - 0.5 * bc.x, a.y - 0.5 * bc.y};
        // sign * i * s3 * (b - c)
        const zd u = {-sign * s3 * bmc.y, sign * s3 * bmc.x};
        x[0] = sz::cadd(a, bc);
        x[1] = sz::cadd(t, u);
        x[2] = sz::csub(t, u);
    } else {  // r == 4
        const zd a = x[0], b = x[1], c = x[2], d = x[3];
        const zd apc = sz::cadd(a, c), amc = sz::csub(a, c);
        const zd bpd = sz::cadd(b, d), bmd = sz::csub(b, d);
        const zd ib = {-sign * bmd.y, sign * bmd.x};  // sign * i * (b - d)
        x[0] = sz::cadd(apc, bpd);
        x[1] = sz::cadd(amc, ib);
        x[2] = sz::csub(apc, bpd);
        x[3] = sz::csub(amc, ib);
    }
}

// ntr transforms of length n stored t-major (a[t*n + e]) in LDS; ping-pongs
// between a and b and returns the buffer holding the result.
__device__ zd *lds_fft(zd *a, zd *b, const radix_plan &P, int ntr,
                       const zd *tw, int sign)
{
    const int n = P.n;
    int p = 1;
    for (int s = 0; s < P.nf; ++s) {
        const int r = P.f[s];
        const int nr = n / r;
        for (int it = threadIdx.x; it < ntr * nr; it += NT) {
            const int t = it / nr, i = it - t * nr;
            const int k = i % p;
            const zd *in = a + t * n;
            // radix r <= 4 with constant indices (a register array indexed
            // by a runtime count lives in scratch memory)
            zd x[4];
            const int tstep = k * (n / (p * r));
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                x[q] = zd{0, 0};
                if (q < r) {
                    zd v = in[i + q * nr];
                    if (q > 0 && k > 0) v = sz::cmul(v, twiddle(tw, (q * tstep) % n, sign));
                    x[q] = v;
                }
            }
            dft_small(r, sign, x);
            zd *out = b + t * n;
            const int j = (i - k) * r + k;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (q < r) out[j + q * p] = x[q];
        }
        __syncthreads();
        zd *tmp = a; a = b; b = tmp;
        p *= r;
    }
    return a;
}

struct fft_geom {
    int Ny, Nx, dNx, Nz, dNz, Xw, xkeep, zabs, yt, ytx;   // y lines per block: z, x
};

__device__ inline bool z_retained(const fft_geom &g, int kz)
{
    const int w = kz < g.dNz / 2 + 1 ? kz : g.dNz - kz;
    return w <= g.zabs;
}

// ---- c2c along z for the retained kx: wave <-> mixed.
// dir = +1: wave (retained kz) -> mixed (all z); dir = -1: mixed -> wave,
// zeros outside the retained modes (blocks beyond xkeep zero kx >= xkeep).
__global__ __launch_bounds__(NT)
void k_fft_z(fft_geom g, radix_plan P, const zd *__restrict__ twz, int dir,
             const zd *__restrict__ in, long long sin_, zd *__restrict__ out,
             long long sout)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = g.dNz, yt = g.yt;
    zd *tw = reinterpret_cast<zd *>(smem);
    zd *a = tw + n;
    zd *b = a + yt * n;
    const int ntile = (g.Ny + yt - 1) / yt;
    const int kx = blockIdx.x / ntile;
    const int y0 = (blockIdx.x - kx * ntile) * yt;
    const int f = blockIdx.y;
    in += (size_t)f * sin_;
    out += (size_t)f * sout;
    const int ny = min(yt, g.Ny - y0);
    if (kx >= g.xkeep) {
        // forward only: zero the dealiased kx columns of the wave output
        for (int e = threadIdx.x; e < ny * n; e += NT) {
            const int z = e / ny, yy = e - z * ny;
            out[(size_t)(y0 + yy) + (size_t)g.Ny * (kx + (size_t)g.Xw * z)] = zd{0, 0};
        }
        return;
    }
    for (int e = threadIdx.x; e < n; e += NT) tw[e] = twz[e];
    // load: a[t*n + z] for t = y line
    // component-wise: a struct assigned on several paths goes through
    // scratch memory, and each scratch access waits for every load in flight
    const size_t zs = (size_t)g.Ny * (dir > 0 ? g.Xw : g.xkeep);
    for (int e = threadIdx.x; e < yt * n; e += NT) {
        const int z = e / yt, yy = e - z * yt;
        const bool ok = yy < ny && (dir <= 0 || z_retained(g, z));
        double vx = 0, vy = 0;
        if (ok) {
            const zd *src = in + (size_t)(y0 + yy) + (size_t)g.Ny * kx + zs * z;
            vx = src->x;
            vy = src->y;
        }
        a[yy * n + z] = zd{vx, vy};
    }
    __syncthreads();
    zd *res = lds_fft(a, b, P, yt, tw, dir);
    for (int e = threadIdx.x; e < yt * n; e += NT) {
        const int z = e / yt, yy = e - z * yt;
        if (yy >= ny) continue;
        const zd v = res[yy * n + z];
        const bool keep = dir > 0 || z_retained(g, z);
        const size_t os = (size_t)g.Ny * (dir > 0 ? g.xkeep : g.Xw);
        out[(size_t)(y0 + yy) + (size_t)g.Ny * kx + os * z] =
            zd{keep ? v.x : 0.0, keep ? v.y : 0.0};
    }
}

// ---- c2r along x: mixed (retained kx) -> physical, two y lines per
// complex transform: Z_k = X1_k + i X2_k with Hermitian extension.
__global__ __launch_bounds__(NT)
void k_fft_x_c2r(fft_geom g, radix_plan P, const zd *__restrict__ twx,
                 const zd *__restrict__ mixed, long long smix,
                 double *__restrict__ phys, long long sphys)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = g.dNx, yt = g.ytx, np = yt / 2;
    zd *tw = reinterpret_cast<zd *>(smem);
    zd *a = tw + n;
    zd *b = a + np * n;
    zd *spec = b + np * n;                  // [kx][yy], xkeep x yt
    const int ntile = (g.Ny + yt - 1) / yt;
    const int z = blockIdx.x / ntile;
    const int y0 = (blockIdx.x - z * ntile) * yt;
    const int f = blockIdx.y;
    mixed += (size_t)f * smix;
    phys += (size_t)f * sphys;
    const int ny = min(yt, g.Ny - y0);
    for (int e = threadIdx.x; e < n; e += NT) tw[e] = twx[e];
    for (int e = threadIdx.x; e < g.xkeep * yt; e += NT) {
        const int kx = e / yt, yy = e - kx * yt;
        spec[e] = yy < ny ? mixed[(size_t)(y0 + yy) +
                                  (size_t)g.Ny * (kx + (size_t)g.xkeep * z)]
                          : zd{0, 0};
    }
    __syncthreads();
    for (int e = threadIdx.x; e < np * n; e += NT) {
        const int t = e / n, k = e - t * n;
        // X_k for k <= n/2 (retained), conj(X_{n-k}) above; imaginary parts
        // of X_0 and X_{n/2} ignored
        const int kk = k <= n / 2 ? k : n - k;
        zd x1 = {0, 0}, x2 = {0, 0};
        if (kk < g.xkeep) {
            x1 = spec[kk * yt + 2 * t];
            x2 = spec[kk * yt + 2 * t + 1];
            if (k > n / 2) { x1.y = -x1.y; x2.y = -x2.y; }
            if (k == 0 || 2 * k == n) { x1.y = 0; x2.y = 0; }
        }
        a[t * n + k] = zd{x1.x - x2.y, x1.y + x2.x};   // x1 + i x2
    }
    __syncthreads();
    zd *res = lds_fft(a, b, P, np, tw, +1);
    for (int e = threadIdx.x; e < yt * n; e += NT) {
        const int yy = e / n, x = e - yy * n;
        if (yy >= ny) continue;
        const zd v = res[(yy >> 1) * n + x];
        phys[(size_t)x + (size_t)n * (z + (size_t)g.dNz * (y0 + yy))] =
            (yy & 1) ? v.y : v.x;
    }
}

// ---- r2c along x: physical -> mixed (retained kx), two y lines per
// complex transform: X1_k = (Z_k + conj Z_{n-k})/2, X2_k = (Z_k - conj
// Z_{n-k})/(2i).
__global__ __launch_bounds__(NT)
void k_fft_x_r2c(fft_geom g, radix_plan P, const zd *__restrict__ twx,
                 const double *__restrict__ phys, long long sphys,
                 zd *__restrict__ mixed, long long smix)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = g.dNx, yt = g.ytx, np = yt / 2;
    zd *tw = reinterpret_cast<zd *>(smem);
    zd *a = tw + n;
    zd *b = a + np * n;
    const int ntile = (g.Ny + yt - 1) / yt;
    const int z = blockIdx.x / ntile;
    const int y0 = (blockIdx.x - z * ntile) * yt;
    const int f = blockIdx.y;
    phys += (size_t)f * sphys;
    mixed += (size_t)f * smix;
    const int ny = min(yt, g.Ny - y0);
    for (int e = threadIdx.x; e < n; e += NT) tw[e] = twx[e];
    for (int e = threadIdx.x; e < np * n; e += NT) {
        const int t = e / n, x = e - t * n;
        const int ya = 2 * t, yb = 2 * t + 1;
        const double p1 = ya < ny ? phys[(size_t)x + (size_t)n * (z + (size_t)g.dNz * (y0 + ya))] : 0.0;
        const double p2 = yb < ny ? phys[(size_t)x + (size_t)n * (z + (size_t)g.dNz * (y0 + yb))] : 0.0;
        a[t * n + x] = zd{p1, p2};
    }
    __syncthreads();
    zd *res = lds_fft(a, b, P, np, tw, -1);
    for (int e = threadIdx.x; e < g.xkeep * yt; e += NT) {
        const int kx = e / yt, yy = e - kx * yt;
        if (yy >= ny) continue;
        const int t = yy >> 1;
        const zd zk = res[t * n + kx];
        const zd zm = res[t * n + (kx == 0 ? 0 : n - kx)];
        zd v;
        if ((yy & 1) == 0) v = zd{0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y)};
        else               v = zd{0.5 * (zk.y + zm.y), 0.5 * (zm.x - zk.x)};
        mixed[(size_t)(y0 + yy) + (size_t)g.Ny * (kx + (size_t)g.xkeep * z)] = v;
    }
}

// ------------------------------------------------- two register passes
// N = N1 N2, n = n2 + N2 n1, k = k1 + N1 k2:
//   X_k = sum_n2 w_N2^(n2 k2) [ w_N^(n2 k1) sum_n1 x_n w_N1^(n1 k1) ].
// Pass 1: one thread makes the N1-point sum of one (line, n2) in registers,
// its N1 loads straight from global memory and in flight together; the
// twiddled sums cross through LDS once; pass 2: one thread makes the N2-point
// sum of one (line, k1) and stores its N2 results.  HBM bound: an element
// touches LDS twice and its block waits at one barrier.  As radix-4/2/3 passes
// in LDS (twelve accesses and eleven barriers at length 288) the 46 backward
// transforms of a 192^3 substep took 2.7 ms in z and 3.5 ms in x, 2.4 and 2.8
// TB/s; now 1.5 and 2.3 ms, both 4.3 TB/s (a large copy: 4.7).  Length 108,
// which had only the run-time-size kernels, 38-44 us for 5 fields of 97 x 108
// x 96 in x, now 15-18.

// cos(2 pi j / 144) for j = 0 .. 36
constexpr double COS144[37] = {
    1.0, 0.99904822158185776240, 0.99619469809174553229, 0.99144486137381041114,
    0.98480775301220805936, 0.97629600711993336597, 0.96592582628906828674, 0.95371695074822692114,
    0.93969262078590838405, 0.92387953251128675612, 0.90630778703664996324, 0.88701083317822170105,
    0.86602540378443864676, 0.84339144581288570127, 0.81915204428899178968, 0.79335334029123516457,
    0.76604444311897803520, 0.73727733681012404138, 0.70710678118654752440, 0.67559020761566024434,
    0.64278760968653932632, 0.60876142900872063941, 0.57357643635104609610, 0.53729960834682383184,
    0.5, 0.46174861323503393056, 0.42261826174069943618, 0.38268343236508977172,
    0.34202014332566873304, 0.30070579950427312162, 0.25881904510252076234, 0.21643961393810287975,
    0.17364817766693034885, 0.13052619222005159154, 0.08715574274765817355, 0.04361938736533599978,
    0.0};

// cos(2 pi j / n), n a divisor of 144
constexpr double cos_of(int j, int n)
{
    j = j * (144 / n) % 144;
    if (j > 72) j = 144 - j;
    return j <= 36 ? COS144[j] : -COS144[72 - j];
}
constexpr double sin_of(int j, int n) { return cos_of(j * (144 / n) + 108, 144); }

template <int... I, typename F>
__device__ __forceinline__ void sfor_impl(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}

template <int K, typename F>
__device__ __forceinline__ void sfor(F &&f)
{
    sfor_impl(f, std::make_integer_sequence<int, K>{});
}

constexpr int first_factor(int r) { return r % 4 == 0 ? 4 : r % 2 == 0 ? 2 : 3; }

// where X_k of an R-point transform ends up in its array
constexpr int dft_at(int r, int k)
{
    if (r <= 4) return k;
    const int a = first_factor(r), b = r / a;
    return b * (k % a) + dft_at(b, k / a);
}

// X_k = sum_n x_n exp(S 2 pi i n k / R) of the R elements from O on, in place:
// n in natural order, X_k left at O + dft_at(R, k).  Component arrays, every
// index a constant, no copies (local copies of parts of the arrays left dead
// stores to scratch behind).
template <int R, int S, int O = 0, int L>
__device__ __forceinline__ void dft(double (&x)[L], double (&y)[L])
{
    constexpr int A = first_factor(R), B = R / A;
    sfor<B>([&](auto n_) __attribute__((always_inline)) {
        constexpr int n = decltype(n_)::value, i0 = O + n, i1 = i0 + B;
        if constexpr (A == 2) {
            const double ax = x[i0], ay = y[i0];
            x[i0] = ax + x[i1];
            y[i0] = ay + y[i1];
            x[i1] = ax - x[i1];
            y[i1] = ay - y[i1];
        } else if constexpr (A == 3) {
            constexpr int i2 = i1 + B;
            constexpr double s3 = 0.86602540378443864676;
            const double bx = x[i1] + x[i2], by = y[i1] + y[i2];
            const double dx = x[i1] - x[i2], dy = y[i1] - y[i2];
            const double tx = fma(-0.5, bx, x[i0]), ty = fma(-0.5, by, y[i0]);
            x[i0] += bx;
            y[i0] += by;
            x[i1] = fma(-S * s3, dy, tx);
            y[i1] = fma(S * s3, dx, ty);
            x[i2] = fma(S * s3, dy, tx);
            y[i2] = fma(-S * s3, dx, ty);
        } else {
            constexpr int i2 = i1 + B, i3 = i2 + B;
            const double px = x[i0] + x[i2], py = y[i0] + y[i2];
            const double mx = x[i0] - x[i2], my = y[i0] - y[i2];
            const double qx = x[i1] + x[i3], qy = y[i1] + y[i3];
            const double nx = x[i1] - x[i3], ny = y[i1] - y[i3];
            x[i0] = px + qx;
            y[i0] = py + qy;
            x[i1] = mx - S * ny;
            y[i1] = my + S * nx;
            x[i2] = px - qx;
            y[i2] = py - qy;
            x[i3] = mx + S * ny;
            y[i3] = my - S * nx;
        }
        if constexpr (n > 0) {
            sfor<A - 1>([&](auto k_) __attribute__((always_inline)) {
                constexpr int k = 1 + decltype(k_)::value, i = i0 + B * k;
                constexpr double c = cos_of(n * k, R), s = S * sin_of(n * k, R);
                const double ax = x[i], ay = y[i];
                x[i] = fma(c, ax, -(s * ay));
                y[i] = fma(c, ay, s * ax);
            });
        }
    });
    if constexpr (B > 1)
        sfor<A>([&](auto k_) __attribute__((always_inline)) {
            dft<B, S, O + B * decltype(k_)::value>(x, y);
        });
}

// Lines (pairs of lines in x) a block transforms: runs of at least 128 bytes
// and at most 40 KB of LDS up to length 288, so that four blocks fit a CU; 384
// takes 48 to 51 KB, three blocks.
constexpr int fft_lines(int n) { return n >= 160 ? 8 : n >= 48 ? 16 : 32; }
constexpr int fft_threads(int n1, int n2)
{
    return fft_lines(n1 * n2) * (n1 > n2 ? n1 : n2);
}

// multiply by w^m, w = exp(S 2 pi i / N), from the plan's table
template <int S>
__device__ __forceinline__ void twiddled(double &x, double &y, const zd *tw, int m)
{
    const double c = tw[m].x, s = S * tw[m].y;
    const double a = x, b = y;
    x = fma(c, a, -(s * b));
    y = fma(c, b, s * a);
}

// c2c along z, wave <-> mixed.  For one z the retained (y, kx) of either array
// are one run of P = Ny xkeep elements, so a line is an element of that run
// and tiles need no rounding to Ny.  S = +1: wave (retained kz) -> mixed (all
// z); S = -1: mixed -> wave, zeros outside the retained modes (the tiles past
// P zero kx >= xkeep).
template <int N1, int N2, int S>
__global__ __launch_bounds__(fft_threads(N1, N2))
void k_fft_z2(fft_geom g, const zd *__restrict__ tw, const zd *__restrict__ in,
              long long sin_, zd *__restrict__ out, long long sout)
{
    constexpr int N = N1 * N2, W = fft_lines(N);
    __shared__ zd ex[N * W];                 // [k1][n2][line]
    const int l = threadIdx.x % W, c = threadIdx.x / W;
    const long long P = (long long)g.Ny * g.xkeep, Q = (long long)g.Ny * g.Xw;
    const long long p = (long long)blockIdx.x * W + l;
    in += (size_t)blockIdx.y * sin_;
    out += (size_t)blockIdx.y * sout;
    if ((long long)blockIdx.x * W >= P) {    // S = -1: only kx >= xkeep
        for (int z = c; z < N; z += fft_threads(N1, N2) / W)
            if (p < Q) out[p + Q * z] = zd{0, 0};
        return;
    }
    const bool line = p < P;
    const long long zi = S > 0 ? Q : P, zo = S > 0 ? P : Q;
    if (c < N2) {
        const zd *src = in + (line ? p : 0);
        double x[N1], y[N1];
        sfor<N1>([&](auto n_) __attribute__((always_inline)) {
            // dealiased modes are not read: their lanes repeat mode 0
            const int n = c + N2 * decltype(n_)::value;
            const bool ok = S < 0 || z_retained(g, n);
            const zd *v = src + zi * (ok ? n : 0);
            const double vx = v->x, vy = v->y;
            x[decltype(n_)::value] = ok ? vx : 0.0;
            y[decltype(n_)::value] = ok ? vy : 0.0;
        });
        dft<N1, S>(x, y);
        sfor<N1>([&](auto k_) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value, i = dft_at(N1, k);
            if constexpr (k > 0) twiddled<S>(x[i], y[i], tw, c * k);
            ex[(k * N2 + c) * W + l] = zd{x[i], y[i]};
        });
    }
    __syncthreads();
    if (c < N1) {
        double x[N2], y[N2];
        sfor<N2>([&](auto n_) __attribute__((always_inline)) {
            constexpr int n = decltype(n_)::value;
            x[n] = ex[(c * N2 + n) * W + l].x;
            y[n] = ex[(c * N2 + n) * W + l].y;
        });
        dft<N2, S>(x, y);
        if (line) {
            sfor<N2>([&](auto k_) __attribute__((always_inline)) {
                constexpr int i = dft_at(N2, decltype(k_)::value);
                const int k = c + N1 * decltype(k_)::value;
                const bool keep = S > 0 || z_retained(g, k);
                const double vx = x[i], vy = y[i];
                out[p + zo * k] = zd{keep ? vx : 0.0, keep ? vy : 0.0};
            });
        }
    }
    // a tile across P also zeroes its share of kx >= xkeep
    if (S < 0 && !line && p < Q)
        for (int z = c; z < N; z += fft_threads(N1, N2) / W) out[p + Q * z] = zd{0, 0};
}

// Line pair q of all (z, y pairs): z and the even y of the pair.
struct line_pair {
    int z, y;
    bool odd;                                // the pair's second line exists
};
__device__ __forceinline__ line_pair pair_of(const fft_geom &g, int q)
{
    const int np = (g.Ny + 1) / 2, z = q / np, y = 2 * (q - z * np);
    return line_pair{z, y, y + 1 < g.Ny};
}

// c2r along x: mixed (retained kx) -> physical, the y lines 2h and 2h+1 of one
// z as one complex transform Z_k = X1_k + i X2_k with Hermitian extension; a
// spectral pair (32 bytes) is read by the threads of k and of N - k.
template <int N1, int N2>
__global__ __launch_bounds__(fft_threads(N1, N2))
void k_fft_c2r2(fft_geom g, const zd *__restrict__ tw, const zd *__restrict__ mixed,
                long long smix, double *__restrict__ phys, long long sphys)
{
    constexpr int N = N1 * N2, W = fft_lines(N), ST = N1 + 1;
    __shared__ zd ex[N2 * ST * W];           // [pair][n2][k1], rows padded by one
    mixed += (size_t)blockIdx.y * smix;
    phys += (size_t)blockIdx.y * sphys;
    const int npair = g.dNz * ((g.Ny + 1) / 2), q0 = blockIdx.x * W;
    if (const int h = threadIdx.x % W, c = threadIdx.x / W; c < N2) {
        const line_pair L = pair_of(g, min(q0 + h, npair - 1));
        const zd *src = mixed + (size_t)L.y + (size_t)g.Ny * ((size_t)g.xkeep * L.z);
        const int second = L.odd ? 1 : 0;
        double x[N1], y[N1];
        sfor<N1>([&](auto n_) __attribute__((always_inline)) {
            constexpr int i = decltype(n_)::value;
            const int k = c + N2 * i, kk = k <= N / 2 ? k : N - k;
            const bool ok = kk < g.xkeep;    // others repeat mode 0 and count as zero
            const zd *m = src + (size_t)g.Ny * (ok ? kk : 0);
            const double ax = m[0].x, ay = m[0].y, bx = m[second].x, by = m[second].y;
            // conj above N/2; the imaginary parts of k = 0 and N/2 ignored
            const bool real = k == 0 || 2 * k == N, conj = k > N / 2;
            const double a1 = real ? 0.0 : conj ? -ay : ay;
            const double b0 = L.odd ? bx : 0.0;
            const double b1 = real || !L.odd ? 0.0 : conj ? -by : by;
            x[i] = ok ? ax - b1 : 0.0;
            y[i] = ok ? a1 + b0 : 0.0;
        });
        dft<N1, +1>(x, y);
        sfor<N1>([&](auto k_) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value, i = dft_at(N1, k);
            if constexpr (k > 0) twiddled<+1>(x[i], y[i], tw, c * k);
            ex[(h * N2 + c) * ST + k] = zd{x[i], y[i]};
        });
    }
    __syncthreads();
    const int c = threadIdx.x % N1, h = threadIdx.x / N1;
    if (h < W && q0 + h < npair) {
        double x[N2], y[N2];
        sfor<N2>([&](auto n_) __attribute__((always_inline)) {
            constexpr int n = decltype(n_)::value;
            x[n] = ex[(h * N2 + n) * ST + c].x;
            y[n] = ex[(h * N2 + n) * ST + c].y;
        });
        dft<N2, +1>(x, y);
        const line_pair L = pair_of(g, q0 + h);
        double *dst = phys + (size_t)N * (L.z + (size_t)g.dNz * L.y) + c;
        double *dst2 = dst + (size_t)N * g.dNz;
        sfor<N2>([&](auto k_) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value, i = dft_at(N2, k);
            dst[N1 * k] = x[i];
            if (L.odd) dst2[N1 * k] = y[i];
        });
    }
}

// r2c along x: physical -> mixed (retained kx), two y lines per complex
// transform: X1_k = (Z_k + conj Z_{N-k})/2, X2_k = (Z_k - conj Z_{N-k})/(2i).
template <int N1, int N2>
__global__ __launch_bounds__(fft_threads(N1, N2))
void k_fft_r2c2(fft_geom g, const zd *__restrict__ tw, const double *__restrict__ phys,
                long long sphys, zd *__restrict__ mixed, long long smix)
{
    constexpr int N = N1 * N2, W = fft_lines(N), ST = N2 + 1, BT = fft_threads(N1, N2);
    constexpr int EX = N1 * ST > N ? N1 * ST : N;
    __shared__ zd ex[EX * W];                // [pair][k1][n2], then [k][pair]
    phys += (size_t)blockIdx.y * sphys;
    mixed += (size_t)blockIdx.y * smix;
    const int npair = g.dNz * ((g.Ny + 1) / 2), q0 = blockIdx.x * W;
    if (const int c = threadIdx.x % N2, h = threadIdx.x / N2; h < W) {
        const line_pair L = pair_of(g, min(q0 + h, npair - 1));
        const double *src = phys + (size_t)N * (L.z + (size_t)g.dNz * L.y) + c;
        const double *src2 = src + (L.odd ? (size_t)N * g.dNz : 0);
        double x[N1], y[N1];
        sfor<N1>([&](auto n_) __attribute__((always_inline)) {
            constexpr int i = decltype(n_)::value;
            x[i] = src[N2 * i];
            y[i] = src2[N2 * i];
            y[i] = L.odd ? y[i] : 0.0;
        });
        dft<N1, -1>(x, y);
        sfor<N1>([&](auto k_) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value, i = dft_at(N1, k);
            if constexpr (k > 0) twiddled<-1>(x[i], y[i], tw, c * k);
            ex[(h * N1 + k) * ST + c] = zd{x[i], y[i]};
        });
    }
    __syncthreads();
    const int h = threadIdx.x % W, c = threadIdx.x / W;
    double x[N2], y[N2];
    if (c < N1) {
        sfor<N2>([&](auto n_) __attribute__((always_inline)) {
            constexpr int n = decltype(n_)::value;
            x[n] = ex[(h * N1 + c) * ST + n].x;
            y[n] = ex[(h * N1 + c) * ST + n].y;
        });
        dft<N2, -1>(x, y);
    }
    __syncthreads();
    if (c < N1) {
        sfor<N2>([&](auto k_) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value, i = dft_at(N2, k);
            ex[(c + N1 * k) * W + h] = zd{x[i], y[i]};
        });
    }
    __syncthreads();
    if (q0 + h >= npair) return;
    const line_pair L = pair_of(g, q0 + h);
    zd *dst = mixed + (size_t)L.y + (size_t)g.Ny * ((size_t)g.xkeep * L.z);
    for (int k = c; k < g.xkeep; k += BT / W) {
        const zd a = ex[k * W + h], b = ex[(k == 0 ? 0 : N - k) * W + h];
        dst[(size_t)g.Ny * k] = zd{0.5 * (a.x + b.x), 0.5 * (a.y - b.y)};
        if (L.odd) dst[(size_t)g.Ny * k + 1] = zd{0.5 * (a.y + b.y), 0.5 * (b.x - a.x)};
    }
}

// The lengths run as two register passes and their factors: the 3/2 rule's
// lengths of grids of 8, 12, 16, 24, 32, 36, 48, 64, 72, 96, 108, 128, 144, 192
// and 256 points, those of this repository's channels, ensembles and tests.  A
// choice of what to instantiate, not what the method can take: any length of two
// factors up to 24 could be added (32 = 8 4, 64 = 8 8, 128 = 16 8, 256 = 16 16,
// 324 = 18 18, 432 = 24 18, 576 = 24 24).  Measured over both passes, 5 fields of
// 4 million points, backward and forward: these from 24 up at 4.0 to 5.8 and 3.8
// to 6.2 TB/s, but 162 at 2.7 and 3.4 and 384 at 3.5 and 3.6; the run-time-size
// kernels at 1.6 to 2.2 and 1.9 to 2.7 (32 to 256) and 0.9 to 1.4 and 1.1 to 1.6
// TB/s (324 to 768), the rate they had before.
#define SZ_FFT_TWO_PASS(X)                                                      \
    X(12, 4, 3) X(18, 6, 3) X(24, 6, 4) X(36, 6, 6) X(48, 8, 6) X(54, 9, 6)      \
    X(72, 9, 8) X(96, 12, 8) X(108, 12, 9) X(144, 16, 9) X(162, 18, 9)           \
    X(192, 16, 12) X(216, 18, 12) X(288, 16, 18) X(384, 24, 16)

// Calls f(N1, N2) as constants when n is one of those lengths; else false.
template <typename F>
bool two_pass(int n, F &&f)
{
#define SZ_FFT_CALL(NV, AV, BV)                                                 \
    if (n == NV) {                                                             \
        static_assert(AV * BV == NV, "factors");                               \
        f(std::integral_constant<int, AV>{}, std::integral_constant<int, BV>{}); \
        return true;                                                           \
    }
    SZ_FFT_TWO_PASS(SZ_FFT_CALL)
#undef SZ_FFT_CALL
    return false;
}

}  // namespace

struct sz_fft_plan {
    fft_geom g;
    radix_plan px, pz;
    zd *twx = nullptr, *twz = nullptr;
    int dev = -1;
};

namespace {

std::vector<zd> twiddles(int n)
{
    std::vector<zd> t((size_t)n);
    for (int m = 0; m < n; ++m) {
        const long double a = 2.0L * 3.14159265358979323846264338327950288L * m / n;
        t[(size_t)m] = zd{(double)cosl(a), (double)sinl(a)};
    }
    return t;
}

size_t lds_z_for(int dNz, int yt)
{
    return ((size_t)dNz + 2 * (size_t)yt * dNz) * sizeof(zd);
}

size_t lds_x_for(int dNx, int xkeep, int yt)
{
    return ((size_t)dNx + 2 * (size_t)(yt / 2) * dNx + (size_t)xkeep * yt) * sizeof(zd);
}

size_t lds_z(const sz_fft_plan *p) { return lds_z_for(p->g.dNz, p->g.yt); }

size_t lds_x(const sz_fft_plan *p) { return lds_x_for(p->g.dNx, p->g.xkeep, p->g.ytx); }

}  // namespace

extern "C" {

sz_fft_plan *sz_fft_plan_create(int Ny, int Nx, int dNx, int Nz, int dNz,
                                int *info)
{
    int dummy;
    if (!info) info = &dummy;
    *info = 0;
    if (Ny < 1) { *info = -1; return nullptr; }
    if (Nx < 1 || dNx < Nx || dNx % 2) { *info = -3; return nullptr; }
    if (Nz < 1 || dNz < Nz) { *info = -5; return nullptr; }
    sz_fft_plan *p = new (std::nothrow) sz_fft_plan();
    if (!p) { *info = SZ_ERR_ALLOC; return nullptr; }
    if (!make_plan(dNx, p->px) || !make_plan(dNz, p->pz)) {
        delete p;
        *info = -99;   // lengths must be 2^a 3^b
        return nullptr;
    }
    fft_geom &g = p->g;
    g.Ny = Ny; g.Nx = Nx; g.dNx = dNx; g.Nz = Nz; g.dNz = dNz;
    g.Xw = dNx / 2 + 1;
    g.xkeep = (Nx - 1) / 2 + 1;
    g.zabs = (Nz - 1) / 2;
    // tiles of the run-time-size kernels (the two-pass ones have their own).
    // z: 16 lines per block (256-byte runs of y), or 8 with SZ_FFT_ZLINES=8; x: 8
    int yt = 16;
    if (const char *e = std::getenv("SZ_FFT_ZLINES"))
        if (std::atoi(e) == 8) yt = 8;
    while (yt > 2 && lds_z_for(dNz, yt) > FFT_LDS) yt /= 2;
    int ytx = 8;
    while (ytx > 2 && lds_x_for(dNx, g.xkeep, ytx) > FFT_LDS) ytx /= 2;
    g.yt = yt;
    g.ytx = ytx;
    if (lds_z(p) > 160 * 1024 || lds_x(p) > 160 * 1024) {
        delete p;
        *info = SZ_ERR_LDS;
        return nullptr;
    }
    const auto tx = twiddles(dNx), tz = twiddles(dNz);
    if (hipMalloc(&p->twx, tx.size() * sizeof(zd)) != hipSuccess ||
        hipMalloc(&p->twz, tz.size() * sizeof(zd)) != hipSuccess) {
        if (p->twx) (void)hipFree(p->twx);
        delete p;
        *info = SZ_ERR_ALLOC;
        return nullptr;
    }
    (void)hipMemcpy(p->twx, tx.data(), tx.size() * sizeof(zd), hipMemcpyHostToDevice);
    (void)hipMemcpy(p->twz, tz.data(), tz.size() * sizeof(zd), hipMemcpyHostToDevice);
    (void)hipGetDevice(&p->dev);
    return p;
}

void sz_fft_plan_free(sz_fft_plan *p)
{
    if (!p) return;
    if (p->twx) (void)hipFree(p->twx);
    if (p->twz) (void)hipFree(p->twz);
    delete p;
}

/* Complex elements of the intermediate (mixed) array per field. */
long long sz_fft_mixed_elements(const sz_fft_plan *p)
{
    return (long long)p->g.Ny * p->g.xkeep * p->g.dNz;
}

int sz_fft_wave_to_physical(const sz_fft_plan *p, int nfields,
                            const void *wave, long long swave, void *mixed,
                            long long smixed, double *phys, long long sphys,
                            void *stream)
{
    if (!p) return -1;
    if (nfields < 0) return -2;
    if (nfields == 0) return 0;
    const fft_geom &g = p->g;
    const int ntile = (g.Ny + g.yt - 1) / g.yt, ntx = (g.Ny + g.ytx - 1) / g.ytx;
    hipStream_t st = (hipStream_t)stream;
    const zd *w = reinterpret_cast<const zd *>(wave);
    zd *m = reinterpret_cast<zd *>(mixed);
    if (!two_pass(g.dNz, [&](auto a, auto b) {
            constexpr int A = decltype(a)::value, B = decltype(b)::value, L = fft_lines(A * B);
            const long long tiles = ((long long)g.Ny * g.xkeep + L - 1) / L;
            hipLaunchKernelGGL((k_fft_z2<A, B, +1>), dim3((unsigned)tiles, nfields),
                               dim3(fft_threads(A, B)), 0, st, g, p->twz, w, swave, m, smixed);
        }))
        hipLaunchKernelGGL(k_fft_z, dim3(g.xkeep * ntile, nfields), dim3(NT), lds_z(p), st,
                           g, p->pz, p->twz, +1, w, swave, m, smixed);
    if (!two_pass(g.dNx, [&](auto a, auto b) {
            constexpr int A = decltype(a)::value, B = decltype(b)::value, L = fft_lines(A * B);
            const long long tiles = ((long long)g.dNz * ((g.Ny + 1) / 2) + L - 1) / L;
            hipLaunchKernelGGL((k_fft_c2r2<A, B>), dim3((unsigned)tiles, nfields),
                               dim3(fft_threads(A, B)), 0, st, g, p->twx, m, smixed, phys,
                               sphys);
        }))
        hipLaunchKernelGGL(k_fft_x_c2r, dim3(g.dNz * ntx, nfields), dim3(NT), lds_x(p), st,
                           g, p->px, p->twx, m, smixed, phys, sphys);
    return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
}

int sz_fft_physical_to_wave(const sz_fft_plan *p, int nfields,
                            const double *phys, long long sphys, void *mixed,
                            long long smixed, void *wave, long long swave,
                            void *stream)
{
    if (!p) return -1;
    if (nfields < 0) return -2;
    if (nfields == 0) return 0;
    const fft_geom &g = p->g;
    const int ntile = (g.Ny + g.yt - 1) / g.yt, ntx = (g.Ny + g.ytx - 1) / g.ytx;
    hipStream_t st = (hipStream_t)stream;
    zd *w = reinterpret_cast<zd *>(wave), *m = reinterpret_cast<zd *>(mixed);
    if (!two_pass(g.dNx, [&](auto a, auto b) {
            constexpr int A = decltype(a)::value, B = decltype(b)::value, L = fft_lines(A * B);
            const long long tiles = ((long long)g.dNz * ((g.Ny + 1) / 2) + L - 1) / L;
            hipLaunchKernelGGL((k_fft_r2c2<A, B>), dim3((unsigned)tiles, nfields),
                               dim3(fft_threads(A, B)), 0, st, g, p->twx, phys, sphys, m,
                               smixed);
        }))
        hipLaunchKernelGGL(k_fft_x_r2c, dim3(g.dNz * ntx, nfields), dim3(NT), lds_x(p), st,
                           g, p->px, p->twx, phys, sphys, m, smixed);
    if (!two_pass(g.dNz, [&](auto a, auto b) {
            constexpr int A = decltype(a)::value, B = decltype(b)::value, L = fft_lines(A * B);
            const long long tiles = ((long long)g.Ny * g.Xw + L - 1) / L;
            hipLaunchKernelGGL((k_fft_z2<A, B, -1>), dim3((unsigned)tiles, nfields),
                               dim3(fft_threads(A, B)), 0, st, g, p->twz, m, smixed, w, swave);
        }))
        hipLaunchKernelGGL(k_fft_z, dim3(g.Xw * ntile, nfields), dim3(NT), lds_z(p), st,
                           g, p->pz, p->twz, -1, m, smixed, w, swave);
    return hipGetLastError() == hipSuccess ? 0 : SZ_ERR_LAUNCH;
}

}  // extern "C"
