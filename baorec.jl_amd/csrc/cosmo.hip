// Sky <-> Cartesian conversion on the GPU: the comoving-distance table of
// BAOrec.Cosmology (src/cosmo.jl:64-98) built by FP64 Gauss-Legendre
// quadrature per table interval plus an ordered prefix sum, and the per-galaxy
// conversions of the reference's lightcone driver (examples/lightcone.jl:30-80).
#include <math.h>

#include "kernels.hpp"

namespace baorec {

// 1 / H(z) in s Mpc / km, src/cosmo.jl:74-85: E(z) sums the densities in the
// reference's order; every term is FP64 (the Float32 parameters promote).
__device__ __forceinline__ double inv_hubble(const CosmoArgs &c, double z) {
    const double zp = 1.0 + z;
    const double z2 = zp * zp, z3 = z2 * zp, z4 = z2 * z2;
    const double a = 1.0 / zp;
    // f_DE(a) (src/cosmo.jl:80); at a = 1 the wa term is 0 * NaN, but
    // (1 + z)^f with z = 0 is 1 for any f, which pow() also returns
    const double fde = -3.0 * (1.0 + c.w0) + 3.0 * c.wa * ((a - 1.0) / log(a) - 1.0);
    const double ol = c.omega_l0 * pow(zp, -fde);
    const double e = sqrt(c.omega_nu0 * z4 + c.omega_g0 * z4 + c.omega_b0 * z3 + c.omega_c0 * z3 +
                          c.omega_k0 * z2 + ol);
    return 1.0 / (c.h100 * e);
}

// 4-point Gauss-Legendre rule on [a, b] of c / H (Mpc).
__device__ __forceinline__ double gl4(const CosmoArgs &c, double a, double b) {
    const double x1 = 0.33998104358485626, x2 = 0.86113631159405258;
    const double w1 = 0.65214515486254614, w2 = 0.34785484513745386;
    const double m = 0.5 * (a + b), h = 0.5 * (b - a);
    const double s = w2 * (inv_hubble(c, m - h * x2) + inv_hubble(c, m + h * x2)) +
                     w1 * (inv_hubble(c, m - h * x1) + inv_hubble(c, m + h * x1));
    return kSpeedOfLightKms * h * s;
}

// The knots (z, r) of the table stand side by side: a conversion's two knots
// are 32 bytes, one line of memory most of the time.

// kn[i].x = z[i]
__global__ void k_cosmo_knots(const double *__restrict__ z, double2 *__restrict__ kn, int num) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < num) kn[i].x = z[i];
}

// seg[i] = integral over [z of knot i, z of knot i + 1], i < num - 1
__global__ void k_cosmo_seg(CosmoArgs c, const double2 *__restrict__ kn, double *__restrict__ seg, int num) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num - 1) return;
    seg[i] = gl4(c, kn[i].x, kn[i + 1].x);
}

// kn[k].y = r0 + sum_{i<k} seg[i], with r0 the integral over [0, kn[0].x]; one
// workgroup, fixed summation order (deterministic).
constexpr int kScanThreads = 1024;
__global__ void __launch_bounds__(kScanThreads) k_cosmo_scan(CosmoArgs c, double2 *__restrict__ kn,
                                                            const double *__restrict__ seg, int num) {
    __shared__ double part[kScanThreads];
    const int t = threadIdx.x;
    // r0: [0, zk[0]] in kScanThreads * 4 sub-intervals, tree-reduced
    double s0 = 0.0;
    if (kn[0].x > 0.0) {
        const double h = kn[0].x / (kScanThreads * 4);
        for (int j = 0; j < 4; j++) {
            const double a = (t * 4 + j) * h;
            s0 += gl4(c, a, a + h);
        }
    }
    part[t] = s0;
    __syncthreads();
    for (int o = kScanThreads / 2; o > 0; o >>= 1) {
        if (t < o) part[t] += part[t + o];
        __syncthreads();
    }
    const double r0 = part[0];
    __syncthreads();
    // chunked exclusive scan of the num - 1 segments
    const int nseg = num - 1;
    const int chunk = (nseg + kScanThreads - 1) / kScanThreads;
    const int b = t * chunk, e = min(nseg, b + chunk);
    double cs = 0.0;
    for (int i = b; i < e; i++) cs += seg[i];
    part[t] = cs;
    __syncthreads();
    if (t == 0) {
        double run = r0;
        for (int i = 0; i < kScanThreads; i++) {
            const double v = part[i];
            part[i] = run;
            run += v;
        }
    }
    __syncthreads();
    double run = part[t];
    if (t == 0) kn[0].y = r0;
    for (int i = b; i < e; i++) {
        run += seg[i];
        kn[i + 1].y = run;
    }
}

// Linear interpolation on the increasing knots (z -> r, or r -> z with BYR) in
// two parts, so that work that does not need the knots stands between their
// loads and their use.
template <bool BYR>
struct Interp {
    double x;
    int i;
    bool in;        // inside the table (the reference raises BoundsError)
    double2 a, b;   // knots i and i + 1: (abscissa, ordinate)
    __device__ __forceinline__ static double2 knot(const CosmoTable &t, int k) {
        const double2 v = t.kn[k];
        return BYR ? make_double2(v.y, v.x) : v;
    }
    __device__ __forceinline__ void load(const CosmoTable &t, double xv) {
        x = xv;
        in = x >= knot(t, 0).x && x <= knot(t, t.num - 1).x;
        if constexpr (BYR) {
            // guess from the guide table, linear between points uniform in r
            // (r(z) is smooth: within about a knot at 100000 knots).  The
            // table's 8 KB stay in L1, where an entry per knot took a line of
            // L2 per conversion.
            const double p = (x - t.r0) * t.dr_inv;
            const int j = max(min((int)p, kCosmoGuide - 1), 0);
            const float2 g = t.guide[j];
            i = (int)(g.x + (float)(p - j) * g.y);
        } else {
            i = (int)((x - t.z0) * t.dz_inv);   // the knots are uniform in z
        }
        i = max(min(i, t.num - 2), 0);
        a = knot(t, i);
        b = knot(t, i + 1);
    }
    // The interval as Interpolations.Gridded(Linear()) picks it: the last
    // i <= num - 2 with knot i <= x.  False outside the table.
    __device__ __forceinline__ bool get(const CosmoTable &t, double &y) {
        if (!in) return false;
        while (i > 0 && a.x > x) {
            i--;
            b = a;
            a = knot(t, i);
        }
        while (i < t.num - 2 && b.x <= x) {
            i++;
            a = b;
            b = knot(t, i + 1);
        }
        const double w = (x - a.x) / (b.x - a.x);
        y = a.y + w * (b.y - a.y);
        return true;
    }
};

// guide[j] = (index, its change over one step) at r0 + j / dr_inv, the index
// with its fraction between knots (binary search)
__global__ void k_cosmo_guide(CosmoTable t, float2 *guide) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= kCosmoGuide) return;
    double at[2];
    for (int e = 0; e < 2; e++) {
        const double r = t.r0 + (double)(j + e) / t.dr_inv;
        int lo = 0, hi = t.num - 1;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (t.kn[mid].y <= r)
                lo = mid;
            else
                hi = mid;
        }
        at[e] = lo + (r - t.kn[lo].y) / (t.kn[lo + 1].y - t.kn[lo].y);
    }
    guide[j] = make_float2((float)at[0], (float)(at[1] - at[0]));
}

__global__ void k_comoving_distance(CosmoTable t, const double *__restrict__ z, double *__restrict__ r,
                                    int64_t n, int *err) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double v = 0.0;
    Interp<false> p;
    p.load(t, z[i]);
    if (!p.get(t, v)) {
        atomicOr(err, 1);
        v = NAN;
    }
    r[i] = v;
}

// a b + c with the constant c in scalar registers: left to the compiler each
// coefficient of a Horner chain cost two vector moves beside its fma.
__device__ __forceinline__ double fma_k(double a, double b, double c) {
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
    return r;
}

// n / d to about an ulp (d normal and well inside the range): v_rcp_f64, two
// Newton steps and a correction of the quotient.
__device__ __forceinline__ double div_ulp(double n, double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    r = fma(fma(-d, r, 1.0), r, r);
    const double q = n * r;
    return fma(fma(-d, q, n), r, q);
}

// sin and cos in FP64 of an FP32 angle: x = k pi/2 + r with pi/2 in two parts
// (exact products by fma, so r holds to an ulp for |x| <= 2^17), then the
// Taylor series of both on |r| <= pi/4, truncated below 6e-17 relative.  Beyond,
// and for infinities and NaN, the library's functions.  About 40 vector
// instructions; the library's reduction for any argument took 190.
__device__ __forceinline__ void sincos_f32(float xf, double &s, double &c) {
    const double x = (double)xf;
    if (!(fabsf(xf) <= 131072.0f)) {
        sincos(x, &s, &c);
        return;
    }
    const double k = rint(x * 0.63661977236758134308);   // 2 / pi
    double r = fma(-k, 1.57079632679489655800, x);
    r = fma(-k, 6.12323399573676603587e-17, r);
    const double r2 = r * r;
    double ps = -1.0 / 1307674368000.0;
    ps = fma_k(ps, r2, 1.0 / 6227020800.0);
    ps = fma_k(ps, r2, -1.0 / 39916800.0);
    ps = fma_k(ps, r2, 1.0 / 362880.0);
    ps = fma_k(ps, r2, -1.0 / 5040.0);
    ps = fma_k(ps, r2, 1.0 / 120.0);
    ps = fma_k(ps, r2, -1.0 / 6.0);
    const double sn = fma(ps * r2, r, r);
    double pc = 1.0 / 20922789888000.0;
    pc = fma_k(pc, r2, -1.0 / 87178291200.0);
    pc = fma_k(pc, r2, 1.0 / 479001600.0);
    pc = fma_k(pc, r2, -1.0 / 3628800.0);
    pc = fma_k(pc, r2, 1.0 / 40320.0);
    pc = fma_k(pc, r2, -1.0 / 720.0);
    pc = fma_k(pc, r2, 1.0 / 24.0);
    pc = fma_k(pc, r2, -0.5);
    const double cs = fma(pc, r2, 1.0);
    const int q = (int)k;
    const double a = q & 1 ? cs : sn, b = q & 1 ? sn : cs;
    s = q & 2 ? -a : a;
    c = (q + 1) & 2 ? -b : b;
}

// atan2 in FP64 of FP32 arguments.  With a = min, b = max of the
// magnitudes, atan(a / b) = pi/4 + atan((a - b) / (a + b)) beyond tan(pi/8),
// so one division and |u| <= tan(pi/8); atan(u) / u is a polynomial of degree
// 11 in u^2, the Chebyshev fit on that interval (1.3e-18), below the rounding of
// its evaluation.  Signs, zeros, infinities, NaN and quadrants as atan2's.
__device__ __forceinline__ double atan2_f32(float yf, float xf) {
    double y = fabs((double)yf), x = fabs((double)xf);
    const double sum = x + y;
    if (__builtin_expect(!(sum < HUGE_VAL), 0)) {   // infinities: the angle of their directions
        if (sum != sum) return sum;
        x = x < HUGE_VAL ? 0.0 : 1.0;
        y = y < HUGE_VAL ? 0.0 : 1.0;
    }
    const double a = fmin(x, y), b = fmax(x, y);
    const bool far = a > 0.41421356237309503 * b;
    const double n = far ? a - b : a, d = far ? a + b : b;
    const double u = b == 0.0 ? 0.0 : div_ulp(n, d), u2 = u * u;
    double p = -0.017805395704537506;
    p = fma_k(p, u2, 0.037965256099576565);
    p = fma_k(p, u2, -0.050351024039430294);
    p = fma_k(p, u2, 0.05846878285787001);
    p = fma_k(p, u2, -0.06662951812061838);
    p = fma_k(p, u2, 0.07692045330765912);
    p = fma_k(p, u2, -0.09090896809056438);
    p = fma_k(p, u2, 0.11111110744919396);
    p = fma_k(p, u2, -0.1428571427925024);
    p = fma_k(p, u2, 0.1999999999994089);
    p = fma_k(p, u2, -0.3333333333333312);
    double r = fma(p * u2, u, u);
    if (far) r += 0.78539816339744828;
    if (y > x) r = 1.57079632679489656 - r;
    if (signbit(xf)) r = 3.14159265358979312 - r;
    return copysign(r, (double)yf);
}

// a / b in FP32 from inv = 1 / b rounded to FP64: the product is off by at most
// 2^-52 relative, and no quotient of two FP32 numbers lies that close to the
// middle of two neighbouring FP32 numbers (2^-49), so this is the IEEE quotient
// (of normal size).
__device__ __forceinline__ float div_f32(float a, double inv) { return (float)((double)a * inv); }

// The conversions below move 24 bytes per galaxy and gather two neighbouring
// knots; what bounded them was the library's FP64 trigonometry (190 and 130
// instructions a call, FP64 at the rate of FP32) and a chain of dependent
// table loads.  The knots' loads are now in flight during the trigonometry,
// and the streams, read once, do not displace the table from L2.  22 million
// galaxies: sky_to_cartesian 470 -> 209 us, cartesian_to_sky 538 -> 211 us
// (528 MB each, 112 us at the copy rate; the rest is the gather's lines and
// 200 instructions per galaxy).

// sky_to_cartesian, examples/lightcone.jl:30-48: angles in FP32 as the driver
// computes them (ra * pi / 180 with pi rounded to Float32), trigonometric
// functions evaluated in FP64 and rounded (Julia's Float32 cos/sin are
// correctly rounded in practice), products dist * cos(dec) * cos(ra) * h in
// FP64 (dist is the FP64 table value), stored as FP32.
__global__ void k_sky_to_cart(CosmoTable t, float hh, const float *__restrict__ ra, const float *__restrict__ dec,
                              const float *__restrict__ red, float *__restrict__ x, float *__restrict__ y,
                              float *__restrict__ z, int64_t n, int *err) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float av = __builtin_nontemporal_load(&ra[i]), dv = __builtin_nontemporal_load(&dec[i]);
    const float zv = __builtin_nontemporal_load(&red[i]);
    Interp<false> p;
    p.load(t, (double)zv);
    const float pif = 3.14159265358979323846f;
    const float rar = div_f32(av * pif, 1.0 / 180.0);
    const float der = div_f32(dv * pif, 1.0 / 180.0);
    double sd, cd, sr, cr;
    sincos_f32(der, sd, cd);
    sincos_f32(rar, sr, cr);
    sd = (double)(float)sd;
    cd = (double)(float)cd;
    sr = (double)(float)sr;
    cr = (double)(float)cr;
    double dist = 0.0;
    if (!p.get(t, dist)) {
        atomicOr(err, 1);
        dist = NAN;
    }
    x[i] = (float)(((dist * cd) * cr) * (double)hh);
    y[i] = (float)(((dist * cd) * sr) * (double)hh);
    z[i] = (float)((dist * sd) * (double)hh);
}

// cartesian_to_sky, examples/lightcone.jl:50-80: r = |pos| / h in FP32, the
// redshift interpolated on the distance table, RA = rem(lon - 360, 360) as
// the driver writes it (values in (-360, 0]), Dec from atan(z, s).
__global__ void k_cart_to_sky(CosmoTable t, double h_inv, const float *__restrict__ x, const float *__restrict__ y,
                              const float *__restrict__ z, float *__restrict__ ra, float *__restrict__ dec,
                              float *__restrict__ red, int64_t n, int *err) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float xv = __builtin_nontemporal_load(&x[i]), yv = __builtin_nontemporal_load(&y[i]);
    const float zv = __builtin_nontemporal_load(&z[i]);
    Interp<true> p;
    p.load(t, (double)div_f32(sqrtf((xv * xv + yv * yv) + zv * zv), h_inv));
    const float s = sqrtf(xv * xv + yv * yv);
    const float pif = 3.14159265358979323846f;
    float lon = (float)atan2_f32(yv, xv);
    float lat = (float)atan2_f32(zv, s);
    lon = div_f32(lon * 180.0f, 1.0 / (double)pif);
    lat = div_f32(lat * 180.0f, 1.0 / (double)pif);
    // fmodf(lon, 360) of lon in (-720, 0): the sum is exact
    lon = lon - 360.0f;
    if (lon <= -360.0f) lon = copysignf(lon + 360.0f, -1.0f);
    double zz = 0.0;
    if (!p.get(t, zz)) {
        atomicOr(err, 1);
        zz = NAN;
    }
    ra[i] = lon;
    dec[i] = lat;
    red[i] = (float)zz;
}

static inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

hipError_t launch_cosmo_table(const CosmoArgs &c, double *seg, double2 *kn, int num, hipStream_t s) {
    hipLaunchKernelGGL(k_cosmo_knots, dim3(blocks_for(num)), dim3(256), 0, s, seg, kn, num);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_cosmo_seg, dim3(blocks_for(num)), dim3(256), 0, s, c, kn, seg, num);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_cosmo_scan, dim3(1), dim3(kScanThreads), 0, s, c, kn, seg, num);
    return hipGetLastError();
}

hipError_t launch_cosmo_guide(const CosmoTable &t, float2 *guide, hipStream_t s) {
    hipLaunchKernelGGL(k_cosmo_guide, dim3(blocks_for(kCosmoGuide)), dim3(256), 0, s, t, guide);
    return hipGetLastError();
}

hipError_t launch_comoving_distance(const CosmoTable &t, const double *z, double *r, int64_t n, int *err,
                                    hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_comoving_distance, dim3(blocks_for(n)), dim3(256), 0, s, t, z, r, n, err);
    return hipGetLastError();
}

hipError_t launch_sky_to_cart(const CosmoTable &t, float hh, const float *ra, const float *dec, const float *red,
                              float *x, float *y, float *z, int64_t n, int *err, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sky_to_cart, dim3(blocks_for(n)), dim3(256), 0, s, t, hh, ra, dec, red, x, y, z, n, err);
    return hipGetLastError();
}

hipError_t launch_cart_to_sky(const CosmoTable &t, float h, const float *x, const float *y, const float *z,
                              float *ra, float *dec, float *red, int64_t n, int *err, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_cart_to_sky, dim3(blocks_for(n)), dim3(256), 0, s, t, 1.0 / (double)h, x, y, z, ra, dec, red,
                       n, err);
    return hipGetLastError();
}

}  // namespace baorec
