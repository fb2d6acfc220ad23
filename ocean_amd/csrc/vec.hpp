// Vector layer (OCEAN_vector ops of OCEAN2/OCEAN_psi.f90), Haydock recurrence
// kernels, continued fraction, and the load-time layout transforms.
//
// Reductions are deterministic: a fixed grid of kRedBlocks workgroups writes
// partials, and every consumer sums them in the same order.
#pragma once
#include "action.hpp"
#include "common.hpp"

namespace og {

// <p|q> partials: (sum p_r q_r + p_i q_i, sum p_r q_i - p_i q_r)   OCEAN_psi.f90:1930-2126
__global__ __launch_bounds__(kBlock) void k_dot_part(const double2* __restrict__ p,
                                                      const double2* __restrict__ q, size_t n,
                                                      double* __restrict__ part) {
  __shared__ double lds[8 * 2];
  double v[2] = {0.0, 0.0};
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const double2 a = p[i], b = q[i];
    v[0] = fma(a.x, b.x, v[0]); v[0] = fma(a.y, b.y, v[0]);
    v[1] = fma(a.x, b.y, v[1]); v[1] = fma(-a.y, b.x, v[1]);
  }
  block_sum<2>(v, lds);
  if (threadIdx.x == 0) { part[2 * blockIdx.x] = v[0]; part[2 * blockIdx.x + 1] = v[1]; }
}

// one wave per value: out[j] = sum_b part[b*nv + j]
__global__ void k_finish(const double* __restrict__ part, int nblk, int nv, double* __restrict__ out) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int j = wid; j < nv; j += nw) {
    const double s = wave_sum_parts(part, nblk, nv, j, lane);
    if (lane == 0) out[j] = s;
  }
}

// squared norm partials   OCEAN_psi.f90:1673-1760
__global__ __launch_bounds__(kBlock) void k_nrm_part(const double2* __restrict__ p, size_t n,
                                                      double* __restrict__ part) {
  __shared__ double lds[8];
  double v[1] = {0.0};
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const double2 a = p[i];
    v[0] = fma(a.x, a.x, v[0]); v[0] = fma(a.y, a.y, v[0]);
  }
  block_sum<1>(v, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = v[0];
}

// y += (ar + i ai) x      OCEAN_psi.f90:1386-1458
__global__ void k_axpy(double ar, double ai, const double2* __restrict__ x, double2* __restrict__ y, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const double2 xv = x[i];
    double2 yv = y[i];
    yv.x += ar * xv.x; yv.y += ar * xv.y;
    yv.x += -ai * xv.y; yv.y += ai * xv.x;
    y[i] = yv;
  }
}

__global__ void k_scal(double a, double2* __restrict__ x, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    double2 v = x[i]; v.x *= a; v.y *= a; x[i] = v;
  }
}

// y = (r + i i) x - z  (OCEAN_psi_axmz, OCEAN_psi.f90:1571-1670; z = y gives OCEAN_psi_axmy,
// :1468-1562, whose buffer order (r x - y) -/+ i x is the same arithmetic)
__global__ void k_axmz(double r, double i, const double2* __restrict__ x, const double2* z, double2* y, size_t n) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const double2 xv = x[e], zv = z[e];
    double2 o;
    o.x = (r * xv.x - zv.x) - i * xv.y;
    o.y = (r * xv.y - zv.y) + i * xv.x;
    y[e] = o;
  }
}

// x = x / (r + i i) with the reference's branches (OCEAN_psi_divide, OCEAN_psi.f90:1764-1874):
// which = 1: x * (1/r); 2: (x_i/i, -x_r/i); 3: x * conj(r + i i) / (r^2 + i^2)
__global__ void k_divide(double r, double i, int which, double2* __restrict__ x, size_t n) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const double2 v = x[e];
    double2 o;
    if (which == 1) {
      const double rn = 1.0 / r;
      o = make_double2(rn * v.x, rn * v.y);
    } else if (which == 2) {
      const double in = 1.0 / i;
      o = make_double2(v.y * in, -in * v.x);
    } else {
      const double den = r * r + i * i, rn = r / den, in = i / den;
      o.x = rn * v.x + in * v.y;
      o.y = -in * v.x + rn * v.y;
    }
    x[e] = o;
  }
}

__global__ void k_copy(double2* __restrict__ dst, const double2* __restrict__ src, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

__global__ void k_fill(double2* __restrict__ dst, double2 v, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = v;
}

__global__ void k_fill_d(double* __restrict__ dst, double v, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = v;
}

// ---------------------------------------------------------------------------
// The Haydock two-term step's own pass, the rest of which rides on the action (HayFuse):
//   a(i) = Re<h|psi> from the adjoint's partials; h -= a(i) psi; partials of |h|^2
// h and psi are the stored vectors, n elements per right-hand side; the workgroup lb of
// kRedBlocks always takes the same elements.  The first elements are in flight while
// the partials are summed.
// ---------------------------------------------------------------------------
struct HayArgs {
  HayFuse f;
  double2* h;
  const double2* psi;
  size_t n;
};

__device__ __forceinline__ void hay2_body(const HayArgs& A, int q, int lb, int it) {
  constexpr int U = 2;
  __shared__ double lds[8 * 2];
  __shared__ double s_a;
  double* s = A.f.s + (size_t)q * A.f.stride;
  const int n1 = A.f.n1, np1 = A.f.np1;
  const double* part1 = s + 4 * n1;
  double* part2 = s + 4 * n1 + 2 * np1;
  double2* h = A.h + (size_t)q * A.n;
  const double2* psi = A.psi + (size_t)q * A.n;
  const size_t n = A.n, st = (size_t)kRedBlocks * blockDim.x;
  size_t i = (size_t)lb * blockDim.x + threadIdx.x;
  double2 hv[U], pv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const size_t e = min(i + u * st, n - 1);
    hv[u] = h[e];
    pv[u] = psi[e];
  }
  const double sc = s[3 * n1 + it - 1];
  double p[2] = {0.0, 0.0};
  for (int m = threadIdx.x; m < np1; m += blockDim.x) { p[0] += part1[2 * m]; p[1] += part1[2 * m + 1]; }
  block_sum<2>(p, lds);
  if (threadIdx.x == 0) {
    s_a = p[0];
    if (lb == 0) { s[it - 1] = p[0]; s[n1 + it - 1] = p[1]; }
  }
  __syncthreads();
  const double ma = -s_a;
  double v[1] = {0.0};
  for (; i < n; i += U * st) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t e = i + u * st;
      if (e < n) {
        const double2 a = make_double2(fma(ma, pv[u].x * sc, hv[u].x), fma(ma, pv[u].y * sc, hv[u].y));
        h[e] = a;
        v[0] = fma(a.x, a.x, v[0]); v[0] = fma(a.y, a.y, v[0]);
      }
      const size_t en = min(e + U * st, n - 1);
      hv[u] = h[en];
      pv[u] = psi[en];
    }
  }
  block_sum<1>(v, lds);
  if (threadIdx.x == 0) part2[lb] = v[0];
}

// one problem, all its right-hand sides
__global__ __launch_bounds__(kBlock) void k_hay2(const HayArgs A) {
  hay2_body(A, blockIdx.x / kRedBlocks, blockIdx.x % kRedBlocks, A.f.it);
}
__global__ __launch_bounds__(kBlock) void k_hay_fin(const HayFuse F, int j, int R) { hay_fin(F, j, R); }

// Many problems of one right-hand side each, with the same partition as on their own, so a
// batched recursion reproduces each problem's stand-alone coefficients bit for bit.
__global__ __launch_bounds__(kBlock) void k_hay2_batch(const HayArgs* __restrict__ As, int* __restrict__ itp) {
  const int it = itp[1];
  if (blockIdx.x == 0 && threadIdx.x == 0) itp[0] = it + 1;
  hay2_body(As[blockIdx.x / kRedBlocks], 0, blockIdx.x % kRedBlocks, it);
}
__global__ __launch_bounds__(kBlock) void k_hay_fin_batch(const HayArgs* __restrict__ As, int j) {
  hay_fin(As[blockIdx.x].f, j, 1);
}

// ---------------------------------------------------------------------------
// Continued fraction with the square-root terminator (write_core,
// OCEAN2/OCEAN_haydock.f90:1801-1894), one thread per energy.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double2 c_sqrt(double2 z) {
  const double r = hypot(z.x, z.y);
  if (r == 0.0) return make_double2(0.0, 0.0);
  if (z.x >= 0.0) {
    const double t = sqrt(0.5 * (r + z.x));
    return make_double2(t, z.y / (2.0 * t));
  }
  const double t = sqrt(0.5 * (r - z.x));
  return make_double2(fabs(z.y) / (2.0 * t), copysign(t, z.y));
}

// a / b by Smith's method
__device__ __forceinline__ double2 c_div(double2 a, double2 b) {
  if (fabs(b.y) <= fabs(b.x)) {
    const double r = b.y / b.x, den = b.x + b.y * r;
    return make_double2((a.x + a.y * r) / den, (a.y - a.x * r) / den);
  }
  const double r = b.x / b.y, den = b.y + b.x * r;
  return make_double2((a.x * r + a.y) / den, (a.y * r - a.x) / den);
}

__device__ __forceinline__ double f32r(double v) { return (double)(float)v; }

// ---------------------------------------------------------------------------
// Non-Hermitian (bi-Lanczos) Haydock step, haydock_abc_1 (OCEAN2/OCEAN_haydock.f90:
// 1250-1433), over the forward vectors v (psi, old, h = H psi) and the backward ones
// w (bpsi, bold, bh = H^+ bpsi), in three passes with fixed-order reductions:
//   1: h, bh *= allow; partials of alpha = <bpsi|h>
//   2: alpha; h += -b(i-1) old; bh += -conj(c(i-1)) bold; h += -alpha psi;
//      bh += -conj(alpha) bpsi; h, bh *= allow; partials of r = <bh|h>
//   3: r; c(i) = sqrt(r) (principal root as written), b(i) = conj(r / c(i));
//      bh /= (Re b(i) - i Im b(i)); h /= c(i)
// Each axpy and divide keeps OCEAN_psi_axpy's and OCEAN_psi_divide's operation order.
// coef: [ra, ia, rb, ib, rc, ic], n1 entries each.
// ---------------------------------------------------------------------------
struct AbcArgs {
  double2* h;
  double2* bh;
  const double2* old;
  const double2* bold;
  const double2* psi;
  const double2* bpsi;
  const double* allow;
  double* coef;
  double* part1;  // [2 kRedBlocks]
  double* part2;  // [2 kRedBlocks]
  size_t n;
  int n1;
};

__device__ __forceinline__ double2 axpy_elem(double ar, double ai, double2 x, double2 y) {
  y.x += ar * x.x; y.y += ar * x.y;
  y.x += -ai * x.y; y.y += ai * x.x;
  return y;
}

// x / (r + i i) as OCEAN_psi_divide with both parts given (OCEAN_psi.f90:1797-1810)
__device__ __forceinline__ double2 divide_elem(double r, double i, double2 v) {
  const double den = r * r + i * i, rn = r / den, in = i / den;
  return make_double2(rn * v.x + in * v.y, -in * v.x + rn * v.y);
}

__global__ __launch_bounds__(kBlock) void k_abc1(AbcArgs A) {
  __shared__ double lds[8 * 2];
  double v[2] = {0.0, 0.0};
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < A.n; i += (size_t)gridDim.x * blockDim.x) {
    const double m = A.allow[i];
    double2 a = A.h[i], b = A.bh[i];
    a.x *= m; a.y *= m; b.x *= m; b.y *= m;
    A.h[i] = a;
    A.bh[i] = b;
    const double2 w = A.bpsi[i];
    v[0] = fma(w.x, a.x, v[0]); v[0] = fma(w.y, a.y, v[0]);
    v[1] = fma(w.x, a.y, v[1]); v[1] = fma(-w.y, a.x, v[1]);
  }
  block_sum<2>(v, lds);
  if (threadIdx.x == 0) { A.part1[2 * blockIdx.x] = v[0]; A.part1[2 * blockIdx.x + 1] = v[1]; }
}

__global__ __launch_bounds__(kBlock) void k_abc2(AbcArgs A, int it) {
  __shared__ double lds[8 * 2];
  __shared__ double s_a[2];
  if (threadIdx.x < 64) {
    const double ar = wave_sum_parts(A.part1, kRedBlocks, 2, 0, threadIdx.x);
    const double ai = wave_sum_parts(A.part1, kRedBlocks, 2, 1, threadIdx.x);
    if (threadIdx.x == 0) {
      s_a[0] = ar; s_a[1] = ai;
      if (blockIdx.x == 0) { A.coef[it - 1] = ar; A.coef[A.n1 + it - 1] = ai; }
    }
  }
  __syncthreads();
  const double ar = s_a[0], ai = s_a[1];
  const double* c = A.coef;
  const int n1 = A.n1;
  const double brm = -c[2 * n1 + it - 1], bim = -c[3 * n1 + it - 1];
  const double crm = -c[4 * n1 + it - 1], cim = c[5 * n1 + it - 1];
  double v[2] = {0.0, 0.0};
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < A.n; i += (size_t)gridDim.x * blockDim.x) {
    const double m = A.allow[i];
    double2 a = axpy_elem(brm, bim, A.old[i], A.h[i]);
    double2 b = axpy_elem(crm, cim, A.bold[i], A.bh[i]);
    a = axpy_elem(-ar, -ai, A.psi[i], a);
    b = axpy_elem(-ar, ai, A.bpsi[i], b);
    a.x *= m; a.y *= m; b.x *= m; b.y *= m;
    A.h[i] = a;
    A.bh[i] = b;
    v[0] = fma(b.x, a.x, v[0]); v[0] = fma(b.y, a.y, v[0]);
    v[1] = fma(b.x, a.y, v[1]); v[1] = fma(-b.y, a.x, v[1]);
  }
  block_sum<2>(v, lds);
  if (threadIdx.x == 0) { A.part2[2 * blockIdx.x] = v[0]; A.part2[2 * blockIdx.x + 1] = v[1]; }
}

__global__ __launch_bounds__(kBlock) void k_abc3(AbcArgs A, int it) {
  __shared__ double s_c[4];
  if (threadIdx.x < 64) {
    const double rr = wave_sum_parts(A.part2, kRedBlocks, 2, 0, threadIdx.x);
    const double ri = wave_sum_parts(A.part2, kRedBlocks, 2, 1, threadIdx.x);
    if (threadIdx.x == 0) {
      const double mag = sqrt(rr * rr + ri * ri);
      const double cr = sqrt((mag + rr) / 2.0), ci = copysign(sqrt((mag - rr) / 2.0), ri);
      // r / c in complex(DP) division, then b = conj
      const double2 t = c_div(make_double2(rr, ri), make_double2(cr, ci));
      s_c[0] = t.x; s_c[1] = -t.y; s_c[2] = cr; s_c[3] = ci;
      if (blockIdx.x == 0) {
        const int n1 = A.n1;
        A.coef[2 * n1 + it] = t.x; A.coef[3 * n1 + it] = -t.y;
        A.coef[4 * n1 + it] = cr; A.coef[5 * n1 + it] = ci;
      }
    }
  }
  __syncthreads();
  const double br = s_c[0], bi = s_c[1], cr = s_c[2], ci = s_c[3];
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < A.n; i += (size_t)gridDim.x * blockDim.x) {
    A.bh[i] = divide_elem(br, -bi, A.bh[i]);
    A.h[i] = divide_elem(cr, ci, A.h[i]);
  }
}

// (ar + i ai)(br + i bi) in single precision with every product and sum rounded on
// its own (Fortran complex(4) arithmetic).  The operators are written here under
// contract(off): a fused multiply-add would round the product and the sum once.
__device__ __forceinline__ double2 cmul32(float ar, float ai, float br, float bi) {
#pragma clang fp contract(off)
  const float re = ar * br - ai * bi;
  const float im = ar * bi + ai * br;
  return make_double2((double)re, (double)im);
}

// b(j) c(j) of the fraction: b = c real for the Hermitian recursion (ib == nullptr),
// complex b and c for the bi-Lanczos one (write_core, OCEAN_haydock.f90:1846-1847,
// :1870); literal rounds the kind-less cmplx() operands and products to single
// precision as OCEAN2's build does
__device__ __forceinline__ double2 cf_bc(const double* __restrict__ rb, const double* __restrict__ ib,
                                         const double* __restrict__ rc, const double* __restrict__ ic, int j,
                                         double scale, int literal) {
  if (ib == nullptr) {
    if (literal) {
      const float b32 = (float)rb[j];
      return make_double2((double)(((float)scale * b32) * b32), 0.0);
    }
    return make_double2(scale * rb[j] * rb[j], 0.0);
  }
  if (literal) {
    const float s = (float)scale;
    return cmul32(__fmul_rn(s, (float)rb[j]), __fmul_rn(s, (float)ib[j]), (float)rc[j], (float)ic[j]);
  }
  const double br = scale * rb[j], bi = scale * ib[j];
  return make_double2(br * rc[j] - bi * ic[j], br * ic[j] + bi * rc[j]);
}

// delta(e) of the n-level fraction with its square-root terminator; the spectrum
// is kpref |Im delta| / |delta|^2 and SPKK kpref Re delta / |delta|^2.
__device__ double2 cf_delta(const double* __restrict__ ra, const double* __restrict__ rb,
                            const double* __restrict__ ia, int n, double e, double gam, int literal,
                            const double* __restrict__ ib = nullptr, const double* __restrict__ rc = nullptr,
                            const double* __restrict__ ic = nullptr) {
  double2 ct = make_double2(e - ra[n - 1], gam + ia[n - 1]);
  const double2 fourbc = cf_bc(rb, ib, rc, ic, n, 4.0, literal);
  double2 z2 = make_double2(ct.x * ct.x - ct.y * ct.y - fourbc.x, 2.0 * ct.x * ct.y - fourbc.y);
  const double2 disc = c_sqrt(z2);
  double2 delta = (disc.y > 0.0) ? make_double2(0.5 * (ct.x + disc.x), 0.5 * (ct.y + disc.y))
                                 : make_double2(0.5 * (ct.x - disc.x), 0.5 * (ct.y - disc.y));
  for (int jj = n - 1; jj >= 0; --jj) {
    const double2 bc = cf_bc(rb, ib, rc, ic, jj + 1, 1.0, literal);
    double2 z;
    if (literal) {
      z = make_double2(f32r(e - ra[jj]), f32r(gam + ia[jj]));
    } else {
      z = make_double2(e - ra[jj], gam + ia[jj]);
    }
    const double2 q = c_div(bc, delta);
    delta = make_double2(z.x - q.x, z.y - q.y);
  }
  return delta;
}

__global__ void k_cfrac(const double* __restrict__ ra, const double* __restrict__ rb,
                        const double* __restrict__ ia, int n, double kpref, double gam, double el,
                        double eh, int ne, int literal, double hartree2ev, double* __restrict__ out,
                        const double* __restrict__ ib = nullptr, const double* __restrict__ rc = nullptr,
                        const double* __restrict__ ic = nullptr) {
  const int ie = blockIdx.x * blockDim.x + threadIdx.x;
  if (ie > ne) return;
  const double e = el + (eh - el) * (double)(2 * ie) / (double)(2 * ne);
  const double2 delta = cf_delta(ra, rb, ia, n, e, gam, literal, ib, rc, ic);
  const double dr = delta.x, di = fabs(delta.y);
  const double den = dr * dr + di * di;
  const double sp = kpref * di / den, kk = kpref * dr / den;
  double* o = out + (size_t)ie * 5;
  o[0] = hartree2ev * e;
  o[1] = sp; o[2] = sp; o[3] = kk; o[4] = kk;
}

// Plasmon-pole lifetime broadening (CNBSE/zcmsnmult/zf90/gamfcn.f90:8-42): energy e
// (Hartree) above the Fermi level, valence density n (bohr^-3), dielectric e0.
__device__ double gamfcn_dev(double e, double n, double e0) {
  const double pi = 3.14159265358979;
  const double kf = pow(3.0 * pi * pi * n, 1.0 / 3.0);
  const double wp = sqrt(4.0 * pi * n);
  double k = kf * kf / 2.0 + e;
  if (k < kf * kf / 2.0) return 0.0;
  k = sqrt(2.0 * k);
  const double wf = kf * kf / 2.0;
  const double lam = sqrt(wp * wp / (wf * wf * (e0 - 1.0)));
  const double dq = 0.005 * kf;
  double q = 0.5 * dq, su = 0.0;
  bool test1 = true;
  while (test1) {
    const double qq = q / kf;
    const double xp = qq * (2.0 + qq) / lam, xm = qq * (2.0 - qq) / lam;
    const double q3 = qq * qq * qq, q5 = q3 * qq * qq;
    const double term1 = lam / (2.0 * q3) * (atan(xp) + atan(xm));
    const double term2 = (0.125 * lam * lam / q5 + 0.5 / q3 - 0.125 / qq) * log((1.0 + xp * xp) / (1.0 + xm * xm));
    const double epsq = 1.0 + 2.0 / (pi * kf) * (1.0 / (qq * qq) - term1 + term2);
    const double wq = wp / sqrt(1.0 - 1.0 / epsq);
    test1 = k * k - kf * kf - 2.0 * wq > 0.0;
    const bool test2 = k * q - wq - q * q / 2.0 > 0.0;
    if (test1 && test2) su += dq / (q * wq);
    q += dq;
  }
  return wp * wp * su / (2.0 * k);
}

// Spectrum rows as OCEAN 3.2.1's write_core writes them (OCEAN_haydock.f90:1801-1894),
// one thread per energy: (E, Spect, Spect(0), SPKK, SPKK(0), sigma a.u.^2, sigma cm^2,
// sigma^2 a.u.^5, sigma^2 cm^4 s).  Spect/SPKK carry gamfcn when old_broaden.
struct SpectConst {
  double hartree2ev, ev2hartree, alpha, bohr, pi, au2sec;
};
__global__ void k_write_core(const double* __restrict__ ra, const double* __restrict__ rb,
                             const double* __restrict__ ia, int n, double kpref, double gam0, double el,
                             double eh, int ne, double ebase_ev, int old_broaden, double nval, double eps,
                             double ucvol, int literal, SpectConst K, double* __restrict__ out) {
  const int ie = blockIdx.x * blockDim.x + threadIdx.x;
  if (ie > ne) return;
  const double e = el + (eh - el) * (double)(2 * ie) / (double)(2 * ne);
  double spct[2], spkk[2];
  for (int jd = 0; jd <= (old_broaden ? 1 : 0); ++jd) {
    const double gam = gam0 + (jd ? gamfcn_dev(e, nval, eps) : 0.0);
    const double2 d = cf_delta(ra, rb, ia, n, e, gam, literal);
    const double dr = d.x, di = fabs(d.y), den = dr * dr + di * di;
    spct[jd] = kpref * di / den;
    spkk[jd] = kpref * dr / den;
  }
  if (!old_broaden) { spct[1] = spct[0]; spkk[1] = spkk[0]; }
  const double ener = ebase_ev + K.hartree2ev * e;
  const double a_by_v = K.ev2hartree * K.alpha * ucvol;
  const double bsq = K.bohr * K.bohr * 1.e-16;
  const double tpa = (K.alpha * K.alpha * 2.0 * K.pi) * ucvol;
  const double tpacm4 = tpa * bsq * bsq * K.au2sec;
  const double sigma = a_by_v * ener * spct[0];
  double* o = out + (size_t)ie * 9;
  o[0] = ener; o[1] = spct[1]; o[2] = spct[0]; o[3] = spkk[1]; o[4] = spkk[0];
  o[5] = sigma; o[6] = sigma * bsq; o[7] = spct[0] * tpa; o[8] = spct[0] * tpacm4;
}

// write_core_Voigt (OCEAN_haydock.f90:1896-1989), one thread per output point p.  The
// reference walks a fine grid of step estep around each output energy and reuses it,
// shifted by nratio, for the next point: the value at offset ii of point p was last
// computed at the point q whose freshly computed window [nstep - nratio, nstep] (all
// of [-nstep, nstep] at q = 0) held offset o = ii + (p - q) nratio.  Each thread
// evaluates exactly those (q, o) energies and sums in the reference's ii order, so
// the rows equal the sequential reuse.  The printed energy is the last fine energy
// of the point's loop, ee_p + nstep estep, as the reference prints it.
__global__ void k_write_core_voigt(const double* __restrict__ ra, const double* __restrict__ rb,
                                   const double* __restrict__ ia, int n, double kpref, double gam0,
                                   double el, double eh, int ne, double ebase_ev, double nval, double eps,
                                   int literal, double estep, int nratio, int nstep, double prefactor,
                                   double inv2s2, double hartree2ev, double* __restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p > ne) return;
  double s[2] = {0.0, 0.0}, k[2] = {0.0, 0.0};
  for (int ii = -nstep; ii <= nstep; ++ii) {
    int d = 0;
    if (nstep - nratio - ii > 0) d = (nstep - nratio - ii + nratio - 1) / nratio;
    int q = p - d, o = ii + d * nratio;
    if (q < 1) { q = 0; o = ii + p * nratio; }
    const double eeq = el + (eh - el) * (double)(2 * q) / (double)(2 * ne);
    const double e = eeq + (double)o * estep;
    const double pref = exp(-(double)(ii * ii) * (estep * estep) * inv2s2);
    for (int jd = 0; jd <= 1; ++jd) {
      const double gam = gam0 + (jd ? gamfcn_dev(e, nval, eps) : 0.0);
      const double2 dl = cf_delta(ra, rb, ia, n, e, gam, literal);
      const double dr = dl.x, di = fabs(dl.y), den = dr * dr + di * di;
      s[jd] += pref * (prefactor * kpref * di / den);
      k[jd] += pref * (prefactor * kpref * dr / den);
    }
  }
  const double ee = el + (eh - el) * (double)(2 * p) / (double)(2 * ne);
  double* o5 = out + (size_t)p * 5;
  o5[0] = ebase_ev + hartree2ev * (ee + (double)nstep * estep);
  o5[1] = s[1]; o5[2] = s[0]; o5[3] = k[1]; o5[4] = k[0];
}

// o_spect's core branch (OCEAN2/o_spect.f90:228-266), one thread per output energy:
// the it-level fraction in full FP64 complex arithmetic, gam0 and gam0 + gamfcn, and
// with ebase > 0.01 the anti-resonant fraction md (poles mirrored to -(a + 2 ebase)).
// Both SPKK columns carry -Re(eps) of the broadened pass.
__global__ void k_ospect_core(const double* __restrict__ ra, const double* __restrict__ rb, int it,
                              double kpref, double el, double eh, int ne, double gam0, double ebase,
                              double nval, double eps0, double hartree2ev, double* __restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p > ne) return;
  const double e = el + (eh - el) * (double)(2 * p) / (double)(2 * ne);
  double sp[2] = {0.0, 0.0};
  double2 eps = make_double2(0.0, 0.0);
  for (int jd = 0; jd <= 1; ++jd) {
    const double gam = gam0 + (jd ? gamfcn_dev(e, nval, eps0) : 0.0);
    const double2 ct = make_double2(e - ra[it - 1], gam);
    const double2 disc = c_sqrt(make_double2(ct.x * ct.x - ct.y * ct.y - 4.0 * (rb[it] * rb[it]), 2.0 * ct.x * ct.y));
    double2 delta = (disc.y > 0.0) ? make_double2(0.5 * (ct.x + disc.x), 0.5 * (ct.y + disc.y))
                                   : make_double2(0.5 * (ct.x - disc.x), 0.5 * (ct.y - disc.y));
    double2 md = make_double2(delta.x - e - 2.0 * ebase, delta.y - gam);
    for (int jj = it - 1; jj >= 0; --jj) {
      const double bb = rb[jj + 1] * rb[jj + 1];
      const double2 q = c_div(make_double2(bb, 0.0), delta);
      const double2 qm = c_div(make_double2(bb, 0.0), md);
      delta = make_double2((e - ra[jj]) - q.x, gam - q.y);
      md = make_double2((-e - ra[jj] - 2.0 * ebase) - qm.x, -gam - qm.y);
    }
    eps = c_div(make_double2(-kpref, 0.0), delta);
    if (ebase > 0.01) {
      const double2 t = c_div(make_double2(kpref, 0.0), md);
      eps = make_double2(eps.x - t.x, eps.y - t.y);
    }
    sp[jd] = eps.y;
  }
  double* o5 = out + (size_t)p * 5;
  o5[0] = (e + ebase) * hartree2ev;
  o5[1] = sp[1]; o5[2] = sp[0]; o5[3] = -eps.x; o5[4] = -eps.x;
}

// o_spect's valence branch (OCEAN2/o_spect.f90:166-222) at the ne midpoint energies:
// eps = 1 - f/al - f/be with the resonant (al) and anti-resonant (be) fractions, then
// n, kappa, mu, reflectivity and the loss function.
__global__ void k_ospect_val(const double* __restrict__ ra, const double* __restrict__ rb, int it,
                             double kpref, double ucvol, double el, double eh, int ne, double gam0,
                             double hartree2ev, double mu_den, double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ne) return;
  const double w = el + (eh - el) * (double)(2 * i + 1) / (double)(2 * ne);
  const double fact = kpref * ucvol * 2.0;
  const double at = ra[it - 1];
  const double2 arg = c_sqrt(make_double2((w - at) * (w - at) - 4.0 * (rb[it] * rb[it]), 0.0));
  const double2 rp = make_double2(0.5 * (w - at + arg.x), 0.5 * arg.y);
  const double2 rm = make_double2(0.5 * (w - at - arg.x), -0.5 * arg.y);
  const double2 rrr = (rp.y < 0.0) ? rp : rm;
  double2 al = make_double2((w - at) - rrr.x, gam0 - rrr.y);
  double2 be = make_double2((-w - at) - rrr.x, -gam0 - rrr.y);
  for (int j = it - 1; j >= 0; --j) {
    const double bb = rb[j + 1] * rb[j + 1];
    const double2 qa = c_div(make_double2(bb, 0.0), al);
    const double2 qb = c_div(make_double2(bb, 0.0), be);
    al = make_double2((w - ra[j]) - qa.x, gam0 - qa.y);
    be = make_double2((-w - ra[j]) - qb.x, -gam0 - qb.y);
  }
  const double2 fa = c_div(make_double2(fact, 0.0), al), fb = c_div(make_double2(fact, 0.0), be);
  const double re = (1.0 - fa.x) - fb.x, im = (-fa.y) - fb.y;
  const double loss = im / (re * re + im * im);
  const double rad = sqrt(re * re + im * im);
  const double th = acos(re / rad) / 2.0;
  const double nref = sqrt(rad) * cos(th), kap = sqrt(rad) * sin(th);
  const double2 N = c_sqrt(make_double2(re, im));
  const double2 r = c_div(make_double2(N.x - 1.0, N.y), make_double2(N.x + 1.0, N.y));
  double* o8 = out + (size_t)i * 8;
  o8[0] = w * hartree2ev;
  o8[1] = re; o8[2] = im; o8[3] = nref; o8[4] = kap;
  o8[5] = 2.0 * w * hartree2ev * N.y / mu_den;
  o8[6] = r.x * r.x + r.y * r.y;
  o8[7] = loss;
}

// Eigenvalues of the (n+1) x (n+1) Lanczos matrix redtrid builds (diagonal a(0:n),
// off-diagonals b(1:n); OCEAN_haydock.f90:2273-2316, solved there by EISPACK's elsch),
// by Sturm-sequence bisection: thread j brackets the j-th smallest eigenvalue inside
// the Gershgorin interval until the bracket stops shrinking in FP64.
__device__ int sturm_below(const double* __restrict__ a, const double* __restrict__ b, int m, double x, double pivmin) {
  int cnt = 0;
  double q = a[0] - x;
  if (fabs(q) < pivmin) q = -pivmin;
  if (q < 0.0) ++cnt;
  for (int i = 1; i < m; ++i) {
    q = (a[i] - x) - b[i] * b[i] / q;
    if (fabs(q) < pivmin) q = -pivmin;
    if (q < 0.0) ++cnt;
  }
  return cnt;
}

__global__ void k_tridiag_eigs(const double* __restrict__ a, const double* __restrict__ b, int m, double lo0,
                               double hi0, double pivmin, double* __restrict__ w) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= m) return;
  double lo = lo0, hi = hi0;
  for (int it = 0; it < 200; ++it) {
    const double mid = 0.5 * (lo + hi);
    if (!(mid > lo && mid < hi)) break;  // the bracket is two adjacent doubles
    if (sturm_below(a, b, m, mid, pivmin) > j) hi = mid; else lo = mid;
  }
  w[j] = 0.5 * (lo + hi);
}

// Early-exit test of the Haydock loop (check_convergence + calc_spect_core,
// OCEAN2/OCEAN_haydock.f90:1608-1661, :1991-2027): the spectra of iterations n1 and
// n2 at the ne midpoint energies e = el + (eh - el)(2 ie + 1)/(2 ne).  Partials per
// workgroup: sum |sp1 - sp2|, sum |sp1|, sum |sp2|, max |sp1 - sp2|.
__global__ __launch_bounds__(kBlock) void k_conv_part(const double* __restrict__ ra, const double* __restrict__ rb,
                                                      const double* __restrict__ ia, int n1, int n2,
                                                      double kpref, double gam, double el, double eh, int ne,
                                                      double* __restrict__ part) {
  __shared__ double lds[4 * 4];
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  for (int ie = blockIdx.x * blockDim.x + threadIdx.x; ie < ne; ie += gridDim.x * blockDim.x) {
    const double e = el + (eh - el) * (double)(2 * ie + 1) / (double)(2 * ne);
    const double2 d1 = cf_delta(ra, rb, ia, n1, e, gam, 1);
    const double2 d2 = cf_delta(ra, rb, ia, n2, e, gam, 1);
    const double i1 = fabs(d1.y), i2 = fabs(d2.y);
    const double s1 = kpref * i1 / (d1.x * d1.x + i1 * i1);
    const double s2 = kpref * i2 / (d2.x * d2.x + i2 * i2);
    const double df = fabs(s1 - s2);
    v[0] += df;
    v[1] += fabs(s1);
    v[2] += fabs(s2);
    v[3] = fmax(v[3], df);
  }
  // max via the sum helper would be wrong: reduce it on its own
  double mx = v[3];
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
  double s3[3] = {v[0], v[1], v[2]};
  block_sum<3>(s3, lds);
  __shared__ double mw[4];
  if ((threadIdx.x & 63) == 0) mw[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) mx = fmax(mx, mw[w]);
    double* o = part + 4 * (size_t)blockIdx.x;
    o[0] = s3[0]; o[1] = s3[1]; o[2] = s3[2]; o[3] = fmax(mw[0], mx);
  }
}

// conv[0] = relArea = 2 sum|diff| / (sum|sp1| + sum|sp2|), conv[1] = maxDiff
__global__ void k_conv_fin(const double* __restrict__ part, int nblk, double* __restrict__ conv) {
  if (threadIdx.x != 0) return;
  double a = 0.0, b = 0.0, c = 0.0, m = 0.0;
  for (int i = 0; i < nblk; ++i) {
    a += part[4 * i];
    b += part[4 * i + 1];
    c += part[4 * i + 2];
    m = fmax(m, part[4 * i + 3]);
  }
  conv[0] = 2.0 * a / (b + c);
  conv[1] = m;
}

// ---------------------------------------------------------------------------
// Load-time transforms
// ---------------------------------------------------------------------------
// Reference u (nb, nk, nx, ns) column-major planes -> device [s][k][n][x] complex.
// Tiled 32x32 transpose of the (x, n) plane of each (s, k).
template <typename T2>
__global__ void k_load_u(const double* __restrict__ re, const double* __restrict__ im,
                         T2* __restrict__ u, int nb, int nk, int nx, int ldu) {
  using T = typename Scalar<T2>::T;
  __shared__ double2 tile[32][33];
  const int sk = blockIdx.z;  // s*nk + k
  const int s = sk / nk, k = sk - s * nk;
  const int n0 = blockIdx.x * 32, x0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 256 threads: ty 0..7
  for (int r = ty; r < 32; r += 8) {
    const int x = x0 + r, n = n0 + tx;
    if (x < nx && n < nb) {
      const size_t off = (((size_t)s * nx + x) * nk + k) * nb + n;
      tile[r][tx] = make_double2(re[off], im[off]);
    }
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int n = n0 + r, x = x0 + tx;
    if (x < nx && n < nb) {
      const double2 v = tile[tx][r];
      u[(((size_t)s * nk + k) * nb + n) * ldu + x] = cmake<T2>((T)v.x, (T)v.y);
    }
  }
}

// Same, applying the supercell phase of OCEAN_bloch_lrLOAD (OCEAN2/OCEAN_bloch.f90:177-203)
// from the wrapped x offsets xoff(3, nx).
template <typename T2>
__global__ void k_load_u_phase(const double* __restrict__ re, const double* __restrict__ im,
                               const int* __restrict__ xoff, T2* __restrict__ u, int nb, int nk,
                               int nx, int K1, int K2, int K3, int X1, int X2, int X3, int ldu) {
  using T = typename Scalar<T2>::T;
  __shared__ double2 tile[32][33];
  const int sk = blockIdx.z;
  const int s = sk / nk, k = sk - s * nk;
  const int q1 = k / (K2 * K3), q2 = (k / K3) % K2, q3 = k % K3;
  const int n0 = blockIdx.x * 32, x0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const double twopi = 6.283185307179586476925286766559;
  for (int r = ty; r < 32; r += 8) {
    const int x = x0 + r, n = n0 + tx;
    if (x < nx && n < nb) {
      const size_t off = (((size_t)s * nx + x) * nk + k) * nb + n;
      const double px = twopi * (double)(xoff[3 * x + 0] * q1) / (double)(X1 * K1);
      const double py = twopi * (double)(xoff[3 * x + 1] * q2) / (double)(X2 * K2);
      const double pz = twopi * (double)(xoff[3 * x + 2] * q3) / (double)(X3 * K3);
      double sp, cp;
      sincos(px + py + pz, &sp, &cp);
      const double vr = re[off], vi = im[off];
      tile[r][tx] = make_double2(cp * vr - sp * vi, cp * vi + sp * vr);
    }
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int n = n0 + r, x = x0 + tx;
    if (x < nx && n < nb) {
      const double2 v = tile[tx][r];
      u[(((size_t)s * nk + k) * nb + n) * ldu + x] = cmake<T2>((T)v.x, (T)v.y);
    }
  }
}

// Transposed copy uT[s][k][x][n] (band index fastest) from the reference planes,
// optionally phased: the reference's (n, k, x, s) order already has bands
// fastest, so this is a permutation of whole band rows (k, x) -> (x, k).
template <typename T2>
__global__ void k_load_uT(const double* __restrict__ re, const double* __restrict__ im,
                          const int* __restrict__ xoff, T2* __restrict__ uT, int nb, int nk, int nx,
                          int ns, int K1, int K2, int K3, int X1, int X2, int X3, int ldT) {
  using T = typename Scalar<T2>::T;
  const size_t tot = (size_t)ns * nk * nx * nb;
  const double twopi = 6.283185307179586476925286766559;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (size_t)gridDim.x * blockDim.x) {
    const int n = (int)(e % nb);
    size_t r = e / nb;
    const int x = (int)(r % nx);
    r /= nx;
    const int k = (int)(r % nk);
    const int s = (int)(r / nk);
    const size_t off = (((size_t)s * nx + x) * nk + k) * nb + n;
    double vr = re[off], vi = im[off];
    if (xoff) {
      const int q1 = k / (K2 * K3), q2 = (k / K3) % K2, q3 = k % K3;
      const double px = twopi * (double)(xoff[3 * x + 0] * q1) / (double)(X1 * K1);
      const double py = twopi * (double)(xoff[3 * x + 1] * q2) / (double)(X2 * K2);
      const double pz = twopi * (double)(xoff[3 * x + 2] * q3) / (double)(X3 * K3);
      double sp, cp;
      sincos(px + py + pz, &sp, &cp);
      const double tr = cp * vr - sp * vi, ti = cp * vi + sp * vr;
      vr = tr;
      vi = ti;
    }
    uT[((size_t)s * nk + k) * ldT + (size_t)x * nb + n] = cmake<T2>((T)vr, (T)vi);
  }
}

// W(k,x) from the radial table (lr_populate_W2 + intval 'cap','cap'), keeping the
// bracket and hat weights for dW/dptab.
__global__ void k_build_w(const double* __restrict__ rdist, const double* __restrict__ rtab,
                          const double* __restrict__ ptab, int nptab, double epsi, double scale,
                          size_t nel, double* __restrict__ W, int* __restrict__ i0,
                          double* __restrict__ w0, double* __restrict__ w1) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < nel; e += (size_t)gridDim.x * blockDim.x) {
    const double r = rdist[e];
    double pot, a0 = 0.0, a1 = 0.0;
    int j = 0;
    if (r > rtab[nptab - 1]) {
      pot = epsi / r;
    } else if (r < rtab[0]) {
      pot = ptab[0];
      a0 = 1.0;
    } else {
      int lo = 0, hi = nptab - 1;  // first index with rtab >= r, minus one
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (rtab[mid] < r) lo = mid; else hi = mid;
      }
      j = (rtab[0] >= r) ? 0 : lo;
      const double rat = (r - rtab[j]) / (rtab[j + 1] - rtab[j]);
      pot = ptab[j] + rat * (ptab[j + 1] - ptab[j]);
      a0 = 1.0 - rat;
      a1 = rat;
    }
    W[e] = pot * scale;
    i0[e] = j;
    w0[e] = a0 * scale;
    w1[e] = a1 * scale;
  }
}

template <typename T>
__global__ void k_cast(const double* __restrict__ src, T* __restrict__ dst, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = (T)src[i];
}

}  // namespace og
