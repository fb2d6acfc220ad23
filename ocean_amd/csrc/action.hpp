// Kernels of the core-level BSE action H.psi (OCEAN_xact, OCEAN2/OCEAN_action.f90:286-618).
//
// Device layouts (chosen for gfx950, not the reference's):
//   u   [s][k][n][x]  x fastest: the projection streams rows over x with lanes over x,
//                     the adjoint streams the same rows and reduces over x per wave.
//                     One copy serves both passes, so the second pass can hit the
//                     256 MB Infinity Cache when u fits (FP32 form).
//   phi [k][x][a]     projection output / FFT in-out (columns c = x*na + a)
//   W   [x][k]        = the reference's W(nk, nx) column-major
//   psi [a][k][n]     interleaved complex, = OCEAN_vector %r/%i order
//   c   [s][k][p][n]  compact projector index p = (l, m, nu)
#pragma once
#include "common.hpp"

namespace og {

enum ActFlags : int {
  F_LR = 1, F_FG = 2, F_SO = 4, F_E0 = 8, F_BACK = 16,
};

// GMRES control state on the device: the solve of one energy enqueues several
// iterations ahead and every kernel of them returns at once when `done` is set, so
// the host reads the state back once per block of iterations, not per iteration.
struct GmCtl {
  int done;     // 0 running, 1 converged, 2 least-squares pivot failure
  int conv_it;  // the iteration (1..depth of its cycle) at which it converged
  int info;     // zhptrf-style pivot index of a failure
  int pad1;     // (keeps the doubles 16-byte aligned)
  double gval, rval, ival, pad2;  // |g|^2, Re / Im <rhs|x> of the last residual
  double rxr, rxi, pad3, pad4;    // <rhs|x_b> of the materialised x (x = x_b + sum_i C_i U_i)
};

// The finish of a GMRES residual step: the residual kernel wrote one partial triple
// per workgroup; the finish sums them in a fixed order and, by mode:
//   kResX   (x materialised, C = 0): v = (|g|^2, <rhs|x>); <rhs|x> becomes <rhs|x_b>;
//   kResU   v = (|g|^2, <rhs|U_slot>) (slot < 0: no new vector); <rhs|x> is
//           <rhs|x_b> + sum_{i<m} C_i <rhs|U_i>;
//   kDotU   v = (0, <rhs|U_slot>): the dot only.
// kResX and kResU store |g|^2 and <rhs|x> and, with check, apply the reference's
// stopping test (OCEAN_gmres.f90:845-852): |g|^2 < ffff and (-|g|^2 / Im<rhs|x> < 0.001
// or |g|^2 < ffff / 10).  It runs as its own one-workgroup kernel or, inside a
// restart cycle, in workgroup 0 of the next action's projection (c == nullptr: none).
enum { kResX = 0, kResU = 1, kDotU = 2 };
struct GmFin {
  GmCtl* c = nullptr;
  const double* part = nullptr;
  const double2* C = nullptr;
  double2* rU = nullptr;
  double ffff = 0.0;
  int nblk = 0, it = 0, check = 0, mode = 0, m = 0, slot = -1;
};

// One workgroup of any size (one wave or more).
__device__ __noinline__ void gm_finish(const GmFin F) {
  GmCtl* c = F.c;
  if (c->done) return;
  __shared__ double sv[5];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int task = w; task < 4; task += nw) {
    if (task < 3) {
      double acc = 0.0;
      for (int b = lane; b < F.nblk; b += 64) acc += F.part[3 * b + task];
      acc = wave_sum(acc);
      if (lane == 0) sv[task] = acc;
    } else if (F.mode == kResU) {
      // sum_{i<m} C_i <rhs|U_i>, lane-strided then a butterfly (fixed order)
      double ar = 0.0, ai = 0.0;
      for (int i = lane; i < F.m; i += 64) {
        const double2 ci = F.C[i], u = F.rU[i];
        ar += ci.x * u.x - ci.y * u.y;
        ai += ci.x * u.y + ci.y * u.x;
      }
      ar = wave_sum(ar);
      ai = wave_sum(ai);
      if (lane == 0) { sv[3] = ar; sv[4] = ai; }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (F.slot >= 0) F.rU[F.slot] = make_double2(sv[1], sv[2]);
    if (F.mode != kDotU) {
      double rr, ri;
      if (F.mode == kResX) {
        rr = sv[1]; ri = sv[2];
        c->rxr = rr; c->rxi = ri;
      } else {
        rr = c->rxr + sv[3]; ri = c->rxi + sv[4];
      }
      c->gval = sv[0];
      c->rval = rr;
      c->ival = ri;
      if (F.check && sv[0] < F.ffff) {
        const double rel = -sv[0] / ri;
        if (rel < 0.001 || sv[0] < F.ffff / 10.0) {
          c->done = 1;
          c->conv_it = F.it;
        }
      }
    }
  }
  __syncthreads();
}

// A Haydock iteration fused into the action (OCEAN_hay_ab_twoterm, OCEAN2/OCEAN_haydock.f90:
// 824-938).  The recursion's vectors stay as they are before their division by b: vector
// psi_i is the stored one times inv(i - 1) = 1 / b(i - 1).  The transform's grid has one
// more workgroup that finishes b(i - 1) from the partials of |h|^2; the adjoint's
// epilogue scales H psi, subtracts b(i - 1) psi_(i-1) and writes the partials of <h|psi>;
// k_hay2 (vec.hpp) takes a(i) from them, subtracts a(i) psi and writes the partials of
// |h|^2.  As three passes over the vectors of their own after the action these steps
// took 14.5 us of a 135 us iteration at 131 072 elements and 10.6 of 34 at 4 096.
// Scalars of right-hand side q at s + q stride: a(0:niter), imag a, b, inv (n1 each), part1
// [np1][2], part2 [kRedBlocks].  The iteration number is `it`, or *itp where one captured
// iteration is replayed; the adjoint then copies it to itp[1] for k_hay2, which advances
// itp[0].
struct HayFuse {
  double* s = nullptr;  // nullptr: no recursion
  const double2* old = nullptr;
  int* itp = nullptr;
  int it = 0, n1 = 0, np1 = 0, stride = 0;
};
struct HayScal { double sc, so, mb; };  // of psi, of old, -b(i - 1)

__device__ __forceinline__ int hay_it(const HayFuse& F) { return F.itp ? F.itp[0] : F.it; }
__device__ __forceinline__ HayScal hay_scal(const HayFuse& F, int it, int q) {
  if (F.s == nullptr) return {1.0, 0.0, 0.0};
  const double* s = F.s + (size_t)q * F.stride + 2 * F.n1;
  return {s[F.n1 + it - 1], s[F.n1 + max(it - 2, 0)], -s[it - 1]};
}
// h = r - b psi_old of one element, and its term of <h|psi>
__device__ __forceinline__ double2 hay_elem(const HayScal& c, double2 pv, double2 ov, double2& r) {
  r.x = fma(c.mb, ov.x * c.so, r.x);
  r.y = fma(c.mb, ov.y * c.so, r.y);
  return make_double2(fma(r.y, pv.y, r.x * pv.x), fma(-r.y, pv.x, r.x * pv.y));
}
// partial `idx` of right-hand side q: wave q of the workgroup sums n terms
__device__ __forceinline__ void hay_part(const HayFuse& F, const double2* t, int n, int q, int idx) {
  const int lane = threadIdx.x & 63;
  double x = 0.0, y = 0.0;
  for (int e = lane; e < n; e += 64) { x += t[e].x; y += t[e].y; }
  x = wave_sum(x);
  y = wave_sum(y);
  double* p = F.s + (size_t)q * F.stride + 4 * F.n1 + 2 * idx;
  if (lane == 0) { p[0] = x; p[1] = y; }
}
// b(j) = sqrt(|h|^2) and 1 / b(j) of every right-hand side (one workgroup)
__device__ __forceinline__ void hay_fin(const HayFuse& F, int j, int R) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  for (int q = threadIdx.x >> 6; q < R; q += nw) {
    double* s = F.s + (size_t)q * F.stride;
    const double b = sqrt(wave_sum_parts(s + 4 * F.n1 + 2 * F.np1, kRedBlocks, 1, 0, lane));
    if (lane == 0) { s[2 * F.n1 + j] = b; s[3 * F.n1 + j] = 1.0 / b; }
  }
}

// Everything one problem's action kernels read: pointers into its device state,
// its sizes and its launch geometry.  Passed by value to the single-problem
// kernels; the batched kernels read an array of them, one per problem.
template <typename T2>
struct ActArgs {
  using T = typename Scalar<T2>::T;
  const T2* u;                // [s][k][n][x], row stride ldu
  const T2* uT;               // [s][k][x][n], k-slab stride ldT
  T2* phi;                    // [k][x][a], row stride ldphi
  const T* W;                 // [x][k]
  const double2* psi;         // in  [a][k][n]
  double2* out;               // out [a][k][n]
  const double2* energy;
  const double* allow;
  const double2* cproj;       // [s][k][p][n]
  double2* apart;             // [nm][a*P+p] multiplet partials
  const double2* Kmat;        // (na P)^2
  double2* hmult;             // [a*P+p]
  const double2* S;           // [a][b] over the na0 alphas of one right-hand side
  double mul;                 // inter_scale / (N_k celvol)
  int nb, nk, nx, na, ns, P, nj;
  int na0;                    // alphas per right-hand side: alpha a of a vector belongs to
                              // right-hand side a / na0 (na = na0 for one right-hand side)
  int ldu, ldT, ldphi;
  int flags;
  int px;                     // projection x-tiles per k (one wave tile per wave)
  int tput;                   // projection: phi tiles go out through LDS (one spin, where it fits)
  int nm, nmb;                // multiplet workgroups per spin and 16 projectors, and in all
  int G, ncol, nfft, nred;    // transform: columns per strip, strips, reduction workgroups
  int K1, K2, K3;
  int XC, JR;                 // adjoint: phi' chunk, alphas per reduction round
  const T2* phs;              // OBF form: supercell phase [x][k] applied around the transform
  const int* skip;            // nullable: when *skip != 0 every kernel of the action returns at once
                              // (a solver that has converged on the device drops the work it
                              // enqueued ahead)
  int axmy;                   // 1: the adjoint writes c psi - H psi instead of H psi
  double2 axmy_c;             // c = E + i gamma of a GMRES step (OCEAN_psi_axmy)
  HayFuse hay;                // hay.s != nullptr: a Haydock iteration rides on the action
  int nfin;                   // 1: the transform's grid finishes the previous iteration's b
  GmFin fin;                  // fin.c != nullptr: workgroup 0 of the projection first runs
                              // the previous GMRES residual step's finish
};

// out = c psi - r in OCEAN_psi_axmy's operation order (OCEAN2/OCEAN_psi.f90:1468-1562)
template <typename T2>
__device__ __forceinline__ double2 axmy_epilogue(const ActArgs<T2>& A, double2 pv, double2 r) {
  if (!A.axmy) return r;
  const double br = A.axmy_c.x * pv.x - r.x, bi = A.axmy_c.x * pv.y - r.y;
  return make_double2(br - A.axmy_c.y * pv.y, bi + A.axmy_c.y * pv.x);
}

template <typename T2>
__device__ __forceinline__ bool skipped(const ActArgs<T2>& A) {
  return A.skip != nullptr && *A.skip != 0;
}

// Problem p of a batched launch owns workgroups [off[p], off[p+1]).
__device__ __forceinline__ int find_problem(const int* __restrict__ off, int np, int b) {
  int lo = 0, hi = np - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// ---------------------------------------------------------------------------
// Multiplet projection partials: amplitude (a, p) = sum_{k,n} c(n,k,p) (A psi)(n,k,a)
//   OCEAN_multiplet.f90:1730-1783 (no conjugation)
// as an FP64 matrix-core GEMM (M = 16 projectors, N = the 2 nalpha real columns of a
// spin, K = bands and k).  Workgroup blk = (s, projector tile, m): its waves take units
// of one k and up to 64 bands, m nw + w first and nm nw apart, with kB steps of four
// bands in flight; their sums are added in LDS in wave order into apart[m].  These
// workgroups come first in the projection's grid, so that they run beside the u
// stream: at the end of the slab workgroups (a butterfly of 16 sums per alpha and
// wave, after the slab) the same sums cost 5 us of a 31 us FP32 projection at 64
// bands, 31 of 163 us at the L2,3 edge with 128 bands; here 4 and 8.
// ---------------------------------------------------------------------------
template <int NA>
constexpr int mult_lds_per_wave() { return ((2 * NA + 15) / 16) * 4 * 64 * (int)sizeof(double); }

template <int NA>
__device__ __forceinline__ void mult_body(const double2* __restrict__ c, const double2* __restrict__ psi,
                                          const double* __restrict__ allow, double2* __restrict__ apart, int nb,
                                          int nk, int na, int ns, int P, int nm, int blk, double* red) {
  constexpr int NT = (2 * NA + 15) / 16, kB = NT == 1 ? 8 : 4;
  const int npt = (P + 15) >> 4;
  const int s = blk / (nm * npt), pt = (blk / nm) % npt, m = blk % nm;
  const int astep = (ns == 2) ? 2 : 1;
  const int acnt = (ns == 2) ? na / 2 : na;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const int i = lane & 15, kk = lane >> 4;
  const bool im = i & 1;
  const int nch = (nb + 63) >> 6, units = nk * nch;
  og_d4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = og_d4{0, 0, 0, 0};
  for (int un = m * nw + w; un < units; un += nm * nw) {
    const int k = un / nch, n00 = (un - k * nch) * 64, n1 = min(nb, n00 + 64);
    const double2* cb = c + ((size_t)(s * nk + k) * P + min(16 * pt + i, P - 1)) * nb;
    for (int n0 = n00; n0 < n1; n0 += 4 * kB) {
      double2 cv[kB], pv[kB][NT];
      double mv[kB][NT];
#pragma unroll
      for (int q = 0; q < kB; ++q) {
        const int n = min(n0 + 4 * q + kk, nb - 1);
        cv[q] = ld_stream(cb + n);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int j = min((16 * t + i) >> 1, acnt - 1);
          const size_t off = ((size_t)(s + j * astep) * nk + k) * nb + n;
          pv[q][t] = psi[off];
          mv[q][t] = allow[off];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < kB; ++q) {
        // rows past the unit's bands contribute zeros on both sides
        const bool ok = n0 + 4 * q + kk < n1;
        const double cx = ok ? cv[q].x : 0.0, cy = ok ? cv[q].y : 0.0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const double pr = ok ? pv[q][t].x * mv[q][t] : 0.0, pi = ok ? pv[q][t].y * mv[q][t] : 0.0;
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(cx, im ? pi : pr, acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(cy, im ? pr : -pi, acc[t], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[((w * NT + t) * 4 + r) * 64 + lane] = acc[t][r];
  __syncthreads();
  for (int e = threadIdx.x; e < NT * 256; e += blockDim.x) {
    const int l = e & 63, r = (e >> 6) & 3, t = e >> 8;
    double v = 0.0;
    for (int q = 0; q < nw; ++q) v += red[((q * NT + t) * 4 + r) * 64 + l];
    const int G = 16 * t + (l & 15), p = 16 * pt + Mf<double>::row(l >> 4, r);
    if ((G >> 1) < acnt && p < P)
      reinterpret_cast<double*>(apart + (size_t)m * na * P + (s + (G >> 1) * astep) * P + p)[G & 1] = v;
  }
}

template <int NA>
__global__ __launch_bounds__(kBlock) void k_mproj(const double2* __restrict__ c, const double2* __restrict__ psi,
                                                  const double* __restrict__ allow, double2* __restrict__ apart,
                                                  int nb, int nk, int na, int ns, int P, int nm) {
  __shared__ double red[mult_lds_per_wave<NA>() / 8 * (kBlock / 64)];
  mult_body<NA>(c, psi, allow, apart, nb, nk, na, ns, P, nm, blockIdx.x, red);
}

// ---------------------------------------------------------------------------
// Projection: phi(k,x,a) = sum_n u(n,k,x) (A psi)(n,k,a)
//   long_range.f90:897-906 (no conjugation of u).
// Per (k, s) a GEMM on the matrix cores in the precision of the stored u, M = x, N = the
// 2 nalpha real columns (G = 2 a + re/im), K = bands with the complex parts unrolled:
// lane l supplies u(n, x) for x = l % 16, n = l / 16 and, from A psi staged in LDS as
// Bs[n][a], column l % 16 of B; columns past 2 nalpha compute values nobody stores.
// Each wave takes one tile of kProjNL loads: 16 x points each in FP64, 32 in FP32 (a
// 16-byte load holds u(n, x) and u(n, x + 1), which feed an even and an odd tile), with
// a ring of kProjD steps of four bands in registers, so that kProjD - 1 are in flight
// while one is multiplied.  It is bound by HBM: reading u alone runs at 6.5-7 TB/s and
// writing phi beside it adds about a byte's read time per two thirds of a byte.  256
// threads: at 512 the tail of the grid is coarser (L2,3 edge, 128 bands, 213 -> 222 us
// FP64, 125 -> 142 FP32).  Phi goes out through a wave-private LDS transpose as whole
// contiguous rows (118 -> 115 us there in FP32).  Against streaming FMAs below six
// alphas and matrix-core forms with one load per step and k-strided stores above,
// at 512 k points (us before -> after):
//   64 bands, 512 x, 4 alphas: FP64 50 -> 50, FP32 31 -> 27 (100 bands: FP64 46 -> 37)
//   64 bands, 512 x, 12 / 24 alphas: FP64 66 -> 63 / 128 -> 93, FP32 (24) 66 -> 53
//   128 bands, 1000 x, 12 alphas: FP64 221 -> 213, FP32 163 -> 125
//   64 k points, 16 bands, 216 x, 4 alphas: FP64 8.1 -> 4.4
// ---------------------------------------------------------------------------
constexpr int kProjNL = 2;  // loads per step and wave (one: 222 -> 244 us, 130 -> 151 us at the L2,3 edge)
constexpr int kProjD = 4;   // ring steps (three: equal to 1 us; six at three waves per SIMD: slower)

template <typename T2> struct ProjLoad;
template <> struct ProjLoad<double2> {
  using F = double2;
  static constexpr int X = 16;  // x points per load
};
template <> struct ProjLoad<float2> {
  using F = float4;
  static constexpr int X = 32;
};
// x points per wave
template <typename T2> constexpr int proj_xt() { return ProjLoad<T2>::X * kProjNL; }

template <typename T2, int NA>
__device__ __forceinline__ void proj_body(const ActArgs<T2>& A, int bx, int k, int s, unsigned char* smem) {
  using T = typename Scalar<T2>::T;
  using M = Mf<T>;
  using V = typename M::V;
  using F = typename ProjLoad<T2>::F;
  constexpr int NT = (2 * NA + 15) / 16, NL = kProjNL, D = kProjD, XL = ProjLoad<T2>::X;
  constexpr int Q = sizeof(T) == 8 ? 1 : 2;  // matrix-core tiles per load
  const int nb = A.nb, nk = A.nk, nx = A.nx, na = A.na, ns = A.ns;
  const int astep = (ns == 2) ? 2 : 1;
  const int acnt = (ns == 2) ? na / 2 : na;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const int i = lane & 15, kk = lane >> 4;
  const bool im = i & 1;
  const int S = (nb + 3) >> 2;  // steps of four bands; B rows past nb are zero
  T2* Bs = reinterpret_cast<T2*>(smem);
  const int x0 = (bx * nw + w) * XL * NL;
  const bool on = x0 < nx;
  const T2* __restrict__ ub = A.u + (size_t)(s * nk + k) * nb * A.ldu;
  int xo[NL];
#pragma unroll
  for (int l = 0; l < NL; ++l)
    xo[l] = sizeof(T) == 8 ? min(x0 + 16 * l + i, nx - 1) : min(x0 + 32 * l + 2 * i, A.ldu - 2);
  int ln = kk;
  auto load = [&](F(&f)[NL]) {
    const T2* row = ub + (size_t)min(ln, nb - 1) * A.ldu;
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      if constexpr (sizeof(T) == 8) f[l] = ld_stream(row + xo[l]);
      else f[l] = ld_stream4(row + xo[l]);
    }
    ln += 4;
  };
  // the first steps of the stream are in flight while A psi is staged
  F f[D][NL];
  if (on) {
#pragma unroll
    for (int d = 0; d < D - 1; ++d) load(f[d]);
  }
  const int nel = 4 * S * acnt;
  constexpr int kF = 4;
  for (int i0 = threadIdx.x; i0 < nel; i0 += kF * blockDim.x) {
    double2 pv[kF];
    double mv[kF];
#pragma unroll
    for (int q = 0; q < kF; ++q) {
      const int e = min(i0 + q * (int)blockDim.x, nel - 1);
      const int j = e / (4 * S), n = min(e - j * 4 * S, nb - 1);
      const size_t off = ((size_t)(s + j * astep) * nk + k) * nb + n;
      pv[q] = A.psi[off];
      mv[q] = A.allow[off];
    }
#pragma unroll
    for (int q = 0; q < kF; ++q) {
      const int e = i0 + q * (int)blockDim.x;
      if (e < nel) {
        const int j = e / (4 * S), n = e - j * 4 * S;
        Bs[n * acnt + j] = n < nb ? cmake<T2>((T)(pv[q].x * mv[q]), (T)(pv[q].y * mv[q])) : cmake<T2>(0, 0);
      }
    }
  }
  __syncthreads();
  if (!on) return;
  V acc[NT][NL * Q];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < NL * Q; ++m) acc[t][m] = V{0, 0, 0, 0};
  const T2* bp[NT];
  bool jok[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int G = 16 * t + i;
    jok[t] = (G >> 1) < acnt;
    bp[t] = Bs + kk * acnt + min(G >> 1, acnt - 1);
  }
  // u B: re: ur br - ui bi, im: ur bi + ui br
  auto step = [&](const F(&g)[NL], int st) {
    T b0[NT], b1[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const T2 b = bp[t][4 * st * acnt];
      b0[t] = im ? b.y : b.x;
      b1[t] = im ? b.x : -b.y;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int l = 0; l < NL; ++l) {
        acc[t][l * Q] = M::step(g[l].x, b0[t], acc[t][l * Q]);
        if constexpr (Q == 2) acc[t][l * 2 + 1] = M::step(g[l].z, b0[t], acc[t][l * 2 + 1]);
      }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int l = 0; l < NL; ++l) {
        acc[t][l * Q] = M::step(g[l].y, b1[t], acc[t][l * Q]);
        if constexpr (Q == 2) acc[t][l * 2 + 1] = M::step(g[l].w, b1[t], acc[t][l * 2 + 1]);
      }
  };
  int st = 0;
  for (; st + D <= S; st += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(f[(d + D - 1) % D]);
      __builtin_amdgcn_sched_barrier(0);  // keep the ring's loads ahead of this step's products
      step(f[d], st + d);
    }
  }
#pragma unroll
  for (int d = 0; d < D - 1; ++d)
    if (st + d < S) step(f[d], st + d);
  if (A.tput) {
    T2* tw = reinterpret_cast<T2*>(smem + (((size_t)nel * sizeof(T2) + 15) & ~(size_t)15)) + w * XL * acnt;
    T* o = reinterpret_cast<T*>(tw);
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      const int xl = x0 + XL * l;
      if (xl >= nx) break;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (jok[t]) {
#pragma unroll
          for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[(Q * M::row(kk, r) + q) * 2 * acnt + 16 * t + i] = acc[t][l * Q + q][r];
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const int n16 = min(XL, nx - xl) * acnt * (int)sizeof(T2) / 16;
      const float4* src = reinterpret_cast<const float4*>(tw);
      float4* dst = reinterpret_cast<float4*>(A.phi + (size_t)k * A.ldphi + (size_t)xl * na);
#pragma unroll
      for (int e = lane; e < XL * NA * (int)sizeof(T2) / 16; e += 64)
        if (e < n16) dst[e] = src[e];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  } else {
    T* ph = reinterpret_cast<T*>(A.phi + (size_t)k * A.ldphi);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (!jok[t]) continue;
      T* o = ph + 2 * (s + ((16 * t + i) >> 1) * astep) + (im ? 1 : 0);
#pragma unroll
      for (int m = 0; m < NL * Q; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int x = x0 + XL * (m / Q) + Q * M::row(kk, r) + m % Q;
          if (x < nx) o[(size_t)x * na * 2] = acc[t][m][r];
        }
    }
  }
}

// Workgroup b of a projection launch of n: the multiplet workgroups, then slab tile bx of
// (k, s).  Workgroups are dispatched round-robin over the 8 XCDs; with remap each XCD
// gets a contiguous range of tiles, so the px tiles of one k (which stage the same A
// psi) share an L2.
template <typename T2, int NA>
__device__ __forceinline__ void proj_dispatch(const ActArgs<T2>& A, int b, int n, bool remap) {
  extern __shared__ __align__(16) unsigned char smem[];
  if (b < A.nmb) {
    mult_body<NA>(A.cproj, A.psi, A.allow, A.apart, A.nb, A.nk, A.na, A.ns, A.P, A.nm, b,
                  reinterpret_cast<double*>(smem));
    return;
  }
  b -= A.nmb;
  n -= A.nmb;
  if (remap && (n & 7) == 0) b = (b & 7) * (n >> 3) + (b >> 3);
  const int r = b / A.px, bx = b - r * A.px, k = r % A.nk, s = r / A.nk;
  proj_body<T2, NA>(A, bx, k, s, smem);
}

// Four waves per SIMD at every alpha count.  At 24 the cap makes the compiler spill 17
// registers per lane in FP64 and 8 in FP32; three waves spill none.  us, capped -> not: 512
// k points, 512 x, 64 bands FP64 86.5 -> 83, FP32 52 -> 50.5; 256 bands 336 -> 327, 160 ->
// 163; 64 k points, 1000 x, 64 bands 33.0 -> 33.9, 24.8 -> 26.1.
template <typename T2, int NA>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_proj(const ActArgs<T2> A) {
  if (skipped(A)) return;
  if (A.fin.c != nullptr && blockIdx.x == 0) gm_finish(A.fin);
  proj_dispatch<T2, NA>(A, blockIdx.x, gridDim.x, true);
}

// Many problems: workgroup b belongs to the problem whose range holds it.
template <typename T2, int NA>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_proj_batch(
    const ActArgs<T2>* __restrict__ As, const int* __restrict__ off, int np) {
  const int p = find_problem(off, np, blockIdx.x);
  const ActArgs<T2> A = As[p];
  if (skipped(A)) return;
  proj_dispatch<T2, NA>(A, blockIdx.x - off[p], 0, false);
}

// ---------------------------------------------------------------------------
// Batched 3-D DFT over the k-mesh, staged in LDS, fused with the W multiply:
//   phi' = (1/N_k) F_- [ W(:,x) . F_+ phi ]    long_range.f90:920-939
// F_+ = FFTW_BACKWARD (exp +2 pi i), F_- = FFTW_FORWARD, k3 fastest
// (Modules/FFT_wrapper.f90:67-72, :185-215).  One pencil per thread; edge classes
// LMAX = 8, 16 and 24 (radix 2 for powers of two up to 16, direct sums otherwise).
// FP32 took as long as FP64 although it moves half the bytes: instructions bound it, most
// of them index arithmetic (two run-time divisions per pencil and a shift, a multiply
// and two adds per element), and, in small problems and with many amplitudes, the
// workgroups of the multiplet reduction in its grid.  With linear tile strides, divisions
// by multiplication, halved direct sums and reduction workgroups that do not wait for
// each other, per launch between events, us (before -> after):
//   512 k points, 2 048 columns: FP64 18.2 -> 15.3, FP32 16.9 -> 13.0
//   512 k points, 12 000 columns, 192 amplitudes: FP64 54.8 -> 45.9, FP32 47.7 -> 27.4
//   64 k points, 864 columns, FP64: 12.6 -> 7.1
// The FP64 24-edge class holds two arrays of 24 values: all 256 registers, 2 to 7 of them
// spilled, and half the time of the plain sums (24 x 24 x 2 k points, 864 columns: 119 ->
// 55; 24 x 4 x 4: 27 -> 14).
// ---------------------------------------------------------------------------
template <int L>
__device__ __forceinline__ constexpr int bitrev(int i) {
  int r = 0;
  for (int b = 1; b < L; b <<= 1) { r = (r << 1) | (i & 1); i >>= 1; }
  return r;
}

// n / d for the small tile indices, from r = 1 / d rounded to FP32: (n + 1/2) / d is at
// least 1 / (2 d) away from a whole number, more than its rounding error for n < 2^21
// (three instructions; a division by a run-time value takes about thirty, and every
// pencil of every pass needs one or two).
__device__ __forceinline__ int qdiv(int n, float r) { return (int)(((float)n + 0.5f) * r); }

// The strip in LDS: element (k1, k2, k3, g) at k1 P1 + k2 P2 + k3 G + g.  An even K3
// gets one more group of G per (k1, k2) row, so that the pencils of neighbouring rows
// along k3 start on different banks (P2 / G is odd); every stride is linear, so a
// pencil's addresses are one sum each.
__host__ __device__ __forceinline__ int tile_pad(int K3, int G) { return (K3 & 1) ? 0 : G; }
__host__ __device__ __forceinline__ size_t tile_size(int K1, int K2, int K3, int G) {
  return (size_t)K1 * K2 * (K3 * G + tile_pad(K3, G));
}

// Pencil q of a pass along one dimension of the LDS tile: q + (q / D) M is the LDS
// index of its first element and st the stride.
template <typename T2>
struct LdsPencil {
  T2* p;
  int st;
  __device__ __forceinline__ T2 ld(int j) const { return p[j * st]; }
  __device__ __forceinline__ void put(int j, T2 v) const { p[j * st] = v; }
};
template <typename T2>
struct LdsPass {
  T2* base;
  float rD;
  int M, st;
  __device__ __forceinline__ LdsPencil<T2> at(int q) const { return {base + q + qdiv(q, rD) * M, st}; }
};

// Pencil q = r G + g of the phi columns in HBM, its rows starting at r * k0 with stride ks;
// columns past the strip's gcnt repeat the last one and are not written back.
template <typename T2>
struct HbmPencil {
  T2* p;
  size_t st;
  bool ok;
  __device__ __forceinline__ T2 ld(int j) const { return p[j * st]; }
  __device__ __forceinline__ void put(int j, T2 v) const { if (ok) p[j * st] = v; }
};
template <typename T2>
struct HbmPass {
  T2* base;
  size_t ld;
  float rG;
  int G, gcnt, k0, ks;
  __device__ __forceinline__ HbmPencil<T2> at(int q) const {
    const int r = qdiv(q, rG), g = q - r * G;
    return {base + (size_t)(r * k0) * ld + min(g, gcnt - 1), ks * ld, g < gcnt};
  }
};

// W of the pencils along k1 (q = lo G + g, lo = (k2, k3)): wl holds W(x, :) of the strip's
// x points, the strip's column g belonging to x (off + g) / na.
template <typename T>
struct WPencil {
  const T* p;
  int st;
  __device__ __forceinline__ T ld(int j) const { return p[j * st]; }
};
template <typename T>
struct WPass {
  const T* wl;
  float rG, rna;
  int G, gcnt, off, nk, st;
  __device__ __forceinline__ WPencil<T> at(int q) const {
    const int lo = qdiv(q, rG), g = q - lo * G;
    return {wl + qdiv(off + min(g, gcnt - 1), rna) * nk + lo, st};
  }
};

// The OBF form's phi columns along k3: multiplied by the phase phs(k, x) as they are read,
// by its conjugate as they are written; both forms scale by inv on the way out.
template <typename T2, bool PHS>
struct PhiPencil {
  using T = typename Scalar<T2>::T;
  HbmPencil<T2> h;
  const T2* ph;
  T inv;
  __device__ __forceinline__ T2 ld(int j) const {
    const T2 v = h.ld(j);
    if constexpr (PHS) return cmul(v, ph[j]);
    else return v;
  }
  __device__ __forceinline__ void put(int j, T2 v) const {
    if (!h.ok) return;
    if constexpr (PHS) {
      const T2 p = ph[j];
      v = cmake<T2>(v.x * p.x + v.y * p.y, v.y * p.x - v.x * p.y);
    }
    h.p[j * h.st] = cmake<T2>(v.x * inv, v.y * inv);
  }
};
template <typename T2, bool PHS>
struct PhiPass {
  using T = typename Scalar<T2>::T;
  HbmPass<T2> h;
  const T2* phs;  // phs(0, x) of the strip's first x
  float rna;
  int off, nk, K3;
  T inv;
  __device__ __forceinline__ PhiPencil<T2, PHS> at(int q) const {
    const T2* ph = nullptr;
    if constexpr (PHS) {
      const int r = qdiv(q, h.rG), g = q - r * h.G;
      ph = phs + (size_t)qdiv(off + min(g, h.gcnt - 1), rna) * nk + r * K3;
    }
    return {h.at(q), ph, inv};
  }
};

// One pass of length-L pencils along one k dimension, over the G columns of the strip:
// out[m] = sum_j v[j] w^(j m), w = exp(sign 2 pi i / L), tw[m] = w^m from LDS.
// Power-of-two L: radix-2 decimation in time on data loaded in bit-reversed order;
// otherwise the direct sum.  src and dst give a pencil's accessor (LdsPass, HbmPass),
// so the first pass reads HBM straight into the pencil registers and the last writes
// HBM from them.
// cos and sin of 2 pi m / 16, correctly rounded (c1 = cos(pi/8), s1 = sin(pi/8),
// r = sqrt(2)/2): the power-of-two twiddles
#define OG_C1 0.92387953251128674
#define OG_S1 0.38268343236508978
#define OG_R2 0.70710678118654752
__device__ constexpr double kCos16[16] = {1.0, OG_C1, OG_R2, OG_S1, 0.0, -OG_S1, -OG_R2, -OG_C1,
                                          -1.0, -OG_C1, -OG_R2, -OG_S1, 0.0, OG_S1, OG_R2, OG_C1};
__device__ constexpr double kSin16[16] = {0.0, OG_S1, OG_R2, OG_C1, 1.0, OG_C1, OG_R2, OG_S1,
                                          0.0, -OG_S1, -OG_R2, -OG_C1, -1.0, -OG_C1, -OG_R2, -OG_S1};
#undef OG_C1
#undef OG_S1
#undef OG_R2

// v * w^m, w = exp(SIGN 2 pi i / L), L a power of two <= 16.  After unrolling m is
// a constant, so the multiplications by 1, -1 and +-i fold away and the others
// use literal twiddles.
template <int SIGN, int L, typename T2>
__device__ __forceinline__ T2 tw_mul(int m, T2 v) {
  using T = typename Scalar<T2>::T;
  const int idx = (m * (16 / L)) & 15;
  if (idx == 0) return v;
  if (idx == 8) return cmake<T2>(-v.x, -v.y);
  if (idx == 4) return SIGN > 0 ? cmake<T2>(-v.y, v.x) : cmake<T2>(v.y, -v.x);
  if (idx == 12) return SIGN > 0 ? cmake<T2>(v.y, -v.x) : cmake<T2>(-v.y, v.x);
  const T c = (T)kCos16[idx], sn = (T)(SIGN * kSin16[idx]);
  return cmake<T2>(c * v.x - sn * v.y, c * v.y + sn * v.x);
}

// In-register radix-2 DFT of L (a power of two) values given in bit-reversed order;
// the result is in natural order.
template <int SIGN, int L, typename T2>
__device__ __forceinline__ void fft_regs(T2 (&v)[L]) {
#pragma unroll
  for (int len = 2; len <= L; len <<= 1) {
    const int half = len / 2, step = L / len;
#pragma unroll
    for (int i = 0; i < L; i += len) {
#pragma unroll
      for (int j = 0; j < half; ++j) {
        const T2 t = tw_mul<SIGN, L>(j * step, v[i + j + half]);
        const T2 u = v[i + j];
        v[i + j] = cmake<T2>(u.x + t.x, u.y + t.y);
        v[i + j + half] = cmake<T2>(u.x - t.x, u.y - t.y);
      }
    }
  }
}

// DFT of L values, L not a power of two, by direct sums over the pairs j, L - j:
// w^(jm) v_j + w^(-jm) v_(L-j) = c (v_j + v_(L-j)) + i s (v_j - v_(L-j)), and outputs m and
// L - m share both sums: four multiply-adds for each of the (L/2)^2 pairs instead of
// four for each of the L^2 terms.  tw[m] = (c, s) of m (s carries the sign), in LDS.
template <int L, typename T2>
__device__ __forceinline__ void dft_regs(const T2* __restrict__ tw, T2 (&v)[L]) {
  constexpr int H = (L - 1) / 2;
  T2 a[H + 1], b[H + 1];
#pragma unroll
  for (int j = 1; j <= H; ++j) {
    a[j] = cmake<T2>(v[j].x + v[L - j].x, v[j].y + v[L - j].y);
    b[j] = cmake<T2>(v[j].x - v[L - j].x, v[j].y - v[L - j].y);
  }
  const T2 v0 = v[0], vh = v[L / 2];  // vh: the unpaired middle value of an even L
  T2 sum = v0, alt = v0;
#pragma unroll
  for (int j = 1; j <= H; ++j) {
    sum.x += a[j].x; sum.y += a[j].y;
    alt.x += (j & 1) ? -a[j].x : a[j].x;
    alt.y += (j & 1) ? -a[j].y : a[j].y;
  }
#pragma unroll
  for (int m = 1; m <= H; ++m) {
    T2 e = v0;
    if constexpr ((L & 1) == 0) {
      e.x += (m & 1) ? -vh.x : vh.x;
      e.y += (m & 1) ? -vh.y : vh.y;
    }
    T2 o = cmake<T2>(0, 0);
#pragma unroll
    for (int j = 1; j <= H; ++j) {
      const T2 w = tw[(j * m) % L];
      e.x = fma(w.x, a[j].x, e.x); e.y = fma(w.x, a[j].y, e.y);
      o.x = fma(-w.y, b[j].y, o.x); o.y = fma(w.y, b[j].x, o.y);
    }
    v[m] = cmake<T2>(e.x + o.x, e.y + o.y);
    v[L - m] = cmake<T2>(e.x - o.x, e.y - o.y);
  }
  v[0] = sum;
  if constexpr ((L & 1) == 0) {
    v[0] = cmake<T2>(sum.x + vh.x, sum.y + vh.y);
    constexpr bool neg = ((L / 2) & 1) != 0;
    v[L / 2] = cmake<T2>(alt.x + (neg ? -vh.x : vh.x), alt.y + (neg ? -vh.y : vh.y));
  }
}

template <typename T2, int L, int SIGN, typename Src, typename Dst>
__device__ __forceinline__ void dft_pass(const T2* __restrict__ tw, int npen, const Src& src, const Dst& dst) {
  for (int q = threadIdx.x; q < npen; q += blockDim.x) {
    const auto sp = src.at(q);
    const auto dp = dst.at(q);
    T2 v[L];
    if constexpr ((L & (L - 1)) == 0) {
#pragma unroll
      for (int j = 0; j < L; ++j) v[bitrev<L>(j)] = sp.ld(j);
      fft_regs<SIGN, L>(v);
#pragma unroll
      for (int m = 0; m < L; ++m) dp.put(m, v[m]);
    } else {
#pragma unroll
      for (int j = 0; j < L; ++j) v[j] = sp.ld(j);
      dft_regs<L>(tw, v);
#pragma unroll
      for (int m = 0; m < L; ++m) dp.put(m, v[m]);
    }
  }
}

// The last forward pass, the W product and the first backward pass fused along one
// k dimension: each thread keeps its pencil in registers through F_+, W and F_-, so
// the W product costs no LDS round trip (the 3-D transform is separable: the
// backward passes may run in the reverse dimension order).
template <typename T2, int L, typename Acc, typename Wf>
__device__ __forceinline__ void dft_pass_w(const T2* __restrict__ twp, const T2* __restrict__ twm, int npen,
                                           const Acc& acc_, const Wf& wf) {
  using T = typename Scalar<T2>::T;
  for (int q = threadIdx.x; q < npen; q += blockDim.x) {
    const auto p = acc_.at(q);
    const auto wp = wf.at(q);
    T2 v[L], u[L];
    if constexpr ((L & (L - 1)) == 0) {
#pragma unroll
      for (int j = 0; j < L; ++j) v[bitrev<L>(j)] = p.ld(j);
      fft_regs<1, L>(v);
#pragma unroll
      for (int m = 0; m < L; ++m) {
        const T w = wp.ld(m);
        u[bitrev<L>(m)] = cmake<T2>(v[m].x * w, v[m].y * w);
      }
      fft_regs<-1, L>(u);
#pragma unroll
      for (int m = 0; m < L; ++m) p.put(m, u[m]);
    } else {
#pragma unroll
      for (int j = 0; j < L; ++j) v[j] = p.ld(j);
      dft_regs<L>(twp, v);
#pragma unroll
      for (int m = 0; m < L; ++m) {
        const T w = wp.ld(m);
        u[m] = cmake<T2>(v[m].x * w, v[m].y * w);
      }
      dft_regs<L>(twm, u);
#pragma unroll
      for (int m = 0; m < L; ++m) p.put(m, u[m]);
    }
  }
}

template <typename T2, int LMAX, typename Acc, typename Wf>
__device__ __forceinline__ void dft_run_w(const T2* twp, const T2* twm, int npen, int L, const Acc& acc,
                                          const Wf& wf) {
  switch (L) {
    case 1: dft_pass_w<T2, 1>(twp, twm, npen, acc, wf); break;
    case 2: dft_pass_w<T2, 2>(twp, twm, npen, acc, wf); break;
    case 3: dft_pass_w<T2, 3>(twp, twm, npen, acc, wf); break;
    case 4: dft_pass_w<T2, 4>(twp, twm, npen, acc, wf); break;
    case 5: dft_pass_w<T2, 5>(twp, twm, npen, acc, wf); break;
    case 6: dft_pass_w<T2, 6>(twp, twm, npen, acc, wf); break;
    case 7: dft_pass_w<T2, 7>(twp, twm, npen, acc, wf); break;
    case 8: dft_pass_w<T2, 8>(twp, twm, npen, acc, wf); break;
    default:
      if constexpr (LMAX > 8) {
        switch (L) {
          case 9: dft_pass_w<T2, 9>(twp, twm, npen, acc, wf); break;
          case 10: dft_pass_w<T2, 10>(twp, twm, npen, acc, wf); break;
          case 12: dft_pass_w<T2, 12>(twp, twm, npen, acc, wf); break;
          case 16: dft_pass_w<T2, 16>(twp, twm, npen, acc, wf); break;
          default:
            if constexpr (LMAX > 16) {
              switch (L) {
                case 15: dft_pass_w<T2, 15>(twp, twm, npen, acc, wf); break;
                case 18: dft_pass_w<T2, 18>(twp, twm, npen, acc, wf); break;
                case 20: dft_pass_w<T2, 20>(twp, twm, npen, acc, wf); break;
                case 24: dft_pass_w<T2, 24>(twp, twm, npen, acc, wf); break;
                default: break;  // rejected on the host
              }
            }
            break;
        }
      }
      break;
  }
}

template <typename T2, int LMAX, int SIGN, typename Src, typename Dst>
__device__ __forceinline__ void dft_run(const T2* tw, int npen, int L, const Src& src, const Dst& dst) {
  switch (L) {
    case 1: dft_pass<T2, 1, SIGN>(tw, npen, src, dst); break;
    case 2: dft_pass<T2, 2, SIGN>(tw, npen, src, dst); break;
    case 3: dft_pass<T2, 3, SIGN>(tw, npen, src, dst); break;
    case 4: dft_pass<T2, 4, SIGN>(tw, npen, src, dst); break;
    case 5: dft_pass<T2, 5, SIGN>(tw, npen, src, dst); break;
    case 6: dft_pass<T2, 6, SIGN>(tw, npen, src, dst); break;
    case 7: dft_pass<T2, 7, SIGN>(tw, npen, src, dst); break;
    case 8: dft_pass<T2, 8, SIGN>(tw, npen, src, dst); break;
    default:
      if constexpr (LMAX > 8) {
        switch (L) {
          case 9: dft_pass<T2, 9, SIGN>(tw, npen, src, dst); break;
          case 10: dft_pass<T2, 10, SIGN>(tw, npen, src, dst); break;
          case 12: dft_pass<T2, 12, SIGN>(tw, npen, src, dst); break;
          case 16: dft_pass<T2, 16, SIGN>(tw, npen, src, dst); break;
          default:
            if constexpr (LMAX > 16) {
              switch (L) {
                case 15: dft_pass<T2, 15, SIGN>(tw, npen, src, dst); break;
                case 18: dft_pass<T2, 18, SIGN>(tw, npen, src, dst); break;
                case 20: dft_pass<T2, 20, SIGN>(tw, npen, src, dst); break;
                case 24: dft_pass<T2, 24, SIGN>(tw, npen, src, dst); break;
                default: break;  // rejected on the host
              }
            }
            break;
        }
      }
      break;
  }
}

__device__ void mred_rows(const double2* __restrict__ apart, const double2* __restrict__ K,
                          double2* __restrict__ hmult, int np, int nj, int nj0, double mul, int r, double2* lds);

// Strip of G consecutive phi columns (c = x*na + a) per workgroup, all nk rows:
//   pass 1 (K3, F_+): HBM -> registers -> LDS, with W(x, :) staged beside it
//   pass 2 (K2, F_+)
//   pass 3 (K1): F_+, the W product and F_- on each pencil in registers
//   passes 4, 5 (K2, K3, F_-), the last one scaling by 1/N_k into HBM.
// nred > 0 prepends that many workgroups running the multiplet reduction, which
// is independent of phi and overlaps the transform.
// PHS (the OBF form, long_range.f90:388-406): phi is multiplied by phs(k, x) as it
// is read and the result by conj(phs(k, x)) as it is written.
template <typename T2, int LMAX, bool PHS = false>
__device__ __forceinline__ void fft_body(const ActArgs<T2>& A, int blk) {
  using T = typename Scalar<T2>::T;
  extern __shared__ __align__(16) unsigned char smem[];
  // the reduction workgroups come first so that they are dispatched first
  const int nred = A.nred, nfft = A.nfft;
  if (blk < nred) {
    mred_rows(A.apart, A.Kmat, A.hmult, A.nm, A.nj, A.na0 * A.P, A.mul, blk, reinterpret_cast<double2*>(smem));
    return;
  }
  if (blk < nred + A.nfin) {
    const int it = hay_it(A.hay);
    if (it >= 2) hay_fin(A.hay, it - 1, A.na / A.na0);
    return;
  }
  const int nk = A.nk, ncol = A.ncol, na = A.na, G = A.G, ldphi = A.ldphi;
  const int K1 = A.K1, K2 = A.K2, K3 = A.K3;
  T2* phi = A.phi;
  const T* W = A.W;
  // twiddles: [dim][sign][m], dims ordered (K3, K2, K1), 2 * LMAX per dim
  T2* twl = reinterpret_cast<T2*>(smem);
  T2* lds = twl + 6 * LMAX;                               // [k][g], rows padded (tile_pad)
  T* wl = reinterpret_cast<T*>(lds + tile_size(K1, K2, K3, G));  // W(x, :) of the strip
  const int Ks[3] = {K3, K2, K1};
  // the LDS twiddle table serves the direct sums of non-power-of-two edges only
  const bool direct = ((K1 & (K1 - 1)) | (K2 & (K2 - 1)) | (K3 & (K3 - 1))) != 0;
  for (int t = threadIdx.x; direct && t < 6 * LMAX; t += blockDim.x) {
    const int d = t / (2 * LMAX), rem = t - d * 2 * LMAX, sg = rem / LMAX, m = rem - sg * LMAX;
    const int L = Ks[d];
    T sn = 0, cs = 1;
    if (m < L) {
      if constexpr (sizeof(T) == 8) sincospi((double)(2 * m) / (double)L, &sn, &cs);
      else sincospif((float)(2 * m) / (float)L, &sn, &cs);
    }
    twl[t] = cmake<T2>(cs, sg == 0 ? sn : -sn);  // sg 0: +1 (backward), 1: -1 (forward)
  }
  // Workgroups are dispatched round-robin over the 8 XCDs; remap so that
  // consecutive column strips (which share 128-B lines) run on the same XCD and
  // therefore hit the same L2.
  int b = blk - nred - A.nfin;
  if ((nfft & 7) == 0) b = (b & 7) * (nfft >> 3) + (b >> 3);
  const int c0 = b * G;
  const int gcnt = min(G, ncol - c0);
  const int xlo = c0 / na, xhi = (c0 + gcnt - 1) / na;
  const int nwl = (xhi - xlo + 1) * nk;
  const T* wsrc = W + (size_t)xlo * nk;
  // W loads issued ahead of the first pass, written to LDS after it
  constexpr int kWR = 4;
  T wr[kWR];
#pragma unroll
  for (int i = 0; i < kWR; ++i) wr[i] = wsrc[min((int)threadIdx.x + i * (int)blockDim.x, nwl - 1)];
  __syncthreads();  // twiddles
  const int pad = tile_pad(K3, G), P2 = K3 * G + pad, P1 = K2 * P2, n = nk * G;
  const float rG = 1.0f / (float)G, rG3 = 1.0f / (float)(K3 * G), rna = 1.0f / (float)na;
  const int off = c0 - xlo * na;
  const PhiPass<T2, PHS> hbm{{phi + c0, (size_t)ldphi, rG, G, gcnt, K3, 1},
                             PHS ? A.phs + (size_t)xlo * nk : nullptr, rna, off, nk, K3, (T)1 / (T)nk};
  const LdsPass<T2> l3{lds, rG, P2 - G, G}, l2{lds, rG3, P1 - K3 * G, P2}, l1{lds, rG3, pad, P1};
  dft_run<T2, LMAX, 1>(twl + 0 * LMAX, n / K3, K3, hbm, l3);
#pragma unroll
  for (int i = 0; i < kWR; ++i) {
    const int idx = threadIdx.x + i * blockDim.x;
    if (idx < nwl) wl[idx] = wr[i];
  }
  for (int idx = threadIdx.x + kWR * blockDim.x; idx < nwl; idx += blockDim.x) wl[idx] = wsrc[idx];
  __syncthreads();
  dft_run<T2, LMAX, 1>(twl + 2 * LMAX, n / K2, K2, l2, l2);
  __syncthreads();
  // K1: F_+, W, F_- in registers
  dft_run_w<T2, LMAX>(twl + 4 * LMAX, twl + 5 * LMAX, n / K1, K1, l1,
                      WPass<T>{wl, rG, rna, G, gcnt, off, nk, K2 * K3});
  __syncthreads();
  dft_run<T2, LMAX, -1>(twl + 3 * LMAX, n / K2, K2, l2, l2);
  __syncthreads();
  dft_run<T2, LMAX, -1>(twl + 1 * LMAX, n / K3, K3, l3, hbm);
}

template <typename T2, int LMAX, bool PHS = false>
__global__ __launch_bounds__(256) void k_fft_w(const ActArgs<T2> A) {
  if (skipped(A)) return;
  fft_body<T2, LMAX, PHS>(A, blockIdx.x);
}

template <typename T2, int LMAX>
__global__ __launch_bounds__(256) void k_fft_w_batch(const ActArgs<T2>* __restrict__ As,
                                                     const int* __restrict__ off, int np) {
  const int p = find_problem(off, np, blockIdx.x);
  const ActArgs<T2> A = As[p];
  if (skipped(A)) return;
  fft_body<T2, LMAX>(A, blockIdx.x - off[p]);
}

// ---------------------------------------------------------------------------
// Differentiation: the forward half of the transform, P = F_+ (U A v), with no W
// and no scaling (in place on phi), and the contraction of two such fields into
// the W-derivative of <y|H_lr|x>:
//   d<y|H_lr|x>/dW(k,x) = -(1/N_k) sum_a conj(P_y(k,x,a)) P_x(k,x,a)
// (H_lr = -sum_x A U_x^+ (N_k^-1 F_- W_x F_+) U_x A with F_- = F_+^+).
// ---------------------------------------------------------------------------
template <typename T2, int LMAX>
__global__ __launch_bounds__(256) void k_fft_fwd(const ActArgs<T2> A) {
  using T = typename Scalar<T2>::T;
  extern __shared__ __align__(16) unsigned char smem[];
  T2* twl = reinterpret_cast<T2*>(smem);  // [dim][m], exp(+2 pi i m / L), dims (K3, K2, K1)
  T2* lds = twl + 3 * LMAX;
  const int nk = A.nk, ncol = A.ncol, G = A.G, ldphi = A.ldphi;
  const int Ks[3] = {A.K3, A.K2, A.K1};
  const bool direct = ((A.K1 & (A.K1 - 1)) | (A.K2 & (A.K2 - 1)) | (A.K3 & (A.K3 - 1))) != 0;
  for (int t = threadIdx.x; direct && t < 3 * LMAX; t += blockDim.x) {
    const int d = t / LMAX, m = t - d * LMAX;
    const int L = Ks[d];
    T sn = 0, cs = 1;
    if (m < L) {
      if constexpr (sizeof(T) == 8) sincospi((double)(2 * m) / (double)L, &sn, &cs);
      else sincospif((float)(2 * m) / (float)L, &sn, &cs);
    }
    twl[t] = cmake<T2>(cs, sn);
  }
  __syncthreads();
  int b = blockIdx.x;
  const int nfft = gridDim.x;
  if ((nfft & 7) == 0) b = (b & 7) * (nfft >> 3) + (b >> 3);
  const int c0 = b * G;
  const int gcnt = min(G, ncol - c0);
  const int K1 = A.K1, K2 = A.K2, K3 = A.K3;
  const int pad = tile_pad(K3, G), P2 = K3 * G + pad, P1 = K2 * P2, n = nk * G;
  const float rG = 1.0f / (float)G, rG3 = 1.0f / (float)(K3 * G);
  const HbmPass<T2> h3{A.phi + c0, (size_t)ldphi, rG, G, gcnt, K3, 1};
  const HbmPass<T2> h1{A.phi + c0, (size_t)ldphi, rG, G, gcnt, 1, K2 * K3};
  const LdsPass<T2> l3{lds, rG, P2 - G, G}, l2{lds, rG3, P1 - K3 * G, P2}, l1{lds, rG3, pad, P1};
  dft_run<T2, LMAX, 1>(twl + 0 * LMAX, n / K3, K3, h3, l3);
  __syncthreads();
  dft_run<T2, LMAX, 1>(twl + 1 * LMAX, n / K2, K2, l2, l2);
  __syncthreads();
  dft_run<T2, LMAX, 1>(twl + 2 * LMAX, n / K1, K1, l1, h1);
}

// Q[k][x] += coef * Im sum_a conj(PY(k,x,a)) PX(k,x,a); one thread per (k, x), each
// element updated by one thread per launch (deterministic over energies).
template <typename T2>
__global__ void k_wgrad(const T2* __restrict__ PX, const T2* __restrict__ PY, int nk, int nx, int na,
                        int ldphi, double coef, double* __restrict__ Q) {
  const size_t tot = (size_t)nk * nx;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (size_t)gridDim.x * blockDim.x) {
    const int k = (int)(e / nx), x = (int)(e - (size_t)k * nx);
    const T2* px = PX + (size_t)k * ldphi + (size_t)x * na;
    const T2* py = PY + (size_t)k * ldphi + (size_t)x * na;
    double im = 0.0;
    for (int a = 0; a < na; ++a) {
      const T2 p = px[a], q = py[a];
      im += (double)q.x * (double)p.y - (double)q.y * (double)p.x;
    }
    Q[e] += coef * im;
  }
}

// h(i) = mul * sum_j K(i, j) amp(j): direct -mpm a plus exchange X a
// (OCEAN_multiplet.f90:1812-1936), where amp are the summed partials.  With several
// right-hand sides K is block diagonal over blocks of nj0 amplitudes and a row sums its own
// block only (so a NaN in one right-hand side stays there).  Run by extra workgroups of
// another kernel's grid, or on their own (k_mred): workgroup r forms
// kRedPerBlock rows of h.  Every workgroup sums the np partials of all nj0 amplitudes of
// its rows' right-hand side (64 x 64 to 64 x 192 values, from L2) and applies its rows of
// K to them, so that no workgroup waits for another: with the amplitudes shared out
// over the workgroups and K applied by the last to arrive, the chain of partials,
// counter, amplitudes and K was the longest workgroup of a small problem's transform.
// The four waves of a workgroup sum 16 partials each, pairwise; their sums are added in
// order.
constexpr int kRedPerBlock = 4;

// LDS of one reduction workgroup of nw waves
constexpr size_t mred_lds(int nj0, int nw) { return (size_t)nj0 * nw * sizeof(double2); }

__device__ void mred_rows(const double2* __restrict__ apart, const double2* __restrict__ K,
                          double2* __restrict__ hmult, int np, int nj, int nj0, double mul, int r, double2* lds) {
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const int i0 = r * kRedPerBlock, jb = i0 - i0 % nj0;  // nj0 is a multiple of the four rows
  constexpr int MW = kMultBlocks / (kBlock / 64), B = 8;
  for (int j = lane; j < nj0; j += 64) {
    double2 a = make_double2(0.0, 0.0);
#pragma unroll 1
    for (int m0 = wid * MW; m0 < min(wid * MW + MW, np); m0 += B) {
      double2 v[B];
#pragma unroll
      for (int q = 0; q < B; ++q) v[q] = apart[(size_t)min(m0 + q, np - 1) * nj + jb + j];
#pragma unroll
      for (int q = 0; q < B; ++q)
        if (m0 + q >= np) v[q] = make_double2(0.0, 0.0);
#pragma unroll
      for (int d = 1; d < B; d <<= 1)
#pragma unroll
        for (int q = 0; q < B; q += 2 * d) { v[q].x += v[q + d].x; v[q].y += v[q + d].y; }
      a.x += v[0].x; a.y += v[0].y;
    }
    lds[wid * nj0 + j] = a;
  }
  __syncthreads();
  for (int i = i0 + wid; i < min(i0 + kRedPerBlock, nj); i += nw) {
    double2 acc = make_double2(0.0, 0.0);
    for (int j = lane; j < nj0; j += 64) {
      const double2 kv = K[(size_t)i * nj + jb + j];
      double2 a = lds[j];
      for (int q = 1; q < nw; ++q) { a.x += lds[q * nj0 + j].x; a.y += lds[q * nj0 + j].y; }
      cfma(acc, kv, a);
    }
    acc.x = wave_sum(acc.x);
    acc.y = wave_sum(acc.y);
    if (lane == 0) hmult[i] = make_double2(acc.x * mul, acc.y * mul);
  }
}

// The reduction on its own, where the long-range term is off and there is no transform to
// ride on: rows of four per workgroup as there.  With all rows in one workgroup the 64 partials
// of an amplitude were one thread's serial chain: 64 amplitudes 20.0 -> 4.0 us (and 12.8 with
// one partial per k, before they were blocked).
__global__ __launch_bounds__(kBlock) void k_mred(const double2* __restrict__ apart, const double2* __restrict__ K,
                                                 double2* __restrict__ hmult, int np, int nj, int nj0, double mul) {
  extern __shared__ __align__(16) unsigned char smem[];
  mred_rows(apart, K, hmult, np, nj, nj0, mul, blockIdx.x, reinterpret_cast<double2*>(smem));
}

// ---------------------------------------------------------------------------
// Adjoint projection fused with the whole epilogue of OCEAN_xact:
//   lr(n,k,a)  = - sum_x conj(u(n,k,x)) phi'(k,x,a)         long_range.f90:943-961
//   fg(n,k,a)  =   sum_p conj(c(n,k,p)) h(p,a)               OCEAN_multiplet.f90:1943-1998
//   out        =   E.psi + A.(fg + lr) + S psi                OCEAN_action.f90:337-372, :596-608
// Reads the transposed copy uT[s][k][x][n] (band index fastest): lanes run over
// bands, so every wave load is a contiguous band row, phi'(k,x,:) is the same
// for all lanes of a row (an LDS broadcast), and no cross-lane reduction is
// needed until the XS x-splits of the workgroup are summed once at the end.
// The projector rows c(:,k,p) have the same band-fastest shape and are streamed
// by the same threads (p split like x).  Every operand of the epilogue and the
// projector rows are loaded before the u stream starts, so their latency hides
// under it: with one k per workgroup the whole grid is resident at once and any
// load left to the end would be paid by every workgroup together.
// One workgroup per k; threads (n, xs) with n fastest, in whole waves (the threads past
// nb XS only stage and finish).  JR alphas per reduction round through LDS (the
// reduction buffer reuses the phi' staging area).
// ---------------------------------------------------------------------------
template <typename T2, int NA, bool HAY>
__device__ __forceinline__ void adj_body(const ActArgs<T2>& A, int blk) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int nb = A.nb, nk = A.nk, nx = A.nx, na = A.na, ns = A.ns, P = A.P;
  const int XC = A.XC, JR = A.JR, flags = A.flags, ldT = A.ldT, ldphi = A.ldphi;
  const T2* __restrict__ uT = A.uT;
  const T2* __restrict__ phi = A.phi;
  const double2* __restrict__ psi = A.psi;
  const double2* __restrict__ energy = A.energy;
  const double* __restrict__ allow = A.allow;
  const double2* __restrict__ cproj = A.cproj;
  const double2* __restrict__ hmult = A.hmult;
  const double2* __restrict__ S = A.S;
  double2* __restrict__ out = A.out;
  const int XS = blockDim.x / nb;  // x-splits (host guarantees nb <= blockDim.x)
  double2* res = reinterpret_cast<double2*>(smem);           // [na][nb]
  T2* ph = reinterpret_cast<T2*>(res + na * nb);              // [XC][NA] during the stream
  double2* red = res + na * nb;                               // [XS][JR][nb] afterwards
  // XCD-major workgroup order so that consecutive k share an XCD (phi' rows of
  // neighbouring k are adjacent in memory)
  int kk = blk;
  const int nblk = nk;
  if ((nblk & 7) == 0) kk = (kk & 7) * (nblk >> 3) + (kk >> 3);
  const int k = kk;
  const int t = threadIdx.x, bd = blockDim.x;
  const int n = t % nb, xs = t / nb;
  const bool active = xs < XS;
  const bool lr = (flags & F_LR) != 0;
  const bool fg = (flags & F_FG) != 0;
  const int nel = na * nb;
  const int na0 = A.na0;
  // epilogue operands of the first kEP elements owned by this thread
  constexpr int kEP = HAY ? 1 : 2;  // (a recursion holds more per element)
  const int it = HAY ? hay_it(A.hay) : 0;
  HayScal hs0 = {1.0, 0.0, 0.0};
  double2 e_psi[kEP], e_en[kEP], e_old[kEP];
  double e_m[kEP];
  auto operands = [&]() {
#pragma unroll
    for (int i = 0; i < kEP; ++i) {
      const int e = min(t + i * bd, nel - 1);
      const int a = e / nb, nn = e - a * nb;
      const size_t off = ((size_t)a * nk + k) * nb + nn;
      e_psi[i] = psi[off];
      e_en[i] = energy[off];
      e_m[i] = allow[off];
    }
  };
  // Beside a recursion's own operands these cost registers: a second workgroup per CU was
  // lost with all of them held through the stream (a batch of FP32 problems 92 -> 127
  // us).  So the recursion's come behind it, in FP64 the others too (50.6 against 51.7 us
  // at 512 k points and 64 bands; FP32 31.7 against 31.2).
  constexpr bool kPre = !HAY || sizeof(T2) == 8;
  if constexpr (kPre) operands();

  const int astep = (ns == 2) ? 2 : 1;
  const int acnt = (ns == 2) ? na / 2 : na;
  for (int s = 0; s < ns; ++s) {
    // projector rows p = xs + i XS of this spin, issued first
    constexpr int kCP = 2;
    const double2* cb = cproj + ((size_t)s * nk + k) * P * nb + n;
    double2 cpre[kCP];
    if (fg && P > 0) {
#pragma unroll
      for (int i = 0; i < kCP; ++i) cpre[i] = cb[(size_t)min(xs + i * XS, P - 1) * nb];
    }
    T2 acc[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) acc[j] = cmake<T2>(0, 0);
    if (lr) {
      const T2* ub = uT + ((size_t)s * nk + k) * ldT;
      for (int x0 = 0; x0 < nx; x0 += XC) {
        const int xc = min(XC, nx - x0);
        const int tot = xc * acnt;
        __syncthreads();
        for (int e0 = t; e0 < tot; e0 += 4 * bd) {
          T2 v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int e = min(e0 + i * bd, tot - 1);
            const int xl = e / acnt, j = e - xl * acnt;
            v[i] = phi[(size_t)k * ldphi + (size_t)(x0 + xl) * na + s + j * astep];
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int e = e0 + i * bd;
            if (e < tot) {
              const int xl = e / acnt, j = e - xl * acnt;
              ph[xl * NA + j] = v[i];
            }
          }
        }
        __syncthreads();
        if (active) {
          // kB independent row loads in flight per wave (addresses clamped, use
          // predicated): 128 bytes per lane in both precisions
          constexpr int kB = sizeof(T2) == 16 ? 8 : 16;
          for (int xb = xs; xb < xc; xb += kB * XS) {
            T2 uv[kB];
#pragma unroll
            for (int i = 0; i < kB; ++i) {
              const int xl = min(xb + i * XS, xc - 1);
              uv[i] = ld_stream(ub + (size_t)(x0 + xl) * nb + n);
            }
            __builtin_amdgcn_sched_barrier(0);
            // one row's NA phi' values at a time: with many alphas, letting the
            // compiler hoist the LDS reads of several rows costs occupancy
#pragma unroll
            for (int i = 0; i < kB; ++i) {
              const int xl = xb + i * XS;
              if (xl < xc) {
                if constexpr (NA >= 6) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < NA; ++j) cfmac(acc[j], uv[i], ph[xl * NA + j]);
              }
            }
          }
        }
      }
    }
    // this thread's share: fg - lr per alpha, in FP64
    double2 part[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) part[j] = make_double2(-(double)acc[j].x, -(double)acc[j].y);
    if (fg && active) {
#pragma unroll
      for (int i = 0; i < kCP; ++i) {
        const int p = xs + i * XS;
        if (p < P) {
#pragma unroll
          for (int j = 0; j < NA; ++j)
            if (j < acnt) cfmac(part[j], cpre[i], hmult[(s + j * astep) * P + p]);
        }
      }
      for (int p = xs + kCP * XS; p < P; p += XS) {
        const double2 cv = cb[(size_t)p * nb];
#pragma unroll
        for (int j = 0; j < NA; ++j)
          if (j < acnt) cfmac(part[j], cv, hmult[(s + j * astep) * P + p]);
      }
    }
    // sum the x-splits, JR alphas per round
    for (int j0 = 0; j0 < acnt; j0 += JR) {
      __syncthreads();
      if (active) {
#pragma unroll
        for (int j = 0; j < NA; ++j)
          if (j >= j0 && j < j0 + JR && j < acnt) red[(xs * JR + (j - j0)) * nb + n] = part[j];
      }
      __syncthreads();
      const int jn = min(JR, acnt - j0);
      for (int e = t; e < jn * nb; e += bd) {
        const int jj = e / nb, nn = e - jj * nb;
        double2 sum = make_double2(0.0, 0.0);
        for (int q = 0; q < XS; ++q) {
          const double2 r = red[(q * JR + jj) * nb + nn];
          sum.x += r.x;
          sum.y += r.y;
        }
        res[(s + (j0 + jj) * astep) * nb + nn] = sum;
      }
    }
  }
  if constexpr (HAY) {
    if constexpr (!kPre) operands();
    hs0 = hay_scal(A.hay, it, 0);
#pragma unroll
    for (int i = 0; i < kEP; ++i) {
      const int e = min(t + i * bd, nel - 1), a = e / nb;
      e_old[i] = A.hay.old[((size_t)a * nk + k) * nb + e - a * nb];
    }
  }
  __syncthreads();
  const bool back = (flags & F_BACK) != 0;
  auto finish = [&](int e, double2 pv, double2 ev, double am, double2 ov) {
    const int a = e / nb, nn = e - a * nb;
    const size_t off = ((size_t)a * nk + k) * nb + nn;
    double2 inter = res[e];
    inter.x *= am;
    inter.y *= am;
    if (flags & F_SO) {
      // S mixes the alphas of one right-hand side: rows a0 .. a0 + na0 - 1
      const int ar = a % na0, a0 = a - ar;
      for (int b = 0; b < na0; ++b) {
        double2 sab = S[ar * na0 + b];
        if (back) sab.y = -sab.y;
        cfma(inter, sab, psi[((size_t)(a0 + b) * nk + k) * nb + nn]);
      }
    }
    HayScal hs = hs0;
    if constexpr (HAY) {
      if (a >= na0) hs = hay_scal(A.hay, it, a / na0);
      pv.x *= hs.sc; pv.y *= hs.sc;
      inter.x *= hs.sc; inter.y *= hs.sc;
    }
    double2 r = inter;
    if (flags & F_E0) {
      if (back) ev.y = -ev.y;
      r.x = ev.x * pv.x - ev.y * pv.y + inter.x;
      r.y = ev.x * pv.y + ev.y * pv.x + inter.y;
    }
    if constexpr (HAY) res[e] = hay_elem(hs, pv, ov, r);
    out[off] = axmy_epilogue(A, pv, r);
  };
#pragma unroll
  for (int i = 0; i < kEP; ++i)
    if (t + i * bd < nel) finish(t + i * bd, e_psi[i], e_en[i], e_m[i], e_old[i]);
  for (int e = t + kEP * bd; e < nel; e += bd) {
    const int a = e / nb, nn = e - a * nb;
    const size_t off = ((size_t)a * nk + k) * nb + nn;
    finish(e, psi[off], energy[off], allow[off], HAY ? A.hay.old[off] : make_double2(0.0, 0.0));
  }
  if constexpr (HAY) {
    __syncthreads();
    // one wave per right-hand side: bd is a whole number of waves, at least one
    for (int q = t >> 6; q < na / na0; q += bd >> 6) hay_part(A.hay, res + q * na0 * nb, na0 * nb, q, k);
    if (A.hay.itp && blk == 0 && t == 0) A.hay.itp[1] = it;
  }
}

// One problem: one workgroup per k.
template <typename T2, int NA, bool HAY>
__global__ __launch_bounds__(512) void k_adj(const ActArgs<T2> A) {
  if (skipped(A)) return;
  adj_body<T2, NA, HAY>(A, blockIdx.x);
}

template <typename T2, int NA, bool HAY>
__global__ __launch_bounds__(512) void k_adj_batch(const ActArgs<T2>* __restrict__ As,
                                                   const int* __restrict__ off, int np) {
  const int p = find_problem(off, np, blockIdx.x);
  const ActArgs<T2> A = As[p];
  if (skipped(A)) return;
  adj_body<T2, NA, HAY>(A, blockIdx.x - off[p]);
}

}  // namespace og
