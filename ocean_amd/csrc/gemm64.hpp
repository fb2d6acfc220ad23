// FP64 matrix-core GEMM pieces shared by the OBF x-side products and the matrix-core
// adjoint of the many-alpha edges.
#pragma once
#include "action.hpp"
#include "common.hpp"

namespace og {

// Complex GEMMs on the FP64 matrix cores: v_mfma_f64_16x16x4f64, where lane l
// supplies A[l % 16][l / 16] and B[l / 16][l % 16] and receives D[l / 16 + 4 r]
// [l % 16], r = 0..3 (measured on gfx950; the FP32 16x16x4 form returns rows
// 4 (l / 16) + r instead).  The complex product is a real GEMM with the complex parts
// unrolled along K: for every group of four K indices (kk = l / 16) the first
// instruction takes the real parts of A and the second the imaginary parts, with
// B[(kk, re)][(col, c)] and B[(kk, im)][(col, c)] formed from the lane's own complex
// B element, so each lane loads one complex A element per M tile and one complex B
// element per group.  Output columns are flattened as G = 2 (k nalpha + a) + c
// (c = real/imaginary part); an N tile is 16 consecutive G.

struct MfCol {
  int k, a, c;
  bool ok;
};
__device__ __forceinline__ MfCol mf_col(int G, int na, int nk) {
  MfCol r;
  r.k = G / (2 * na);
  r.a = (G >> 1) % na;
  r.c = G & 1;
  r.ok = r.k < nk;
  r.k = min(r.k, nk - 1);
  return r;
}

// The adjoint for the many-alpha edges (one spin), on the matrix cores:
//   lr(n, k, a) = sum_x conj(uT(k, x, n)) phi'(k, x, a)          (long_range.f90:943-961)
// as a GEMM per k (M = bands, N = the 2 nalpha real columns, K = x) in the precision
// of the stored u (FP64, or FP32 accumulating in FP32 for the mixed form), followed
// in the same workgroup by the rest of OCEAN_xact for its 64 bands:
//   fg(n, k, a)  = sum_p conj(c(n, k, p)) h(p, a)                  OCEAN_multiplet.f90:1943-1998
//   out          = E psi + A (fg - lr) + S psi                     OCEAN_action.f90:337-372, :596-608
// (and c psi - H psi for a GMRES step).  The VALU adjoint reads each phi'(k, x, :) as
// nalpha LDS broadcasts per band row, which bounds it at twelve alphas; here
// phi'(k, x, :) is the B operand.  Workgroup: 64 bands (four M tiles) by all N tiles
// of one k on four waves, so every uT element is read once; a grid that would leave
// compute units idle takes 32 bands on eight waves instead (60 k points, 37 bands, 1000
// x: FP64 52 -> 30 us, FP32 53 -> 27).  Its waves take the x groups in turn, so that it
// reads one contiguous stretch of uT at a time, and their tiles are added in LDS in a
// fixed order.  The epilogue then gives a thread one band and every AS-th alpha: rows
// of c and the element's own psi, E and allow are coalesced band rows, h(p, a) is
// uniform across a wave of 64 bands, and the spin-orbit term reads psi(:, k, n) and S
// staged in the LDS area the tiles leave free.
// It is bound by the uT stream, in FP64 with the matrix cores half busy beside it.  512 k
// points, 128 bands, 1000 x, 12 alphas, us: FP64 242 -> 227 (5.3 TB/s), FP32 153 -> 132
// (16-byte loads; 4.8 TB/s); 64 bands, 512 x: 12 alphas 71 and 50 -> 47, 24 alphas
// 100 -> 86 and 61 -> 60.

// Loads of uT: 16 bytes per lane, one band in FP64, two adjacent ones in FP32 (a row of
// an odd number of bands starts on 8 bytes; the last pair may take one element past the
// row, which ldT's padding covers on the last row of a slab).
template <typename T2> struct AdjLoad;
template <> struct AdjLoad<double2> {
  using F = double2;
  static constexpr int N = 1;
  static __device__ __forceinline__ F ld(const double2* p) { return ld_stream(p); }
};
template <> struct AdjLoad<float2> {
  using F = float4;
  static constexpr int N = 2;
  static __device__ __forceinline__ F ld(const float2* p) {
    typedef float v4f __attribute__((ext_vector_type(4), aligned(8)));
    const v4f t = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(p));
    return make_float4(t.x, t.y, t.z, t.w);
  }
};

// LDS of the adjoint: two waves' tiles, later psi and S for the spin-orbit term
template <typename T, int NA, int MT>
constexpr size_t adj_lr_lds() {
  const size_t tiles = 2 * ((2 * NA + 15) / 16) * 4 * MT * 64 * sizeof(T);
  const size_t so = sizeof(double2) * (NA * 16 * MT + 12 * 12);
  return tiles > so ? tiles : so;
}

// MT M tiles of 16 bands and W waves per workgroup, D groups of four x in a wave's ring.
template <typename T2, int NA, int MT, int W, int D>
__device__ __forceinline__ void adj_lr_body(const ActArgs<T2>& A, int bx, int k) {
  using T = typename Scalar<T2>::T;
  using M = Mf<T>;
  using V = typename M::V;
  using L = AdjLoad<T2>;
  using F = typename L::F;
  constexpr int NT = (2 * NA + 15) / 16, NL = MT / L::N, BN = 16 * MT;
  __shared__ __align__(16) unsigned char smem[adj_lr_lds<T, NA, MT>()];
  T(*part)[NT * 4 * MT][64] = reinterpret_cast<T(*)[NT * 4 * MT][64]>(smem);
  const T2* __restrict__ uT = A.uT;
  const T2* __restrict__ phi = A.phi;
  const int nb = A.nb, nk = A.nk, nx = A.nx, ldT = A.ldT, ldphi = A.ldphi;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, kk = lane >> 4;
  const int n0 = bx * BN;
  int cc[NT];
  const T2* yp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int G = t * 16 + i;
    cc[t] = G & 1;
    yp[t] = phi + (size_t)k * ldphi + min(G >> 1, NA - 1);
  }
  const T2* __restrict__ ap = uT + (size_t)k * ldT;
  int nrow[NL];
#pragma unroll
  for (int m = 0; m < NL; ++m) nrow[m] = min(n0 + 16 * L::N * m + L::N * i, nb - 1);
  // wave w takes groups w, w + W, ... of four x, so that the workgroup reads one
  // contiguous stretch of rows at a time
  const int xa = 4 * w, xst = 4 * W;
  // epilogue: thread (band nl, alphas a0 + AS j); the element's own operands are in flight
  // during the stream, or every workgroup of a grid that is resident at once would wait
  // for them together at its end
  constexpr int AS = 64 * W / BN, APW = (NA + AS - 1) / AS;
  const int nl = threadIdx.x % BN, n = n0 + nl, nn = min(n, nb - 1);
  const int a0 = BN == 64 ? w : (int)threadIdx.x / BN;
  const bool hay = A.hay.s != nullptr;
  const int it = hay_it(A.hay);
  double2 pv[APW], ev[APW], ov[APW];
  double am[APW];
#pragma unroll
  for (int j = 0; j < APW; ++j) {
    const int a = min(a0 + AS * j, NA - 1);
    const size_t off = ((size_t)a * nk + k) * nb + nn;
    pv[j] = A.psi[off];
    ev[j] = A.energy[off];
    am[j] = A.allow[off];
    ov[j] = hay ? A.hay.old[off] : make_double2(0.0, 0.0);
  }
  V acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = V{0, 0, 0, 0};
  // without the long-range term (nhflag) only the epilogue runs: lr = 0
  if (A.flags & F_LR) {
    // a ring of D groups of four x in registers: the loads of group g + D - 1 are issued
    // before the products of group g
    T2 yv[D][NT];
    F av[D][NL];
    auto load = [&](int xs, T2 (&yn)[NT], F (&an)[NL]) {
      const int x = max(min(xs + kk, nx - 1), 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) yn[t] = yp[t][(size_t)x * NA];
#pragma unroll
      for (int m = 0; m < NL; ++m) an[m] = L::ld(ap + (size_t)x * nb + nrow[m]);
    };
    // C = conj(A) Y: re: ar yr + ai yi, im: ar yi - ai yr
    auto step = [&](int xs, const T2 (&yv)[NT], const F (&av)[NL]) {
      const bool ok = xs + kk < nx;
      T b0[NT], b1[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const T2 y = ok ? yv[t] : cmake<T2>(0, 0);
        b0[t] = cc[t] ? y.y : y.x;
        b1[t] = cc[t] ? -y.x : y.y;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < NL; ++m) {
          acc[t][L::N * m] = M::step(av[m].x, b0[t], acc[t][L::N * m]);
          if constexpr (L::N == 2) acc[t][2 * m + 1] = M::step(av[m].z, b0[t], acc[t][2 * m + 1]);
        }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < NL; ++m) {
          acc[t][L::N * m] = M::step(av[m].y, b1[t], acc[t][L::N * m]);
          if constexpr (L::N == 2) acc[t][2 * m + 1] = M::step(av[m].w, b1[t], acc[t][2 * m + 1]);
        }
    };
#pragma unroll
    for (int d = 0; d < D - 1; ++d) load(xa + xst * d, yv[d], av[d]);
    for (int xs = xa; xs < nx; xs += xst * D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        load(xs + xst * (d + D - 1), yv[(d + D - 1) % D], av[(d + D - 1) % D]);
        asm volatile("" ::: "memory");  // keep the later groups' loads ahead of this group's products
        step(xs + xst * d, yv[d], av[d]);
      }
    }
  }
  // pairs of waves pass their tiles to waves 0 and 1, whose sums the epilogue adds (parking
  // every wave's tiles held the FP64 form to two workgroups per CU)
  auto park = [&](int q) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[q][4 * (MT * t + m) + r][lane] = acc[t][m][r];
  };
#pragma unroll
  for (int q = W - 2; q > 0; q -= 2) {
    if (w == q || w == q + 1) park(w - q);
    __syncthreads();
    if (w < 2) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[t][m][r] += part[w][4 * (MT * t + m) + r][lane];
    }
    if (q > 2) __syncthreads();
  }
  if (w < 2) park(w);
  __syncthreads();

  // ---- epilogue ----
  // lr of this thread's band: column G = 2 a + c of tile t = G / 16 sits at lane group
  // i = G % 16; band row nl = N (16 (m / N) + the instruction's output row of (kk, r)) + m % N
  const int mrow = L::N * (nl / (16 * L::N)) + nl % L::N, row = (nl / L::N) & 15;
  const int lkk = M::kk_of(row), lr_ = M::r_of(row);
  double2 res[APW];
#pragma unroll
  for (int j = 0; j < APW; ++j) {
    const int a = min(a0 + AS * j, NA - 1);
    double v[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int G = 2 * a + c, t = G >> 4, gi = G & 15;
      const int rr = 4 * (MT * t + mrow) + lr_, cl = lkk * 16 + gi;
      v[c] = (double)(part[0][rr][cl] + part[1][rr][cl]);
    }
    res[j] = make_double2(-v[0], -v[1]);  // fg - lr starts at -lr
  }
  const int flags = A.flags;
  const bool back = (flags & F_BACK) != 0;
  const bool so = (flags & F_SO) != 0;
  const int na0 = A.na0;
  __syncthreads();  // every lane has its lr: the tile area is free
  double2* Ps = reinterpret_cast<double2*>(smem);            // psi(a, k, n0 + q) at Ps[a * BN + q]
  double2* Ss = Ps + NA * BN;                                 // S (conjugated backwards), na0 x na0
  if (so) {
    for (int e = threadIdx.x; e < NA * BN; e += blockDim.x) {
      const int a = e / BN, q = e % BN;
      Ps[e] = A.psi[((size_t)a * nk + k) * nb + min(n0 + q, nb - 1)];
    }
    for (int e = threadIdx.x; e < na0 * na0; e += blockDim.x) {
      double2 v = A.S[e];
      if (back) v.y = -v.y;
      Ss[e] = v;
    }
  }
  // the projector rows (one spin: c[0][k][p][n])
  if (flags & F_FG) {
    const int P = A.P;
    const double2* __restrict__ cb = A.cproj + (size_t)k * P * nb + nn;
    const double2* __restrict__ hm = A.hmult;
    constexpr int kC = NA > 12 ? 4 : 8;
    for (int p0 = 0; p0 < P; p0 += kC) {
      double2 cv[kC];
#pragma unroll
      for (int q = 0; q < kC; ++q) cv[q] = cb[(size_t)min(p0 + q, P - 1) * nb];
#pragma unroll
      for (int q = 0; q < kC; ++q)
        if (p0 + q < P) {
#pragma unroll
          for (int j = 0; j < APW; ++j)
            if (a0 + AS * j < NA) cfmac(res[j], cv[q], hm[(a0 + AS * j) * P + p0 + q]);
        }
    }
  }
  if (so) __syncthreads();
  double2 dt[APW];
#pragma unroll
  for (int j = 0; j < APW; ++j) {
    const int a = a0 + AS * j;
    dt[j] = make_double2(0.0, 0.0);
    if (a >= NA || n >= nb) continue;
    double2 inter = res[j];
    inter.x *= am[j];
    inter.y *= am[j];
    const int ar = a % na0, ab = a - ar;
    if (so) {
      for (int b = 0; b < na0; ++b) cfma(inter, Ss[ar * na0 + b], Ps[(ab + b) * BN + nl]);
    }
    const HayScal hs = hay_scal(A.hay, it, a / na0);
    pv[j].x *= hs.sc; pv[j].y *= hs.sc;
    inter.x *= hs.sc; inter.y *= hs.sc;
    double2 r = inter;
    if (flags & F_E0) {
      double2 e = ev[j];
      if (back) e.y = -e.y;
      r.x = e.x * pv[j].x - e.y * pv[j].y + inter.x;
      r.y = e.x * pv[j].y + e.y * pv[j].x + inter.y;
    }
    if (hay) dt[j] = hay_elem(hs, pv[j], ov[j], r);
    A.out[((size_t)a * nk + k) * nb + n] = axmy_epilogue(A, pv[j], r);
  }
  if (hay) {
    __syncthreads();  // psi and S of the spin-orbit term have been read
#pragma unroll
    for (int j = 0; j < APW; ++j)
      if (a0 + AS * j < NA) Ps[(a0 + AS * j) * BN + nl] = dt[j];
    __syncthreads();
    const int nbb = (nb + BN - 1) / BN;
    for (int q = w; q < NA / na0; q += W) hay_part(A.hay, Ps + q * na0 * BN, na0 * BN, q, k * nbb + bx);
    if (A.hay.itp && k == 0 && bx == 0 && threadIdx.x == 0) A.hay.itp[1] = it;
  }
}

constexpr int kAdjRing = 3;
// waves per SIMD: FP64 tiles at three waves spill their ring (227 -> 267 us).  24 alphas in
// FP64 spill 34 registers at two waves and are faster with them than at one wave without:
// 512 k points, 512 x, 64 / 128 / 256 bands 92 / 186 / 336 us against 103 / 199 / 386.
template <typename T2, int NA> constexpr int adj_lr_waves() { return sizeof(T2) == 8 && NA <= 12 ? 4 : 2; }

template <typename T2, int NA, int MT, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(adj_lr_waves<T2, NA>()))) void k_adj_lr(
    const ActArgs<T2> A) {
  if (skipped(A)) return;
  // consecutive workgroups take the band blocks of one k, then the next k, each XCD a
  // contiguous range: the band blocks of a k share its phi' rows through one L2
  const int nbb = (A.nb + 16 * MT - 1) / (16 * MT), n = gridDim.x;
  int b = blockIdx.x;
  if ((n & 7) == 0) b = (b & 7) * (n >> 3) + (b >> 3);
  adj_lr_body<T2, NA, MT, W, kAdjRing>(A, b % nbb, b / nbb);
}

// Batched form: problem p owns workgroups [off[p], off[p+1]), numbered band block
// fastest, then k.
template <typename T2, int NA, int MT, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(adj_lr_waves<T2, NA>()))) void k_adj_lr_batch(
    const ActArgs<T2>* __restrict__ As, const int* __restrict__ off, int np) {
  const int p = find_problem(off, np, blockIdx.x);
  const ActArgs<T2> A = As[p];
  if (skipped(A)) return;
  const int nbb = (A.nb + 16 * MT - 1) / (16 * MT);
  const int loc = blockIdx.x - off[p];
  adj_lr_body<T2, NA, MT, W, kAdjRing>(A, loc % nbb, loc / nbb);
}

}  // namespace og
