// Device code shared by the generated Rys-quadrature kernels
// (codegen/gen_rys.py): nodes and weights, synchronisation within a block,
// the J/K digest of a quartet block held in LDS.
#pragma once
#include "eri_device.h"

#define L2G_RYS_NI 128  // unit intervals of T in the table (codegen/rys_table.py)
#define L2G_RYS_ND 12   // coefficients per polynomial

// l2g_uniform_cart_scale for l <= 3
static __constant__ double l2g_uniform_scale[4][10] = {
    {1.0},
    {1.0, 1.0, 1.0},
    {1.0, 1.7320508075688772, 1.7320508075688772, 1.0, 1.7320508075688772, 1.0},
    {1.0, 2.23606797749979, 2.23606797749979, 2.23606797749979, 3.872983346207417, 2.23606797749979, 1.0,
     2.23606797749979, 2.23606797749979, 1.0}};

// Order between LDS writes and reads of different lanes of a block.  A block
// of one wave needs no barrier: its LDS operations complete in order, so only
// the compiler has to keep them.
template <int NW>
__device__ __forceinline__ void rys_sync() {
  if (NW == 1) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// Node u (= t^2) and weight w of root r of the NR-point rule at T; tab is the
// rule's section of the table.
template <int NR>
__device__ __forceinline__ void rys_root(double T, const double* __restrict__ tab, int r, double& u, double& w) {
  const int iv = T < (double)L2G_RYS_NI ? (int)T : L2G_RYS_NI;
  const double* __restrict__ c = tab + ((size_t)iv * NR + r) * (2 * L2G_RYS_ND);
  if (iv == L2G_RYS_NI) {
    const double rs = rsqrt(T);
    u = c[0] * (rs * rs);
    w = c[L2G_RYS_ND] * rs;
    return;
  }
  const double x = fma(2.0, T - (double)iv, -1.0);
  const double2* __restrict__ c2 = reinterpret_cast<const double2*>(c);
  double2 a[L2G_RYS_ND];
#pragma unroll
  for (int k = 0; k < L2G_RYS_ND; ++k) a[k] = c2[k];
  double p = a[L2G_RYS_ND / 2 - 1].y, q = a[L2G_RYS_ND - 1].y;
#pragma unroll
  for (int k = L2G_RYS_ND / 2 - 1; k >= 0; --k) {
    if (k < L2G_RYS_ND / 2 - 1) {
      p = fma(p, x, a[k].y);
      q = fma(q, x, a[L2G_RYS_ND / 2 + k].y);
    }
    p = fma(p, x, a[k].x);
    q = fma(q, x, a[L2G_RYS_ND / 2 + k].x);
  }
  u = p;
  w = q;
}

// One primitive quartet as a Rys kernel's primitive stage leaves it in LDS:
// per axis PA, QC, P - Q, then eta/(zeta+eta), zeta/(zeta+eta), 1/2zeta,
// 1/2eta, the rule's argument T and the prefactor (0: screened out).
#define L2G_RYS_REC 15

// Shell quartet of a work item (LDS, one per quartet of the block).
struct RysItem {
  int pb0, pk0, npk, pbeg, pend, bp, kp, meta;
  int qi;       // index in the work list, -1 past its end
  int nsurv;    // non-zero once a primitive quartet survived the screening
  double lnprec, qprec, npbk, rnpk;
};

// The work items of a block of Q slots.  The list is sorted by decreasing
// primitive count and its first rys_deep[0] items take min(16, Q) slots each,
// the next rys_deep[1] min(4, Q), the rest one: a deep quartet's primitive
// loop would otherwise run serially on one slot while the chip drains, and
// its sums are shorter.  The share depends on the quartet alone
// (rys_tier_of), so its bits do not depend on the batch it is in.
// The finish launch after pieces has few quartets with many partial sums
// each: a block per quartet.
template <int Q>
struct RysTier {
  static constexpr int S0 = Q < 16 ? Q : 16, S1 = Q < 4 ? Q : 4;
  int S, NI, first, end;
  static __host__ __device__ int ceil_div(int a, int b) { return (a + b - 1) / b; }
  static int blocks(const L2gEriArgs& A) {
    if (A.gpart_mode == 2) return A.n;
    const int a = A.rys_deep[0], b = A.rys_deep[1];
    return ceil_div(a, Q / S0) + ceil_div(b, Q / S1) + ceil_div(A.n - a - b, Q);
  }
  __device__ __forceinline__ RysTier(const L2gEriArgs& A, int blk) {
    const int a = A.rys_deep[0], b = A.rys_deep[1], na = ceil_div(a, Q / S0), nb = ceil_div(b, Q / S1);
    if (A.gpart_mode == 2) {
      S = 1, NI = 1, first = blk, end = A.n;
    } else if (blk < na) {
      S = S0, NI = Q / S0, first = blk * NI, end = a;
    } else if (blk < na + nb) {
      S = S1, NI = Q / S1, first = a + (blk - na) * NI, end = a + b;
    } else {
      S = 1, NI = Q, first = a + b + (blk - na - nb) * Q, end = A.n;
    }
  }
};

// Sum of one value over n pieces, in piece order; the loads of 16 pieces are
// in flight together (one after the other, the sums of the 85 pieces of a
// 4096-primitive (dp|ff) quartet took 0.6 ms).
__device__ __forceinline__ double rys_piece_sum(const double* __restrict__ g, long long stride, int n) {
  double s = 0.0;
#pragma unroll 1
  for (int x = 0; x < n; x += 16, g += 16 * stride) {
    double v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = x + k < n ? g[k * stride] : 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) s += v[k];
  }
  return s;
}

// Primitive quartet p of an item: screening as the per-lane kernels do it,
// and the record.  Past the item's end (act false) a stand-in with prefactor 0.
// erfc(w r)/r takes each primitive quartet twice, p even with 1/r and p odd
// with -erf(w r)/r: the sums are never larger than the values, and one launch
// does both operators.
__device__ __forceinline__ void rys_prim(const L2gEriArgs& A, RysItem& I, int p, double* rec) {
  const bool act = p < I.pend, erf = A.omega > 0 && (!A.erfc || (p & 1));
  p >>= A.erfc;
  // p / npk: the half keeps the product off the integers by more than its rounding error
  const int ib = act ? (int)(((double)p + 0.5) * I.rnpk) : 0;
  const int gb = act ? I.pb0 + ib : 0, gk = act ? I.pk0 + (p - ib * I.npk) : 0;
  const double4 P = A.pp_P[gb], PA = A.pp_PA[gb], Q = A.pp_P[gk], QC = A.pp_PA[gk];
  const double2 xb = A.pp_aux[gb], xk = A.pp_aux[gk];
  const double rs = rsqrt(P.w + Q.w);
  const double oos = rs * rs;
  double pf = PA.w * QC.w * rs * A.scale;
  bool ok = act && xb.x + xk.x > I.lnprec;
  if (A.method == L2G_SCREEN_ORIGINAL)
    ok = ok && !(fabs(pf) < I.qprec);
  else if (A.method == L2G_SCREEN_CONSERVATIVE)
    ok = ok && !(fabs(pf) * fmax(1.0, A.pp_nonsph[gb] * A.pp_nonsph[gk]) * I.npbk < I.qprec);
  // contraction is off in the including files (copies of this code have to
  // round alike): the fused operations are written out
  const double PQx = P.x - Q.x, PQy = P.y - Q.y, PQz = P.z - Q.z;
  double goq = Q.w * oos, gop = P.w * oos;
  const double rho = P.w * Q.w * oos;
  double T = rho * fma(PQz, PQz, fma(PQy, PQy, PQx * PQx));
  if (erf) {  // erf(w r)/r: nodes s u(sT), weights sqrt(s) w(sT), s = w^2 / (w^2 + rho)
    const double s = A.omega * A.omega / fma(A.omega, A.omega, rho);
    T *= s;
    goq *= s;  // the nodes enter as u goq and u gop only
    gop *= s;
    pf *= A.erfc ? -sqrt(s) : sqrt(s);
  }
  if (ok) I.nsurv = 1;
  rec[0] = PA.x, rec[1] = QC.x, rec[2] = PQx;
  rec[3] = PA.y, rec[4] = QC.y, rec[5] = PQy;
  rec[6] = PA.z, rec[7] = QC.z, rec[8] = PQz;
  rec[9] = goq, rec[10] = gop, rec[11] = xb.y, rec[12] = xk.y;
  rec[13] = ok ? T : 0.0, rec[14] = ok ? pf : 0.0;
}

// Integrals of a canonical quartet with the pure flags of meta.
__device__ __forceinline__ int rys_size(int meta, int l1, int l2, int l3, int l4) {
  return ((meta >> 3) & 1 ? 2 * l1 + 1 : l2g_ncart(l1)) * ((meta >> 4) & 1 ? 2 * l2 + 1 : l2g_ncart(l2)) *
         ((meta >> 5) & 1 ? 2 * l3 + 1 : l2g_ncart(l3)) * ((meta >> 6) & 1 ? 2 * l4 + 1 : l2g_ncart(l4));
}

// A canonical quartet's four shells for the digest (LDS): sizes, first
// functions, strides in the block V[i1][i2][i3][i4], and the offsets of the
// six shell-pair blocks 12 34 13 14 23 24 in their concatenation.
struct RysDigest {
  int n[4], l[4], bf[4], sv[4], off[7], nv;
  long long mo, N;
  double deg;
  __device__ __forceinline__ int fn(int k, int i, int gauss) const {
    const int m = i - l[k];  // l < 0: Cartesian, or the Standard order
    return bf[k] + (!gauss || l[k] < 0 ? i : (m == 0 ? 0 : (m > 0 ? 2 * m - 1 : -2 * m)));
  }
  __device__ __forceinline__ int block(int o) const {
    return (o >= off[1]) + (o >= off[2]) + (o >= off[3]) + (o >= off[4]) + (o >= off[5]);
  }
};
__device__ __forceinline__ int rys_bi(int b) { return (0x110020 >> (4 * b)) & 3; }
__device__ __forceinline__ int rys_bj(int b) { return (0x323231 >> (4 * b)) & 3; }

__device__ __forceinline__ void rys_digest_setup(const L2gEriArgs& A, const RysItem& I, int l1, int l2, int l3, int l4,
                                                 RysDigest& g) {
  const int ll[4] = {l1, l2, l3, l4};
  const int4 bf = A.q_bf[I.qi];
  const int b[4] = {bf.x, bf.y, bf.z, bf.w};
  int n[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int pure = (I.meta >> (3 + k)) & 1;
    n[k] = pure ? 2 * ll[k] + 1 : l2g_ncart(ll[k]);
    g.n[k] = n[k];
    g.l[k] = pure ? ll[k] : -1;
    g.bf[k] = b[k];
  }
  g.sv[0] = n[1] * n[2] * n[3], g.sv[1] = n[2] * n[3], g.sv[2] = n[3], g.sv[3] = 1;
  g.nv = n[0] * g.sv[0];
  g.off[0] = 0;
  g.off[1] = n[0] * n[1];
  g.off[2] = g.off[1] + n[2] * n[3];
  g.off[3] = g.off[2] + n[0] * n[2];
  g.off[4] = g.off[3] + n[0] * n[3];
  g.off[5] = g.off[4] + n[1] * n[2];
  g.off[6] = g.off[5] + n[1] * n[3];
  const L2gMatDesc md = A.mats[A.q_req ? A.q_req[I.qi] : 0];
  g.mo = md.off, g.N = md.n;
  g.deg = A.q_scale[I.qi];
}

// Element o of the six blocks of the density.
__device__ __forceinline__ double rys_density(const L2gEriArgs& A, const RysDigest& g, int o) {
  const int b = g.block(o), i = rys_bi(b), j = rys_bj(b), k = o - g.off[b];
  const int r = k / g.n[j], c = k - r * g.n[j];
  return A.dens[g.mo + g.fn(i, r, A.shg_gaussian) * g.N + g.fn(j, c, A.shg_gaussian)];
}

// Element o of the six blocks of a quartet's J and K contributions, from its
// integrals V and density blocks D: J12 takes D34, K13 takes D24, and so on,
// as compute_2body_fock digests them (tests/hartree-fock/
// hartree-fock++.cc:1709-1743).  A lane sums one element over the two shells
// of the partner block, so a quartet leaves one atomic per element.
__device__ __forceinline__ void rys_digest(const L2gEriArgs& A, const RysDigest& g, int o, const double* V,
                                           const double* D) {
  const int b = g.block(o), i = rys_bi(b), j = rys_bj(b), k = o - g.off[b];
  const int r = k / g.n[j], c = k - r * g.n[j];
  const int pb = b < 2 ? 1 - b : 7 - b, pi = rys_bi(pb), pj = rys_bj(pb);
  const int nx = g.n[pi], ny = g.n[pj], sx = g.sv[pi], sy = g.sv[pj];
  const double* v = V + r * g.sv[i] + c * g.sv[j];
  const double* d = D + g.off[pb];
  double s = 0.0;
  for (int x = 0; x < nx; ++x, v += sx, d += ny)
    for (int y = 0; y < ny; ++y) s = fma(d[y], v[y * sy], s);
  double* m = b < 2 ? A.jg : A.kg;
  l2g_acc(&m[g.mo + g.fn(i, r, A.shg_gaussian) * g.N + g.fn(j, c, A.shg_gaussian)], g.deg * s, A.fx_hoff);
}

// The same for a block of quartets of solid harmonics (and s, p), whose
// shell sizes are then the class's: block B of the density into LDS, and
// block B's contributions.  A loop per block has no divergence and constant
// strides; the general loops above spend 260 instructions an element on
// decoding it.  Each sum runs in the general loop's order.
template <int NT, int B, int N0, int N1, int N2, int N3>
struct RysBlock {
  static constexpr int n[4] = {N0, N1, N2, N3}, sv[4] = {N1 * N2 * N3, N2 * N3, N3, 1}, nv = N0 * N1 * N2 * N3;
  static constexpr int bi[6] = {0, 2, 0, 0, 1, 1}, bj[6] = {1, 3, 2, 3, 2, 3};
  static constexpr int first(int b) { return b == 0 ? 0 : first(b - 1) + n[bi[b - 1]] * n[bj[b - 1]]; }
  static constexpr int i = bi[B], j = bj[B], size = n[i] * n[j];
  static constexpr int pb = B < 2 ? 1 - B : 7 - B, pi = bi[pb], pj = bj[pb], nx = n[pi], ny = n[pj];

  static __device__ __forceinline__ long long at(const L2gEriArgs& A, const RysDigest& g, int k) {
    const int r = k / n[j], c = k - r * n[j];
    const int fr = A.shg_gaussian ? g.fn(i, r, 1) : g.bf[i] + r, fc = A.shg_gaussian ? g.fn(j, c, 1) : g.bf[j] + c;
    return g.mo + (long long)fr * (int)g.N + fc;
  }
  static __device__ __forceinline__ void density(const L2gEriArgs& A, const RysItem* items, const RysDigest* dig, int qn,
                                                 double* V, int region) {
    for (int it = threadIdx.x; it < qn * size; it += NT) {
      const int q = it / size, k = it - q * size;
      if (items[q].nsurv) V[q * region + nv + first(B) + k] = A.dens[at(A, dig[q], k)];
    }
  }
  static __device__ __forceinline__ void digest(const L2gEriArgs& A, const RysItem* items, const RysDigest* dig, int qn,
                                                const double* V, int region) {
    for (int it = threadIdx.x; it < qn * size; it += NT) {
      const int q = it / size, k = it - q * size;
      if (!items[q].nsurv) continue;
      const int r = k / n[j], c = k - r * n[j];
      const double* v = V + q * region + r * sv[i] + c * sv[j];
      const double* d = V + q * region + nv + first(pb);
      double s = 0.0;
#pragma unroll nx * ny <= 25 ? nx : 1
      for (int x = 0; x < nx; ++x)
#pragma unroll
        for (int y = 0; y < ny; ++y) s = fma(d[x * ny + y], v[x * sv[pi] + y * sv[pj]], s);
      l2g_acc(&(B < 2 ? A.jg : A.kg)[at(A, dig[q], k)], dig[q].deg * s, A.fx_hoff);
    }
  }
};

template <int NT, int NW, int N0, int N1, int N2, int N3>
__device__ __forceinline__ void rys_digest_pure(const L2gEriArgs& A, const RysItem* items, const RysDigest* dig, int qn,
                                                double* V, int region) {
  RysBlock<NT, 0, N0, N1, N2, N3>::density(A, items, dig, qn, V, region);
  RysBlock<NT, 1, N0, N1, N2, N3>::density(A, items, dig, qn, V, region);
  RysBlock<NT, 2, N0, N1, N2, N3>::density(A, items, dig, qn, V, region);
  RysBlock<NT, 3, N0, N1, N2, N3>::density(A, items, dig, qn, V, region);
  RysBlock<NT, 4, N0, N1, N2, N3>::density(A, items, dig, qn, V, region);
  RysBlock<NT, 5, N0, N1, N2, N3>::density(A, items, dig, qn, V, region);
  rys_sync<NW>();
  RysBlock<NT, 0, N0, N1, N2, N3>::digest(A, items, dig, qn, V, region);
  RysBlock<NT, 1, N0, N1, N2, N3>::digest(A, items, dig, qn, V, region);
  RysBlock<NT, 2, N0, N1, N2, N3>::digest(A, items, dig, qn, V, region);
  RysBlock<NT, 3, N0, N1, N2, N3>::digest(A, items, dig, qn, V, region);
  RysBlock<NT, 4, N0, N1, N2, N3>::digest(A, items, dig, qn, V, region);
  RysBlock<NT, 5, N0, N1, N2, N3>::digest(A, items, dig, qn, V, region);
}
