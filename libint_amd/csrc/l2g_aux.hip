// Small hand-written kernels used by the host code: the Fock finishing step
// and the combination step of first-derivative integrals.
#include "l2g_internal.h"

// In place, for one request block of the Fock arenas: J = (jg + jg^T)/4 into
// jg, K = (kg + kg^T)/8 into kg, G = 2J - K into the density block.  The
// digest kernels add each unique quartet's integrals once with its
// degeneracy factor and without mirroring, which leaves this
// symmetrisation, as in compute_2body_fock
// (tests/hartree-fock/hartree-fock++.cc:1709-1771).
// Thread (i, j) with i <= j owns both mirrored elements, so no element is
// read after another thread wrote it.
__global__ void __launch_bounds__(256) l2g_fock_finish_kernel(double* __restrict__ jg, double* __restrict__ kg,
                                                              double* __restrict__ g, long long N, long long hoff) {
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N * N) return;
  const long long i = idx / N, j = idx - i * N;
  if (j < i) return;
  const long long a = i * N + j, b = j * N + i;
  double ja, jb, ka, kb;
  if (hoff) {  // fixed-point accumulators: low words in place, high words hoff further on
    const unsigned long long* jw = reinterpret_cast<const unsigned long long*>(jg);
    const unsigned long long* kw = reinterpret_cast<const unsigned long long*>(kg);
    ja = l2g_fx_value(jw[a + hoff], jw[a]);
    jb = l2g_fx_value(jw[b + hoff], jw[b]);
    ka = l2g_fx_value(kw[a + hoff], kw[a]);
    kb = l2g_fx_value(kw[b + hoff], kw[b]);
  } else {
    ja = jg[a], jb = jg[b], ka = kg[a], kb = kg[b];
  }
  const double Jv = 0.25 * (ja + jb);
  const double Kv = 0.125 * (ka + kb);
  jg[a] = Jv;
  jg[b] = Jv;
  kg[a] = Kv;
  kg[b] = Kv;
  g[a] = 2.0 * Jv - Kv;
  g[b] = 2.0 * Jv - Kv;
}

// Cartesian component index of x^a y^b z^c in libint's order (x descending,
// then y descending): (l - a)(l - a + 1)/2 + (l - a - b).
__device__ __forceinline__ int l2g_cart_index(int l, int a, int b) { return (l - a) * (l - a + 1) / 2 + (l - a - b); }

// First derivatives of (ab|cd) with respect to the centre k of one shell,
// d/dK_i x_i^n e^{-alpha r^2} = 2 alpha x_i^(n+1) e^{..} - n x_i^(n-1) e^{..}:
// the ERI with shell k raised (l+1, coefficients 2 alpha c) minus n times
// the ERI with shell k lowered (l-1), both Cartesian, then the solid-harmonic
// rows of the pure centres.  Derivative d = 3 k + i of quartet q goes to
// out[d * total + out_off[q] + f], f row-major over the four shells' output
// functions in caller order (the layout of Engine::results()[d] for
// deriv_order = 1, include/libint2/engine.h:779-781).  A block per quartet
// takes as many of the 12 derivatives at a time as its buffers hold, all of
// them for most classes: the Cartesian blocks (two loads per element) into
// LDS, then one centre's solid-harmonic rows after the other between two LDS
// buffers, then the store.  Bound by the barriers' and loads' latency: one
// derivative at a time (60 barriers a quartet, integer divisions for every
// index) took 450 us for 20,000 s/p/d quartets, this 190.  Shells up to l = 2
// (the raised ones up to 3): at most 6^4 Cartesian elements.
constexpr int kDerivMaxCart = 1296;

// x / n and the remainder for x < 2^21: the half keeps the product further
// from the integers than its rounding error
struct FastDiv {
  int n;
  float r;
  __device__ __forceinline__ explicit FastDiv(int n_) : n(n_), r(1.0f / (float)n_) {}
  __device__ __forceinline__ int div(int& x) const {  // x: the remainder
    const int q = (int)(((float)x + 0.5f) * r);
    x -= q * n;
    return q;
  }
};

__global__ void __launch_bounds__(256) l2g_deriv1_combine_kernel(const double* __restrict__ raw,
                                                                 const long long* __restrict__ raw_off,
                                                                 const long long* __restrict__ out_off,
                                                                 const int* __restrict__ qinfo, long long nq,
                                                                 long long total, double* __restrict__ out,
                                                                 l2g_impl::L2gDerivTab tab) {
  __shared__ double buf[2][kDerivMaxCart];
  __shared__ long long ro[8];
  __shared__ double coef[3 * 7 * 4];  // rows of l = 0 .. 2, from the argument once: a load per use is far slower
  __shared__ signed char cidx[3 * 7 * 4], nnz[3 * 7];
  const long long q = blockIdx.x;
  if (q >= nq) return;
  const int info = qinfo[q];
  if (threadIdx.x < 3 * 7 * 4) {
    const int i = threadIdx.x / 28, m = threadIdx.x / 4 % 7, a = threadIdx.x & 3;
    coef[threadIdx.x] = tab.coef[i][m][a];
    cidx[threadIdx.x] = tab.cidx[i][m][a];
    if (a == 0) nnz[threadIdx.x / 4] = tab.nnz[i][m];
  } else if (threadIdx.x >= 128 && threadIdx.x < 136) {
    ro[threadIdx.x - 128] = raw_off[(threadIdx.x - 128) * nq + q];
  }
  __syncthreads();
  auto lof = [&](int k) { return (info >> (4 * k)) & 15; };
  int nc[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) nc[k] = (lof(k) + 1) * (lof(k) + 2) / 2;
  const int ncart = nc[0] * nc[1] * nc[2] * nc[3];
  const long long obase = out_off[q];
  const FastDiv dcart(ncart), d1(nc[1]), d2(nc[2]), d3(nc[3]);
  // as many derivatives at a time as the buffers hold
  const int most = min(12, kDerivMaxCart / ncart);
  for (int d0 = 0; d0 < 12; d0 += most) {
    const int nd = min(most, 12 - d0);
    // Cartesian derivative blocks
    for (int it = threadIdx.x; it < nd * ncart; it += blockDim.x) {
      int f = it;
      const int d = d0 + dcart.div(f), k = d / 3, ax = d - 3 * k;
      int c3 = f;
      int c2 = d3.div(c3), c1 = d2.div(c2);
      const int c0 = d1.div(c1);
      const int lk = lof(k), ck = k == 0 ? c0 : k == 1 ? c1 : k == 2 ? c2 : c3;
      const int r = (ck >= 1) + (ck >= 3) + (ck >= 6);
      const int ez = ck - r * (r + 1) / 2, ey = r - ez, ex = lk - r;
      const int dp = (lk + 2) * (lk + 3) / 2, dm = lk * (lk + 1) / 2;
      auto at = [&](int dk, int u) {  // element with component u (of dk) on centre k
        const int a0 = k == 0 ? u : c0, a1 = k == 1 ? u : c1, a2 = k == 2 ? u : c2, a3 = k == 3 ? u : c3;
        return ((a0 * (k == 1 ? dk : nc[1]) + a1) * (k == 2 ? dk : nc[2]) + a2) * (k == 3 ? dk : nc[3]) + a3;
      };
      double v = raw[ro[k] + at(dp, l2g_cart_index(lk + 1, ex + (ax == 0), ey + (ax == 1)))];
      const int nx = ax == 0 ? ex : ax == 1 ? ey : ez;
      if (nx > 0) v -= nx * raw[ro[4 + k] + at(dm, l2g_cart_index(lk - 1, ex - (ax == 0), ey - (ax == 1)))];
      buf[0][it] = v;
    }
    __syncthreads();
    // solid-harmonic rows, one pure centre at a time
    int dims[4] = {nc[0], nc[1], nc[2], nc[3]};
    int cur = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (!((info >> (16 + j)) & 1)) continue;
      const int lj = lof(j), nout_j = 2 * lj + 1;
      int inner = 1, outer = nd;
#pragma unroll
      for (int t = 0; t < 4; ++t) (t > j ? inner : outer) *= t == j ? 1 : dims[t];
      const FastDiv di(inner), dm(nout_j);
      for (int it = threadIdx.x; it < outer * nout_j * inner; it += blockDim.x) {
        int i_in = it;
        int m = di.div(i_in);
        const int o = dm.div(m);
        double s = 0.0;
        const int row = lj * 7 + m, n = nnz[row];
        for (int a = 0; a < n; ++a)
          s += coef[4 * row + a] * buf[cur][(o * dims[j] + cidx[4 * row + a]) * inner + i_in];
        buf[cur ^ 1][it] = s;
      }
      dims[j] = nout_j;
      cur ^= 1;
      __syncthreads();
    }
    const int nout = dims[0] * dims[1] * dims[2] * dims[3];
    const FastDiv dn(nout);
    for (int it = threadIdx.x; it < nd * nout; it += blockDim.x) {
      int i = it;
      const int d = dn.div(i);
      out[(long long)(d0 + d) * total + obase + i] = buf[cur][it];
    }
    __syncthreads();
  }
}

namespace l2g_impl {

void launch_deriv1_combine(const double* raw, const long long* raw_off, const long long* out_off, const int* qinfo,
                           long long nq, long long total, double* out, const L2gDerivTab& tab, hipStream_t s) {
  if (nq <= 0) return;
  if (nq > 0x7fffffffLL) throw std::invalid_argument("too many quartets for one derivative launch");
  hipLaunchKernelGGL(l2g_deriv1_combine_kernel, dim3((unsigned)nq), dim3(256), 0, s, raw, raw_off, out_off, qinfo, nq,
                     total, out, tab);
  LAUNCHCHK("l2g_deriv1_combine_kernel");
}

namespace {

__global__ void __launch_bounds__(64) schwarz_reduce_kernel(const long long* __restrict__ off,
                                                            const double* __restrict__ vals, int norm,
                                                            const int* __restrict__ first,
                                                            const double* __restrict__ gpart, long long stride, int ne,
                                                            const long long* __restrict__ idx,
                                                            double* __restrict__ out, double* __restrict__ out2) {
  const int i = blockIdx.x;
  double m = 0.0, q = 0.0, h = 0.0;
  for (long long k = off[i] + threadIdx.x; k < off[i + 1]; k += 64) {
    const double v = vals[k];
    m = fmax(m, fabs(v));
    q = fma(v, v, q);
  }
  if (out2)
    for (int e = threadIdx.x; e < ne; e += 64) {
      double s = 0.0;
      for (int x = first[i]; x < first[i + 1]; ++x) s += gpart[x * stride + (long long)e * ne + e];
      h = fmax(h, fabs(s));
    }
  for (int o = 32; o > 0; o >>= 1) {
    m = fmax(m, __shfl_xor(m, o));
    q += __shfl_xor(q, o);
    h = fmax(h, __shfl_xor(h, o));
  }
  if (threadIdx.x == 0) {
    out[idx[i]] = norm ? sqrt(sqrt(q)) : sqrt(m);
    if (out2) out2[idx[i]] = sqrt(h);
  }
}

}  // namespace

void launch_schwarz_reduce(int n, const long long* off, const double* vals, int norm, const int* first,
                           const double* gpart, long long stride, int ne, const long long* idx, double* out,
                           double* out2, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(schwarz_reduce_kernel, dim3((unsigned)n), dim3(64), 0, s, off, vals, norm, first, gpart, stride,
                     ne, idx, out, out2);
  LAUNCHCHK("schwarz_reduce_kernel");
}

void launch_fock_finish(double* jg, double* kg, double* g, long long N, long long hoff, hipStream_t s) {
  if (N <= 0) return;
  const long long n = N * N;
  const int block = 256;
  const long long grid = (n + block - 1) / block;
  hipLaunchKernelGGL(l2g_fock_finish_kernel, dim3((unsigned)grid), dim3(block), 0, s, jg, kg, g, N, hoff);
  LAUNCHCHK("l2g_fock_finish_kernel");
}

}  // namespace l2g_impl
