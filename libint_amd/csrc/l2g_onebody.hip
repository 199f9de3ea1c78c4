// One-body integrals over shell pairs: overlap, kinetic energy and the
// attraction to point charges (Engine(Operator::overlap / kinetic / nuclear),
// engine.impl.h:181-561, as compute_1body_ints assembles them,
// hartree-fock.cc:480-535).
//
// A wave per shell pair, a kernel per pair of angular momenta.  The lanes
// share the primitive pairs (S, T) or the primitive pairs times the charges
// (V); each keeps the Cartesian block of its part in registers and the wave
// sums it at the end.  The attraction is a Rys quadrature,
//   V_ab = -sum_C Z_C sum_p sum_r X_r(ax, bx) Y_r(ay, by) Z_r(az, bz),
// with the two-index recurrences of both centres in registers.  Bound by the
// FP64 VALU.  460 functions and 20 charges: kernels 10 ms as Hermite sums with
// the R tables built level by level in LDS, one charge after another.
#include "l2g_internal.h"
#include "rys_device.h"

using namespace l2g_impl;

namespace {

__constant__ double c_sh1[4][7][10];  // solid-harmonic coefficients, Standard rows

struct CartTab {
  int e[10][3];
};
constexpr CartTab cart_tab(int l) {
  CartTab t{};
  int n = 0;
  for (int x = l; x >= 0; --x)
    for (int y = l - x; y >= 0; --y, ++n) t.e[n][0] = x, t.e[n][1] = y, t.e[n][2] = l - x - y;
  return t;
}

// Sum of acc over the wave into out (LDS).
template <int N>
__device__ __forceinline__ void reduce_to(double* out, const double (&acc)[N], int lane) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const double v = l2g_wave_sum(acc[k]);
    if (lane == (k & 63)) out[k] = v;
  }
}

// g[i][j] of one axis: (i, j) <- D (i, j-1) + B10 (j-1 (i, j-2) + i (i-1, j-1))
template <int I, int J>
__device__ __forceinline__ void two_index(double (&g)[I + 1][J + 1], double g00, double C, double D, double B10) {
  g[0][0] = g00;
#pragma unroll
  for (int i = 0; i < I; ++i) g[i + 1][0] = C * g[i][0] + (i ? i * B10 * g[i ? i - 1 : 0][0] : 0.0);
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int i = 0; i <= I; ++i)
      g[i][j + 1] = D * g[i][j] + B10 * ((j ? j * g[i][j ? j - 1 : 0] : 0.0) + (i ? i * g[i ? i - 1 : 0][j] : 0.0));
}

template <int LA, int LB>
__global__ void __launch_bounds__(64) l2g_onebody_kernel(l2g_impl::L2gOneBodyArgs A, const int2* __restrict__ pairs) {
  constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2, N = NA * NB, NR = (LA + LB) / 2 + 1;
  constexpr CartTab ta = cart_tab(LA), tb = cart_tab(LB);
  __shared__ double cart[3][N];
  const int lane = threadIdx.x;
  const int sa = pairs[blockIdx.x].x, sb = pairs[blockIdx.x].y;
  const int a0 = A.poff[sa], b0 = A.poff[sb], npb = A.poff[sb + 1] - b0, npp = (A.poff[sa + 1] - a0) * npb;
  double Ao[3], Bo[3], AB[3], AB2 = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    Ao[x] = A.origin[3 * sa + x], Bo[x] = A.origin[3 * sb + x], AB[x] = Ao[x] - Bo[x];
    AB2 += AB[x] * AB[x];
  }
#pragma unroll 1
  for (int m = 0; m < 2; ++m) {  // overlap, kinetic energy
    if (!(m ? A.T : A.S)) continue;
    double acc[N];
#pragma unroll
    for (int k = 0; k < N; ++k) acc[k] = 0.0;
#pragma unroll 1
    for (int it = lane; it < npp; it += 64) {
      const int ia = it / npb, ib = it - ia * npb;
      const double a = A.alpha[a0 + ia], b = A.alpha[b0 + ib], oop = 1.0 / (a + b), o2p = 0.5 * oop;
      const double q = 3.14159265358979323846 * oop;
      const double pre = A.coeff[a0 + ia] * A.coeff[b0 + ib] * exp(-a * b * oop * AB2) * q * sqrt(q);
      double s[3][LA + 1][LB + 3];
#pragma unroll
      for (int x = 0; x < 3; ++x)
        two_index<LA, LB + 2>(s[x], x ? 1.0 : pre, -b * oop * AB[x], a * oop * AB[x], o2p);
      if (m == 0) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            acc[i * NB + j] += s[0][ta.e[i][0]][tb.e[j][0]] * s[1][ta.e[i][1]][tb.e[j][1]] * s[2][ta.e[i][2]][tb.e[j][2]];
      } else {
        double t[3][LA + 1][LB + 1];  // -1/2 d^2/dx^2 on the second centre
#pragma unroll
        for (int x = 0; x < 3; ++x)
#pragma unroll
          for (int i = 0; i <= LA; ++i)
#pragma unroll
            for (int j = 0; j <= LB; ++j)
              t[x][i][j] = b * (2 * j + 1) * s[x][i][j] - 2.0 * b * b * s[x][i][j + 2] -
                           (j > 1 ? 0.5 * j * (j - 1) * s[x][i][j > 1 ? j - 2 : 0] : 0.0);
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            const double sx = s[0][ta.e[i][0]][tb.e[j][0]], sy = s[1][ta.e[i][1]][tb.e[j][1]],
                         sz = s[2][ta.e[i][2]][tb.e[j][2]];
            acc[i * NB + j] += t[0][ta.e[i][0]][tb.e[j][0]] * sy * sz + sx * t[1][ta.e[i][1]][tb.e[j][1]] * sz +
                               sx * sy * t[2][ta.e[i][2]][tb.e[j][2]];
          }
      }
    }
    reduce_to<N>(cart[m], acc, lane);
  }
  if (A.V) {
    double acc[N];
#pragma unroll
    for (int k = 0; k < N; ++k) acc[k] = 0.0;
    const int nc = A.ncharge;
    const long long items = (long long)npp * nc;
#pragma unroll 1
    for (long long it = lane; it < items; it += 64) {
      const int pp = (int)(it / nc), c = (int)(it - (long long)pp * nc);
      const int ia = pp / npb, ib = pp - ia * npb;
      const double a = A.alpha[a0 + ia], b = A.alpha[b0 + ib], p = a + b, oop = 1.0 / p, o2p = 0.5 * oop;
      const double pre = -A.q[c] * A.coeff[a0 + ia] * A.coeff[b0 + ib] * exp(-a * b * oop * AB2) *
                         (2.0 * 3.14159265358979323846) * oop;
      double PC[3], PA[3], PB[3], r2 = 0.0;
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        PA[x] = -b * oop * AB[x], PB[x] = a * oop * AB[x];
        PC[x] = Ao[x] + PA[x] - A.qxyz[3 * c + x];
        r2 += PC[x] * PC[x];
      }
      const double T = p * r2;
#pragma unroll 1
      for (int r = 0; r < NR; ++r) {
        double u, w;
        rys_root<NR>(T, A.rys, r, u, w);
        const double B10 = o2p * (1.0 - u);
        double g[3][LA + 1][LB + 1];
#pragma unroll
        for (int x = 0; x < 3; ++x)
          two_index<LA, LB>(g[x], x ? 1.0 : w * pre, PA[x] - u * PC[x], PB[x] - u * PC[x], B10);
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            acc[i * NB + j] += g[0][ta.e[i][0]][tb.e[j][0]] * g[1][ta.e[i][1]][tb.e[j][1]] * g[2][ta.e[i][2]][tb.e[j][2]];
      }
    }
    reduce_to<N>(cart[2], acc, lane);
  }
  __syncthreads();
  // solid harmonics and the store; the mirrored block is the transpose
  const int pa = (A.pure[sa] && LA > 0) ? 1 : 0, pb = (A.pure[sb] && LB > 0) ? 1 : 0;
  const int noa = pa ? 2 * LA + 1 : NA, nob = pb ? 2 * LB + 1 : NB;
  double* out[3] = {A.S, A.T, A.V};
  for (int r = lane; r < noa * nob; r += 64) {
    const int fi = r / nob, fj = r % nob;
    // output position -> row m + l: Standard m = f - l, Gaussian 0, +1, -1, +2, ...
    const int ra = pa ? (A.gauss ? LA + (fi == 0 ? 0 : ((fi & 1) ? (fi + 1) / 2 : -fi / 2)) : fi) : 0;
    const int rb = pb ? (A.gauss ? LB + (fj == 0 ? 0 : ((fj & 1) ? (fj + 1) / 2 : -fj / 2)) : fj) : 0;
    const long long o = (A.bf0[sa] + fi) * A.nbf + A.bf0[sb] + fj;
    const long long ot = (A.bf0[sb] + fj) * A.nbf + A.bf0[sa] + fi;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      if (!out[m]) continue;
      double s = 0.0;
      for (int ca = pa ? 0 : fi; ca < (pa ? NA : fi + 1); ++ca) {
        const double wa = pa ? c_sh1[LA][ra][ca] : 1.0;
        if (wa == 0.0) continue;
        for (int cb = pb ? 0 : fj; cb < (pb ? NB : fj + 1); ++cb) {
          const double wb = pb ? c_sh1[LB][rb][cb] : 1.0;
          if (wb != 0.0) s += wa * wb * cart[m][ca * NB + cb];
        }
      }
      out[m][o] = s;
      if (sa != sb) out[m][ot] = s;  // a diagonal block writes each of its elements itself
    }
  }
}

template <int LA, int LB>
void launch_class(l2g_impl::L2gOneBodyArgs A, const int2* pairs, int n, hipStream_t s) {
  if (n == 0) return;
  // the class's rule in the node table: sections n = 1, 2, .. back to back
  constexpr int NR = (LA + LB) / 2 + 1;
  A.rys += (size_t)(L2G_RYS_NI + 1) * (NR * (NR - 1) / 2) * 2 * L2G_RYS_ND;
  hipLaunchKernelGGL((l2g_onebody_kernel<LA, LB>), dim3(n), dim3(64), 0, s, A, pairs);
  LAUNCHCHK("l2g_onebody_kernel");
}

}  // namespace

namespace l2g_impl {

void onebody_init(const double* sh) { HIPCHK(hipMemcpyToSymbol(HIP_SYMBOL(c_sh1), sh, sizeof(double) * 4 * 7 * 10)); }

void launch_onebody(const L2gOneBodyArgs& A, const int2* pairs, const int (&first)[17], hipStream_t s) {
#define L2G_OB(a, b) launch_class<a, b>(A, pairs + first[a * 4 + b], first[a * 4 + b + 1] - first[a * 4 + b], s)
  L2G_OB(0, 0);
  L2G_OB(1, 0);
  L2G_OB(1, 1);
  L2G_OB(2, 0);
  L2G_OB(2, 1);
  L2G_OB(2, 2);
  L2G_OB(3, 0);
  L2G_OB(3, 1);
  L2G_OB(3, 2);
  L2G_OB(3, 3);
#undef L2G_OB
}

}  // namespace l2g_impl
