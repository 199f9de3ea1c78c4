// Screened Fock quartet list on the GPU: the permutationally-unique quartet
// loop of compute_2body_fock (tests/hartree-fock/hartree-fock++.cc:1628-1696)
// over the significant shell pairs, which are listed in (s1, s2)
// lexicographic order.  In that order the unique quartets are exactly the
// pairs of pairs (p1, p2) with p2 <= p1, so the loop is one triangular index
// t -> (p1, p2) that every thread decodes on its own.
//
// Pass 1 counts the surviving quartets of each block's contiguous t range;
// pass 2 writes them (screening Dnorm1234 K12 K34 >= precision, per-quartet
// precision precision / Dnorm1234, degeneracy, canonical shell order and
// kernel class as the host enumeration in l2g_fock.cpp) at the block's
// offset, with a sort key (class, decreasing primitive-loop length);
// a radix sort by that key then groups the classes and orders each by depth.
#include <hipcub/hipcub.hpp>

#include "l2g_internal.h"

using namespace l2g_impl;

namespace {

constexpr int kEnumThreads = 256;

__device__ __forceinline__ void decode_tri(long long t, long long& p1, long long& p2) {
  long long a = (long long)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while (a * (a + 1) / 2 > t) --a;
  while ((a + 1) * (a + 2) / 2 <= t) ++a;
  p1 = a;
  p2 = t - a * (a + 1) / 2;
}

// Largest |D| of every shell block, and of all of them (dmax: bits of a
// non-negative double, which order as integers)
__global__ void __launch_bounds__(kEnumThreads) shell_norms(const double* __restrict__ D, long long N,
                                                            const int* __restrict__ bf1st, int n,
                                                            double* __restrict__ Dn,
                                                            unsigned long long* __restrict__ dmax) {
  const long long k = (long long)blockIdx.x * kEnumThreads + threadIdx.x;
  double m = 0.0;
  if (k < (long long)n * n) {
    const int s1 = (int)(k / n), s2 = (int)(k - (long long)s1 * n);
    for (int i = bf1st[s1]; i < bf1st[s1 + 1]; ++i)
      for (int j = bf1st[s2]; j < bf1st[s2 + 1]; ++j) m = fmax(m, fabs(D[i * N + j]));
    Dn[k] = m;
  }
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
  if ((threadIdx.x & 63) == 0 && m > 0.0) atomicMax(dmax, (unsigned long long)__double_as_longlong(m));
}

struct Quartet {
  int s1, s2, s3, s4;
  double Dn1234;
};

// screening of one unique quartet; true when it survives
__device__ __forceinline__ bool screen(const l2g_impl::FockEnumArgs& E, long long p1, long long p2, Quartet& q) {
  q.s1 = E.ps1[p1], q.s2 = E.ps2[p1], q.s3 = E.ps1[p2], q.s4 = E.ps2[p2];
  const long long n = E.n;
  const double* Dn = E.Dn;
  const double d = fmax(fmax(fmax(Dn[q.s1 * n + q.s2], Dn[q.s3 * n + q.s4]), fmax(Dn[q.s1 * n + q.s3], Dn[q.s2 * n + q.s3])),
                        fmax(Dn[q.s1 * n + q.s4], Dn[q.s2 * n + q.s4]));
  q.Dn1234 = d;
  return !(d * E.pK[p1] * E.pK[p2] < E.precision);
}

__global__ void __launch_bounds__(kEnumThreads) enum_count(const l2g_impl::FockEnumArgs E, long long total,
                                                              long long chunk, long long* __restrict__ counts) {
  __shared__ long long red[kEnumThreads / 64];
  const long long t0 = (long long)blockIdx.x * chunk, t1 = min(total, t0 + chunk);
  long long c = 0;
  for (long long t = t0 + threadIdx.x; t < t1; t += kEnumThreads) {
    long long p1, p2;
    decode_tri(t, p1, p2);
    Quartet q;
    c += screen(E, p1, p2, q) ? 1 : 0;
  }
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    long long s = 0;
    for (int i = 0; i < kEnumThreads / 64; ++i) s += red[i];
    counts[blockIdx.x] = s;
  }
}

// fills the items of blocks [block0, block0 + gridDim.x) of the count pass's
// partition; base[k] is the first item of block block0 + k within the window
__global__ void __launch_bounds__(kEnumThreads) enum_fill(const l2g_impl::FockEnumArgs E, long long total,
                                                             long long chunk, long long block0,
                                                             const long long* __restrict__ base,
                                                             l2g_impl::FockEnumOut O) {
  __shared__ unsigned int pos;
  __shared__ unsigned int hist[l2g_impl::kEnumClasses];
  __shared__ unsigned long long whist[l2g_impl::kEnumClasses];
  if (threadIdx.x == 0) pos = 0;
  for (int c = threadIdx.x; c < l2g_impl::kEnumClasses; c += kEnumThreads) hist[c] = 0, whist[c] = 0;
  __syncthreads();
  const long long t0 = (block0 + blockIdx.x) * chunk, t1 = min(total, t0 + chunk);
  const long long b0 = base[blockIdx.x];
  for (long long t = t0 + threadIdx.x; t < t1; t += kEnumThreads) {
    long long p1, p2;
    decode_tri(t, p1, p2);
    Quartet q;
    if (!screen(E, p1, p2, q)) continue;
    const int s1 = q.s1, s2 = q.s2, s3 = q.s3, s4 = q.s4;
    const double qprec = q.Dn1234 != 0.0 ? E.precision / q.Dn1234 : E.needed;
    const int deg = (s1 == s2 ? 1 : 2) * (s3 == s4 ? 1 : 2) * (s1 == s3 ? (s2 == s4 ? 1 : 2) : 2);
    const int l1 = E.l[s1], l2 = E.l[s2], l3 = E.l[s3], l4 = E.l[s4];
    const bool stb = E.pswap[p1] != 0, stk = E.pswap[p2] != 0, sbk = (l1 + l2) > (l3 + l4);
    const int b1 = sbk ? (stk ? s4 : s3) : (stb ? s2 : s1);
    const int b2 = sbk ? (stk ? s3 : s4) : (stb ? s1 : s2);
    const int k1 = sbk ? (stb ? s2 : s1) : (stk ? s4 : s3);
    const int k2 = sbk ? (stb ? s1 : s2) : (stk ? s3 : s4);
    const int bp = sbk ? E.pid[p2] : E.pid[p1], kp = sbk ? E.pid[p1] : E.pid[p2];
    const int lk = ((E.l[b1] * 4 + E.l[b2]) * 4 + E.l[k1]) * 4 + E.l[k2];
    // every class up to the compiled l has a kernel; the last class flags none
    int cls = E.clsmap[lk];
    if (E.fp32_thr > 0 && E.pK[p1] * E.pK[p2] < E.fp32_thr && E.pS[p1] * E.pS[p2] < E.hrr_factor * E.fp32_thr &&
        E.cls32map[lk] >= 0)
      cls = E.cls32map[lk];
    if (cls < 0 || cls >= l2g_impl::kEnumClasses - 1) cls = l2g_impl::kEnumClasses - 1;
    auto pb = [&](int sh) { return (E.pure[sh] && E.l[sh] > 0) ? 1 : 0; };
    const int w = E.np[bp] * E.np[kp];
    const long long i = b0 + atomicAdd(&pos, 1u);
    O.bra[i] = bp;
    O.ket[i] = kp;
    O.meta[i] = (pb(b1) << 3) | (pb(b2) << 4) | (pb(k1) << 5) | (pb(k2) << 6);
    O.lnp[i] = qprec > 0 ? log(qprec) : -1.7976931348623157e308;
    O.scale[i] = (double)deg;
    O.bf[i] = int4{E.bf1st[b1], E.bf1st[b2], E.bf1st[k1], E.bf1st[k2]};
    O.pr[i] = int2{0, w};
    O.key[i] = ((unsigned)cls << 13) | (unsigned)(8191 - min(w, 8191));  // kEnumKeyBits bits
    O.idx[i] = (unsigned)i;
    atomicAdd(&hist[cls], 1u);
    atomicAdd(&whist[cls], (unsigned long long)w);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < l2g_impl::kEnumClasses; c += kEnumThreads)
    if (hist[c]) {
      atomicAdd(&O.cls_count[c], (unsigned long long)hist[c]);
      atomicAdd(&O.cls_nprim[c], whist[c]);
    }
}

// the items in sorted order, one launch for their seven arrays
__global__ void __launch_bounds__(kEnumThreads) gather_items(const l2g_impl::FockEnumOut in,
                                                             const unsigned* __restrict__ perm,
                                                             l2g_impl::FockEnumState::Items out, long long n) {
  const long long k = (long long)blockIdx.x * kEnumThreads + threadIdx.x;
  if (k >= n) return;
  const unsigned i = perm[k];
  const int bra = in.bra[i], ket = in.ket[i], meta = in.meta[i];
  const double lnp = in.lnp[i], scale = in.scale[i];
  const int4 bf = in.bf[i];
  const int2 pr = in.pr[i];
  out.bra[k] = bra, out.ket[k] = ket, out.meta[k] = meta, out.lnp[k] = lnp, out.scale[k] = scale, out.bf[k] = bf;
  out.pr[k] = pr;
}

struct SplitChunks {  // largest piece per class
  int c[l2g_impl::kEnumClasses];
};

// Primitive-range split of the sorted items: an item of class c whose
// primitive loop is longer than chunk[c] becomes ceil(len / chunk[c])
// consecutive pieces of near-equal length.
__global__ void __launch_bounds__(kEnumThreads) split_count(long long n, const unsigned* __restrict__ key,
                                                               const int2* __restrict__ pr,
                                                               const SplitChunks chunk,
                                                               unsigned* __restrict__ pieces,
                                                               unsigned long long* __restrict__ cls_pieces) {
  __shared__ unsigned int hist[l2g_impl::kEnumClasses];
  for (int c = threadIdx.x; c < l2g_impl::kEnumClasses; c += kEnumThreads) hist[c] = 0;
  __syncthreads();
  const long long i = (long long)blockIdx.x * kEnumThreads + threadIdx.x;
  if (i < n) {
    const int c = (int)(key[i] >> 13);
    const int len = pr[i].y - pr[i].x, ch = chunk.c[c];
    const unsigned np = len > ch ? (unsigned)((len + ch - 1) / ch) : 1u;
    pieces[i] = np;
    atomicAdd(&hist[c], np);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < l2g_impl::kEnumClasses; c += kEnumThreads)
    if (hist[c]) atomicAdd(&cls_pieces[c], (unsigned long long)hist[c]);
}

__global__ void __launch_bounds__(kEnumThreads) split_fill(long long n, const unsigned* __restrict__ pieces,
                                                              const unsigned long long* __restrict__ at,
                                                              l2g_impl::FockEnumState::Items in,
                                                              l2g_impl::FockEnumState::Items out) {
  const long long i = (long long)blockIdx.x * kEnumThreads + threadIdx.x;
  if (i >= n) return;
  const unsigned np = pieces[i];
  const unsigned long long o = at[i];
  const int b = in.pr[i].x, len = in.pr[i].y - b;
  const int bra = in.bra[i], ket = in.ket[i], meta = in.meta[i];
  const double lnp = in.lnp[i], scale = in.scale[i];
  const int4 bf = in.bf[i];
  for (unsigned k = 0; k < np; ++k) {
    const unsigned long long j = o + k;
    out.bra[j] = bra, out.ket[j] = ket, out.meta[j] = meta, out.lnp[j] = lnp, out.scale[j] = scale, out.bf[j] = bf;
    out.pr[j] = int2{b + (int)((long long)len * k / np), b + (int)((long long)len * (k + 1) / np)};
  }
}

}  // namespace

namespace l2g_impl {

namespace {

// Ranges of one allocation.
struct Arena {
  size_t bytes = 0;
  char* base = nullptr;
  size_t add(size_t b) {
    const size_t at = bytes;
    bytes += (b + 255) & ~size_t(255);
    return at;
  }
  template <class T>
  T* at(size_t o) const {
    return reinterpret_cast<T*>(base + o);
  }
};

// Workspaces up to this size stay with the builder from build to build (an
// allocation and its release cost a small molecule's build 10 us each, and
// there were 28); larger ones are given back.
constexpr size_t kKeepBytes = size_t(64) << 20;

void alloc_items(FockEnumState::Bufs& b, size_t n) {
  b.bra.alloc(n * sizeof(int));
  b.ket.alloc(n * sizeof(int));
  b.meta.alloc(n * sizeof(int));
  b.lnp.alloc(n * sizeof(double));
  b.scale.alloc(n * sizeof(double));
  b.bf.alloc(n * sizeof(int4));
  b.pr.alloc(n * sizeof(int2));
}

unsigned blocks(long long n) { return (unsigned)((n + kEnumThreads - 1) / kEnumThreads); }

}  // namespace

void fock_split_device(FockEnumState& S, const std::vector<int>& chunk, hipStream_t st) {
  const long long n = S.n;
  S.cls_pieces.assign(kEnumClasses, 0ull);
  if (n == 0) return;
  if ((int)chunk.size() != kEnumClasses) throw L2gError(L2G_E_STATE, "split: one chunk per class expected");
  LAUNCHCHK("work before the item split");
  SplitChunks sc;
  std::copy(chunk.begin(), chunk.end(), sc.c);
  Arena a;
  const size_t o_pieces = a.add((size_t)n * sizeof(unsigned)), o_at = a.add((size_t)n * sizeof(unsigned long long)),
               o_cls = a.add(kEnumClasses * sizeof(unsigned long long));
  size_t tmp_bytes = 0;
  HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, (unsigned*)nullptr, (unsigned long long*)nullptr, (int)n,
                                          st));
  const size_t o_tmp = a.add(std::max<size_t>(tmp_bytes, 16));
  S.work.alloc(a.bytes);
  a.base = S.work.as<char>();
  unsigned* const pieces = a.at<unsigned>(o_pieces);
  unsigned long long *const at = a.at<unsigned long long>(o_at), *const cls = a.at<unsigned long long>(o_cls);
  HIPCHK(hipMemsetAsync(cls, 0, kEnumClasses * sizeof(unsigned long long), st));
  hipLaunchKernelGGL(split_count, dim3(blocks(n)), dim3(kEnumThreads), 0, st, n, S.key.as<unsigned>(),
                     S.cur.pr.as<int2>(), sc, pieces, cls);
  LAUNCHCHK("split_count");
  HIPCHK(hipcub::DeviceScan::ExclusiveSum(a.at<char>(o_tmp), tmp_bytes, pieces, at, (int)n, st));
  HIPCHK(hipMemcpyAsync(S.cls_pieces.data(), cls, kEnumClasses * sizeof(unsigned long long), hipMemcpyDeviceToHost,
                        st));
  HIPCHK(hipStreamSynchronize(st));
  unsigned long long total = 0;
  for (int c = 0; c < kEnumClasses; ++c) {
    if (S.cls_pieces[c] < S.cls_count[c])
      throw L2gError(L2G_E_STATE, "split: class " + std::to_string(c) + " has " + std::to_string(S.cls_pieces[c]) +
                                      " pieces for " + std::to_string(S.cls_count[c]) + " items");
    total += S.cls_pieces[c];
  }
  if (total >= (1ull << 31)) throw L2gError(L2G_E_INVALID, "more than 2^31 work items in one Fock build");
  if (total != (unsigned long long)n) {  // else nothing to split
    alloc_items(S.alt, total);
    hipLaunchKernelGGL(split_fill, dim3(blocks(n)), dim3(kEnumThreads), 0, st, n, pieces, at, S.cur.items(),
                       S.alt.items());
    LAUNCHCHK("split_fill");
    std::swap(S.cur, S.alt);
    S.n = (long long)total;
  }
  if (S.work.bytes > kKeepBytes || S.alt.bytes() > kKeepBytes) {
    HIPCHK(hipStreamSynchronize(st));
    S.work = DevBuf();
    S.alt = FockEnumState::Bufs();
  }
}

void fock_count_device(const FockEnumArgs& E, const double* D, long long nbf, double* Dn, FockEnumState& S,
                       hipStream_t st) {
  const long long np = E.npairs;
  S.total_t = np * (np + 1) / 2;
  S.block_count.clear();
  S.nblocks = 0;
  S.tchunk = 0;
  S.dmax = 0.0;
  // 4 quartets a thread in small molecules (64 left a 3-atom molecule one
  // block: 77 us for its list, now 11), more where 8192 blocks are reached
  S.nblocks = (int)std::min<long long>(8192, (S.total_t + kEnumThreads * 4 - 1) / (kEnumThreads * 4));
  if (S.nblocks) S.tchunk = (S.total_t + S.nblocks - 1) / S.nblocks;
  S.counts.alloc((size_t)(S.nblocks + 1) * sizeof(long long));
  long long* const counts = S.counts.as<long long>();  // dmax, then a count per block
  HIPCHK(hipMemsetAsync(counts, 0, sizeof(long long), st));
  if (E.n) {
    hipLaunchKernelGGL(shell_norms, dim3(blocks(E.n * E.n)), dim3(kEnumThreads), 0, st, D, nbf, E.bf1st, (int)E.n, Dn,
                       reinterpret_cast<unsigned long long*>(counts));
    LAUNCHCHK("shell_norms");
  }
  if (S.nblocks) {
    hipLaunchKernelGGL(enum_count, dim3(S.nblocks), dim3(kEnumThreads), 0, st, E, S.total_t, S.tchunk, counts + 1);
    LAUNCHCHK("enum_count");
  }
  S.block_count.resize(S.nblocks + 1);
  HIPCHK(hipMemcpyAsync(S.block_count.data(), counts, (size_t)(S.nblocks + 1) * sizeof(long long),
                        hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  std::memcpy(&S.dmax, S.block_count.data(), sizeof(double));
  S.block_count.erase(S.block_count.begin());
}

void fock_fill_device(const FockEnumArgs& E, FockEnumState& S, int blk0, int blk1, hipStream_t st) {
  S.n = 0;
  S.cls_count.assign(kEnumClasses, 0ull);
  S.cls_nprim.assign(kEnumClasses, 0ull);
  if (blk1 <= blk0) return;
  const int nb = blk1 - blk0;
  std::vector<long long> base(nb);
  long long n = 0;
  for (int b = 0; b < nb; ++b) {
    base[b] = n;
    n += S.block_count[blk0 + b];
  }
  S.n = n;
  if (n == 0) return;
  if (n >= (1ll << 31)) throw L2gError(L2G_E_INVALID, "more than 2^31 screened quartets in one window of a Fock build");
  S.base.alloc((size_t)nb * sizeof(long long));
  HIPCHK(hipMemcpyAsync(S.base.p, base.data(), (size_t)nb * sizeof(long long), hipMemcpyHostToDevice, st));
  // unsorted items, then sorted
  const size_t sz = (size_t)n;
  Arena a;
  const size_t o_bra = a.add(sz * sizeof(int)), o_ket = a.add(sz * sizeof(int)), o_meta = a.add(sz * sizeof(int)),
               o_lnp = a.add(sz * sizeof(double)), o_scale = a.add(sz * sizeof(double)),
               o_bf = a.add(sz * sizeof(int4)), o_pr = a.add(sz * sizeof(int2)), o_key = a.add(sz * sizeof(unsigned)),
               o_idx = a.add(sz * sizeof(unsigned)), o_perm = a.add(sz * sizeof(unsigned)),
               o_stats = a.add(2 * kEnumClasses * sizeof(unsigned long long));
  size_t tmp_bytes = 0;
  HIPCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, (unsigned*)nullptr, (unsigned*)nullptr,
                                            (unsigned*)nullptr, (unsigned*)nullptr, (int)n, 0, kEnumKeyBits, st));
  const size_t o_tmp = a.add(std::max<size_t>(tmp_bytes, 16));
  S.work.alloc(a.bytes);
  a.base = S.work.as<char>();
  S.key.alloc(sz * sizeof(unsigned));
  alloc_items(S.cur, sz);
  FockEnumOut O;
  O.bra = a.at<int>(o_bra);
  O.ket = a.at<int>(o_ket);
  O.meta = a.at<int>(o_meta);
  O.lnp = a.at<double>(o_lnp);
  O.scale = a.at<double>(o_scale);
  O.bf = a.at<int4>(o_bf);
  O.pr = a.at<int2>(o_pr);
  O.key = a.at<unsigned>(o_key);
  O.idx = a.at<unsigned>(o_idx);
  O.cls_count = a.at<unsigned long long>(o_stats);
  O.cls_nprim = O.cls_count + kEnumClasses;
  HIPCHK(hipMemsetAsync(O.cls_count, 0, 2 * kEnumClasses * sizeof(unsigned long long), st));
  hipLaunchKernelGGL(enum_fill, dim3(nb), dim3(kEnumThreads), 0, st, E, S.total_t, S.tchunk, (long long)blk0,
                     S.base.as<long long>(), O);
  LAUNCHCHK("enum_fill");
  // sort the item indices by (class, decreasing depth)
  HIPCHK(hipcub::DeviceRadixSort::SortPairs(a.at<char>(o_tmp), tmp_bytes, O.key, S.key.as<unsigned>(), O.idx,
                                            a.at<unsigned>(o_perm), (int)n, 0, kEnumKeyBits, st));
  hipLaunchKernelGGL(gather_items, dim3(blocks(n)), dim3(kEnumThreads), 0, st, O, a.at<unsigned>(o_perm),
                     S.cur.items(), n);
  LAUNCHCHK("gather_items");
  std::vector<unsigned long long> h(2 * kEnumClasses);
  HIPCHK(hipMemcpyAsync(h.data(), O.cls_count, 2 * kEnumClasses * sizeof(unsigned long long), hipMemcpyDeviceToHost,
                        st));
  HIPCHK(hipStreamSynchronize(st));
  if (S.work.bytes > kKeepBytes) S.work = DevBuf();
  for (int c = 0; c < kEnumClasses; ++c) S.cls_count[c] = h[c], S.cls_nprim[c] = h[kEnumClasses + c];
  if (S.cls_count[kEnumClasses - 1]) throw L2gError(L2G_E_LMAX, "no Fock kernel for an angular momentum class");
}

}  // namespace l2g_impl
