// Sparse matrix times sparse vector (SpMSpV) and top-down BFS for gfx950.
//
// cbx_spmspv replaces the local y = A*x of CombBLAS's SpMV with a sparse
// vector: SpImpl<SR,IT,NUM,IVT,OVT>::SpMXSpV (SpImpl.cpp:55-158) and its
// boolean-matrix form SpImpl<SR,IT,bool,IVT,OVT>::SpMXSpV (SpImpl.cpp:167-213),
// reached through generic_gespmv (Friends.h:448-482).  Output indices are
// ascending, an entry exists wherever some A(i,k) x_k term exists, and a
// boolean A contributes x_k itself (the boolean specialisation never calls
// multiply, SpImpl.cpp:183-188).  The GPU form is a dense accumulator over the
// m rows with a presence bitmap; products are block-flattened across the
// frontier's columns, and the output is compacted in row order by a scan of
// the bitmap's word counts.
//
// The BFS plan runs the level loop of TopDownBFS.cpp:442-448 with
// SelectMaxSRing<bool,int64> (parent = largest frontier neighbour):
//   fringe.setNumToInd(); fringe = SpMV(A, fringe); fringe = EWiseMult(fringe,
//   parents, exclude=true, -1); parents.Set(fringe);
// fused per level into two kernels: expand (every frontier vertex k offers k to
// each unvisited neighbour with an atomic max; the first offer appends the
// neighbour to the next frontier) and finalize (parents = offers; mark
// visited).  Large frontiers of a symmetric pattern go bottom-up instead, from
// and to a bitmap.  Each level is one captured hipGraph, whose last kernel
// reports the next frontier's size and edges to the host's pinned memory (two
// copies took longer than the small levels' kernels).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <cstdlib>
#include <cstring>
#include <limits>
#include <mutex>
#include <type_traits>

#include "cbx_device.h"
#include "cbx_flatten.h"
#include "cbx_index.h"
#include "cbx_semiring.h"
#include "cbx_spgemm.h"

namespace cbx {

// ----------------------------------------------- global-memory accumulation
template <int K, class T>
struct GAcc;
template <>
struct GAcc<kPlusTimes, int64_t> {
  static __device__ void acc(int64_t* p, int64_t v) { atomicAdd((unsigned long long*)p, (unsigned long long)v); }
};
template <>
struct GAcc<kPlusTimes, double> {
  static __device__ void acc(double* p, double v) { atomicAdd(p, v); }
};
template <>
struct GAcc<kPlusTimes, float> {
  static __device__ void acc(float* p, float v) { atomicAdd(p, v); }
};
template <>
struct GAcc<kMinPlus, int64_t> {
  static __device__ void acc(int64_t* p, int64_t v) { atomicMin((long long*)p, (long long)v); }
};
template <>
struct GAcc<kSelectMax, int64_t> {
  static __device__ void acc(int64_t* p, int64_t v) { atomicMax((long long*)p, (long long)v); }
};
// SR::add on a value in memory, which keeps a NaN there; with `empty_nan` a NaN
// is an accumulator without products yet.
template <class F, class U>
__device__ void gcas_minmax(F* p, F v, bool is_min, bool empty_nan = false) {
  U* up = reinterpret_cast<U*>(p);
  U old = __hip_atomic_load(up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  while (true) {
    const F cur = __builtin_bit_cast(F, old);
    if (!((is_min ? (v < cur) : (cur < v)) || (empty_nan && cur != cur))) return;
    if (__hip_atomic_compare_exchange_strong(up, &old, __builtin_bit_cast(U, v), __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      return;
  }
}
template <>
struct GAcc<kMinPlus, double> {
  static __device__ void acc(double* p, double v) { gcas_minmax<double, unsigned long long>(p, v, true); }
};
template <>
struct GAcc<kMinPlus, float> {
  static __device__ void acc(float* p, float v) { gcas_minmax<float, unsigned int>(p, v, true); }
};
template <>
struct GAcc<kSelectMax, double> {
  static __device__ void acc(double* p, double v) { gcas_minmax<double, unsigned long long>(p, v, false); }
};
template <>
struct GAcc<kSelectMax, float> {
  static __device__ void acc(float* p, float v) { gcas_minmax<float, unsigned int>(p, v, false); }
};

// Into an accumulator that started at ident_of().
template <int K, class T>
__device__ __forceinline__ void acc_new(T* p, T v) {
  if constexpr (K == kPlusTimes || !std::is_floating_point<T>::value) {
    GAcc<K, T>::acc(p, v);
  } else {
    using Bits = typename std::conditional<sizeof(T) == 8, unsigned long long, unsigned int>::type;
    gcas_minmax<T, Bits>(p, v, K == kMinPlus, true);
  }
}

namespace {

// What one product's kernels count: the structure check of A (cbx_spgemm.h),
// whether x breaks its rules, the long columns set aside, and y's entries.
struct SpvFlags {
  unsigned long long chk[3];
  int bad_x, nhubs, ny;
  __device__ __host__ bool malformed() const { return chk[0] || chk[1] != chk[2]; }
};

template <class T>
__global__ void k_sv_begin(int32_t* __restrict__ colmap, int64_t n, T* __restrict__ acc, int64_t m, T ident,
                           uint32_t* __restrict__ bits, int64_t nw, SpvFlags* __restrict__ f) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) colmap[i] = -1;
  if (i < m) acc[i] = ident;
  if (i < nw) bits[i] = 0u;
  if (i == 0) *f = SpvFlags{{0ull, 0ull, 0ull}, 0, 0, 0};
}

// A lane's value of the lane STEP before it in its row of sixteen (`none` in the
// row's first lanes), or after it.
template <int STEP>
__device__ __forceinline__ int row_before(int v, int none) {
  return __builtin_amdgcn_update_dpp(none, v, 0x110 + STEP, 0xf, 0xf, false);
}
__device__ __forceinline__ int row_after(int v, int none) {
  return __builtin_amdgcn_update_dpp(none, v, 0x101, 0xf, 0xf, false);
}

template <int STEP>
__device__ __forceinline__ void row_or(int at, uint32_t& mask) {
  const int w = row_before<STEP>(at, -1);
  const uint32_t o = (uint32_t)row_before<STEP>((int)mask, 0);
  if (w == at) mask |= o;
}

// One lane's U products into the accumulator, where there are some (ok), with
// the loads in flight together; e: places in A (valid also without a product),
// consecutive along each row of sixteen lanes.  Whole rows call it.
template <int K, class T, bool BOOLA, int U>
__device__ __forceinline__ void sv_products(const int64_t* __restrict__ ir, const T* __restrict__ val,
                                            const int64_t (&e)[U], const bool (&ok)[U], T x, T* __restrict__ acc,
                                            uint32_t* __restrict__ bits) {
  using SR = Sem<K, T>;
  int64_t r[U];
  T a[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    r[u] = ir[e[u]];
    if constexpr (!BOOLA) a[u] = val[e[u]];
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    pin(r[u]);
    if constexpr (!BOOLA) pin(a[u]);
  }
  // The rows of a step ascend along a row of sixteen lanes, so its lanes with
  // one word of the bitmap are neighbours: they set their bits with one atomic.
  // (Hubs lie next to each other in skewed graphs, and thousands of products
  // meet in one word: 147 K products of R-MAT s18 took 46 us with this, 79 with
  // an atomic each.  Looking first whether the bit is set, or whether a maximum
  // grows, took longer: the loads queue at the same words.)
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int at = ok[u] ? (int)(r[u] >> 5) : -1;
    uint32_t mask = ok[u] ? 1u << (r[u] & 31) : 0u;
    row_or<1>(at, mask);
    row_or<2>(at, mask);
    row_or<4>(at, mask);
    row_or<8>(at, mask);
    if (at >= 0 && row_after(at, -1) != at ) atomicOr(&bits[at], mask);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (!ok[u]) continue;
    T v;
    if constexpr (BOOLA) v = x;
    else v = (T)SR::out(SR::mul(a[u], x));
    acc_new<K, T>(&acc[r[u]], v);
  }
}

// y_acc[i] (+)= A(i,k) (x) x_k for k in x; presence bit per row.  Sixteen lanes
// take an entry of x, 64 products a step; columns longer than kSvHub go to a
// list while it has room (x is short and its columns' lengths skewed: one
// workgroup for 256 entries of x left the chip idle behind the longest column,
// 102 us for the 5242 columns of R-MAT s18 that 27 + 19 us take now; lists from
// 128 or 512 entries on measured the same within 2 us).
// x entries must be valid column indices, ascending and unique.
constexpr int kSvExpandNT = 256, kSvGroup = 16;
constexpr int64_t kSvHub = 256, kSvPiece = 512;
constexpr int kSvMaxHubs = 2048;

template <int K, class T, bool BOOLA>
__global__ __launch_bounds__(kSvExpandNT) void k_sv_expand(const int64_t* __restrict__ cpA,
                                                           const int64_t* __restrict__ irA,
                                                           const void* __restrict__ valA,
                                                           const int32_t* __restrict__ colmap, int64_t n,
                                                           const int32_t* __restrict__ xind,
                                                           const T* __restrict__ xval, int32_t nx,
                                                           T* __restrict__ acc, uint32_t* __restrict__ bits,
                                                           int32_t* __restrict__ hubs, int max_hubs, SpvFlags* f) {
  constexpr int U = 4, GROUPS = kSvExpandNT / kSvGroup;
  if (f->malformed()) return;
  const int l = threadIdx.x % kSvGroup;
  for (int64_t t = (int64_t)blockIdx.x * GROUPS + threadIdx.x / kSvGroup; t < nx; t += (int64_t)gridDim.x * GROUPS) {
    const int32_t k = xind[t], next = t + 1 < nx ? xind[t + 1] : INT32_MAX;
    if (k < 0 || k >= n || next <= k) {
      f->bad_x = 1;
      continue;
    }
    const int32_t p = colmap[k];
    if (p < 0) continue;
    const T x = xval[t];
    const int64_t b = cpA[p];
    int64_t end = cpA[p + 1];
    if (end - b > kSvHub) {
      int slot = 0;
      if (l == 0) slot = atomicAdd(&f->nhubs, 1);
      slot = __shfl(slot, 0, kSvGroup);
      if (slot < max_hubs) {
        if (l == 0) hubs[slot] = (int32_t)t;
        continue;
      }
    }
    for (int64_t i = b; i < end; i += U * kSvGroup) {
      int64_t e[U];
      bool ok[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        ok[u] = i + u * kSvGroup + l < end;
        e[u] = min(i + u * kSvGroup + l, end - 1);
      }
      sv_products<K, T, BOOLA, U>(irA, (const T*)valA, e, ok, x, acc, bits);
    }
  }
}

// The listed columns, in pieces of kSvPiece products, one per workgroup at a time.
template <int K, class T, bool BOOLA>
__global__ __launch_bounds__(kSvExpandNT) void k_sv_expand_hubs(const int64_t* __restrict__ cpA,
                                                                const int64_t* __restrict__ irA,
                                                                const void* __restrict__ valA,
                                                                const int32_t* __restrict__ colmap,
                                                                const int32_t* __restrict__ xind,
                                                                const T* __restrict__ xval, T* __restrict__ acc,
                                                                uint32_t* __restrict__ bits,
                                                                const int32_t* __restrict__ hubs, int max_hubs,
                                                                const SpvFlags* __restrict__ f) {
  constexpr int PT = kSvMaxHubs / kSvExpandNT, U = (int)(kSvPiece / kSvExpandNT);
  __shared__ int off[kSvMaxHubs + 1];
  __shared__ int64_t beg[kSvMaxHubs], end[kSvMaxHubs];
  __shared__ T xs[kSvMaxHubs];
  __shared__ int wsum[kSvExpandNT / kWave];
  const int nh = min(f->nhubs, max_hubs);
  if (nh == 0) return;
  int np[PT], sum = 0;
#pragma unroll
  for (int k = 0; k < PT; ++k) {
    const int h = threadIdx.x * PT + k;
    np[k] = 0;
    if (h < nh) {
      const int32_t t = hubs[h], p = colmap[xind[t]];
      beg[h] = cpA[p];
      end[h] = cpA[p + 1];
      xs[h] = xval[t];
      np[k] = (int)((end[h] - beg[h] + kSvPiece - 1) / kSvPiece);
    }
    sum += np[k];
  }
  int total;
  int ex = block_excl_scan<kSvExpandNT>(sum, wsum, total);
#pragma unroll
  for (int k = 0; k < PT; ++k) {
    off[threadIdx.x * PT + k] = ex;
    ex += np[k];
  }
  if (threadIdx.x == 0) off[kSvMaxHubs] = total;
  __syncthreads();
  for (int piece = blockIdx.x; piece < total; piece += gridDim.x) {
    int lo = 0, hi = nh;  // the last h with off[h] <= piece
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (off[mid] <= piece) lo = mid;
      else hi = mid;
    }
    const int64_t i = beg[lo] + (piece - off[lo]) * kSvPiece;
    int64_t e[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      ok[u] = i + u * kSvExpandNT + (int)threadIdx.x < end[lo];
      e[u] = min(i + u * kSvExpandNT + (int)threadIdx.x, end[lo] - 1);
    }
    sv_products<K, T, BOOLA, U>(irA, (const T*)valA, e, ok, xs[lo], acc, bits);
  }
}

// y's entries in each block of wpb bitmap words; then, with the blocks before
// it summed by every block (at most kSvMaxSums), the entries themselves: a lane
// per row.
constexpr int kSvEmitNT = 256;
constexpr int64_t kSvMaxSums = 4096;

__global__ __launch_bounds__(kSvEmitNT) void k_sv_count(const uint32_t* __restrict__ bits, int64_t nw, int64_t wpb,
                                                        int32_t* __restrict__ sums) {
  __shared__ long long wsum[kSvEmitNT / kWave];
  const int64_t w0 = blockIdx.x * wpb, w1 = min(nw, w0 + wpb);
  long long c = 0;
  for (int64_t w = w0 + threadIdx.x; w < w1; w += kSvEmitNT) c += __popc(bits[w]);
  c = block_sum_ll<kSvEmitNT>(c, wsum);
  if (threadIdx.x == 0) sums[blockIdx.x] = (int32_t)c;
}

template <class T>
__global__ __launch_bounds__(kSvEmitNT) void k_sv_emit(const uint32_t* __restrict__ bits, int64_t nw, int64_t wpb,
                                                       const int32_t* __restrict__ sums, const T* __restrict__ acc,
                                                       int32_t* __restrict__ yind, T* __restrict__ yval, SpvFlags* f) {
  constexpr int NW = kSvEmitNT / kWave, R = kWave / 2 / NW;  // rounds of 64 rows per wave and 64 words
  __shared__ long long wsum[NW];
  if (f->malformed() || f->bad_x) return;  // y is left as it was
  long long before = 0;
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += kSvEmitNT) before += sums[b];
  before = block_sum_ll<kSvEmitNT>(before, wsum);
  int64_t at = before;
  const int64_t w0 = blockIdx.x * wpb, w1 = min(nw, w0 + wpb);
  const int lane = lane_id(), wave = wave_id_uniform();
  for (int64_t w = w0; w < w1; w += kWave) {
    const uint32_t word = w + lane < w1 ? bits[w + lane] : 0u;
    const int incl = wave_incl_scan(__popc(word));
    const int excl = incl - __popc(word);
    T v[R];
    bool in[R];
    unsigned lo[R], hi[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int j = 2 * (wave * R + k);
      lo[k] = (unsigned)__builtin_amdgcn_readlane((int)word, j);
      hi[k] = (unsigned)__builtin_amdgcn_readlane((int)word, j + 1);
      in[k] = ((lane < 32 ? lo[k] : hi[k]) >> (lane & 31)) & 1u;
      v[k] = acc[in[k] ? (w + j) * 32 + lane : 0];
    }
#pragma unroll
    for (int k = 0; k < R; ++k) pin(v[k]);
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int j = 2 * (wave * R + k);
      const int64_t q = at + __builtin_amdgcn_readlane(excl, j) +
                        (int)__builtin_amdgcn_mbcnt_hi(hi[k], __builtin_amdgcn_mbcnt_lo(lo[k], 0u));
      if (in[k]) {
        yind[q] = (int32_t)((w + j) * 32 + lane);
        yval[q] = v[k];
      }
    }
    at += __builtin_amdgcn_readlane(incl, kWave - 1);
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) f->ny = (int)at;
}

inline unsigned nb(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

#define CBX_TRY_SV(x)              \
  do {                             \
    cbx_status st_ = (x);          \
    if (st_ != CBX_OK) return st_; \
  } while (0)

template <int K, class T>
T ident_of() {
  if (K == kPlusTimes) return std::is_floating_point<T>::value ? (T)-0.0 : (T)0;
  if (std::is_floating_point<T>::value) return std::numeric_limits<T>::quiet_NaN();  // (as in cbx_semiring.h)
  if (K == kMinPlus) return std::numeric_limits<T>::max();
  return std::numeric_limits<T>::lowest();
}

// Scratch of one SpMSpV: the column map of A (n), the dense accumulator (m
// values) and presence bitmap (nw words), the flags, and 2 * (nw + 1) words for
// the blocks' sums and the list of long columns.
struct SvWork {
  int32_t *colmap = nullptr, *lists = nullptr;
  void* acc = nullptr;
  uint32_t* bits = nullptr;
  SpvFlags* flags = nullptr;
};

inline int64_t sv_words(int64_t m) { return m / 32 + 1; }

// The product with its scratch in `w` (every array is initialised here, so
// the scratch may hold anything on entry); A has columns and x entries.  The
// structure check of A runs first; what follows it stops at its verdict.
template <int K, class T>
cbx_status spmspv_run(const cbx_dcsc* A, bool boolA, const int32_t* xind, const T* xval, int32_t nx, int32_t* yind,
                      T* yval, int32_t* ny, const SvWork& w, hipStream_t s) {
  const int64_t m = A->m, n = A->n, nw = sv_words(m);
  T* acc = (T*)w.acc;
  const int64_t wpb = kWave * ((nw + kWave * kSvMaxSums - 1) / (kWave * kSvMaxSums));
  const int64_t nblk = (nw + wpb - 1) / wpb;
  int32_t *sums = w.lists, *hubs = w.lists + nblk;
  const int max_hubs = (int)std::min<int64_t>(kSvMaxHubs, 2 * (nw + 1) - nblk);
  k_sv_begin<T><<<nb(std::max(std::max(m, n), nw), 256), 256, 0, s>>>(w.colmap, n, acc, m, ident_of<K, T>(), w.bits,
                                                                     nw, w.flags);
  dcsc_check_structure_launch(A, w.flags->chk, w.colmap, s);
  const unsigned g = std::min(nb(nx, kSvExpandNT / kSvGroup), 16384u), gh = 512;
  if (boolA) {
    k_sv_expand<K, T, true><<<g, kSvExpandNT, 0, s>>>(A->cp, A->ir, A->val, w.colmap, n, xind, xval, nx, acc, w.bits,
                                                     hubs, max_hubs, w.flags);
    k_sv_expand_hubs<K, T, true><<<gh, kSvExpandNT, 0, s>>>(A->cp, A->ir, A->val, w.colmap, xind, xval, acc, w.bits,
                                                           hubs, max_hubs, w.flags);
  } else {
    k_sv_expand<K, T, false><<<g, kSvExpandNT, 0, s>>>(A->cp, A->ir, A->val, w.colmap, n, xind, xval, nx, acc, w.bits,
                                                      hubs, max_hubs, w.flags);
    k_sv_expand_hubs<K, T, false><<<gh, kSvExpandNT, 0, s>>>(A->cp, A->ir, A->val, w.colmap, xind, xval, acc, w.bits,
                                                            hubs, max_hubs, w.flags);
  }
  k_sv_count<<<(unsigned)nblk, kSvEmitNT, 0, s>>>(w.bits, nw, wpb, sums);
  k_sv_emit<T><<<(unsigned)nblk, kSvEmitNT, 0, s>>>(w.bits, nw, wpb, sums, acc, yind, yval, w.flags);
  SpvFlags h{};
  CBX_HIP(hipGetLastError());
  CBX_HIP(hipMemcpyAsync(&h, w.flags, sizeof(h), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  if (h.malformed()) return set_error(CBX_ERR_INVALID, "cbx_dcsc_check: malformed DCSC");
  if (h.bad_x) return set_error(CBX_ERR_INVALID, "cbx_spmspv: x indices must be ascending, unique and below ncols");
  *ny = h.ny;
  return CBX_OK;
}

template <int K, class T>
cbx_status spmspv_typed(const cbx_dcsc* A, bool boolA, const int32_t* xind, const T* xval, int32_t nx, int32_t* yind,
                        T* yval, int32_t* ny, hipStream_t s) {
  const int64_t m = A->m, n = A->n, nw = sv_words(m);
  ScratchSet ws(s);
  SvWork w;
  T* acc = nullptr;
  if (!ws.take(&w.colmap, std::max<int64_t>(n, 1)) || !ws.take(&w.lists, 2 * (nw + 1)) ||
      !ws.take(&acc, std::max<int64_t>(m, 1)) || !ws.take(&w.bits, nw) || !ws.take(&w.flags, 1))
    return set_error(CBX_ERR_NOMEM, "cbx_spmspv: workspace allocation failed");
  w.acc = acc;
  return spmspv_run<K, T>(A, boolA, xind, xval, nx, yind, yval, ny, w, s);
}

// Carves the scratch of one SpMSpV out of one caller-given region; with base
// == null it only adds up the bytes.  Every piece starts on a 256-byte
// boundary.
template <class T>
size_t sv_carve(int64_t m, int64_t n, char* base, SvWork* w) {
  const int64_t nw = sv_words(m);
  size_t used = 0;
  auto take = [&](size_t bytes) -> void* {
    void* p = base ? base + used : nullptr;
    used += (std::max<size_t>(bytes, 1) + 255) & ~(size_t)255;
    return p;
  };
  SvWork t;
  t.colmap = (int32_t*)take(sizeof(int32_t) * std::max<int64_t>(n, 1));
  t.lists = (int32_t*)take(sizeof(int32_t) * 2 * (nw + 1));
  t.acc = take(sizeof(T) * std::max<int64_t>(m, 1));
  t.bits = (uint32_t*)take(sizeof(uint32_t) * nw);
  t.flags = (SpvFlags*)take(sizeof(SpvFlags));
  if (w) *w = t;
  return used;
}

// cbx_spmspv with its scratch in `region` (bytes of device memory): no
// allocation.
template <int K, class T>
cbx_status spmspv_in_region(const cbx_dcsc* A, bool boolA, const int32_t* xind, const T* xval, int32_t nx,
                            int32_t* yind, T* yval, int32_t* ny, char* region, size_t bytes, hipStream_t s) {
  *ny = 0;
  const size_t need = sv_carve<T>(A->m, A->n, nullptr, nullptr);
  CBX_RETURN_IF(need > bytes, CBX_ERR_LIMIT,
                "cbx_spmspv_noalloc: a %lld x %lld matrix needs %zu bytes of scratch, more than the %zu available",
                (long long)A->m, (long long)A->n, need, bytes);
  SvWork w;
  sv_carve<T>(A->m, A->n, region, &w);
  CBX_RETURN_IF(A->nzc == 0 && A->nnz != 0, CBX_ERR_INVALID, "cbx_dcsc_check: nnz without columns");
  if (A->nzc == 0) return CBX_OK;
  if (nx == 0) {  // the structure check all the same
    dcsc_check_launch(A, w.flags->chk, s);
    return dcsc_check_result(w.flags->chk, s);
  }
  return spmspv_run<K, T>(A, boolA, xind, xval, nx, yind, yval, ny, w, s);
}

}  // namespace

// ====================================================================== BFS
namespace {

// The rows of column j: [range[j].x, range[j].y) (empty: both 0).
__global__ void k_bfs_ranges(const int64_t* __restrict__ cp, const int64_t* __restrict__ jc, int64_t nzc,
                             int2* __restrict__ range) {
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p < nzc) range[jc[p]] = make_int2((int)cp[p], (int)cp[p + 1]);
}

// The vertices that no search reaches, as a bitmap: those without neighbours
// in a symmetric pattern (in another a vertex without a column may have rows),
// and the bits from n on.
__global__ __launch_bounds__(256) void k_bfs_isolated(const int2* __restrict__ range, int64_t n, int64_t nw,
                                                      bool symmetric, unsigned long long* __restrict__ isolated) {
  const int64_t w = global_wave();
  if (w >= nw) return;
  const int64_t v = w * kWave + lane_id();
  bool none = true;
  if (v < n) none = symmetric && range[v].x == range[v].y;
  const unsigned long long mask = __ballot(none);
  if (lane_id() == 0) isolated[w] = mask;
}

// Number of positions where two int64 arrays differ (the symmetry check of
// a plan: A's arrays against its transpose's).
__global__ void k_bfs_count_diff(const int64_t* __restrict__ a, const int64_t* __restrict__ b, int64_t n,
                                 unsigned long long* __restrict__ cnt) {
  long long d = 0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    d += a[i] != b[i];
  d = wave_sum_ll(d);
  if (lane_id() == 0 && d) atomicAdd(cnt, (unsigned long long)d);
}

__global__ void k_bfs_rows32(const int64_t* __restrict__ ir, int64_t nnz, int32_t* __restrict__ rows) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < nnz) rows[i] = (int32_t)ir[i];
}

// Frontier vertices with more than kBfsHub neighbours ("hubs") are expanded
// in pieces of kBfsHub edges by k_bfs_expand_hubs, one workgroup per piece,
// instead of by the workgroup that holds them in the frontier: R-MAT hubs have
// 10^5 neighbours and would otherwise keep one workgroup busy long after the
// others finished.  A piece is (vertex << 32 | piece index).
constexpr int64_t kBfsHub = 1024;

__device__ __forceinline__ void bfs_add_pieces(int32_t v, int64_t deg, int32_t* __restrict__ pcount,
                                               long long* __restrict__ pieces) {
  const int np = (int)((deg + kBfsHub - 1) / kBfsHub);
  const int b = atomicAdd(pcount, np);
  for (int k = 0; k < np; ++k) pieces[b + k] = ((long long)v << 32) | k;
}

// What a level's workgroups count: vertices found and their edges, in slots a
// line apart (thousands of workgroups adding to one counter would serialise).
constexpr int kBfsSlots = 64;
struct BfsSlot {
  unsigned long long found, edges, pad[6];
};

// A search's state on the device; k_bfs_level_end brings it from level to level.
struct BfsState {
  BfsSlot slots[kBfsSlots];
  int32_t listed[2], pieces[2];  // entries of the two frontier lists and of their hub pieces
  int32_t size;                  // the current frontier
  int32_t longs[2];              // vertices listed by k_bfs_bottom_up
  unsigned long long levels, reached;
};

// What the host reads (pinned): the next frontier's size and edges, levels and
// vertices reached so far.
struct BfsReport {
  unsigned long long size, edges, levels, reached;
};

__global__ void k_bfs_reset(int64_t n, int32_t* __restrict__ cand, int64_t* __restrict__ parents,
                            unsigned long long* __restrict__ visited,
                            const unsigned long long* __restrict__ isolated, int64_t nw, int32_t* __restrict__ f0,
                            long long* __restrict__ pieces0, const int2* __restrict__ range,
                            BfsState* __restrict__ st, BfsReport* __restrict__ rep, int64_t root) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) {
    cand[i] = -1;
    parents[i] = -1;
  }
  if (i < nw) visited[i] = isolated[i];
  if (i < kBfsSlots) {
    st->slots[i].found = 0ull;
    st->slots[i].edges = 0ull;
  }
  if (i == 0) {
    f0[0] = (int32_t)root;
    st->listed[0] = 1;
    st->listed[1] = 0;
    st->pieces[0] = 0;
    st->pieces[1] = 0;
    st->size = 1;
    st->levels = 0ull;
    st->reached = 0ull;
    st->longs[0] = 0;
    st->longs[1] = 0;
    const int64_t deg = range[root].y - range[root].x;
    if (deg > kBfsHub) bfs_add_pieces((int32_t)root, deg, &st->pieces[0], pieces0);
    rep->size = 1ull;
    rep->edges = (unsigned long long)deg;
  }
}

// Last kernel of a level from frontier `par` to 1 - par: sums the slots, counts
// the level if its frontier was not empty (a level launched after the search
// ended changes nothing), clears what the next level counts in and reports to
// the host.  A bottom-up level (bits) leaves its frontier as a bitmap, its list
// empty.  One wave.
__global__ __launch_bounds__(kWave) void k_bfs_level_end(BfsState* __restrict__ st, int par, bool bits,
                                                         BfsReport* __restrict__ rep) {
  BfsSlot& sl = st->slots[threadIdx.x];
  const long long found = wave_sum_ll((long long)sl.found);
  const long long edges = wave_sum_ll((long long)sl.edges);
  sl.found = 0ull;
  sl.edges = 0ull;
  if (threadIdx.x) return;
  const unsigned long long levels = st->levels + (st->size > 0), reached = st->reached + found;
  st->levels = levels;
  st->reached = reached;
  st->size = (int32_t)found;
  st->listed[par] = 0;
  st->pieces[par] = 0;
  if (bits) {
    st->longs[0] = 0;
    st->longs[1] = 0;
    st->listed[1 - par] = 0;
    st->pieces[1 - par] = 0;
  }
  *rep = BfsReport{(unsigned long long)found, (unsigned long long)edges, levels, reached};
}

// A workgroup's counts into its slot.
template <int NT>
__device__ __forceinline__ void bfs_count(BfsState* st, long long found, long long edges) {
  BfsSlot& sl = st->slots[blockIdx.x % kBfsSlots];
  block_add_counts<NT>(found, edges, &sl.found, &sl.edges);
}

// Frontier vertices offer themselves (k[u]) to neighbours r[u] (ok[u]: there is
// one): SelectMax keeps the largest offer in cand[r]; the first offer appends r
// to the next frontier, one atomic per wave for the appends of this step.  The
// U probes of a lane are in flight together.  All lanes call it.
template <int U>
__device__ __forceinline__ void bfs_offer(const int32_t (&r)[U], const int32_t (&k)[U], const bool (&ok)[U],
                                          const uint32_t* __restrict__ visited, int32_t* __restrict__ cand,
                                          int32_t* __restrict__ fout, int32_t* __restrict__ fout_count) {
  uint32_t word[U];
  int32_t seen[U], old[U];
#pragma unroll
  for (int u = 0; u < U; ++u) word[u] = visited[r[u] >> 5];
#pragma unroll
  for (int u = 0; u < U; ++u) pin(word[u]);
  bool live[U];
  // Offers only grow cand, so a value read without the atomic (possibly
  // stale, never above the true one) that already holds an offer at least
  // this large makes the atomic a no-op: skip it.  Hubs receive thousands
  // of offers per level and only the record-breaking ones reach the
  // serialising atomic.  (Lanes without an unvisited neighbour read cand[0].)
#pragma unroll
  for (int u = 0; u < U; ++u) {
    live[u] = ok[u] && !((word[u] >> (r[u] & 31)) & 1u);
    seen[u] = __hip_atomic_load(&cand[live[u] ? r[u] : 0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) pin(seen[u]);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    old[u] = 0;
    if (live[u] && seen[u] < k[u]) old[u] = atomicMax(&cand[r[u]], k[u]);
  }
  unsigned long long mask[U];
  int total = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    mask[u] = __ballot(old[u] == -1);
    total += __popcll(mask[u]);
  }
  if (!total) return;
  int at = 0;
  if (lane_id() == 0) at = atomicAdd(fout_count, total);
  at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (old[u] == -1)
      fout[at + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask[u] >> 32),
                                               __builtin_amdgcn_mbcnt_lo((unsigned)mask[u], 0u))] = r[u];
    at += __popcll(mask[u]);
  }
}

// One level's SpMV(A, fringe) with SelectMax<bool,int64> fused with the
// EWiseMult(exclude) filter: each frontier vertex k offers k to its unvisited
// neighbours; cand[i] keeps the largest offer; the first offer appends i.
template <int NT, int U>
__global__ __launch_bounds__(NT) void k_bfs_expand(const int2* __restrict__ range, const int32_t* __restrict__ rows,
                                                   const int32_t* __restrict__ fin,
                                                   const int32_t* __restrict__ fin_count,
                                                   const uint32_t* __restrict__ visited, int32_t* __restrict__ cand,
                                                   int32_t* __restrict__ fout, int32_t* __restrict__ fout_count) {
  __shared__ FlatStage<int32_t, NT, true> st;
  const int nf = *fin_count;
  if ((int)blockIdx.x * NT >= nf) return;
  flat_init(st);
  int par = 0;
  for (int c0 = blockIdx.x * NT; c0 < nf; c0 += gridDim.x * NT) {
    const int t = c0 + threadIdx.x;
    int base = 0, len = 0;
    int32_t k = 0;
    if (t < nf) {
      k = fin[t];
      const int2 rg = range[k];
      base = rg.x;
      len = rg.y - rg.x;
      if (len > kBfsHub) len = 0;  // a hub: k_bfs_expand_hubs takes its pieces
    }
    const FlatSeg me = flat_stage<int32_t, NT, true>(st, base, len, k);
    flat_chunk<int32_t, NT, true, U>(st, me, par, [&](const int32_t(&idx)[U], int32_t(&ks)[U], const bool(&ok)[U]) {
      int32_t r[U];
#pragma unroll
      for (int u = 0; u < U; ++u) r[u] = rows[idx[u]];
#pragma unroll
      for (int u = 0; u < U; ++u) pin(r[u]);
      bfs_offer<U>(r, ks, ok, visited, cand, fout, fout_count);
    });
  }
}

// The hubs' pieces of the same level: one workgroup per piece of kBfsHub
// consecutive edges (coalesced row reads, kBfsHub / NT edges per thread).
template <int NT>
__global__ __launch_bounds__(NT) void k_bfs_expand_hubs(const int2* __restrict__ range,
                                                        const int32_t* __restrict__ rows,
                                                        const long long* __restrict__ pieces,
                                                        const int32_t* __restrict__ pcount,
                                                        const uint32_t* __restrict__ visited,
                                                        int32_t* __restrict__ cand, int32_t* __restrict__ fout,
                                                        int32_t* __restrict__ fout_count) {
  static_assert(kBfsHub % NT == 0, "whole rounds per piece");
  constexpr int U = kBfsHub / NT;
  const int np = *pcount;
  for (int p = blockIdx.x; p < np; p += gridDim.x) {
    const long long pc = pieces[p];
    const int32_t v = (int32_t)(pc >> 32);
    const int2 rg = range[v];
    const int e0 = rg.x + (int)((pc & 0xffffffffll) * kBfsHub);
    int32_t r[U], ks[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      ks[u] = v;
      r[u] = rows[entry_from(e0, rg.y, u * NT + (int)threadIdx.x, ok[u])];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) pin(r[u]);
    bfs_offer<U>(r, ks, ok, visited, cand, fout, fout_count);
  }
}

// parents.Set(fringe) (FullyDistVec.cpp:1036) and the visited mark; also
// counts the new frontier and its edges (the host's direction choice).
constexpr int kBfsFinNT = 256;
__global__ __launch_bounds__(kBfsFinNT) void k_bfs_finalize(const int32_t* __restrict__ f,
                                                            const int32_t* __restrict__ count,
                                                            const int32_t* __restrict__ cand,
                                                            const int2* __restrict__ range,
                                                            int64_t* __restrict__ parents,
                                                            uint32_t* __restrict__ visited, BfsState* st,
                                                            int32_t* __restrict__ pcount,
                                                            long long* __restrict__ pieces) {
  const int nf = *count;
  if ((int)blockIdx.x * kBfsFinNT >= nf) return;
  long long deg = 0;
  for (int t = blockIdx.x * kBfsFinNT + threadIdx.x; t < nf; t += gridDim.x * kBfsFinNT) {
    const int32_t i = f[t];
    parents[i] = cand[i];
    atomicOr(&visited[i >> 5], 1u << (i & 31));
    const int2 rg = range[i];
    const int d = rg.y - rg.x;
    deg += d;
    if (d > kBfsHub) bfs_add_pieces(i, d, pcount, pieces);  // the next level expands hubs in pieces
  }
  bfs_count<kBfsFinNT>(st, blockIdx.x == 0 && threadIdx.x == 0 ? nf : 0, deg);
}

// A frontier between its two forms: the list as a bitmap, and back.
__global__ void k_bfs_bits_clear(unsigned long long* __restrict__ bits, int64_t nw) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < nw) bits[i] = 0ull;
}

__global__ void k_bfs_bits_set(const int32_t* __restrict__ f, const int32_t* __restrict__ count,
                               uint32_t* __restrict__ bits) {
  const int nf = *count;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < nf; t += gridDim.x * blockDim.x)
    atomicOr(&bits[f[t] >> 5], 1u << (f[t] & 31));
}

// (The frontiers that go back to a list are small: most words are empty.)
__global__ __launch_bounds__(256) void k_bfs_bits_list(const unsigned long long* __restrict__ bits, int64_t nw,
                                                       const int2* __restrict__ range, int32_t* __restrict__ f,
                                                       int32_t* __restrict__ count, int32_t* __restrict__ pcount,
                                                       long long* __restrict__ pieces) {
  const int64_t w0 = global_wave() * kWave;
  const int64_t i = w0 + lane_id();
  const unsigned long long mine = i < nw ? bits[i] : 0ull;
  unsigned long long some = __ballot(mine != 0ull);
  while (some) {
    const int j = __ffsll(some) - 1;
    some &= some - 1;
    const unsigned long long word = (unsigned long long)readlane_ll((long long)mine, j);
    int at = 0;
    if (lane_id() == 0) at = atomicAdd(count, __popcll(word));
    at = __builtin_amdgcn_readfirstlane(at);
    if ((word >> lane_id()) & 1ull) {
      const int32_t v = (int32_t)((w0 + j) * kWave) + lane_id();
      f[at + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(word >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)word, 0u))] = v;
      const int2 rg = range[v];
      if (rg.y - rg.x > kBfsHub) bfs_add_pieces(v, rg.y - rg.x, pcount, pieces);
    }
  }
}

// Eight consecutive rows from an address of any 4-byte alignment.
struct __attribute__((packed, aligned(4))) BfsRows {
  int32_t r[8];
};
constexpr int kBfsBatch = 8;

// Bottom-up form of the same level (for large frontiers): every unvisited
// vertex scans its neighbours from the largest index down and stops at the
// first one in the frontier -- the largest frontier neighbour, the value
// SelectMax's atomic max gives top-down, so both forms produce the same
// parents and next frontier.
//
// A scan is a chain of two loads (a row, its bit) per step: bound by their
// latency, and by the longest scan of the slowest wave, as vertices with many
// neighbours lie next to each other in skewed graphs.  k_bfs_bottom_up gives a
// vertex with at most kBfsSerialDeg neighbours to a lane, eight a step, and
// lists the others; k_bfs_bottom_up_long spreads those evenly: sixteen lanes
// and 128 neighbours a step, four vertices at once, up to kBfsWaveDeg (from the
// list's front), the whole wave and 512 a step above (from its end).
//
// R-MAT s20, 31 M edges, the first bottom-up level: 386 us with one neighbour a
// step per lane (64 for a wave above 64 neighbours), 164 with the batches alone
// (the slowest waves then scanned 64 vertices of some 1000 neighbours), 36 + 46
// with the list; a level that finds little 9 + 3.  Workgroups of 256 lose more
// to their atomics on the list's ends (55 + 46) than those of 1024 to their
// barriers (36 + 46, but 13 + 4); scan lengths of 16 and 64 for a lane gave
// 32 + 49 and 60 + 34.  A copy of the frontier's bitmap in LDS did not pay: the
// lookups are not what bounds it.
constexpr int kBfsSerialDeg = 32, kBfsWaveDeg = 512;
constexpr int kBfsUpNT = 512;
constexpr unsigned kBfsUpGrid = 4096, kBfsLongGrid = 1024;

// Which of a lane's neighbours r[u] are in the frontier.
template <int U>
__device__ __forceinline__ void bfs_lookup(const uint32_t* __restrict__ fin, const int32_t (&r)[U], bool (&in)[U]) {
  uint32_t word[U];
#pragma unroll
  for (int u = 0; u < U; ++u) word[u] = fin[r[u] >> 5];
#pragma unroll
  for (int u = 0; u < U; ++u) pin(word[u]);
#pragma unroll
  for (int u = 0; u < U; ++u) in[u] = (word[u] >> (r[u] & 31)) & 1u;
}

// A wave has the 64 vertices of one word of the bitmaps: it marks what it found
// visited, writes the next frontier's word and counts without atomics.
__global__ __launch_bounds__(kBfsUpNT) void k_bfs_bottom_up(const int2* __restrict__ range,
                                                            const int32_t* __restrict__ rows, int64_t n, int64_t nw,
                                                            const uint32_t* __restrict__ fin,
                                                            unsigned long long* __restrict__ fout,
                                                            unsigned long long* __restrict__ visited,
                                                            int64_t* __restrict__ parents,
                                                            int32_t* __restrict__ longs, BfsState* st) {
  constexpr int NW = kBfsUpNT / kWave;
  __shared__ int wsum[NW];
  __shared__ int s_at[2];
  const int lane = lane_id();
  long long found = 0, edges = 0;
  for (int64_t w0 = (int64_t)blockIdx.x * NW; w0 < nw; w0 += (int64_t)gridDim.x * NW) {
    const int64_t w = w0 + wave_id_uniform();
    const unsigned long long vis = w < nw ? visited[w] : ~0ull;  // (vertices from n on count as visited)
    const int64_t v = w * kWave + lane;
    int b = 0, e = 0;
    if (~vis) {
      const int2 rg = range[min(v, n - 1)];
      b = rg.x;
      e = ((vis >> lane) & 1ull) ? rg.x : rg.y;
    }
    int32_t par = -1;
    if (e - b <= kBfsSerialDeg) {
      for (int i = e; i > b && par < 0; i -= kBfsBatch) {
        const int s = max(i - kBfsBatch, 0);  // rows has kBfsBatch entries more than the matrix
        const BfsRows a = *(const BfsRows*)(rows + s);
        bool in[kBfsBatch];
        bfs_lookup(fin, a.r, in);
#pragma unroll
        for (int j = 0; j < kBfsBatch; ++j)
          if (s + j >= b && s + j < i && in[j]) par = a.r[j];
      }
    }
    const unsigned long long next = __ballot(par >= 0);
    if (par >= 0) {
      parents[v] = par;
      edges += e - b;
    }
    if (lane == 0 && w < nw) {
      fout[w] = next;
      if (next) visited[w] = vis | next;
      found += __popcll(next);
    }
    // the vertices left to k_bfs_bottom_up_long
    const int kind = e - b <= kBfsSerialDeg ? 0 : e - b <= kBfsWaveDeg ? 1 : 1 << 16;
    int total;
    const int at = block_excl_scan<kBfsUpNT>(kind, wsum, total);
    if (total == 0) continue;
    if (threadIdx.x == 0) {
      s_at[0] = atomicAdd(&st->longs[0], total & 0xffff);
      s_at[1] = total >> 16 ? atomicAdd(&st->longs[1], total >> 16) : 0;
    }
    __syncthreads();
    if (kind == 1) longs[s_at[0] + (at & 0xffff)] = (int32_t)v;
    if (kind > 1) longs[n - 1 - s_at[1] - (at >> 16)] = (int32_t)v;
    __syncthreads();
  }
  bfs_count<kBfsUpNT>(st, found, edges);
}

__global__ __launch_bounds__(kBfsUpNT) void k_bfs_bottom_up_long(const int2* __restrict__ range,
                                                                 const int32_t* __restrict__ rows, int64_t n,
                                                                 const uint32_t* __restrict__ fin,
                                                                 uint32_t* __restrict__ fout,
                                                                 uint32_t* __restrict__ visited,
                                                                 int64_t* __restrict__ parents,
                                                                 const int32_t* __restrict__ longs, BfsState* st) {
  constexpr int U = 8, G = 16;
  const int nmid = st->longs[0], nbig = st->longs[1];
  const int lane = lane_id(), g = lane / G;
  const int nwaves = gridDim.x * (kBfsUpNT / kWave);
  const int wave = wave_id_uniform() * gridDim.x + blockIdx.x;
  long long found = 0, edges = 0;
  auto set = [&](int32_t v, int32_t par, int deg) {
    parents[v] = par;
    atomicOr(&fout[v >> 5], 1u << (v & 31));
    atomicOr(&visited[v >> 5], 1u << (v & 31));
    ++found;
    edges += deg;
  };
  // one vertex at a time
  for (int i = wave; i < nbig; i += nwaves) {
    const int32_t v = longs[n - 1 - i];
    const int2 rg = range[v];
    int32_t got = -1;
    for (int top = rg.y; top > rg.x && got < 0; top -= U * kWave) {
      int32_t u[U];
      bool in[U];
#pragma unroll
      for (int k = 0; k < U; ++k) u[k] = rows[max(top - 1 - k * kWave - lane, rg.x)];
#pragma unroll
      for (int k = 0; k < U; ++k) pin(u[k]);
      bfs_lookup(fin, u, in);
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const unsigned long long hits = __ballot(in[k]);
        if (got < 0 && hits) got = __builtin_amdgcn_readlane(u[k], __ffsll(hits) - 1);
      }
    }
    if (got >= 0 && lane == 0) set(v, got, rg.y - rg.x);
  }
  // four vertices at a time
  for (int i = wave * 4; i < nmid; i += nwaves * 4) {
    const bool mine = i + g < nmid;
    const int32_t v = longs[min(i + g, nmid - 1)];
    const int2 rg = range[v];
    int top = mine ? rg.y : rg.x;
    int32_t got = -1;
    while (__ballot(top > rg.x)) {
      int32_t u[U];
      bool in[U];
#pragma unroll
      for (int k = 0; k < U; ++k) u[k] = rows[max(top - 1 - k * G - (lane & (G - 1)), rg.x)];
#pragma unroll
      for (int k = 0; k < U; ++k) pin(u[k]);
      bfs_lookup(fin, u, in);
      const bool live = top > rg.x;
      int32_t first = -1;
#pragma unroll
      for (int k = 0; k < U; ++k) {
        // (past the list's end a lane has its first entry again)
        const unsigned hits = (unsigned)(__ballot(live && in[k]) >> (g * G)) & 0xffffu;
        const int32_t r = __shfl(u[k], g * G + (hits ? __ffs(hits) - 1 : 0), kWave);
        if (first < 0 && hits) first = r;
      }
      top -= U * G;
      if (first >= 0) {
        got = first;
        top = rg.x;
      }
    }
    if (got >= 0 && (lane & (G - 1)) == 0) set(v, got, rg.y - rg.x);
  }
  bfs_count<kBfsUpNT>(st, found, edges);
}

}  // namespace

}  // namespace cbx

using namespace cbx;

struct cbx_bfs_plan_s {
  int64_t n = 0, nnz = 0, nw = 0;  // nw: 64-bit words of a bitmap
  hipStream_t stream = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};  // around a run
  int2* range = nullptr;
  int64_t* parents = nullptr;
  int32_t *rows = nullptr, *f[2] = {nullptr, nullptr};
  long long* pieces[2] = {nullptr, nullptr};  // hub pieces of the two frontier lists
  int32_t* cand = nullptr;  // the largest offer per vertex (vertex ids fit 32 bits: n < 2^31)
  unsigned long long *visited = nullptr, *isolated = nullptr, *bits[2] = {nullptr, nullptr};
  BfsState* state = nullptr;
  BfsReport* report = nullptr;  // pinned
  int direction = CBX_BFS_DIRECTION_OPTIMIZING;
  // Pattern of A equal to that of its transpose.  Bottom-up levels scan column
  // v of A for frontier rows, which is row v only for a symmetric pattern, so
  // a plan over a directed graph runs every level top-down.
  bool symmetric = true;
  // [the frontier comes as: 0 list, 1 bitmap][direction (0 top-down, 1 bottom-up)][frontier parity]
  hipGraph_t graph[2][2][2] = {};
  hipGraphExec_t exec[2][2][2] = {};
  // top-down only: kBfsTdLevels consecutive levels in one graph, launched
  // until the frontier is empty (levels after the last one do nothing)
  hipGraph_t td_graph = nullptr;
  hipGraphExec_t td_exec = nullptr;
};

static void bfs_plan_free(cbx_bfs_plan_s* p) {
  if (!p) return;
  for (int i = 0; i < 8; ++i) {
    if (p->exec[i >> 2][(i >> 1) & 1][i & 1]) (void)hipGraphExecDestroy(p->exec[i >> 2][(i >> 1) & 1][i & 1]);
    if (p->graph[i >> 2][(i >> 1) & 1][i & 1]) (void)hipGraphDestroy(p->graph[i >> 2][(i >> 1) & 1][i & 1]);
  }
  if (p->td_exec) (void)hipGraphExecDestroy(p->td_exec);
  if (p->td_graph) (void)hipGraphDestroy(p->td_graph);
  for (void* q : {(void*)p->range, (void*)p->parents, (void*)p->rows, (void*)p->f[0], (void*)p->f[1],
                  (void*)p->pieces[0], (void*)p->pieces[1], (void*)p->cand, (void*)p->visited, (void*)p->isolated,
                  (void*)p->bits[0], (void*)p->bits[1], (void*)p->state})
    if (q) (void)hipFree(q);
  if (p->report) (void)hipHostFree(p->report);
  for (hipEvent_t e : p->ev)
    if (e) (void)hipEventDestroy(e);
  if (p->stream) (void)hipStreamDestroy(p->stream);
  delete p;
}

constexpr int kBfsNT = 256;
constexpr unsigned kBfsGrid = 2048;
constexpr unsigned kBfsHubGrid = 2048;  // workgroups over the hubs' pieces
constexpr int64_t kBfsAlpha = 256;
constexpr int kBfsTdLevels = 8;  // even: the frontier parity is 0 again after one top-down graph

// One level from frontier `par` (a list, or a bitmap where `bits`) to 1 - par.
static void bfs_level(cbx_bfs_plan_s* p, bool bits, bool bottom_up, int par, hipStream_t s) {
  BfsState* st = p->state;
  int32_t *cin = &st->listed[par], *cout = &st->listed[1 - par];
  const unsigned words = nb(p->nw, 256);
  if (bottom_up) {
    if (!bits) {
      k_bfs_bits_clear<<<words, 256, 0, s>>>(p->bits[par], p->nw);
      k_bfs_bits_set<<<256, 256, 0, s>>>(p->f[par], cin, (uint32_t*)p->bits[par]);
    }
    const unsigned g = std::min(nb(p->nw * kWave, kBfsUpNT), kBfsUpGrid);
    const uint32_t* fin = (const uint32_t*)p->bits[par];
    int32_t* longs = p->f[1 - par];  // (free: the next frontier is a bitmap)
    k_bfs_bottom_up<<<g, kBfsUpNT, 0, s>>>(p->range, p->rows, p->n, p->nw, fin, p->bits[1 - par], p->visited,
                                           p->parents, longs, st);
    k_bfs_bottom_up_long<<<kBfsLongGrid, kBfsUpNT, 0, s>>>(p->range, p->rows, p->n, fin, (uint32_t*)p->bits[1 - par],
                                                           (uint32_t*)p->visited, p->parents, longs, st);
  } else {
    if (bits)
      k_bfs_bits_list<<<words, 256, 0, s>>>(p->bits[par], p->nw, p->range, p->f[par], cin, &st->pieces[par],
                                            p->pieces[par]);
    k_bfs_expand<kBfsNT, 4><<<kBfsGrid, kBfsNT, 0, s>>>(p->range, p->rows, p->f[par], cin,
                                                       (const uint32_t*)p->visited, p->cand, p->f[1 - par], cout);
    k_bfs_expand_hubs<kBfsNT><<<kBfsHubGrid, kBfsNT, 0, s>>>(p->range, p->rows, p->pieces[par], &st->pieces[par],
                                                             (const uint32_t*)p->visited, p->cand, p->f[1 - par],
                                                             cout);
    k_bfs_finalize<<<256, kBfsFinNT, 0, s>>>(p->f[1 - par], cout, p->cand, p->range, p->parents,
                                             (uint32_t*)p->visited, st, &st->pieces[1 - par], p->pieces[1 - par]);
  }
  k_bfs_level_end<<<1, kWave, 0, s>>>(st, par, bottom_up, p->report);
}

extern "C" cbx_status cbx_bfs_plan_create(const cbx_dcsc* A, cbx_bfs_plan_s** out) {
  CBX_RETURN_IF(!A || !out, CBX_ERR_INVALID, "cbx_bfs_plan_create: null argument");
  *out = nullptr;
  CBX_RETURN_IF(A->location != CBX_DEVICE, CBX_ERR_INVALID, "cbx_bfs_plan_create: expected a device matrix");
  CBX_RETURN_IF(A->m != A->n, CBX_ERR_INVALID, "cbx_bfs_plan_create: the adjacency matrix must be square");
  CBX_RETURN_IF(A->n >= (1ll << 31) || A->nnz >= (1ll << 31), CBX_ERR_LIMIT,
                "cbx_bfs_plan_create: n and nnz must be below 2^31");
  cbx_status st = cbx_dcsc_check(A);
  if (st != CBX_OK) return st;
  // symmetric pattern?  (A's structure against its transpose's)
  bool symmetric = true;
  {
    cbx_dcsc T;
    std::memset(&T, 0, sizeof(T));
    st = cbx_dcsc_transpose(A, &T, nullptr);
    if (st != CBX_OK) return st;
    symmetric = T.nzc == A->nzc && T.nnz == A->nnz;
    if (symmetric && A->nnz) {
      unsigned long long* cnt = nullptr;
      unsigned long long diff = 0;
      if (hipMalloc(&cnt, sizeof(*cnt)) != hipSuccess) {
        cbx_dcsc_free(&T);
        return set_error(CBX_ERR_NOMEM, "cbx_bfs_plan_create: allocation");
      }
      (void)hipMemset(cnt, 0, sizeof(*cnt));
      k_bfs_count_diff<<<1024, 256>>>(A->cp, T.cp, A->nzc + 1, cnt);
      k_bfs_count_diff<<<1024, 256>>>(A->jc, T.jc, A->nzc, cnt);
      k_bfs_count_diff<<<1024, 256>>>(A->ir, T.ir, A->nnz, cnt);
      const hipError_t e = hipMemcpy(&diff, cnt, sizeof(diff), hipMemcpyDeviceToHost);
      (void)hipFree(cnt);
      if (e != hipSuccess) {
        cbx_dcsc_free(&T);
        return set_error(CBX_ERR_HIP, "cbx_bfs_plan_create: symmetry check: %s", hipGetErrorString(e));
      }
      symmetric = diff == 0;
    }
    cbx_dcsc_free(&T);
  }
  auto* p = new cbx_bfs_plan_s();
  p->symmetric = symmetric;
  p->n = A->n;
  p->nnz = A->nnz;
  p->nw = A->n / kWave + 1;
  auto fail = [&](const char* what) {
    bfs_plan_free(p);
    return set_error(CBX_ERR_HIP, "cbx_bfs_plan_create: %s", what);
  };
  if (hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&p->ev[0]) != hipSuccess || hipEventCreate(&p->ev[1]) != hipSuccess)
    return fail("stream");
  const int64_t n = p->n;
  // every hub of a frontier contributes ceil(deg / kBfsHub) <= 2 deg / kBfsHub pieces
  const int64_t max_pieces = 2 * p->nnz / kBfsHub + 2;
  const int64_t n1 = std::max<int64_t>(n, 1);
  if (hipMalloc(&p->range, 8 * n1) || hipMalloc(&p->parents, 8 * n1) ||
      hipMalloc(&p->rows, 4 * (p->nnz + kBfsBatch)) || hipMalloc(&p->f[0], 4 * n1) || hipMalloc(&p->f[1], 4 * n1) ||
      hipMalloc(&p->cand, 4 * n1) || hipMalloc(&p->visited, 8 * p->nw) || hipMalloc(&p->isolated, 8 * p->nw) ||
      hipMalloc(&p->bits[0], 8 * p->nw) || hipMalloc(&p->bits[1], 8 * p->nw) ||
      hipMalloc(&p->pieces[0], 8 * max_pieces) || hipMalloc(&p->pieces[1], 8 * max_pieces) ||
      hipMalloc(&p->state, sizeof(BfsState)) || hipHostMalloc(&p->report, sizeof(BfsReport), hipHostMallocDefault))
    return fail("allocation");
  hipStream_t s = p->stream;
  if (hipMemsetAsync(p->range, 0, 8 * n, s) || hipMemsetAsync(p->rows + p->nnz, 0, 4 * kBfsBatch, s))
    return fail("memset");
  if (A->nzc) k_bfs_ranges<<<nb(A->nzc, 256), 256, 0, s>>>(A->cp, A->jc, A->nzc, p->range);
  if (A->nnz) k_bfs_rows32<<<nb(A->nnz, 256), 256, 0, s>>>(A->ir, A->nnz, p->rows);
  k_bfs_isolated<<<nb(p->nw, 4), 256, 0, s>>>(p->range, n, p->nw, symmetric, p->isolated);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return fail("setup kernels");
  // one graph per form of the frontier, direction and parity
  for (int i = 0; i < 8; ++i) {
    const int from = i >> 2, dir = (i >> 1) & 1, par = i & 1;
    if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) return fail("capture begin");
    bfs_level(p, from, dir, par, s);
    if (hipStreamEndCapture(s, &p->graph[from][dir][par]) != hipSuccess) return fail("capture end");
    if (hipGraphInstantiate(&p->exec[from][dir][par], p->graph[from][dir][par], nullptr, nullptr, 0) != hipSuccess)
      return fail("graph instantiate");
  }
  // kBfsTdLevels top-down levels in one graph, no host round trip between
  // them; the host reads the frontier size once per graph
  if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) return fail("capture begin");
  for (int l = 0; l < kBfsTdLevels; ++l) bfs_level(p, false, false, l & 1, s);
  if (hipStreamEndCapture(s, &p->td_graph) != hipSuccess) return fail("capture end");
  if (hipGraphInstantiate(&p->td_exec, p->td_graph, nullptr, nullptr, 0) != hipSuccess)
    return fail("graph instantiate");
  *out = p;
  return CBX_OK;
}

extern "C" cbx_status cbx_bfs_run(cbx_bfs_plan_s* p, int64_t root, int64_t* parents_dev, cbx_bfs_stats* stats) {
  CBX_RETURN_IF(!p || !parents_dev, CBX_ERR_INVALID, "cbx_bfs_run: null argument");
  CBX_RETURN_IF(root < 0 || root >= p->n, CBX_ERR_INVALID, "cbx_bfs_run: root %lld out of range", (long long)root);
  hipStream_t s = p->stream;
  const volatile BfsReport* rep = p->report;
  CBX_HIP(hipEventRecord(p->ev[0], s));
  k_bfs_reset<<<nb(std::max<int64_t>(p->n, kBfsSlots), 256), 256, 0, s>>>(
      p->n, p->cand, p->parents, p->visited, p->isolated, p->nw, p->f[0], p->pieces[0], p->range, p->state, p->report,
      root);
  // direction per level: bottom-up while the frontier's edges exceed 1/256 of
  // the edges still unexplored.  (Beamer's rule compares the two with a factor
  // 14 for equal per-edge costs; here a top-down edge costs a device atomic on
  // the target, some 20-40 times a bottom-up edge, which is a streamed read.)
  int bottom_up_levels = 0;
  if (p->direction == CBX_BFS_TOP_DOWN || !p->symmetric) {
    // every level top-down: graphs of kBfsTdLevels levels until the frontier
    // is empty (a BFS has at most n levels)
    for (int64_t launched = 0;; launched += kBfsTdLevels) {
      CBX_HIP(hipGraphLaunch(p->td_exec, s));
      CBX_HIP(hipStreamSynchronize(s));
      if (rep->size == 0 || launched > p->n + 1) break;
    }
  } else {
    CBX_HIP(hipGetLastError());
    CBX_HIP(hipStreamSynchronize(s));
    int levels = 0;
    int64_t mu = p->nnz;
    int64_t fe = (int64_t)rep->edges;  // edges of the current frontier
    bool bottom_up = p->direction == CBX_BFS_BOTTOM_UP, bits = false;
    for (int par = 0;; par ^= 1) {
      if (p->direction == CBX_BFS_DIRECTION_OPTIMIZING) bottom_up = fe > mu / kBfsAlpha;
      CBX_HIP(hipGraphLaunch(p->exec[bits][bottom_up][par], s));
      CBX_HIP(hipStreamSynchronize(s));
      ++levels;
      bottom_up_levels += bottom_up;
      bits = bottom_up;
      fe = (int64_t)rep->edges;
      mu -= fe;
      if (rep->size == 0 || levels > p->n + 1) break;
    }
  }
  const int64_t levels = (int64_t)rep->levels, reached = (int64_t)rep->reached;
  CBX_HIP(hipMemcpyAsync(parents_dev, p->parents, sizeof(int64_t) * p->n, hipMemcpyDeviceToDevice, s));
  CBX_HIP(hipEventRecord(p->ev[1], s));
  CBX_HIP(hipStreamSynchronize(s));
  float ms = 0;
  (void)hipEventElapsedTime(&ms, p->ev[0], p->ev[1]);
  if (stats) {
    stats->levels = (int32_t)levels;
    stats->bottom_up_levels = bottom_up_levels;
    stats->reached = reached;
    stats->ms = ms;
  }
  return CBX_OK;
}

extern "C" cbx_status cbx_bfs_plan_set_direction(cbx_bfs_plan_s* p, cbx_bfs_direction direction) {
  CBX_RETURN_IF(!p, CBX_ERR_INVALID, "cbx_bfs_plan_set_direction: null plan");
  CBX_RETURN_IF(direction != CBX_BFS_DIRECTION_OPTIMIZING && direction != CBX_BFS_TOP_DOWN &&
                    direction != CBX_BFS_BOTTOM_UP,
                CBX_ERR_INVALID, "cbx_bfs_plan_set_direction: unknown direction %d", (int)direction);
  CBX_RETURN_IF(direction == CBX_BFS_BOTTOM_UP && !p->symmetric, CBX_ERR_INVALID,
                "cbx_bfs_plan_set_direction: bottom-up levels need a symmetric pattern (this plan's is not)");
  p->direction = direction;
  return CBX_OK;
}

extern "C" void cbx_bfs_plan_destroy(cbx_bfs_plan_s* p) { bfs_plan_free(p); }


// ------------------------------------------------------ SpMV, dense vector
// dcsc_gespmv (Friends.h:63-77): y[i] = add(y[i], multiply(A(i,j), x[j])) for
// every stored entry, y accumulated in place; a boolean A contributes x[j]
// itself.
//
// Tiled form (m <= 2^24): the entries are cut into tiles of kSvTile.  One pass
// over A forms a tile's products, orders them in LDS by the block of rows they
// fall in and writes them, contiguous, to the tile's own place, with the
// blocks' offsets in it; nothing has to be counted beforehand, and every write
// is a full line.  A block's products are then the runs that the tiles hold of
// it: k_svb_cut cuts each block's tiles into chunks of about equal numbers of
// products, and k_svb_accumulate sums a chunk's runs in LDS and updates y once
// per row: a plain read-modify-write when one workgroup owns the block, the
// semiring's device atomic when a hot block is split over several.  Device
// atomics per entry (the direct form below, kept for taller matrices and small
// products) serialise on the hot rows of skewed matrices.
//
// Blocks have 4096 rows up to m = 2^20 and 16384 above: a tile's run of one
// block is then at least four products on average (256 and 1024 blocks), and
// the block's sums still fit LDS.
//
// Counting the tiles' products per block first and scattering each product to
// its block's bucket read the rows twice and wrote two scattered values per
// entry, each with a search for its column and one load in flight at a time:
// at 2^20 rows and 16 M entries (FP64) 0.49 ms a product, 0.36 of them in the
// counting and scattering passes; now 0.21 ms, 0.095 in k_svb_tile (4.4 TB/s)
// and 0.075 in k_svb_accumulate (2.1 TB/s: 40 us of loads, the rest the
// rounds' barriers; chunks of half or twice the size and twice the loads in
// flight measured 75 to 85).
constexpr int kSvLB = 12, kSvLBTall = 14;           // log2 of the rows per block
constexpr int64_t kSvShort = (int64_t)1 << 20;      // up to so many rows blocks have 2^kSvLB
constexpr int kSvMaxBlocks = 1024;                  // tiled form while m <= 2^24
constexpr int kSvTile = 4096, kSvNT = 256;          // entries and threads per tile
constexpr int kSvPer = kSvTile / kSvNT;             // entries per thread
constexpr int kSvChunkLog = 3;                      // log2 of the products per chunk and row of the block
constexpr int64_t kSvMinNnz = 1 << 16;              // below this the direct form is cheaper

template <int K, class T, bool BOOLA>
__global__ void k_spmv_dense(const int64_t* __restrict__ cp, const int64_t* __restrict__ jc,
                             const int64_t* __restrict__ ir, const void* __restrict__ valA_, int64_t nzc,
                             const T* __restrict__ x, T* __restrict__ y) {
  using SR = Sem<K, T>;
  const int64_t q = global_wave();
  if (q >= nzc) return;
  const T xj = x[jc[q]];
  for (int64_t e = cp[q] + lane_id(); e < cp[q + 1]; e += kWave) {
    T prod;
    if constexpr (BOOLA) prod = xj;
    else prod = (T)SR::out(SR::mul(((const T*)valA_)[e], xj));
    GAcc<K, T>::acc(&y[ir[e]], prod);
  }
}

// What the passes report: the structure check's verdicts on columns and on
// entries (a kernel that may find a fault stops only at those of the kernels
// before it, so that a workgroup stops as a whole), and the chunks.
struct SvFlags {
  int bad_columns, bad_entries, nchunks;
};

__global__ void k_svb_begin(SvFlags* __restrict__ f) {
  if (threadIdx.x == 0) *f = SvFlags{0, 0, 0};
}

// The structure check's per-column rules (those of cbx_dcsc_check), and the
// column qs[t] that holds the first entry of tile t.  A column longer than m
// is malformed (its rows could not ascend), so a thread writes at most m /
// kSvTile + 1 of them.
__global__ __launch_bounds__(256) void k_svb_columns(const int64_t* __restrict__ cp, const int64_t* __restrict__ jc,
                                                     int64_t nzc, int64_t nnz, int64_t m, int64_t n,
                                                     int32_t* __restrict__ qs, SvFlags* __restrict__ f) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q >= nzc) return;
  const int64_t b = cp[q], e = cp[q + 1], j = jc[q], jn = q + 1 < nzc ? jc[q + 1] : n;
  const bool err = b < 0 || e <= b || e > nnz || e - b > m || j < 0 || jn <= j || (q == 0 && b != 0) ||
                   (q == nzc - 1 && (e != nnz || j >= n));
  if (err) {
    f->bad_columns = 1;
    return;
  }
  for (int64_t t = (b + kSvTile - 1) / kSvTile; t * kSvTile < e; ++t) qs[t] = (int32_t)q;
}

// Products of one tile, ordered by row block: bval / brow (row in the block)
// from the tile's first entry on, and tbl[b * ntiles + t] = the place of block
// b's first one (b = nblk: the tile's end).  Also the structure check's rules
// for entries: rows in range, ascending but for column starts.
//
// Bound by the bytes of A and of the products; each thread's 16 entries are
// loaded before anything else.  A tile's columns' x values are gathered into
// LDS once per column, and an entry finds its column by counting the column
// starts before it (a bitmap, two mbcnt per entry); consecutive tiles go to
// the same XCD, whose L2 then merges their neighbouring entries of tbl.
template <int K, class T, bool BOOLA>
__global__ __launch_bounds__(kSvNT) void k_svb_tile(const int64_t* __restrict__ cp, const int64_t* __restrict__ jc,
                                                    const int64_t* __restrict__ ir, const void* __restrict__ valA_,
                                                    int64_t nzc, int64_t nnz, int64_t m, const T* __restrict__ x,
                                                    int lb, int nblk, int64_t ntiles,
                                                    const int32_t* __restrict__ qs, uint16_t* __restrict__ tbl,
                                                    uint16_t* __restrict__ brow, T* __restrict__ bval,
                                                    SvFlags* __restrict__ f) {
  using SR = Sem<K, T>;
  constexpr int U = kSvPer, NW = kSvNT / kWave;
  static_assert(kSvTile == kWave * kWave, "one bitmap word per lane");
  static_assert(kSvMaxBlocks % kSvNT == 0, "whole block counts per thread");
  __shared__ T xs[kSvTile + 1];  // x of the tile's columns, then the ordered products
  __shared__ uint16_t srow[kSvTile];
  __shared__ int h[kSvMaxBlocks];
  __shared__ unsigned long long starts[kWave];
  __shared__ int wsum[NW];
  if (f->bad_columns) return;  // cp, jc or qs cannot be trusted as indices
  const int64_t per = (ntiles + 7) / 8;
  const int64_t t = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (t >= ntiles) return;
  const int64_t e0 = t * kSvTile;
  const int cnt = (int)min<int64_t>(nnz - e0, kSvTile);
  const int lane = lane_id(), w = wave_id_uniform();

  int64_t r[U];
  T a[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = min((w * U + u) * kWave + lane, cnt - 1);
    r[u] = ir[e0 + i];
    if constexpr (!BOOLA) a[u] = ((const T*)valA_)[e0 + i];
  }
  // the entry after this wave's last (its own last row + 1 where there is none)
  const int last = (w + 1) * U * kWave;
  const int64_t after = e0 + last < nnz ? ir[e0 + last] : 0;
  const int64_t q0 = qs[t], q1 = t + 1 < ntiles ? qs[t + 1] : nzc - 1;
  const int nq = (int)min<int64_t>(q1 - q0 + 1, kSvTile + 1);
  for (int b = threadIdx.x; b < nblk; b += kSvNT) h[b] = 0;
  if (threadIdx.x < kWave) starts[threadIdx.x] = 0ull;
  __syncthreads();
  for (int i = threadIdx.x; i < nq; i += kSvNT) {
    const int64_t s = cp[q0 + i] - e0, j = jc[q0 + i];
    xs[i] = x[j];
    // bit s - 1: the entries from s on lie past this column's start
    if (i > 0 && s >= 1 && s <= kSvTile) atomicOr(&starts[(s - 1) >> 6], 1ull << ((s - 1) & 63));
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    pin(r[u]);
    if constexpr (!BOOLA) pin(a[u]);
  }
  __syncthreads();
  const unsigned long long word = starts[lane];  // lane i: the starts in (64 i, 64 i + 64]
  const int ones = __popcll(word);
  const int before = wave_incl_scan(ones) - ones;

  bool bad = false;
  int rank[U];
  T prod[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = w * U + u;
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)word, j);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(word >> 32), j);
    const int k = (int)__builtin_amdgcn_mbcnt_hi(
        hi, __builtin_amdgcn_mbcnt_lo(lo, (unsigned)__builtin_amdgcn_readlane(before, j)));
    const int i = j * kWave + lane;
    const bool live = i < cnt;
    // descents: the next entry's row, unless a column starts there (bit i)
    const int64_t nf = u + 1 < U ? readlane_ll(r[u + 1 < U ? u + 1 : u], 0) : after;
    int64_t next = __shfl_down((long long)r[u], 1, kWave);
    if (lane == kWave - 1) next = nf;
    const bool start = ((((unsigned long long)hi << 32) | lo) >> lane) & 1u;
    const bool in = r[u] >= 0 && r[u] < m;
    bad |= live && (!in || (e0 + i + 1 < nnz && next <= r[u] && !start));
    const T xj = xs[k];
    if constexpr (BOOLA) prod[u] = xj;
    else prod[u] = (T)SR::out(SR::mul(a[u], xj));
    rank[u] = live && in ? atomicAdd(&h[r[u] >> lb], 1) : -1;
  }
  if (__ballot(bad) && lane == 0) f->bad_entries = 1;
  __syncthreads();  // the blocks' counts; xs has been read
  {
    constexpr int PT = kSvMaxBlocks / kSvNT;
    int c[PT], sum = 0;
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int b = threadIdx.x * PT + k;
      c[k] = b < nblk ? h[b] : 0;
      sum += c[k];
    }
    int total;
    int ex = block_excl_scan<kSvNT>(sum, wsum, total);
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int b = threadIdx.x * PT + k;
      if (b < nblk) h[b] = ex;
      ex += c[k];
    }
    if (threadIdx.x == 0) tbl[(int64_t)nblk * ntiles + t] = (uint16_t)total;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nblk; b += kSvNT) tbl[(int64_t)b * ntiles + t] = (uint16_t)h[b];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (rank[u] < 0) continue;
    const int p = h[r[u] >> lb] + rank[u];
    xs[p] = prod[u];
    srow[p] = (uint16_t)(r[u] & ((1 << lb) - 1));
  }
  __syncthreads();
  for (int i = threadIdx.x; i < cnt; i += kSvNT) {
    bval[e0 + i] = xs[i];
    brow[e0 + i] = srow[i];
  }
}

// A chunk: the tiles [t0, t1) of a row block, one of n chunks of that block.
struct SvChunk {
  int32_t b, t0, t1, n;
};

// Cuts one row block's tiles into chunks (one workgroup per block): chunk c
// starts at the first tile with at least c << lc products before it, so a
// chunk has at most 2^lc + kSvTile products, and the numbers have no gaps
// (2^lc >= kSvTile).  The chunks' places are taken with one atomic per block.
constexpr int kSvCutNT = 256, kSvCutPer = 8;
__global__ __launch_bounds__(kSvCutNT) void k_svb_cut(const uint16_t* __restrict__ tbl, int64_t ntiles, int lc,
                                                      SvChunk* __restrict__ chunks, SvFlags* __restrict__ f) {
  __shared__ long long wsum[kSvCutNT / kWave];
  __shared__ int s_base;
  if (f->bad_columns || f->bad_entries) return;
  const int b = blockIdx.x;
  const uint16_t* lo = tbl + (int64_t)b * ntiles;
  const uint16_t* hi = lo + ntiles;
  long long all = 0;
  for (int64_t t0 = threadIdx.x; t0 < ntiles; t0 += kSvCutNT * kSvCutPer) {
    uint16_t a[kSvCutPer], z[kSvCutPer];
#pragma unroll
    for (int k = 0; k < kSvCutPer; ++k) {
      const int64_t t = min<int64_t>(t0 + k * kSvCutNT, ntiles - 1);
      a[k] = lo[t];
      z[k] = hi[t];
    }
#pragma unroll
    for (int k = 0; k < kSvCutPer; ++k) {
      pin(a[k]);
      pin(z[k]);
      if (t0 + k * kSvCutNT < ntiles) all += z[k] - a[k];
    }
  }
  all = block_sum_ll<kSvCutNT>(all, wsum);
  if (all == 0) return;
  const int n = (int)((all - (hi[ntiles - 1] - lo[ntiles - 1])) >> lc) + 1;
  if (threadIdx.x == 0) s_base = atomicAdd(&f->nchunks, n);
  __syncthreads();
  SvChunk* out = chunks + s_base;
  long long done = 0;  // products before this round's tiles
  for (int64_t t0 = 0; t0 < ntiles; t0 += kSvCutNT * kSvCutPer) {
    const int64_t tb = t0 + threadIdx.x * kSvCutPer;
    int len[kSvCutPer];
    long long sum = 0;
#pragma unroll
    for (int k = 0; k < kSvCutPer; ++k) {
      const int64_t t = min<int64_t>(tb + k, ntiles - 1);
      len[k] = hi[t] - lo[t];
      if (tb + k >= ntiles) len[k] = 0;
      sum += len[k];
    }
    long long total;
    long long p = done + block_excl_scan_ll<kSvCutNT>(sum, wsum, total);
#pragma unroll
    for (int k = 0; k < kSvCutPer; ++k) {
      // the chunk after this tile's starts at the next tile
      const int c = (int)(p >> lc), d = (int)((p + len[k]) >> lc);
      const int64_t t = tb + k;
      if (t == 0) {
        out[0].b = b;
        out[0].t0 = 0;
        out[0].n = n;
      }
      if (t < ntiles && d != c && d < n) {
        out[c].t1 = (int32_t)(t + 1);
        out[d].b = b;
        out[d].t0 = (int32_t)(t + 1);
        out[d].n = n;
      }
      if (t == ntiles - 1) out[n - 1].t1 = (int32_t)ntiles;
      p += len[k];
    }
    done += total;
  }
}

// One workgroup per chunk: its runs, a tile per thread at a time, flattened.
template <int K, class T, int LB, int NT, int U>
__global__ __launch_bounds__(NT) void k_svb_accumulate(const SvChunk* __restrict__ chunks,
                                                       const SvFlags* __restrict__ f,
                                                       const uint16_t* __restrict__ tbl, int64_t ntiles, int64_t m,
                                                       const uint16_t* __restrict__ brow,
                                                       const T* __restrict__ bval, T* __restrict__ y) {
  using SR = Sem<K, T>;
  using Acc = typename SR::Acc;
  constexpr int BR = 1 << LB;
  __shared__ typename SR::Lds acc[BR];
  __shared__ FlatStage<T, NT, false> st;
  if (f->bad_columns || f->bad_entries || (int)blockIdx.x >= f->nchunks) return;  // malformed: y is left as it was
  const SvChunk ch = chunks[blockIdx.x];
  for (int r = threadIdx.x; r < BR; r += NT) acc[r] = SR::lident();
  flat_init(st);
  const uint16_t* lo = tbl + (int64_t)ch.b * ntiles;
  const uint16_t* hi = lo + ntiles;
  int par = 0;
  const int tf = min(ch.t0 + (int)threadIdx.x, ch.t1 - 1);
  uint16_t na = lo[tf], nz = hi[tf];  // the next round's run
  for (int t0 = ch.t0; t0 < ch.t1; t0 += NT) {
    const int a = na;
    const int len = t0 + (int)threadIdx.x < ch.t1 ? nz - a : 0;
    const int tn = min(t0 + NT + (int)threadIdx.x, ch.t1 - 1);
    na = lo[tn];
    nz = hi[tn];
    const int64_t e0 = (int64_t)t0 * kSvTile;
    const FlatSeg me = flat_stage<T, NT, false>(st, (int)threadIdx.x * kSvTile + a, len, T{});
    flat_chunk<T, NT, false, U>(st, me, par, [&](const int32_t(&idx)[U], T(&)[U], const bool(&ok)[U]) {
      uint16_t r[U];
      T v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        r[u] = brow[e0 + idx[u]];
        v[u] = bval[e0 + idx[u]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        pin(r[u]);
        pin(v[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ok[u]) SR::acc(&acc[r[u]], (Acc)v[u]);
    });
  }
  __syncthreads();
  const int64_t row0 = (int64_t)ch.b * BR;
  using Bits = typename std::conditional<sizeof(Acc) == 8, unsigned long long, unsigned int>::type;
  const Bits id = __builtin_bit_cast(Bits, SR::ident());
  for (int r = threadIdx.x; r < BR && row0 + r < m; r += NT) {
    const Acc a = (Acc)SR::lout(acc[r]);
    if (ch.n == 1) {
      y[row0 + r] = (T)SR::out(SR::add((Acc)y[row0 + r], a));
    } else if (__builtin_bit_cast(Bits, a) != id) {  // the identity changes nothing
      GAcc<K, T>::acc(&y[row0 + r], (T)SR::out(a));
    }
  }
}

template <int K, class T>
static cbx_status spmv_dense_typed(const cbx_dcsc* A, bool boolA, const T* x, T* y, hipStream_t s) {
  if (A->nzc == 0) return CBX_OK;
  const int64_t nnz = A->nnz, m = A->m;
  const int lb = m <= kSvShort ? kSvLB : kSvLBTall;
  const int64_t nblk64 = (m + (1 << lb) - 1) >> lb;
  if (nnz < kSvMinNnz || nblk64 > kSvMaxBlocks) {
    {  // the structure check first: the kernel indexes y by A's rows and x by its columns
      ScratchSet cs(s);
      unsigned long long* chk = nullptr;
      if (!cs.take(&chk, 3)) return set_error(CBX_ERR_NOMEM, "cbx_spmv_dense: workspace allocation failed");
      dcsc_check_launch(A, chk, s);
      const cbx_status cst = dcsc_check_result(chk, s);
      if (cst != CBX_OK) return cst;
    }
    if (boolA)
      k_spmv_dense<K, T, true><<<wave_grid(A->nzc), 256, 0, s>>>(A->cp, A->jc, A->ir, A->val, A->nzc, x, y);
    else
      k_spmv_dense<K, T, false><<<wave_grid(A->nzc), 256, 0, s>>>(A->cp, A->jc, A->ir, A->val, A->nzc, x, y);
    CBX_HIP(hipGetLastError());
    CBX_HIP(hipStreamSynchronize(s));
    return CBX_OK;
  }
  const int nblk = (int)nblk64;
  const int64_t ntiles = (nnz + kSvTile - 1) / kSvTile;
  const int lc = lb + kSvChunkLog;
  const int64_t max_chunks = (nnz >> lc) + nblk;
  CBX_RETURN_IF(ntiles >= (1ll << 31) / nblk || max_chunks >= (1ll << 31), CBX_ERR_LIMIT,
                "cbx_spmv_dense: matrix too large for one launch");
  int32_t* qs = nullptr;
  uint16_t *tbl = nullptr, *brow = nullptr;
  T* bval = nullptr;
  SvChunk* chunks = nullptr;
  SvFlags* flags = nullptr;
  ScratchSet ws(s);
  if (!ws.take(&qs, ntiles) || !ws.take(&tbl, (nblk + 1) * ntiles) || !ws.take(&brow, nnz) || !ws.take(&bval, nnz) ||
      !ws.take(&chunks, max_chunks) || !ws.take(&flags, 1))
    return set_error(CBX_ERR_NOMEM, "cbx_spmv_dense: workspace allocation failed");
  // the structure check (the rules of cbx_dcsc_check) runs inside the
  // launches, and each stops at a verdict of those before it
  k_svb_begin<<<1, 64, 0, s>>>(flags);
  k_svb_columns<<<nb(A->nzc, 256), 256, 0, s>>>(A->cp, A->jc, A->nzc, nnz, m, A->n, qs, flags);
  const unsigned g = (unsigned)((ntiles + 7) / 8 * 8);
  if (boolA)
    k_svb_tile<K, T, true><<<g, kSvNT, 0, s>>>(A->cp, A->jc, A->ir, A->val, A->nzc, nnz, m, x, lb, nblk, ntiles, qs,
                                              tbl, brow, bval, flags);
  else
    k_svb_tile<K, T, false><<<g, kSvNT, 0, s>>>(A->cp, A->jc, A->ir, A->val, A->nzc, nnz, m, x, lb, nblk, ntiles, qs,
                                               tbl, brow, bval, flags);
  k_svb_cut<<<(unsigned)nblk, kSvCutNT, 0, s>>>(tbl, ntiles, lc, chunks, flags);
  if (lb == kSvLB)
    k_svb_accumulate<K, T, kSvLB, 512, 4><<<(unsigned)max_chunks, 512, 0, s>>>(chunks, flags, tbl, ntiles, m, brow,
                                                                           bval, y);
  else
    k_svb_accumulate<K, T, kSvLBTall, 1024, 4><<<(unsigned)max_chunks, 1024, 0, s>>>(chunks, flags, tbl, ntiles, m,
                                                                                 brow, bval, y);
  hipError_t e = hipGetLastError();
  SvFlags h{0, 0, 0};
  if (e == hipSuccess) e = hipMemcpyAsync(&h, flags, sizeof(h), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  ws.release();
  if (e != hipSuccess) return set_error(CBX_ERR_HIP, "cbx_spmv_dense: %s", hipGetErrorString(e));
  if (h.bad_columns || h.bad_entries) return set_error(CBX_ERR_INVALID, "cbx_dcsc_check: malformed DCSC");
  return CBX_OK;
}

extern "C" cbx_status cbx_spmspv(const cbx_dcsc* A, const int32_t* xind, const void* xval, int32_t nx,
                                 cbx_semiring semiring, cbx_dtype xdtype, int32_t* yind, void* yval, int32_t* ny,
                                 void* stream) {
  CBX_RETURN_IF(!A || !ny || (nx > 0 && (!xind || !xval)) || !yind || !yval, CBX_ERR_INVALID,
                "cbx_spmspv: null argument");
  CBX_RETURN_IF(A->location != CBX_DEVICE, CBX_ERR_INVALID, "cbx_spmspv: expected a device matrix");
  CBX_RETURN_IF(A->m >= (1ll << 31) || A->n >= (1ll << 31), CBX_ERR_LIMIT, "cbx_spmspv: dimensions must be below 2^31");
  CBX_RETURN_IF(nx < 0 || nx > A->n, CBX_ERR_INVALID, "cbx_spmspv: bad vector length");
  const bool boolA = A->dtype == CBX_BOOL;
  CBX_RETURN_IF(!boolA && A->dtype != xdtype, CBX_ERR_UNSUPPORTED,
                "cbx_spmspv: A must be boolean or share the vector's dtype");
  *ny = 0;
  if (A->nzc == 0 || nx == 0) {
    const cbx_status st = cbx_dcsc_check(A);  // otherwise with the product
    if (st != CBX_OK) return st;
  }
  const cbx_status init = init_device_once();
  if (init != CBX_OK) return init;
  hipStream_t s = (hipStream_t)stream;
  switch (semiring * 8 + xdtype) {
#define CBX_SV(SRK, SRE, T, DT)                                                                                     \
  case SRE * 8 + DT:                                                                                                \
    if (A->nzc == 0 || nx == 0) return CBX_OK;                                                                      \
    return spmspv_typed<SRK, T>(A, boolA, xind, (const T*)xval, nx, yind, (T*)yval, ny, s);
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, int64_t, CBX_I64)
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, double, CBX_F64)
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, float, CBX_F32)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, int64_t, CBX_I64)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, double, CBX_F64)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, float, CBX_F32)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, int64_t, CBX_I64)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, double, CBX_F64)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, float, CBX_F32)
#undef CBX_SV
  }
  return set_error(CBX_ERR_UNSUPPORTED, "cbx_spmspv: semiring %d with vector dtype %d is not provided", (int)semiring,
                   (int)xdtype);
}

// ------------------------------------------------ allocation-free SpMSpV
// The scratch of cbx_spmspv_noalloc: one static array per GPU, held until the
// process ends.  In host code `scratch` names a host-side stand-in, not device
// memory, so the host never passes it to a kernel or a copy: each device's
// address of the array is looked up once (hipGetSymbolAddress, with that
// device current) and kept in g_scratch_dev.
constexpr size_t kSpmspvScratchBytes = (size_t)CBX_SPMSPV_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kSpmspvScratchBytes];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
char* g_scratch_dev[kMaxScratchDevices] = {};

// Device address of `scratch` on the current device (looked up on the first
// call made with that device current).
cbx_status scratch_region(char** out) {
  int dev = 0;
  CBX_HIP(hipGetDevice(&dev));
  CBX_RETURN_IF(dev < 0 || dev >= kMaxScratchDevices, CBX_ERR_LIMIT, "cbx_spmspv_noalloc: device %d out of range",
                dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error(CBX_ERR_HIP, "cbx_spmspv_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                       hipGetErrorString(e));
    g_scratch_dev[dev] = (char*)p;
  }
  *out = g_scratch_dev[dev];
  return CBX_OK;
}
}  // namespace

extern "C" cbx_status cbx_spmspv_noalloc(const cbx_dcsc* A, const int32_t* xind, const void* xval, int32_t nx,
                                         cbx_semiring semiring, cbx_dtype xdtype, int32_t* yind, void* yval,
                                         int32_t* ny, void* stream) {
  CBX_RETURN_IF(!A || !ny || (nx > 0 && (!xind || !xval)) || !yind || !yval, CBX_ERR_INVALID,
                "cbx_spmspv_noalloc: null argument");
  CBX_RETURN_IF(A->location != CBX_DEVICE, CBX_ERR_INVALID, "cbx_spmspv_noalloc: expected a device matrix");
  CBX_RETURN_IF(A->m < 0 || A->n < 0 || A->nnz < 0 || A->nzc < 0, CBX_ERR_INVALID, "cbx_spmspv_noalloc: negative size");
  CBX_RETURN_IF(A->m >= (1ll << 31) || A->n >= (1ll << 31), CBX_ERR_LIMIT,
                "cbx_spmspv_noalloc: dimensions must be below 2^31");
  CBX_RETURN_IF(nx < 0 || nx > A->n, CBX_ERR_INVALID, "cbx_spmspv_noalloc: bad vector length");
  const bool boolA = A->dtype == CBX_BOOL;
  CBX_RETURN_IF(!boolA && A->dtype != xdtype, CBX_ERR_UNSUPPORTED,
                "cbx_spmspv_noalloc: A must be boolean or share the vector's dtype");
  char* region = nullptr;
  const cbx_status rs = scratch_region(&region);
  if (rs != CBX_OK) return rs;
  hipStream_t s = (hipStream_t)stream;
  switch (semiring * 8 + xdtype) {
#define CBX_SV(SRK, SRE, T, DT)                                                                                      \
  case SRE * 8 + DT:                                                                                                 \
    return spmspv_in_region<SRK, T>(A, boolA, xind, (const T*)xval, nx, yind, (T*)yval, ny, region,                  \
                                    kSpmspvScratchBytes, s);
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, int64_t, CBX_I64)
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, double, CBX_F64)
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, float, CBX_F32)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, int64_t, CBX_I64)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, double, CBX_F64)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, float, CBX_F32)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, int64_t, CBX_I64)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, double, CBX_F64)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, float, CBX_F32)
#undef CBX_SV
  }
  return set_error(CBX_ERR_UNSUPPORTED, "cbx_spmspv_noalloc: semiring %d with vector dtype %d is not provided",
                   (int)semiring, (int)xdtype);
}

extern "C" cbx_status cbx_spmv_dense(const cbx_dcsc* A, const void* x, void* y, cbx_semiring semiring,
                                     cbx_dtype xdtype, void* stream) {
  CBX_RETURN_IF(!A || (A->n > 0 && !x) || (A->m > 0 && !y), CBX_ERR_INVALID, "cbx_spmv_dense: null argument");
  CBX_RETURN_IF(A->location != CBX_DEVICE, CBX_ERR_INVALID, "cbx_spmv_dense: expected a device matrix");
  CBX_RETURN_IF(A->m >= (1ll << 31) || A->n >= (1ll << 31), CBX_ERR_LIMIT,
                "cbx_spmv_dense: dimensions must be below 2^31");
  const bool boolA = A->dtype == CBX_BOOL;
  CBX_RETURN_IF(!boolA && A->dtype != xdtype, CBX_ERR_UNSUPPORTED,
                "cbx_spmv_dense: A must be boolean or share the vectors' dtype");
  // (the structure check, the rules of cbx_dcsc_check, runs with the product)
  CBX_RETURN_IF(A->nzc == 0 && A->nnz != 0, CBX_ERR_INVALID, "cbx_dcsc_check: nnz without columns");
  CBX_RETURN_IF(A->m <= 0 && A->nnz != 0, CBX_ERR_INVALID, "cbx_dcsc_check: nnz without rows");
  const cbx_status init = init_device_once();
  if (init != CBX_OK) return init;
  hipStream_t s = (hipStream_t)stream;
  switch (semiring * 8 + xdtype) {
#define CBX_SV(SRK, SRE, T, DT) \
  case SRE * 8 + DT:            \
    return spmv_dense_typed<SRK, T>(A, boolA, (const T*)x, (T*)y, s);
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, int64_t, CBX_I64)
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, double, CBX_F64)
    CBX_SV(kPlusTimes, CBX_SR_PLUS_TIMES, float, CBX_F32)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, int64_t, CBX_I64)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, double, CBX_F64)
    CBX_SV(kMinPlus, CBX_SR_MIN_PLUS, float, CBX_F32)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, int64_t, CBX_I64)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, double, CBX_F64)
    CBX_SV(kSelectMax, CBX_SR_SELECT_MAX, float, CBX_F32)
#undef CBX_SV
  }
  return set_error(CBX_ERR_UNSUPPORTED, "cbx_spmv_dense: semiring %d with vector dtype %d is not provided",
                   (int)semiring, (int)xdtype);
}
