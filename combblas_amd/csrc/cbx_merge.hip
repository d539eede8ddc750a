// Stage merge: the sum, under a semiring's add, of several sparse matrices of
// one shape, returned as DCSC.
//
// cbx_dcsc_merge replaces MultiwayMerge<SR> (MultiwayMerge.h:428-541; the
// per-split SerialMerge at :193-250) and MultiwayMergeHash with sorted=true
// (:553), which SUMMA uses to combine the local products of its stages, and
// the SpDCCols(SpTuples) conversion after it (SpDCCols.cpp:109-184): entries
// with equal (row, col) are combined with SR::add, nothing is dropped
// (explicit zeros stay), the result is column-major with ascending rows.  The
// reference merges k column-sorted lists with a heap; here the merge of c
// parts P_s (m x n) is the product [P_0 ... P_{c-1}] * B of their column
// concatenation (m x cn) with B (cn x n) stacking c identities whose entries
// are the semiring's multiplicative one (1 for plus-times and select-max,
// -0.0 / 0 for min-plus: x + -0.0 = x keeps a -0.0 entry's sign), so C(:,j)
// combines the parts' columns j with the semiring's add: the SpGEMM's own
// tiers do the merge and write DCSC directly.  Equal entries are combined in
// the accumulation's order, the reference in heap order: this changes only
// floating-point rounding.
//
// cbx_dcsc_from_coo (the Graph500 edge-list constructor, further below) keys
// the entries, radix-sorts them and combines equal neighbours in one pass that
// writes the DCSC.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <type_traits>
#include <vector>

#include "cbx_device.h"
#include "cbx_semiring.h"
#include "cbx_spgemm.h"

namespace cbx {
namespace {

constexpr int kMergeNT = 256;

// The semiring's add on stored values (SR::add of the reference's semirings).
// Min and max keep a NaN on the left and pass over one on the right, which is
// not associative: in a tree, (5 + NaN) + (NaN + 3) would lose the 3.  `join`
// passes over NaN on either side; a run's fold from left to right is then its
// first value if that is NaN, and otherwise the join of all in any shape.
template <int K, class T>
struct SemAdd {
  static constexpr bool kKeepsNan = K != kPlusTimes && std::is_floating_point<T>::value;
  __device__ __forceinline__ T operator()(const T& a, const T& b) const {
    using SR = Sem<K, T>;
    using Acc = typename SR::Acc;
    return (T)SR::out(SR::add((Acc)a, (Acc)b));
  }
  __device__ __forceinline__ T join(const T& a, const T& b) const {
    if (kKeepsNan && a != a) return b;
    return (*this)(a, b);
  }
};

// A value of another lane.
template <class T>
__device__ __forceinline__ T shfl_down(T v, int d) {
  if constexpr (sizeof(T) == 1) return (T)__shfl_down((int)v, d, kWave);
  else return __shfl_down(v, d, kWave);
}
template <class T>
__device__ __forceinline__ T shfl_from(T v, int lane) {
  if constexpr (sizeof(T) == 1) return (T)__shfl((int)v, lane, kWave);
  else return __shfl(v, lane, kWave);
}

// B (c n x n): column j holds c entries, at rows s n + j, each the one.
template <class T>
__global__ void k_stacked_identity(int64_t n, int c, T one, int64_t* __restrict__ cpB, int64_t* __restrict__ jcB,
                                   int64_t* __restrict__ irB, T* __restrict__ valB) {
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j > n) return;
  cpB[j] = j * c;
  if (j == n) return;
  jcB[j] = j;
  for (int p = 0; p < c; ++p) {
    irB[j * c + p] = p * n + j;
    valB[j * c + p] = one;
  }
}

template <int K, class T>
T semiring_one() {
  if constexpr (K == kMinPlus) {
    if constexpr (std::is_floating_point<T>::value) return (T)-0.0;
    else return (T)0;
  } else {
    return (T)1;
  }
}

// The product's kernels hold places in A's entries and A's stored columns as
// 32-bit numbers: so many of either in one concatenation at most.
constexpr int64_t kMergeMost = (1ll << 31) - 1;

// A matrix to merge, or a range of its columns (entries from nz_base on, column
// ids from col_base on).
struct MergePart {
  const int64_t *cp, *jc, *ir;
  const void* val;
  int64_t nnz, nzc, nz_base, col_base;
};

struct MergeResult {
  cbx_dcsc x{};
  MergeResult() = default;
  MergeResult(MergeResult&& o) noexcept : x(o.x) { o.x = cbx_dcsc{}; }
  MergeResult(const MergeResult&) = delete;
  ~MergeResult() { cbx_dcsc_free(&x); }
  MergePart part() const { return MergePart{x.cp, x.jc, x.ir, x.val, x.nnz, x.nzc, 0, 0}; }
};

cbx_status merge_empty(int64_t m, int64_t n, cbx_dtype dtype, cbx_dcsc* out, hipStream_t s) {
  std::memset(out, 0, sizeof(*out));
  out->m = m;
  out->n = n;
  out->dtype = dtype;
  out->location = CBX_DEVICE;
  cbx_status st = CBX_OK;
  if ((st = dev_alloc((void**)&out->cp, sizeof(int64_t))) != CBX_OK ||
      (st = dev_alloc((void**)&out->jc, sizeof(int64_t))) != CBX_OK ||
      (st = dev_alloc((void**)&out->ir, sizeof(int64_t))) != CBX_OK ||
      (st = dev_alloc(&out->val, sizeof(int64_t))) != CBX_OK) {
    cbx_dcsc_free(out);
    return st;
  }
  CBX_HIP(hipMemsetAsync(out->cp, 0, sizeof(int64_t), s));
  CBX_HIP(hipStreamSynchronize(s));
  return CBX_OK;
}

// The merge of n columns as one product.
template <int K, class T>
cbx_status merge_product(const std::vector<MergePart>& parts, int64_t m, int64_t n, cbx_dtype dtype, cbx_dcsc* out,
                         hipStream_t s) {
  const int64_t count = (int64_t)parts.size();
  int64_t nnz = 0, nzc = 0;
  for (const MergePart& P : parts) {
    nnz += P.nnz;
    nzc += P.nzc;
  }
  CBX_RETURN_IF((double)count * (double)n >= 9.0e18, CBX_ERR_LIMIT, "cbx_dcsc_merge: too many columns in the parts");
  cbx_dcsc A{}, B{};
  A.m = m;
  A.n = count * n;
  A.nnz = nnz;
  A.nzc = nzc;
  A.dtype = B.dtype = dtype;
  A.location = B.location = CBX_DEVICE;
  B.m = A.n;
  B.n = n;
  B.nnz = count * n;
  B.nzc = n;
  ScratchSet ws(s);
  int64_t *cpA, *jcA, *cpB, *jcB, *irB;
  int32_t* rowsA;
  T *valA, *valB;
  if (!ws.take(&cpA, nzc + 1) || !ws.take(&jcA, nzc) || !ws.take(&rowsA, nnz) || !ws.take(&valA, nnz) ||
      !ws.take(&cpB, n + 1) || !ws.take(&jcB, n) || !ws.take(&irB, B.nnz) || !ws.take(&valB, B.nnz))
    return set_error(CBX_ERR_NOMEM, "cbx_dcsc_merge: workspace allocation failed");
  A.cp = cpA;
  A.jc = jcA;
  A.val = valA;
  B.cp = cpB;
  B.jc = jcB;
  B.ir = irB;
  B.val = valB;
  // the parts as column blocks of one matrix, each checked against its own
  // bounds (a column id beyond n would fall into the next part's block)
  std::vector<PackSeg> segs((size_t)count);
  int64_t eb = 0, qb = 0;
  for (int64_t i = 0; i < count; ++i) {
    const MergePart& P = parts[i];
    segs[i] = PackSeg{P.cp, P.jc, P.ir, P.val, 0, i * n, eb, qb, m, n, P.nnz, P.nzc, P.nz_base, P.col_base};
    eb += P.nnz;
    qb += P.nzc;
  }
  cbx_status st = pack_members(segs.data(), count, A, rowsA, s);
  if (st != CBX_OK) return st;
  k_stacked_identity<T><<<(unsigned)((n + 1 + kMergeNT - 1) / kMergeNT), kMergeNT, 0, s>>>(
      n, (int)count, semiring_one<K, T>(), cpB, jcB, irB, valB);
  CBX_HIP(hipGetLastError());
  SpgemmConfig cfg = current_config();
  cfg.trusted_a = cfg.trusted_b = true;
  cfg.rows_a = rowsA;
  const cbx_semiring sr = K == kPlusTimes ? CBX_SR_PLUS_TIMES : K == kMinPlus ? CBX_SR_MIN_PLUS : CBX_SR_SELECT_MAX;
  st = spgemm_dispatch(&A, &B, sr, CBX_SPGEMM_TWO_PHASE, cfg, out, nullptr, s);
  if (st != CBX_OK) cbx_dcsc_free(out);
  return st;
}

// Of each part: its first stored column (x) at or after column id `col`, and
// that column's first entry (y), both counted in the part's range.
__global__ __launch_bounds__(kMergeNT) void k_merge_below(const MergePart* __restrict__ parts, int64_t count,
                                                          int64_t col, longlong2* __restrict__ below) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= count) return;
  const MergePart P = parts[i];
  int64_t lo = 0, hi = P.nzc;
  while (lo < hi) {
    const int64_t mid = lo + (hi - lo) / 2;
    if (P.jc[mid] - P.col_base < col) lo = mid + 1;
    else hi = mid;
  }
  below[i] = make_longlong2(lo, P.nzc ? P.cp[lo] - P.nz_base : 0);
}

// A range's columns into the output's arrays at its place (cp: one more, the
// next range's first or the end).
__global__ __launch_bounds__(kMergeNT) void k_merge_columns(const int64_t* __restrict__ cp,
                                                            const int64_t* __restrict__ jc, int64_t nzc,
                                                            int64_t entries, int64_t first, int64_t* __restrict__ ocp,
                                                            int64_t* __restrict__ ojc) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q > nzc) return;
  ocp[q] = cp[q] + entries;
  if (q < nzc) ojc[q] = jc[q] + first;
}

// The merge of n columns whose parts hold too much for one product: column
// ranges that fit, one after the other, and their results one after the other
// in the output.  A single column that does not fit is merged in two halves of
// the parts first.  Nothing of the parts is trusted here beyond their sizes:
// the cuts are checked below, and each range is checked as it is packed.
template <int K, class T>
cbx_status merge_columns(const std::vector<MergePart>& parts, int64_t m, int64_t n, cbx_dtype dtype, int64_t most,
                         cbx_dcsc* out, hipStream_t s) {
  const size_t count = parts.size();
  int64_t nnz = 0, nzc = 0;
  for (const MergePart& P : parts) {
    nnz += P.nnz;
    nzc += P.nzc;
  }
  if (nzc == 0) return merge_empty(m, n, dtype, out, s);
  if (nnz <= most && nzc <= most) return merge_product<K, T>(parts, m, n, dtype, out, s);
  std::memset(out, 0, sizeof(*out));
  cbx_status st = CBX_OK;
  if (n == 1) {
    CBX_RETURN_IF(count < 3, CBX_ERR_LIMIT, "cbx_dcsc_merge: a column of two partial sums holds %lld entries, more than %lld",
                  (long long)nnz, (long long)most);
    MergeResult half[2];
    for (int h = 0; h < 2; ++h) {
      const std::vector<MergePart> some(parts.begin() + (h ? count / 2 : 0), h ? parts.end() : parts.begin() + count / 2);
      if ((st = merge_columns<K, T>(some, m, 1, dtype, most, &half[h].x, s)) != CBX_OK) return st;
    }
    return merge_columns<K, T>({half[0].part(), half[1].part()}, m, 1, dtype, most, out, s);
  }
  ScratchSet ws(s);
  MergePart* dparts;
  longlong2* dbelow;
  if (!ws.take(&dparts, count) || !ws.take(&dbelow, count))
    return set_error(CBX_ERR_NOMEM, "cbx_dcsc_merge: workspace allocation failed");
  CBX_HIP(hipMemcpyAsync(dparts, parts.data(), sizeof(MergePart) * count, hipMemcpyHostToDevice, s));
  std::vector<longlong2> from(count, make_longlong2(0, 0)), to(count);
  // what the columns [from, col) hold; malformed: they are no range of a part
  auto upto = [&](int64_t col, int64_t& entries, int64_t& columns) -> cbx_status {
    if (col == n) {
      for (size_t i = 0; i < count; ++i) to[i] = make_longlong2(parts[i].nzc, parts[i].nnz);
    } else {
      k_merge_below<<<(unsigned)((count + kMergeNT - 1) / kMergeNT), kMergeNT, 0, s>>>(dparts, (int64_t)count, col,
                                                                                     dbelow);
      CBX_HIP(hipGetLastError());
      CBX_HIP(hipMemcpyAsync(to.data(), dbelow, sizeof(longlong2) * count, hipMemcpyDeviceToHost, s));
      CBX_HIP(hipStreamSynchronize(s));
    }
    entries = columns = 0;
    for (size_t i = 0; i < count; ++i) {
      CBX_RETURN_IF(to[i].x < from[i].x || to[i].y < from[i].y || to[i].y > parts[i].nnz, CBX_ERR_INVALID,
                    "cbx_dcsc_check: a part is malformed");
      entries += to[i].y - from[i].y;
      columns += to[i].x - from[i].x;
    }
    return CBX_OK;
  };
  struct Range {
    int64_t first, columns, entries;  // column id, and stored columns and entries before its own in the output
    MergeResult merged;
  };
  std::vector<Range> ranges;
  int64_t cols_out = 0, entries_out = 0;
  for (int64_t c0 = 0; c0 < n;) {
    int64_t lo = c0 + 1, hi = n, entries = 0, columns = 0;  // the last end of a range that fits, one column at least
    while (lo < hi) {
      const int64_t mid = lo + (hi - lo + 1) / 2;
      if ((st = upto(mid, entries, columns)) != CBX_OK) return st;
      if (entries <= most && columns <= most) lo = mid;
      else hi = mid - 1;
    }
    if ((st = upto(lo, entries, columns)) != CBX_OK) return st;
    std::vector<MergePart> some;
    for (size_t i = 0; i < count; ++i) {
      const MergePart& P = parts[i];
      if (to[i].x == from[i].x) {
        CBX_RETURN_IF(to[i].y != from[i].y, CBX_ERR_INVALID, "cbx_dcsc_check: a part is malformed");
        continue;
      }
      some.push_back(MergePart{P.cp + from[i].x, P.jc + from[i].x, P.ir + from[i].y, (const T*)P.val + from[i].y,
                               to[i].y - from[i].y, to[i].x - from[i].x, P.nz_base + from[i].y, P.col_base + c0});
    }
    if (!some.empty()) {
      ranges.push_back(Range{c0, cols_out, entries_out, {}});
      cbx_dcsc& x = ranges.back().merged.x;
      if ((st = merge_columns<K, T>(some, m, lo - c0, dtype, most, &x, s)) != CBX_OK) return st;
      cols_out += x.nzc;
      entries_out += x.nnz;
    }
    c0 = lo;
    from = to;
  }
  ws.release();
  out->m = m;
  out->n = n;
  out->dtype = dtype;
  out->location = CBX_DEVICE;
  // array by array, each range's given back before the next is allocated
  auto fail = [&](cbx_status why) {
    (void)hipStreamSynchronize(s);
    cbx_dcsc_free(out);
    return why;
  };
  if ((st = dev_alloc((void**)&out->cp, sizeof(int64_t) * (size_t)(cols_out + 1))) != CBX_OK ||
      (st = dev_alloc((void**)&out->jc, sizeof(int64_t) * (size_t)std::max<int64_t>(cols_out, 1))) != CBX_OK)
    return fail(st);
  for (const Range& r : ranges)
    k_merge_columns<<<(unsigned)((r.merged.x.nzc + kMergeNT) / kMergeNT), kMergeNT, 0, s>>>(
        r.merged.x.cp, r.merged.x.jc, r.merged.x.nzc, r.entries, r.first, out->cp + r.columns, out->jc + r.columns);
  hipError_t e = hipGetLastError();
  auto gather = [&](auto member, void** to_all, size_t size) -> cbx_status {
    const cbx_status ast = dev_alloc(to_all, size * (size_t)std::max<int64_t>(entries_out, 1));
    if (ast != CBX_OK) return ast;
    for (Range& r : ranges)
      if (e == hipSuccess && r.merged.x.nnz)
        e = hipMemcpyAsync((char*)*to_all + size * (size_t)r.entries, *member(r.merged.x), size * (size_t)r.merged.x.nnz,
                           hipMemcpyDeviceToDevice, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    for (Range& r : ranges) {
      dev_free(*member(r.merged.x));
      *member(r.merged.x) = nullptr;
    }
    return CBX_OK;
  };
  if ((st = gather([](cbx_dcsc& x) { return (void**)&x.ir; }, (void**)&out->ir, sizeof(int64_t))) != CBX_OK ||
      (st = gather([](cbx_dcsc& x) { return &x.val; }, &out->val, sizeof(T))) != CBX_OK)
    return fail(st);
  if (e != hipSuccess) return fail(set_error(CBX_ERR_HIP, "cbx_dcsc_merge: %s", hipGetErrorString(e)));
  out->nnz = entries_out;
  out->nzc = cols_out;
  return CBX_OK;
}

template <int K, class T>
cbx_status merge_typed(int32_t count, const cbx_dcsc* parts, int64_t most, cbx_dcsc* out, hipStream_t s) {
  std::memset(out, 0, sizeof(*out));
  std::vector<MergePart> all((size_t)count);
  for (int32_t i = 0; i < count; ++i)
    all[i] = MergePart{parts[i].cp, parts[i].jc, parts[i].ir, parts[i].val, parts[i].nnz, parts[i].nzc, 0, 0};
  return merge_columns<K, T>(all, parts[0].m, parts[0].n, parts[0].dtype, most, out, s);
}

// ------------------------------------------------------- edge list to DCSC
// Keys of COO entries: column above row in as many bits as the shape needs, as
// every eight bits are a pass of the sort over keys and values (2^20 x 2^20: 40
// bits and five passes of 160 us for 16.8 M entries; 53 and seven with the row
// in a half of its own and a bit for the dropped loops).  A dropped self
// loop's key is the last one, `drop`, that no entry has (coo_typed).  bad[0]
// counts entries out of range, bad[1] the loops dropped.
__global__ __launch_bounds__(kMergeNT) void k_coo_keys(const int64_t* __restrict__ rows,
                                                       const int64_t* __restrict__ cols, int64_t nnz, int64_t m,
                                                       int64_t n, int drop_loops, int row_bits, uint64_t drop,
                                                       uint64_t* __restrict__ keys,
                                                       unsigned long long* __restrict__ bad) {
  constexpr int U = 4;
  long long oob = 0, loops = 0;
  for (int64_t i0 = blockIdx.x * (int64_t)(kMergeNT * U); i0 < nnz; i0 += (int64_t)gridDim.x * (kMergeNT * U)) {
    int64_t r[U], c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = min(i0 + u * kMergeNT + threadIdx.x, nnz - 1);
      r[u] = rows[i];
      c[u] = cols[i];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      pin(r[u]);
      pin(c[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = i0 + u * kMergeNT + threadIdx.x;
      if (i >= nnz) continue;
      const bool ok = r[u] >= 0 && r[u] < m && c[u] >= 0 && c[u] < n;
      const bool loop = drop_loops && r[u] == c[u];
      oob += !ok;
      loops += ok && loop;
      keys[i] = ok && !loop ? ((uint64_t)c[u] << row_bits) | (uint64_t)r[u] : drop;
    }
  }
  block_add_counts<kMergeNT>(oob, loops, &bad[0], &bad[1]);
}

__global__ void k_coo_begin(unsigned long long* __restrict__ bad) {
  if (threadIdx.x < 2) bad[threadIdx.x] = 0ull;
}

// The sorted keys are taken in strips of kStrip entries, one per wave, kStrips
// to a workgroup; a strip's entries are loaded together, 64 at a time to a lane
// each.  A head is an entry whose key differs from the one before.
constexpr int kChunks = 8, kStrip = kChunks * kWave, kStrips = kMergeNT / kWave;
constexpr int kCooTile = kStrip * kStrips;

struct Strip {
  uint64_t key[kChunks];
  unsigned long long heads[kChunks], columns[kChunks], live[kChunks];  // lanes (uniform)
};

__device__ __forceinline__ Strip load_strip(const uint64_t* __restrict__ keys, int64_t e0, int64_t count,
                                            int row_bits) {
  Strip st;
  uint64_t prev[kChunks];
  const int lane = lane_id();
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int64_t i = max(min(e0 + c * kWave + lane, count - 1), (int64_t)0);
    st.key[c] = keys[i];
    prev[c] = keys[max(i - 1, (int64_t)0)];
  }
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    pin(st.key[c]);
    pin(prev[c]);
  }
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int64_t i = e0 + c * kWave + lane;
    const bool live = i < count;
    st.live[c] = __ballot(live);
    st.heads[c] = __ballot(live && (i == 0 || st.key[c] != prev[c]));
    st.columns[c] = __ballot(live && (i == 0 || (st.key[c] >> row_bits) != (prev[c] >> row_bits)));
  }
  return st;
}

// Heads (x) and column heads (y) of each tile.  count = nnz less the loops.
__global__ __launch_bounds__(kMergeNT) void k_coo_count(const uint64_t* __restrict__ keys, int64_t nnz,
                                                        const unsigned long long* __restrict__ bad, int row_bits,
                                                        int2* __restrict__ tiles) {
  __shared__ int sx[kStrips], sy[kStrips];
  const int64_t count = nnz - (int64_t)bad[1];
  const int w = wave_id_uniform();
  const Strip st = load_strip(keys, blockIdx.x * (int64_t)kCooTile + w * kStrip, count, row_bits);
  int x = 0, y = 0;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    x += __popcll(st.heads[c]);
    y += __popcll(st.columns[c]);
  }
  if (lane_id() == 0) {
    sx[w] = x;
    sy[w] = y;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    x = y = 0;
    for (int k = 0; k < kStrips; ++k) {
      x += sx[k];
      y += sy[k];
    }
    tiles[blockIdx.x] = make_int2(x, y);
  }
}

// Exclusive prefix sums of the tiles' counts in place, and what the host needs.
struct CooReport {
  unsigned long long bad[2];
  long long nnz, nzc;
};
constexpr int kCooScanNT = 1024, kCooScanPer = 8;
__global__ __launch_bounds__(kCooScanNT) void k_coo_scan(int2* __restrict__ tiles, int64_t ntiles,
                                                         const unsigned long long* __restrict__ bad,
                                                         CooReport* __restrict__ rep) {
  __shared__ long long wsum[kCooScanNT / kWave];
  long long bx = 0, by = 0;
  for (int64_t t0 = 0; t0 < ntiles; t0 += kCooScanNT * kCooScanPer) {
    const int64_t t = t0 + (int64_t)threadIdx.x * kCooScanPer;
    int2 v[kCooScanPer];
    long long x = 0, y = 0;
#pragma unroll
    for (int k = 0; k < kCooScanPer; ++k) v[k] = tiles[min(t + k, ntiles - 1)];
#pragma unroll
    for (int k = 0; k < kCooScanPer; ++k) {
      pin(v[k].x);
      pin(v[k].y);
      if (t + k >= ntiles) v[k] = make_int2(0, 0);
      x += v[k].x;
      y += v[k].y;
    }
    long long tx, ty;
    long long ex = bx + block_excl_scan_ll<kCooScanNT>(x, wsum, tx);
    long long ey = by + block_excl_scan_ll<kCooScanNT>(y, wsum, ty);
#pragma unroll
    for (int k = 0; k < kCooScanPer; ++k) {
      if (t + k < ntiles) tiles[t + k] = make_int2((int)ex, (int)ey);
      ex += v[k].x;
      ey += v[k].y;
    }
    bx += tx;
    by += ty;
  }
  if (threadIdx.x == 0) *rep = CooReport{{bad[0], bad[1]}, bx, by};
}

// A value that may be absent (a semiring's add has no identity that every
// stored value leaves alone: infinity against min-plus's largest number).
template <class T>
struct Maybe {
  T v;
  bool some;
};

// What strip s adds to the run that reaches it from the left, and whether that
// run takes all of it.
template <class T>
struct StripLead {
  T v;
  int some, whole;
};

// The DCSC from the sorted entries: each run of equal keys is combined (vals:
// null for ones) and written at its rank, columns at theirs.  A run is combined
// within 64 entries by steps that double, as many as its longest run needs;
// chunks of a strip pass what they add to the run on their left; strips leave
// it in `lead` for k_coo_join.  Bound by the bytes read and written once: 16.8 M
// entries (R-MAT s20, int64) take 96 us, and 31 in k_coo_count; the library's
// reduce-by-key and run lengths, the extraction of rows and a copy of the
// values, with two waits between, took some 600.
template <int K, class T>
__global__ __launch_bounds__(kMergeNT) void k_coo_assemble(const uint64_t* __restrict__ keys,
                                                           const T* __restrict__ vals, int64_t count, int row_bits,
                                                           const int2* __restrict__ tiles, int64_t nnz, int64_t nzc,
                                                           int64_t* __restrict__ cp, int64_t* __restrict__ jc,
                                                           int64_t* __restrict__ ir, T* __restrict__ val,
                                                           StripLead<T>* __restrict__ lead) {
  __shared__ int sx[kStrips], sy[kStrips];
  const SemAdd<K, T> add;
  const int w = wave_id_uniform(), lane = lane_id();
  const int64_t strip = blockIdx.x * (int64_t)kStrips + w, e0 = strip * kStrip;
  T v[kChunks];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    v[c] = (T)1;
    if (vals) v[c] = vals[min(e0 + c * kWave + lane, count - 1)];
  }
  const Strip st = load_strip(keys, e0, count, row_bits);
#pragma unroll
  for (int c = 0; c < kChunks; ++c) pin(v[c]);
  int x = 0, y = 0;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    x += __popcll(st.heads[c]);
    y += __popcll(st.columns[c]);
  }
  if (lane == 0) {
    sx[w] = x;
    sy[w] = y;
  }
  __syncthreads();
  int64_t rank = tiles[blockIdx.x].x, crank = tiles[blockIdx.x].y;  // after this strip
  for (int k = 0; k <= w; ++k) {
    rank += sx[k];
    crank += sy[k];
  }
  Maybe<T> carry{T{}, false};  // from the chunk on the right
  bool whole = true;
#pragma unroll
  for (int c = kChunks - 1; c >= 0; --c) {
    const unsigned long long heads = st.heads[c], live = st.live[c];
    rank -= __popcll(heads);
    crank -= __popcll(st.columns[c]);
    // the first lane after this one's run
    const unsigned long long ends = lane == kWave - 1 ? 0ull : (heads | ~live) >> (lane + 1);
    const int end = ends ? lane + __ffsll(ends) : kWave;
    const T own = v[c];
    for (int d = 1; __ballot(lane + d < end); d *= 2) {
      const T o = shfl_down(v[c], d);
      if (lane + d < end) v[c] = add.join(v[c], o);
    }
    if (end == kWave && carry.some) v[c] = add.join(v[c], carry.v);
    const bool head = (heads >> lane) & 1ull;
    if (head) {
      const int64_t q = rank + __popcll(heads & ((1ull << lane) - 1ull));
      ir[q] = (int64_t)(st.key[c] & ((1ull << row_bits) - 1ull));
      val[q] = add.kKeepsNan && own != own ? own : v[c];
      if ((st.columns[c] >> lane) & 1ull) {
        const int64_t k = crank + __popcll(st.columns[c] & ((1ull << lane) - 1ull));
        jc[k] = (int64_t)(st.key[c] >> row_bits);
        cp[k] = q;
      }
    }
    carry.some = (live & 1ull) && !(heads & 1ull);
    carry.v = shfl_from(v[c], 0);
    whole = whole && !heads && !~live;
  }
  if (lane == 0) lead[strip] = StripLead<T>{carry.v, carry.some, whole};
  if (blockIdx.x == 0 && threadIdx.x == 0) cp[nzc] = nnz;
}

// Runs over the ends of strips: the strip in which one has its head adds what
// the following strips left, up to the first that it does not take whole.  One
// wave per strip; the last run of strip s is the entry before the strip's end
// rank, `tiles` and the strips' heads giving that as in the kernel above.
template <int K, class T>
__global__ __launch_bounds__(kMergeNT) void k_coo_join(const uint64_t* __restrict__ keys, int64_t count, int row_bits,
                                                       const int2* __restrict__ tiles, int64_t nstrips,
                                                       const StripLead<T>* __restrict__ lead, T* __restrict__ val) {
  __shared__ int sx[kStrips];
  const SemAdd<K, T> add;
  const int w = wave_id_uniform(), lane = lane_id();
  const int64_t strip = blockIdx.x * (int64_t)kStrips + w;
  const bool open = strip + 1 < nstrips && lead[strip + 1].some && !lead[strip].whole;
  __shared__ int any;
  if (threadIdx.x == 0) any = 0;
  __syncthreads();
  if (open && lane == 0) any = 1;
  __syncthreads();
  if (!any) return;
  const Strip st = load_strip(keys, strip * kStrip, count, row_bits);
  int x = 0;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) x += __popcll(st.heads[c]);
  if (lane == 0) sx[w] = x;
  __syncthreads();
  if (!open) return;
  int64_t q = (int64_t)tiles[blockIdx.x].x - 1;
  for (int k = 0; k <= w; ++k) q += sx[k];
  T sum = val[q];
  for (int64_t s0 = strip + 1; s0 < nstrips; s0 += kWave) {
    const bool in = s0 + lane < nstrips;
    const StripLead<T> l = lead[min(s0 + lane, nstrips - 1)];
    // lanes up to the first that is not whole
    const unsigned long long stop = __ballot(!in || !l.whole);
    const int n = stop ? __ffsll(stop) : kWave;
    const unsigned long long some = __ballot(in && lane < n && l.some);
    const int terms = some ? kWave - __clzll(some) : 0;  // (all lanes before the last one have a value)
    T v = l.v;
    for (int d = 1; d < terms; d *= 2) {
      const T o = shfl_down(v, d);
      if (lane + d < terms) v = add.join(v, o);
    }
    if (terms) sum = add(sum, shfl_from(v, 0));  // (a NaN so far is the run's first)
    if (stop) break;
  }
  if (lane == 0) val[q] = sum;
}

int bits_for(int64_t v) {  // bits to hold 0..v
  int b = 1;
  while (b < 62 && (int64_t(1) << b) <= v) ++b;
  return b;
}

template <int K, class T>
cbx_status coo_typed(int64_t m, int64_t n, const int64_t* rows, const int64_t* cols, const T* vals, int64_t nnz,
                     int drop_loops, cbx_dcsc* out, hipStream_t s) {
  const char* who = "cbx_dcsc_from_coo";
  const int N = (int)nnz;
  const int row_bits = bits_for(std::max<int64_t>(m - 1, 0));
  int end_bit = row_bits + bits_for(std::max<int64_t>(n - 1, 0));
  // dropped loops sort to the end: the last key of so many bits is the entry
  // (2^row_bits - 1, 2^col_bits - 1), which is out of range or, in a square
  // matrix, a loop itself; otherwise one bit more
  if (drop_loops && m != n && m == (int64_t)1 << row_bits && n == (int64_t)1 << (end_bit - row_bits)) ++end_bit;
  const uint64_t drop = (1ull << end_bit) - 1;
  const int64_t ntiles = (nnz + kCooTile - 1) / kCooTile, nstrips = ntiles * kStrips;
  uint64_t *k0 = nullptr, *k1 = nullptr;
  T* v1 = nullptr;
  int2* tiles = nullptr;
  StripLead<T>* lead = nullptr;
  unsigned long long* bad = nullptr;
  CooReport* rep = nullptr;
  void* tmp = nullptr;
  size_t tb = 0;
  if (vals) CBX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, k0, k1, vals, v1, N, 0, end_bit, s));
  else CBX_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, tb, k0, k1, N, 0, end_bit, s));
  ScratchSet ws(s);
  if (!ws.take(&k0, N) || !ws.take(&k1, N) || (vals && !ws.take(&v1, N)) || !ws.take(&tiles, ntiles) ||
      !ws.take(&lead, nstrips) || !ws.take(&bad, 2) || !ws.take(&rep, 1) ||
      !ws.take_bytes(&tmp, std::max<size_t>(tb, 16))) {
    (void)hipGetLastError();
    return set_error(CBX_ERR_NOMEM, "cbx_dcsc_from_coo: workspace allocation failed");
  }
  k_coo_begin<<<1, 64, 0, s>>>(bad);
  const unsigned g = (unsigned)std::min<int64_t>((nnz + kMergeNT * 4 - 1) / (kMergeNT * 4), 2048);
  k_coo_keys<<<g, kMergeNT, 0, s>>>(rows, cols, nnz, m, n, drop_loops, row_bits, drop, k0, bad);
  CBX_HIP(hipGetLastError());
  if (vals) CBX_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, k0, k1, vals, v1, N, 0, end_bit, s));
  else CBX_HIP(hipcub::DeviceRadixSort::SortKeys(tmp, tb, k0, k1, N, 0, end_bit, s));
  k_coo_count<<<(unsigned)ntiles, kMergeNT, 0, s>>>(k1, nnz, bad, row_bits, tiles);
  k_coo_scan<<<1, kCooScanNT, 0, s>>>(tiles, ntiles, bad, rep);
  CooReport h{};
  CBX_HIP(hipGetLastError());
  CBX_HIP(hipMemcpyAsync(&h, rep, sizeof(h), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  if (h.bad[0])
    return set_error(CBX_ERR_INVALID, "cbx_dcsc_from_coo: %llu entries outside the %lld x %lld shape", h.bad[0],
                     (long long)m, (long long)n);
  const int64_t count = nnz - (int64_t)h.bad[1];
  cbx_status st = CBX_OK;
  const int64_t held = std::max<int64_t>(h.nnz, 1);
  if ((st = dev_alloc((void**)&out->cp, sizeof(int64_t) * (h.nzc + 1))) != CBX_OK ||
      (st = dev_alloc((void**)&out->jc, sizeof(int64_t) * std::max<int64_t>(h.nzc, 1))) != CBX_OK ||
      (st = dev_alloc((void**)&out->ir, sizeof(int64_t) * held)) != CBX_OK ||
      (st = dev_alloc(&out->val, sizeof(T) * held)) != CBX_OK) {
    cbx_dcsc_free(out);
    return st;
  }
  hipError_t e = hipSuccess;
  if (count > 0) {
    k_coo_assemble<K, T><<<(unsigned)ntiles, kMergeNT, 0, s>>>(k1, vals ? v1 : nullptr, count, row_bits, tiles, h.nnz,
                                                              h.nzc, out->cp, out->jc, out->ir, (T*)out->val, lead);
    k_coo_join<K, T><<<(unsigned)ntiles, kMergeNT, 0, s>>>(k1, count, row_bits, tiles, nstrips, lead, (T*)out->val);
    e = hipGetLastError();
  } else {  // every entry a dropped loop
    e = hipMemsetAsync(out->cp, 0, sizeof(int64_t), s);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    cbx_dcsc_free(out);
    return set_error(CBX_ERR_HIP, "%s: %s", who, hipGetErrorString(e));
  }
  out->nnz = h.nnz;
  out->nzc = h.nzc;
  return CBX_OK;
}

}  // namespace
}  // namespace cbx

using namespace cbx;

extern "C" cbx_status cbx_dcsc_merge(int32_t count, const cbx_dcsc* parts, cbx_semiring semiring, cbx_dcsc* out,
                                     void* stream) {
  return cbx_dcsc_merge_in_ranges(count, parts, semiring, kMergeMost, out, stream);
}

extern "C" cbx_status cbx_dcsc_merge_in_ranges(int32_t count, const cbx_dcsc* parts, cbx_semiring semiring,
                                               int64_t max_entries, cbx_dcsc* out, void* stream) {
  CBX_RETURN_IF(max_entries < 1 || max_entries > kMergeMost, CBX_ERR_INVALID,
                "cbx_dcsc_merge_in_ranges: max_entries must be in [1, 2^31)");
  CBX_RETURN_IF(!parts || !out || count < 1, CBX_ERR_INVALID, "cbx_dcsc_merge: need at least one part and an output");
  cbx_status st = init_device_once();
  if (st != CBX_OK) return st;
  for (int32_t i = 0; i < count; ++i) {
    if ((st = check_dcsc(&parts[i], "part", CBX_DEVICE)) != CBX_OK) return st;
    CBX_RETURN_IF(parts[i].m != parts[0].m || parts[i].n != parts[0].n || parts[i].dtype != parts[0].dtype,
                  CBX_ERR_INVALID, "cbx_dcsc_merge: part %d differs in shape or dtype from part 0", i);
  }
  hipStream_t s = (hipStream_t)stream;
  const cbx_dtype dt = parts[0].dtype;
  switch (semiring * 8 + dt) {
#define CBX_MG(SRK, SRE, T, DT) \
  case SRE * 8 + DT:            \
    return merge_typed<SRK, T>(count, parts, max_entries, out, s);
    CBX_MG(kPlusTimes, CBX_SR_PLUS_TIMES, int64_t, CBX_I64)
    CBX_MG(kPlusTimes, CBX_SR_PLUS_TIMES, double, CBX_F64)
    CBX_MG(kPlusTimes, CBX_SR_PLUS_TIMES, float, CBX_F32)
    CBX_MG(kPlusTimes, CBX_SR_PLUS_TIMES, uint8_t, CBX_BOOL)
    CBX_MG(kMinPlus, CBX_SR_MIN_PLUS, int64_t, CBX_I64)
    CBX_MG(kMinPlus, CBX_SR_MIN_PLUS, double, CBX_F64)
    CBX_MG(kMinPlus, CBX_SR_MIN_PLUS, float, CBX_F32)
    CBX_MG(kSelectMax, CBX_SR_SELECT_MAX, int64_t, CBX_I64)
    CBX_MG(kSelectMax, CBX_SR_SELECT_MAX, double, CBX_F64)
    CBX_MG(kSelectMax, CBX_SR_SELECT_MAX, float, CBX_F32)
#undef CBX_MG
  }
  return set_error(CBX_ERR_UNSUPPORTED, "cbx_dcsc_merge: semiring %d with dtype %d is not provided", (int)semiring,
                   (int)dt);
}

extern "C" cbx_status cbx_dcsc_from_coo(int64_t m, int64_t n, const int64_t* rows, const int64_t* cols,
                                        const void* vals, int64_t nnz, cbx_dtype dtype, cbx_semiring semiring,
                                        int32_t remove_loops, cbx_dcsc* out, void* stream) {
  CBX_RETURN_IF(!out || (nnz > 0 && (!rows || !cols)), CBX_ERR_INVALID, "cbx_dcsc_from_coo: null argument");
  CBX_RETURN_IF(m < 0 || n < 0 || nnz < 0, CBX_ERR_INVALID, "cbx_dcsc_from_coo: negative size");
  CBX_RETURN_IF(m >= (1ll << 31) || n >= (1ll << 31), CBX_ERR_LIMIT, "cbx_dcsc_from_coo: dimensions must be below 2^31");
  CBX_RETURN_IF(nnz >= (1ll << 31), CBX_ERR_LIMIT, "cbx_dcsc_from_coo: at most 2^31 - 1 entries");
  cbx_status st = init_device_once();
  if (st != CBX_OK) return st;
  std::memset(out, 0, sizeof(*out));
  out->m = m;
  out->n = n;
  out->dtype = dtype;
  out->location = CBX_DEVICE;
  hipStream_t s = (hipStream_t)stream;
  if (nnz == 0) {  // an empty m x n matrix
    if ((st = dev_alloc((void**)&out->cp, sizeof(int64_t))) != CBX_OK ||
        (st = dev_alloc((void**)&out->jc, sizeof(int64_t))) != CBX_OK ||
        (st = dev_alloc((void**)&out->ir, sizeof(int64_t))) != CBX_OK ||
        (st = dev_alloc(&out->val, sizeof(int64_t))) != CBX_OK) {
      cbx_dcsc_free(out);
      return st;
    }
    CBX_HIP(hipMemsetAsync(out->cp, 0, sizeof(int64_t), s));
    CBX_HIP(hipStreamSynchronize(s));
    return CBX_OK;
  }
  const int loops = remove_loops ? 1 : 0;
  switch (semiring * 8 + dtype) {
#define CBX_CO(SRK, SRE, T, DT) \
  case SRE * 8 + DT:            \
    return coo_typed<SRK, T>(m, n, rows, cols, (const T*)vals, nnz, loops, out, s);
    CBX_CO(kPlusTimes, CBX_SR_PLUS_TIMES, int64_t, CBX_I64)
    CBX_CO(kPlusTimes, CBX_SR_PLUS_TIMES, double, CBX_F64)
    CBX_CO(kPlusTimes, CBX_SR_PLUS_TIMES, float, CBX_F32)
    CBX_CO(kPlusTimes, CBX_SR_PLUS_TIMES, uint8_t, CBX_BOOL)
    CBX_CO(kMinPlus, CBX_SR_MIN_PLUS, int64_t, CBX_I64)
    CBX_CO(kMinPlus, CBX_SR_MIN_PLUS, double, CBX_F64)
    CBX_CO(kMinPlus, CBX_SR_MIN_PLUS, float, CBX_F32)
    CBX_CO(kSelectMax, CBX_SR_SELECT_MAX, int64_t, CBX_I64)
    CBX_CO(kSelectMax, CBX_SR_SELECT_MAX, double, CBX_F64)
    CBX_CO(kSelectMax, CBX_SR_SELECT_MAX, float, CBX_F32)
#undef CBX_CO
  }
  return set_error(CBX_ERR_UNSUPPORTED, "cbx_dcsc_from_coo: semiring %d with dtype %d is not provided", (int)semiring,
                   (int)dtype);
}
