// Batches of independent local products, the transpose, and the batched
// Galerkin triple product for gfx950.
//
// Many small products (one per stencil in a multigrid hierarchy, one per
// process block) are run as ONE product of block-diagonal operands: the
// batch is packed into a single DCSC with row and column offsets (one launch
// per array kind for the whole batch), every tier of the SpGEMM then runs
// once over all columns of all products, and the result is split back into
// per-product matrices with one launch per array kind.  Column results do
// not depend on which other columns share a launch, so each product is
// exactly what a separate call would return.
//
// Transpose (SpDCCols::Transpose, include/CombBLAS/SpDCCols.cpp:871-1011)
// sorts the entries by row with a (stable) device radix sort and rebuilds DCSC.
//
// Galerkin (ReleaseTests/GalerkinNew.cpp:94-112): T = R^T is given, S = T
// transposed, AT = A*T, SAT = S*AT, all with PlusTimes<double>.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>
#include <vector>

#include "cbx_device.h"
#include "cbx_spgemm.h"

namespace cbx {
namespace {

constexpr int kMaxBatch = 4096;

#define CBX_TRY(x)                 \
  do {                             \
    cbx_status st_ = (x);          \
    if (st_ != CBX_OK) return st_; \
  } while (0)

inline unsigned nblocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

struct OutSeg {
  int64_t* cp;
  int64_t* jc;
  int64_t* ir;
  void* val;
  int64_t row_off, col_off;
  int64_t nz_off, c_off, nnz, nzc;
};

// The last segment s with off(s) <= x among all, and this workgroup's: the
// number of segments that start at or before x (uniform; a barrier each 256).
template <class F>
__device__ __forceinline__ int find_seg(int count, int64_t x, F&& off) {
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off(mid) <= x) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}
template <class F>
__device__ __forceinline__ int block_find_seg(int count, int64_t x, F&& off) {
  int n = 0;
  for (int s0 = 0; s0 < count; s0 += 256) {
    const int s = s0 + (int)threadIdx.x;
    const int here = __syncthreads_count(s < count && off(s) <= x);
    n += here;
    if (here < 256) break;
  }
  return __builtin_amdgcn_readfirstlane(n - 1);
}

// Entries and columns are taken in tiles of one workgroup; nearly every tile
// lies in one member, whose pointers are then the same for all lanes and a
// thread's entries are in flight together.  (A search per entry, with one entry
// in flight, moved 1.3 TB/s.)
constexpr int kPackNT = 256, kPackPer = 8, kPackTile = kPackNT * kPackPer;

// chk: as in the product's validation, [0] violations, [1] descents of rows,
// [2] those at column starts.
template <class V>
__global__ __launch_bounds__(kPackNT) void k_pack_entries(const PackSeg* __restrict__ segs, int count, int64_t total,
                                                          int64_t* __restrict__ ir, int32_t* __restrict__ rows32,
                                                          V* __restrict__ val, unsigned long long* __restrict__ chk) {
  auto off = [&](int s) { return segs[s].nz_off; };
  long long bad = 0, desc = 0;
  for (int64_t e0 = blockIdx.x * (int64_t)kPackTile; e0 < total; e0 += gridDim.x * (int64_t)kPackTile) {
    const int s0 = block_find_seg(count, e0, off);
    const bool one = s0 + 1 == count || segs[s0 + 1].nz_off >= min(e0 + kPackTile, total);
    int64_t r[kPackPer], next[kPackPer];
    V v[kPackPer];
    if (one) {
      const PackSeg g = segs[s0];
      const int64_t i0 = e0 - g.nz_off, left = g.nnz - 1;
#pragma unroll
      for (int u = 0; u < kPackPer; ++u) {
        const int64_t i = i0 + u * kPackNT + threadIdx.x;
        r[u] = g.ir[min(i, left)];
        next[u] = g.ir[min(i + 1, left)];
        v[u] = ((const V*)g.val)[min(i, left)];
      }
#pragma unroll
      for (int u = 0; u < kPackPer; ++u) {
        pin(r[u]);
        pin(next[u]);
        pin(v[u]);
      }
#pragma unroll
      for (int u = 0; u < kPackPer; ++u) {
        const int64_t i = i0 + u * kPackNT + threadIdx.x;
        if (i > left) continue;
        bad += r[u] < 0 || r[u] >= g.m;
        desc += i < left && next[u] <= r[u];
        r[u] += g.row_off;
      }
    } else {
#pragma unroll
      for (int u = 0; u < kPackPer; ++u) {
        const int64_t e = e0 + u * kPackNT + threadIdx.x;
        if (e >= total) continue;
        const PackSeg& g = segs[find_seg(count, e, off)];
        const int64_t i = e - g.nz_off;
        r[u] = g.ir[i];
        v[u] = ((const V*)g.val)[i];
        bad += r[u] < 0 || r[u] >= g.m;
        desc += i + 1 < g.nnz && g.ir[i + 1] <= r[u];
        r[u] += g.row_off;
      }
    }
#pragma unroll
    for (int u = 0; u < kPackPer; ++u) {
      const int64_t e = e0 + u * kPackNT + threadIdx.x;
      if (e >= total) continue;
      if (ir) ir[e] = r[u];
      if (rows32) rows32[e] = (int32_t)r[u];
      val[e] = v[u];
    }
  }
  block_add_counts<kPackNT>(bad, desc, &chk[0], &chk[1]);
}

// The column arrays, and the check's rules for columns, of each member.
__global__ __launch_bounds__(kPackNT) void k_pack_cols(const PackSeg* __restrict__ segs, int count, int64_t total,
                                                       int64_t total_nnz, int64_t* __restrict__ cp,
                                                       int64_t* __restrict__ jc,
                                                       unsigned long long* __restrict__ chk) {
  constexpr int PER = 2;
  auto off = [&](int s) { return segs[s].c_off; };
  long long bad = 0, desc = 0;
  for (int64_t q0 = blockIdx.x * (int64_t)(kPackNT * PER); q0 < total; q0 += gridDim.x * (int64_t)(kPackNT * PER)) {
    const int s0 = block_find_seg(count, q0, off);
    const bool one = s0 + 1 == count || segs[s0 + 1].c_off >= min(q0 + kPackNT * PER, total);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int64_t q = q0 + u * kPackNT + threadIdx.x;
      if (q >= total) continue;
      const PackSeg& g = segs[one ? s0 : find_seg(count, q, off)];
      const int64_t i = q - g.c_off;
      const int64_t b = g.cp[i] - g.nz_base, e = g.cp[i + 1] - g.nz_base, j = g.jc[i] - g.col_base;
      bool err = b < 0 || e < b || e > g.nnz || j < 0 || j >= g.n || (i == 0 && b != 0) ||
                 (i + 1 == g.nzc && e != g.nnz);
      if (i + 1 < g.nzc) err |= g.jc[i + 1] - g.col_base <= j;
      bad += err;
      // a column start with another column's entry before it
      if (!err && i > 0 && b > 0 && b < g.nnz && g.cp[i - 1] - g.nz_base < b) desc += g.ir[b] <= g.ir[b - 1];
      cp[q] = b + g.nz_off;
      jc[q] = j + g.col_off;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) cp[total] = total_nnz;
  block_add_counts<kPackNT>(bad, desc, &chk[0], &chk[2]);
}

// qb[s] = first stored column of the packed matrix with column id >= bound[s].
__global__ void k_seg_bounds(const int64_t* __restrict__ jc, int64_t nzc, const int64_t* __restrict__ bound,
                             int count, const int64_t* __restrict__ cp, int64_t* __restrict__ qb,
                             int64_t* __restrict__ nzb) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s > count) return;
  const int64_t b = bound[s];
  int64_t lo = 0, hi = nzc;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (jc[mid] < b) lo = mid + 1;
    else hi = mid;
  }
  qb[s] = lo;
  nzb[s] = cp[lo];
}

template <class V>
__global__ __launch_bounds__(kPackNT) void k_unpack_entries(const OutSeg* __restrict__ segs, int count, int64_t total,
                                                            const int64_t* __restrict__ ir,
                                                            const V* __restrict__ val) {
  const int64_t e0 = blockIdx.x * (int64_t)kPackTile;
  auto off = [&](int s) { return segs[s].nz_off; };
  const int s0 = block_find_seg(count, e0, off);
  const bool one = s0 + 1 == count || segs[s0 + 1].nz_off >= min(e0 + kPackTile, total);
  int64_t r[kPackPer];
  V v[kPackPer];
#pragma unroll
  for (int u = 0; u < kPackPer; ++u) {
    const int64_t e = min(e0 + u * kPackNT + threadIdx.x, total - 1);
    r[u] = ir[e];
    v[u] = val[e];
  }
#pragma unroll
  for (int u = 0; u < kPackPer; ++u) {
    pin(r[u]);
    pin(v[u]);
  }
#pragma unroll
  for (int u = 0; u < kPackPer; ++u) {
    const int64_t e = e0 + u * kPackNT + threadIdx.x;
    if (e >= total) continue;
    const OutSeg& g = segs[one ? s0 : find_seg(count, e, off)];
    g.ir[e - g.nz_off] = r[u] - g.row_off;
    ((V*)g.val)[e - g.nz_off] = v[u];
  }
}

__global__ __launch_bounds__(256) void k_unpack_cols(const OutSeg* __restrict__ segs, int count, int64_t total,
                                                     const int64_t* __restrict__ cp, const int64_t* __restrict__ jc) {
  auto off = [&](int s) { return segs[s].c_off; };
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < total; q += (int64_t)gridDim.x * blockDim.x) {
    const int s = find_seg(count, q, off);
    const int64_t i = q - segs[s].c_off;
    segs[s].cp[i] = cp[q] - segs[s].nz_off;
    segs[s].jc[i] = jc[q] - segs[s].col_off;
  }
  // closing pointer of every product
  for (int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; s < count; s += (int64_t)gridDim.x * blockDim.x)
    segs[s].cp[segs[s].nzc] = segs[s].nnz;
}

// Transpose helpers.  The entries come ordered by column, so a stable sort by
// row alone puts them in the transpose's order: 32-bit keys of the row's bits
// (three passes up to 2^24 rows; seven over (row, column) keys of 64 bits took
// 0.43 ms for 4.7 M entries, these 0.20).  The payload is the entry's place
// and column.  G lanes take a column (a wave per column of 8 entries waited for
// its cp: 0.11 ms, now 0.02), up to 64 entries of it; the wave takes the rest of
// its longer columns together, four loads of a lane in flight.  (With sixteen
// lanes on the longest of R-MAT s18's columns, 15,803 entries where the mean is
// 26, the transpose took 0.65 ms; with a wave per column, one load in flight,
// 0.61; so 0.39.)
template <int G>
__global__ __launch_bounds__(256) void k_entry_keys(const int64_t* __restrict__ cp, const int64_t* __restrict__ jc,
                                                    const int64_t* __restrict__ ir, int64_t nzc,
                                                    uint32_t* __restrict__ key, uint64_t* __restrict__ from) {
  const int lane = lane_id();
  const int64_t q = (global_wave() * kWave + lane) / G;
  int64_t b = 0, end = 0;
  uint32_t c = 0;
  if (q < nzc) {
    b = cp[q];
    end = cp[q + 1];
    c = (uint32_t)jc[q];
  }
  const int64_t own = min(end, b + kWave);
  for (int64_t e = b + lane % G; e < own; e += G) {
    key[e] = (uint32_t)ir[e];
    from[e] = ((uint64_t)e << 32) | c;
  }
  unsigned long long more = __ballot(lane % G == 0 && own < end);
  while (more) {
    const int l = __ffsll(more) - 1;
    more &= more - 1;
    const int64_t e1 = readlane_ll(end, l);
    const uint64_t col = (uint32_t)__builtin_amdgcn_readlane((int)c, l);
    constexpr int U = 4;
    for (int64_t e0 = readlane_ll(own, l); e0 < e1; e0 += U * kWave) {
      int64_t r[U];
#pragma unroll
      for (int u = 0; u < U; ++u) r[u] = ir[min(e0 + u * kWave + lane, e1 - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) pin(r[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t e = e0 + u * kWave + lane;
        if (e >= e1) continue;
        key[e] = (uint32_t)r[u];
        from[e] = ((uint64_t)e << 32) | col;
      }
    }
  }
}

__global__ void k_col_heads(const uint32_t* __restrict__ key, int64_t nnz, int32_t* __restrict__ head) {
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e < nnz) head[e] = (e == 0 || key[e] != key[e - 1]) ? 1 : 0;
  if (e == nnz) head[e] = 0;
}

template <class V>
__global__ void k_transpose_write(const uint32_t* __restrict__ key, const uint64_t* __restrict__ from,
                                  const int32_t* __restrict__ hpos, int64_t nnz, const V* __restrict__ val,
                                  int64_t* __restrict__ ocp, int64_t* __restrict__ ojc, int64_t* __restrict__ oir,
                                  V* __restrict__ oval) {
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= nnz) return;
  const uint64_t f = from[e];
  oir[e] = (int64_t)(f & 0xffffffffull);
  oval[e] = val[f >> 32];
  if (hpos[e + 1] != hpos[e]) {
    ojc[hpos[e]] = (int64_t)key[e];
    ocp[hpos[e]] = e;
  }
  if (e == nnz - 1) ocp[hpos[nnz]] = nnz;
}

cbx_status alloc_dev_dcsc(cbx_dcsc* X, int64_t m, int64_t n, int64_t nnz, int64_t nzc, cbx_dtype dt,
                          bool rows = true) {
  std::memset(X, 0, sizeof(*X));
  X->m = m;
  X->n = n;
  X->nnz = nnz;
  X->nzc = nzc;
  X->dtype = dt;
  X->location = CBX_DEVICE;
  cbx_status st;
  if ((st = dev_alloc((void**)&X->cp, sizeof(int64_t) * (size_t)(nzc + 1))) ||
      (st = dev_alloc((void**)&X->jc, sizeof(int64_t) * (size_t)std::max<int64_t>(nzc, 1))) ||
      (rows && (st = dev_alloc((void**)&X->ir, sizeof(int64_t) * (size_t)std::max<int64_t>(nnz, 1)))) ||
      (st = dev_alloc(&X->val, dtype_size(dt) * (size_t)std::max<int64_t>(nnz, 1)))) {
    cbx_dcsc_free(X);
    return st;
  }
  return CBX_OK;
}

struct Owned {
  cbx_dcsc x{};
  ~Owned() { cbx_dcsc_free(&x); }
};

struct DevMem {
  void* p = nullptr;
  ~DevMem() { dev_free(p); }
  template <class X>
  cbx_status get(X** out, size_t count) {
    CBX_TRY(dev_alloc(&p, sizeof(X) * std::max<size_t>(count, 1)));
    *out = (X*)p;
    return CBX_OK;
  }
};

unsigned grid_for(int64_t n) { return (unsigned)std::min<int64_t>(std::max<int64_t>(nblocks(n, 256), 1), 65536); }

unsigned pack_tiles(int64_t total) { return nblocks(total, kPackTile); }
constexpr unsigned kPackGrid = 2048;  // checking workgroups (each adds to the counters once)

template <class V>
void launch_pack_entries(const PackSeg* segs, int count, const cbx_dcsc& out, int32_t* rows32,
                         unsigned long long* chk, hipStream_t s) {
  if (out.nnz)
    k_pack_entries<V><<<std::min(pack_tiles(out.nnz), kPackGrid), kPackNT, 0, s>>>(segs, count, out.nnz, out.ir, rows32, (V*)out.val, chk);
}

template <class V>
cbx_status launch_unpack_entries(const OutSeg* segs, int count, int64_t total, const int64_t* ir, const void* val,
                                 hipStream_t s) {
  if (total) k_unpack_entries<V><<<pack_tiles(total), kPackNT, 0, s>>>(segs, count, total, ir, (const V*)val);
  CBX_HIP(hipGetLastError());
  return CBX_OK;
}

__global__ void k_pack_begin(unsigned long long* __restrict__ chk) {
  if (threadIdx.x < 3) chk[threadIdx.x] = 0ull;
}

}  // namespace

cbx_status pack_members(const PackSeg* segs, int64_t count, const cbx_dcsc& out, int32_t* rows32, hipStream_t s) {
  for (int64_t i = 0; i < count; ++i)
    CBX_RETURN_IF(segs[i].nzc == 0 && segs[i].nnz != 0, CBX_ERR_INVALID, "cbx_dcsc_check: nnz without columns");
  DevMem dsegs, dchk;
  PackSeg* d;
  unsigned long long* chk;
  CBX_TRY(dsegs.get(&d, count));
  CBX_TRY(dchk.get(&chk, 3));
  CBX_HIP(hipMemcpyAsync(d, segs, sizeof(PackSeg) * count, hipMemcpyHostToDevice, s));
  k_pack_begin<<<1, 64, 0, s>>>(chk);
  k_pack_cols<<<std::min(std::max(nblocks(out.nzc, kPackNT * 2), 1u), kPackGrid), kPackNT, 0, s>>>(d, (int)count, out.nzc, out.nnz, out.cp,
                                                                            out.jc, chk);
  switch (dtype_size(out.dtype)) {
    case 8: launch_pack_entries<uint64_t>(d, (int)count, out, rows32, chk, s); break;
    case 4: launch_pack_entries<uint32_t>(d, (int)count, out, rows32, chk, s); break;
    default: launch_pack_entries<uint8_t>(d, (int)count, out, rows32, chk, s); break;
  }
  CBX_HIP(hipGetLastError());
  unsigned long long h[3] = {0, 0, 0};
  CBX_HIP(hipMemcpyAsync(h, chk, sizeof(h), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));  // the segment table and counters are released at return
  // (a member's descents at column starts are among its descents: the sums
  // agree only if every member's do)
  return h[0] || h[1] != h[2] ? set_error(CBX_ERR_INVALID, "cbx_dcsc_check: a member is malformed") : CBX_OK;
}

// Packs X[0..count) into one block-diagonal DCSC (rows and columns offset by
// the running sums of m and n); with rows32 its rows are written there, as 32
// bits, and it has no ir.
static cbx_status pack(const cbx_dcsc* X, int64_t count, cbx_dcsc* out, DevMem* rows32, int32_t** rows,
                       hipStream_t s) {
  std::vector<PackSeg> segs(count);
  int64_t m = 0, n = 0, nnz = 0, nzc = 0;
  for (int64_t i = 0; i < count; ++i) {
    segs[i] = PackSeg{X[i].cp, X[i].jc, X[i].ir, X[i].val, m, n, nnz, nzc, X[i].m, X[i].n, X[i].nnz, X[i].nzc,
                      0, 0};
    m += X[i].m;
    n += X[i].n;
    nnz += X[i].nnz;
    nzc += X[i].nzc;
  }
  CBX_TRY(alloc_dev_dcsc(out, m, n, nnz, nzc, X[0].dtype, rows32 == nullptr));
  if (rows32) CBX_TRY(rows32->get(rows, nnz));
  return pack_members(segs.data(), count, *out, rows32 ? *rows : nullptr, s);
}

// Splits a packed product into count matrices: product i owns the columns
// [col_bound[i], col_bound[i+1]) and rows offset by row_off[i].
static cbx_status unpack(const cbx_dcsc* P, int64_t count, const std::vector<int64_t>& col_bound,
                         const std::vector<int64_t>& row_off, const std::vector<int64_t>& ms,
                         const std::vector<int64_t>& ns, cbx_dcsc* out, hipStream_t s) {
  DevMem dbound, dqb, dnzb;
  int64_t *bound, *qb, *nzb;
  CBX_TRY(dbound.get(&bound, count + 1));
  CBX_TRY(dqb.get(&qb, count + 1));
  CBX_TRY(dnzb.get(&nzb, count + 1));
  CBX_HIP(hipMemcpyAsync(bound, col_bound.data(), sizeof(int64_t) * (count + 1), hipMemcpyHostToDevice, s));
  k_seg_bounds<<<nblocks(count + 1, 256), 256, 0, s>>>(P->jc, P->nzc, bound, (int)count, P->cp, qb, nzb);
  CBX_HIP(hipGetLastError());
  std::vector<int64_t> hqb(count + 1), hnzb(count + 1);
  CBX_HIP(hipMemcpyAsync(hqb.data(), qb, sizeof(int64_t) * (count + 1), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipMemcpyAsync(hnzb.data(), nzb, sizeof(int64_t) * (count + 1), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  std::vector<OutSeg> segs(count);
  for (int64_t i = 0; i < count; ++i) {
    const int64_t nzc = hqb[i + 1] - hqb[i], nnz = hnzb[i + 1] - hnzb[i];
    cbx_status st = alloc_dev_dcsc(&out[i], ms[i], ns[i], nnz, nzc, P->dtype);
    if (st) {
      for (int64_t k = 0; k < i; ++k) cbx_dcsc_free(&out[k]);
      return st;
    }
    segs[i] = OutSeg{out[i].cp, out[i].jc, out[i].ir, out[i].val, row_off[i], col_bound[i],
                     hnzb[i], hqb[i], nnz, nzc};
  }
  DevMem dsegs;
  OutSeg* d;
  CBX_TRY(dsegs.get(&d, count));
  CBX_HIP(hipMemcpyAsync(d, segs.data(), sizeof(OutSeg) * count, hipMemcpyHostToDevice, s));
  k_unpack_cols<<<grid_for(std::max<int64_t>(P->nzc, count)), 256, 0, s>>>(d, (int)count, P->nzc, P->cp, P->jc);
  CBX_HIP(hipGetLastError());
  switch (dtype_size(P->dtype)) {
    case 8: CBX_TRY(launch_unpack_entries<uint64_t>(d, (int)count, P->nnz, P->ir, P->val, s)); break;
    case 4: CBX_TRY(launch_unpack_entries<uint32_t>(d, (int)count, P->nnz, P->ir, P->val, s)); break;
    default: CBX_TRY(launch_unpack_entries<uint8_t>(d, (int)count, P->nnz, P->ir, P->val, s)); break;
  }
  CBX_HIP(hipStreamSynchronize(s));
  return CBX_OK;
}

template <class V>
static cbx_status transpose_typed(const cbx_dcsc* X, cbx_dcsc* out, hipStream_t s) {
  const int64_t nnz = X->nnz, nzc = X->nzc;
  DevMem dk0, dk1, df0, df1, dh, dhp, dtmp;
  uint32_t *k0, *k1;
  uint64_t *f0, *f1;
  int32_t *head, *hpos;
  CBX_TRY(dk0.get(&k0, nnz));
  CBX_TRY(dk1.get(&k1, nnz));
  CBX_TRY(df0.get(&f0, nnz));
  CBX_TRY(df1.get(&f1, nnz));
  CBX_TRY(dh.get(&head, nnz + 1));
  CBX_TRY(dhp.get(&hpos, nnz + 1));
  if (nzc && nnz / nzc < 8) k_entry_keys<4><<<wave_grid((nzc + 15) / 16), 256, 0, s>>>(X->cp, X->jc, X->ir, nzc, k0, f0);
  else if (nzc && nnz / nzc < 32)
    k_entry_keys<16><<<wave_grid((nzc + 3) / 4), 256, 0, s>>>(X->cp, X->jc, X->ir, nzc, k0, f0);
  else if (nzc)
    k_entry_keys<kWave><<<wave_grid(nzc), 256, 0, s>>>(X->cp, X->jc, X->ir, nzc, k0, f0);
  CBX_HIP(hipGetLastError());
  int rbits = 1;
  while (rbits < 31 && ((int64_t)1 << rbits) < X->m) ++rbits;
  size_t tb = 0, tb2 = 0;
  hipcub::DoubleBuffer<uint32_t> keys(k0, k1);
  hipcub::DoubleBuffer<uint64_t> from(f0, f1);
  CBX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, keys, from, (int)nnz, 0, rbits, s));
  CBX_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb2, head, hpos, (int)(nnz + 1), s));
  uint8_t* tmp;
  CBX_TRY(dtmp.get(&tmp, std::max(tb, tb2)));
  tb = std::max(tb, tb2);
  CBX_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, keys, from, (int)nnz, 0, rbits, s));
  k_col_heads<<<nblocks(nnz + 1, 256), 256, 0, s>>>(keys.Current(), nnz, head);
  CBX_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tb, head, hpos, (int)(nnz + 1), s));
  int32_t ncols = 0;
  CBX_HIP(hipMemcpyAsync(&ncols, hpos + nnz, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  CBX_TRY(alloc_dev_dcsc(out, X->n, X->m, nnz, ncols, X->dtype));
  if (nnz)
    k_transpose_write<V><<<nblocks(nnz, 256), 256, 0, s>>>(keys.Current(), from.Current(), hpos, nnz,
                                                         (const V*)X->val, out->cp, out->jc, out->ir, (V*)out->val);
  else
    CBX_HIP(hipMemsetAsync(out->cp, 0, sizeof(int64_t), s));
  CBX_HIP(hipGetLastError());
  CBX_HIP(hipStreamSynchronize(s));
  return CBX_OK;
}

static cbx_status transpose(const cbx_dcsc* X, cbx_dcsc* out, hipStream_t s) {
  switch (dtype_size(X->dtype)) {
    case 8: return transpose_typed<uint64_t>(X, out, s);
    case 4: return transpose_typed<uint32_t>(X, out, s);
    default: return transpose_typed<uint8_t>(X, out, s);
  }
}

static void add_stats(cbx_spgemm_stats* acc, const cbx_spgemm_stats& s) {
  acc->flops += s.flops;
  acc->nnz += s.nnz;
  acc->nzc += s.nzc;
  acc->overflow_cols += s.overflow_cols;
  acc->predicted_nnz += s.predicted_nnz;
  acc->learned_fallback += s.learned_fallback;
  acc->units_light += s.units_light;
  acc->units_heavy += s.units_heavy;
  acc->nnz_main += s.nnz_main;
  acc->ms_setup += s.ms_setup;
  acc->ms_symbolic += s.ms_symbolic;
  acc->ms_alloc += s.ms_alloc;
  acc->ms_numeric += s.ms_numeric;
  acc->ms_main_kernel += s.ms_main_kernel;
}

static cbx_status check_batch(int64_t count, const cbx_dcsc* X, const char* name) {
  CBX_RETURN_IF(count < 1 || count > kMaxBatch, CBX_ERR_LIMIT, "batch size must be in [1, %d]", kMaxBatch);
  CBX_RETURN_IF(!X, CBX_ERR_INVALID, "%s is null", name);
  int64_t nnz = 0, m = 0, n = 0;
  for (int64_t i = 0; i < count; ++i) {
    CBX_TRY(check_dcsc(&X[i], name, CBX_DEVICE));
    CBX_RETURN_IF(X[i].dtype != X[0].dtype, CBX_ERR_UNSUPPORTED, "%s: batch members must share a dtype", name);
    nnz += X[i].nnz;
    m += X[i].m;
    n += X[i].n;
  }
  CBX_RETURN_IF(nnz >= (1ll << 31) || m >= (1ll << 31) || n >= (1ll << 31), CBX_ERR_LIMIT,
                "%s: the packed batch must hold fewer than 2^31 rows, columns and nonzeros", name);
  return CBX_OK;
}

static cbx_status spgemm_batched(int64_t count, const cbx_dcsc* A, const cbx_dcsc* B, cbx_semiring sr,
                                 cbx_spgemm_mode mode, const SpgemmConfig& cfg, cbx_dcsc* C,
                                 cbx_spgemm_stats* st, hipStream_t s) {
  Owned PA, PB, PC;
  DevMem rows;
  int32_t* rows_a = nullptr;
  CBX_TRY(pack(A, count, &PA.x, &rows, &rows_a, s));
  CBX_TRY(pack(B, count, &PB.x, nullptr, nullptr, s));
  SpgemmConfig packed = cfg;
  packed.trusted_a = packed.trusted_b = true;
  packed.rows_a = rows_a;
  cbx_spgemm_stats one;
  CBX_TRY(spgemm_dispatch(&PA.x, &PB.x, sr, mode, packed, &PC.x, &one, s));
  add_stats(st, one);
  std::vector<int64_t> bound(count + 1, 0), roff(count, 0), ms(count), ns(count);
  for (int64_t i = 0; i < count; ++i) {
    bound[i + 1] = bound[i] + B[i].n;
    roff[i] = i ? roff[i - 1] + A[i - 1].m : 0;
    ms[i] = A[i].m;
    ns[i] = B[i].n;
  }
  return unpack(&PC.x, count, bound, roff, ms, ns, C, s);
}

static cbx_status galerkin_batched(int64_t count, const cbx_dcsc* A, const cbx_dcsc* T, const SpgemmConfig& cfg,
                                   cbx_dcsc* SAT, cbx_spgemm_stats* st, hipStream_t s) {
  Owned PA, PT, PS, PAT, PSAT;
  DevMem rows;
  int32_t* rows_a = nullptr;
  CBX_TRY(pack(A, count, &PA.x, &rows, &rows_a, s));
  CBX_TRY(pack(T, count, &PT.x, nullptr, nullptr, s));
  CBX_TRY(transpose(&PT.x, &PS.x, s));
  cbx_spgemm_stats one;
  // the packed operands are checked; S (a transpose) and A*T (a product) come from this library
  SpgemmConfig cfg2 = cfg;
  cfg2.trusted_a = cfg2.trusted_b = true;
  SpgemmConfig packed = cfg2;
  packed.rows_a = rows_a;
  CBX_TRY(spgemm_dispatch(&PA.x, &PT.x, CBX_SR_PLUS_TIMES, CBX_SPGEMM_TWO_PHASE, packed, &PAT.x, &one, s));
  add_stats(st, one);
  CBX_TRY(spgemm_dispatch(&PS.x, &PAT.x, CBX_SR_PLUS_TIMES, CBX_SPGEMM_TWO_PHASE, cfg2, &PSAT.x, &one, s));
  add_stats(st, one);
  std::vector<int64_t> bound(count + 1, 0), roff(count, 0), ms(count), ns(count);
  for (int64_t i = 0; i < count; ++i) {
    bound[i + 1] = bound[i] + T[i].n;
    roff[i] = bound[i];
    ms[i] = T[i].n;
    ns[i] = T[i].n;
  }
  return unpack(&PSAT.x, count, bound, roff, ms, ns, SAT, s);
}

}  // namespace cbx

using namespace cbx;

namespace {
struct Span {
  hipEvent_t a = nullptr, b = nullptr;
  hipStream_t s;
  explicit Span(hipStream_t st) : s(st) {
    (void)hipEventCreate(&a);
    (void)hipEventCreate(&b);
    (void)hipEventRecord(a, s);
  }
  double stop() {
    float f = 0;
    (void)hipEventRecord(b, s);
    (void)hipEventSynchronize(b);
    (void)hipEventElapsedTime(&f, a, b);
    return f;
  }
  ~Span() {
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
  }
};
}  // namespace

extern "C" cbx_status cbx_dcsc_transpose(const cbx_dcsc* X, cbx_dcsc* out, void* stream) {
  cbx_status st;
  if ((st = check_dcsc(X, "X", CBX_DEVICE))) return st;
  CBX_RETURN_IF(!out, CBX_ERR_INVALID, "cbx_dcsc_transpose: out is null");
  CBX_RETURN_IF(X->nnz >= (1ll << 31), CBX_ERR_LIMIT, "cbx_dcsc_transpose: at most 2^31-1 nonzeros");
  if ((st = init_device_once())) return st;
  return transpose(X, out, (hipStream_t)stream);
}

extern "C" cbx_status cbx_spgemm_batched(int64_t count, const cbx_dcsc* A, const cbx_dcsc* B, cbx_semiring semiring,
                                         cbx_spgemm_mode mode, cbx_dcsc* C, cbx_spgemm_stats* stats, void* stream) {
  cbx_status st;
  if ((st = check_batch(count, A, "A")) || (st = check_batch(count, B, "B"))) return st;
  CBX_RETURN_IF(!C, CBX_ERR_INVALID, "cbx_spgemm_batched: C is null");
  for (int64_t i = 0; i < count; ++i)
    CBX_RETURN_IF(A[i].n != B[i].m, CBX_ERR_INVALID, "cbx_spgemm_batched: product %lld: inner dimensions differ",
                  (long long)i);
  CBX_RETURN_IF(A[0].dtype != B[0].dtype, CBX_ERR_UNSUPPORTED, "cbx_spgemm_batched: A and B must share a dtype");
  CBX_RETURN_IF(mode != CBX_SPGEMM_TWO_PHASE && mode != CBX_SPGEMM_UNSORTED && mode != CBX_SPGEMM_LEARNED,
                CBX_ERR_INVALID, "cbx_spgemm_batched: unknown mode %d", (int)mode);
  if ((st = init_device_once())) return st;
  SpgemmConfig cfg = current_config();
  CBX_RETURN_IF(mode == CBX_SPGEMM_LEARNED && !cfg.predictor && cfg.sampling_rounds == 0, CBX_ERR_INVALID,
                "cbx_spgemm_batched: learned mode needs a predictor (cbx_spgemm_set_predictor)");
  cbx_spgemm_stats local;
  cbx_spgemm_stats* sp = stats ? stats : &local;
  std::memset(sp, 0, sizeof(*sp));
  for (int64_t i = 0; i < count; ++i) std::memset(&C[i], 0, sizeof(cbx_dcsc));
  Span span((hipStream_t)stream);
  st = spgemm_batched(count, A, B, semiring, mode, cfg, C, sp, (hipStream_t)stream);
  sp->ms_total = span.stop();
  return st;
}

extern "C" cbx_status cbx_galerkin_batched(int64_t count, const cbx_dcsc* A, const cbx_dcsc* T, cbx_dcsc* SAT,
                                           cbx_spgemm_stats* stats, void* stream) {
  cbx_status st;
  if ((st = check_batch(count, A, "A")) || (st = check_batch(count, T, "T"))) return st;
  CBX_RETURN_IF(!SAT, CBX_ERR_INVALID, "cbx_galerkin_batched: SAT is null");
  CBX_RETURN_IF(A[0].dtype != CBX_F64 && A[0].dtype != CBX_F32, CBX_ERR_UNSUPPORTED,
                "cbx_galerkin_batched: values must be float64 or float32");
  CBX_RETURN_IF(A[0].dtype != T[0].dtype, CBX_ERR_UNSUPPORTED, "cbx_galerkin_batched: A and T must share a dtype");
  for (int64_t i = 0; i < count; ++i)
    CBX_RETURN_IF(A[i].m != A[i].n || A[i].n != T[i].m, CBX_ERR_INVALID,
                  "cbx_galerkin_batched: product %lld: A must be square with as many rows as T", (long long)i);
  if ((st = init_device_once())) return st;
  SpgemmConfig cfg = current_config();
  cbx_spgemm_stats local;
  cbx_spgemm_stats* sp = stats ? stats : &local;
  std::memset(sp, 0, sizeof(*sp));
  for (int64_t i = 0; i < count; ++i) std::memset(&SAT[i], 0, sizeof(cbx_dcsc));
  Span span((hipStream_t)stream);
  st = galerkin_batched(count, A, T, cfg, SAT, sp, (hipStream_t)stream);
  sp->ms_total = span.stop();
  return st;
}
