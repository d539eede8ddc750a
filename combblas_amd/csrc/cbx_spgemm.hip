// Local semiring SpGEMM C = A*B on DCSC blocks for gfx950.
//
// Replaces CombBLAS's LocalHybridSpGEMM<SR,NTO> (include/CombBLAS/mtSpGEMM.h:213-460)
// and LocalSpGEMMHash (mtSpGEMM.h:463-656).  The reference runs, per
// non-empty column j of B:
//   estimateFLOP     flop_j = sum_{k in B(:,j)} nnz(A(:,k))      (mtSpGEMM.h:1057-1134)
//   estimateNNZ_Hash nnz_j  = distinct rows of the products       (mtSpGEMM.h:806-933)
//   prefixsum        column pointers of C                          (mtSpGEMM.h:23-70)
//   numeric          heap merge or hash + sort, rows ascending     (mtSpGEMM.h:289-441)
// This file keeps those phases but maps them to the GPU as follows.
//
// Column tiers (by flop_j, after sorting columns by flop descending):
//   tiny tier  flop_j <= tiny_flop: one wave per column (k_tiny).
//   sort tier  flop_j <= small_flop_max: one workgroup per column; the rows
//              are counted in an LDS linear-probing hash table, and the
//              products sorted by row in LDS (k_num_sort).
//   unit tier  the rest: a symbolic pass cuts each column into row ranges
//              (units) of one workgroup each, which accumulate in LDS.  The
//              A entries of a row range are found through a precomputed
//              tile-pointer table.  (Matrices taller than 2^24 rows walk
//              dense row tiles per column instead.)
// The A-column segments of a workgroup's B entries are flattened, so that all
// lanes work on products even when most segments are short (R-MAT columns
// are).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <type_traits>
#include <cstdint>
#include <cstring>
#include <vector>

#include "cbx_device.h"
#include "cbx_flatten.h"
#include "cbx_index.h"
#include "cbx_semiring.h"
#include "cbx_spgemm.h"

namespace cbx {

// ------------------------------------------------------------------ utils
template <class T>
__device__ __forceinline__ T shfl_any(T v, int src) {
  if constexpr (sizeof(T) == 8) {
    long long x = __builtin_bit_cast(long long, v);
    x = __shfl(x, src, kWave);
    return __builtin_bit_cast(T, x);
  } else if constexpr (sizeof(T) == 4) {
    int x = __builtin_bit_cast(int, v);
    x = __shfl(x, src, kWave);
    return __builtin_bit_cast(T, x);
  } else {
    int x = (int)v;
    x = __shfl(x, src, kWave);
    return (T)x;
  }
}

// Visits the A entries of up to 64 segments, one segment per lane
// ([lo, lo+len) with multiplier bv).  All lanes of the wave must call it.
// f(idx, bv) runs once per entry; entries are spread over all lanes.
template <class T, class F>
__device__ __forceinline__ void wave_visit(int64_t lo, int len, T bv, F&& f) {
  const int lane = lane_id();
  const int incl = wave_incl_scan(len);
  const int total = __shfl(incl, kWave - 1, kWave);
  const int excl = incl - len;
  for (int tb = 0; tb < total; tb += kWave) {
    const int t = tb + lane;
    int L = 0;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) {
      const int cand = L + step;
      const int ex = __shfl(excl, cand, kWave);
      if (ex <= t) L = cand;
    }
    const int64_t loL = shfl_any(lo, L);
    const int exL = __shfl(excl, L, kWave);
    const T bvL = shfl_any(bv, L);
    if (t < total) f(loL + (int64_t)(t - exL), bvL);
  }
}

__device__ __forceinline__ uint32_t hash_slot(int32_t r, int lg) {
  return ((uint32_t)r * 2654435761u) >> (32 - lg);
}

__device__ __forceinline__ int ceil_log2_dev(long long x) {
  int lg = 0;
  while ((1ll << lg) < x) ++lg;
  return lg;
}

// ============================================================ unit tier
// Row-range units.  The symbolic pass builds, per column, the full presence
// bitmap of its output rows in LDS, counts the rows of every block of kBR
// rows, and cuts the column into units: runs of consecutive blocks holding
// at most KMAX outputs and spanning at most RBLK blocks.  The numeric pass
// runs one workgroup per unit.  A unit's accumulator is compact: the value of
// row r lives at rank(r) = number of output rows of the unit below r, read
// from the unit's presence bitmap with per-word prefix counts, so the unit
// is emitted in row order without sorting and LDS holds only real outputs.
constexpr int kBR = 4096;        // rows per block (also the tile-pointer granularity)
constexpr int kBRW = kBR / 32;   // 32-bit bitmap words per block
// Row lists (k_sym_units) cover the blocks with at most this many outputs:
// sixteen denser blocks already fill a small unit, so a unit holding a
// denser block spans at most 16 blocks and takes its ranks from a bitmap.
constexpr int kListBlockMax = 256;

struct Unit {
  int32_t col;     // B stored-column position
  int32_t blk_lo;  // first block
  int32_t blk_hi;  // one past the last block
  int32_t cnt;     // outputs in the unit
  int32_t off;     // offset of the unit's first output within the column
  int32_t slot;    // the column's row-map slot (its workgroup in the symbolic launch)
};

// The unit of workgroup b (of n) when runs of g consecutive units go to one
// XCD.  The hardware deals a launch's workgroups to the 8 XCDs in turn
// (workgroup b runs on XCD b % 8), so with units sorted by row block the
// identity mapping spreads every row band over all eight L2 caches; here,
// within each super-group of 8g workgroups, XCD x takes units x*g .. x*g+g-1,
// and the runs still interleave across the XCDs.  The tail after the last
// full super-group keeps the identity; g = 0 is the identity.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_unit(int b, int n, int g) {
  if (g <= 0) return b;
  const int sg = kXcds * g;
  if (b >= n / sg * sg) return b;
  const int r = b % sg;
  return b - r + (r % kXcds) * g + r / kXcds;
}

// Fused threshold of the MCL expansion (MCLPruneRecoverySelect's hard
// threshold, ParFriends.h:185-345, when no column can need recovery): with
// `on`, the numeric kernels emit only the entries with !(v < thr) of every
// output range they own, compacted at the range's start, and append the
// range (start, kept count, column) to a run list; the host code then gathers
// the runs into the product.  The epilogue on that product keeps exactly what
// it keeps on the unfiltered one (its statistics count only entries > thr and
// its cuts are never below thr), and the product's writes shrink to the kept
// entries.
template <class T>
struct Filter {
  int on = 0;
  T thr{};
  int64_t* run_src = nullptr;
  int32_t* run_kept = nullptr;
  int32_t* run_col = nullptr;
  int* run_count = nullptr;
  int run_cap = 0;
  // entries the staged tiny tier left out (its kept counts size the columns,
  // so the product's unfiltered size is the scan's total plus these)
  unsigned long long* dropped = nullptr;
};

template <class T>
__device__ __forceinline__ void filter_add_run(const Filter<T>& f, int64_t src, int kept, int col, int* err) {
  if (kept <= 0) return;
  const int k = atomicAdd(f.run_count, 1);
  if (k < f.run_cap) {
    f.run_src[k] = src;
    f.run_kept[k] = kept;
    f.run_col[k] = col;
  } else {
    atomicOr(err, 1024);
  }
}

// Writes the kept ones (!(v < thr)) of the items i in [0, n) that item(i, v)
// has, in order and with their rows row_of(i), at `out` (at most cap of them),
// and appends the range to the run list.  Every wave takes one contiguous share of the
// items and goes over it twice, counting and then writing, with one barrier
// between.  `isum`: LDS that no thread still reads.
template <class T, int NT, class G, class R>
__device__ __forceinline__ void emit_filtered(int n, int cap, G&& item, R&& row_of, int64_t out, int64_t* __restrict__ irC,
                                              T* __restrict__ valC, const Filter<T>& flt, int col, int* isum,
                                              int* err) {
  constexpr int NW = NT / kWave;
  const int w = wave_id_uniform(), lane = lane_id();
  const int share = (n + NT - 1) / NT * kWave;
  const int i0 = w * share, i1 = min(n, i0 + share);
  int count = 0;
  for (int i = i0; i < i1; i += kWave) {
    T v{};
    const bool keep = i + lane < i1 && item(i + lane, v) && !(v < flt.thr);
    count += __popcll(__ballot(keep));
  }
  if (lane == 0) isum[w] = count;
  __syncthreads();
  const int incl = wave_incl_scan(lane < NW ? isum[lane] : 0);
  int pos = w ? __builtin_amdgcn_readlane(incl, w - 1) : 0;
  const int total = __builtin_amdgcn_readlane(incl, NW - 1);
  if (count)
    for (int i = i0; i < i1; i += kWave) {
      T v{};
      const bool keep = i + lane < i1 && item(i + lane, v) && !(v < flt.thr);
      const unsigned long long m = __ballot(keep);
      const int at = pos + __popcll(m & ((1ull << lane) - 1ull));
      if (keep && at < cap) {
        irC[out + at] = row_of(i + lane);
        valC[out + at] = v;
      }
      pos += __popcll(m);
    }
  if (threadIdx.x == 0) filter_add_run(flt, out, min(total, cap), col, err);
}

// Tile pointers of the unit tier: at[t * ncols + p] is the index of the first
// entry of A's p-th stored column with row >= t * kBR (t = 0 .. S; the index
// runs over all of A's entries).  Tile-major: the units in flight share a few
// tiles (they are sorted by first block), so a look-up's lines stay in the
// L2 caches (4 B per stored column and tile, 1.4 MB at R-MAT s19).  Stored
// column by column, every look-up fetched a line of its own for two of its
// words, and the column's start another.
struct Tiles {
  const int32_t* at = nullptr;
  int64_t ncols = 0;
};

// Segment of B entry e restricted to tiles [t_lo, t_hi) (or the whole A
// column when `full`).
template <class T, bool VAL>
__device__ __forceinline__ void load_seg(int64_t e, int64_t b1, const int32_t* __restrict__ bpos,
                                         const int64_t* __restrict__ cpA, const Tiles& P, int t_lo, int t_hi,
                                         bool full, const T* __restrict__ valB, int64_t& base, int& len, T& bv) {
  base = 0;
  len = 0;
  bv = T{};
  if (e < b1) {
    const int32_t p = bpos[e];
    if (p >= 0) {
      if (full) {
        base = cpA[p];
        len = (int)(cpA[p + 1] - base);
      } else {
        const int32_t a0 = P.at[t_lo * P.ncols + p];
        base = a0;
        len = P.at[t_hi * P.ncols + p] - a0;
      }
      if constexpr (VAL) bv = valB[e];
    }
  }
}

// Rows (less row0) and values of U entries of A, all loads in flight together.
template <int U>
__device__ __forceinline__ void load_rows(const int32_t* __restrict__ rowsA, int32_t row0, const int32_t (&idx)[U],
                                          int32_t (&r)[U]) {
#pragma unroll
  for (int u = 0; u < U; ++u) r[u] = rowsA[idx[u]];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    pin(r[u]);
    r[u] -= row0;
  }
}
template <class T, int U>
__device__ __forceinline__ void load_entries(const int32_t* __restrict__ rowsA, const T* __restrict__ valA,
                                             int32_t row0, const int32_t (&idx)[U], T (&bvs)[U], int32_t (&r)[U],
                                             T (&a)[U]) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    r[u] = rowsA[idx[u]];
    a[u] = valA[idx[u]];
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    pin(r[u]);
    pin(a[u]);
    pin(bvs[u]);
    r[u] -= row0;
  }
}

// Lanes of the wave with the same value of the low `width` bits of d, among
// `valid` ones.
__device__ __forceinline__ unsigned long long wave_match(uint32_t d, int width, unsigned long long valid) {
  unsigned long long same = valid;
  for (int b = 0; b < width; ++b) {
    const bool bit = (d >> b) & 1u;
    const unsigned long long m = __ballot(bit);
    same &= bit ? m : ~m;
  }
  return same;
}

// ------------------------------------------------------------------ setup
__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Input validation (the reference's preconditions, mtSpGEMM.h / dcsc.h):
// cp starts at 0, ends at nnz and never decreases (empty columns allowed); jc
// strictly increasing and below ncols; rows of every column strictly
// increasing and below nrows.  One fully parallel pass: per entry, rows in
// range and every adjacent descent ir[e+1] <= ir[e] counted; per column, cp
// and jc, and the descents at the positions where a column begins (each
// distinct start counted once).  With cp valid those are the only places a
// descent is allowed, so the rows ascend within columns iff the two counts
// agree.  cnt[0] violations, cnt[1] descents, cnt[2] descents at starts.
// With rows32 the pass also writes the rows as 32-bit (garbage where a row is
// out of range; nothing uses it then): one reading of ir instead of two.
constexpr int kValNT = 256, kValBlocks = 2048, kValPer = 4;  // kValPer entries of a thread in flight together

__global__ __launch_bounds__(kValNT) void k_validate(const int64_t* __restrict__ cp, const int64_t* __restrict__ jc,
                                                     const int64_t* __restrict__ ir, int64_t nzc, int64_t nnz,
                                                     int64_t nrows, int64_t ncols, int eblocks,
                                                     int32_t* __restrict__ rows32,
                                                     unsigned long long* __restrict__ cnt) {
  long long bad = 0, desc = 0;
  if ((int)blockIdx.x < eblocks) {  // entries
    const int64_t stride = (int64_t)eblocks * (kValNT * kValPer);
    for (int64_t e0 = blockIdx.x * (int64_t)(kValNT * kValPer); e0 < nnz; e0 += stride) {
      int64_t r[kValPer], next[kValPer];
#pragma unroll
      for (int u = 0; u < kValPer; ++u) {
        const int64_t e = e0 + u * kValNT + threadIdx.x;
        r[u] = ir[min(e, nnz - 1)];
        next[u] = ir[min(e + 1, nnz - 1)];
      }
#pragma unroll
      for (int u = 0; u < kValPer; ++u) {
        pin(r[u]);
        pin(next[u]);
      }
#pragma unroll
      for (int u = 0; u < kValPer; ++u) {
        const int64_t e = e0 + u * kValNT + threadIdx.x;
        bad += e < nnz && (r[u] < 0 || r[u] >= nrows);
        desc += e + 1 < nnz && next[u] <= r[u];
        if (rows32 && e < nnz) rows32[e] = (int32_t)r[u];
      }
    }
    block_add_counts<kValNT>(bad, desc, &cnt[0], &cnt[1]);
  } else {  // columns
    const int64_t stride = (int64_t)(gridDim.x - eblocks) * kValNT;
    for (int64_t q = ((int64_t)blockIdx.x - eblocks) * kValNT + threadIdx.x; q < nzc; q += stride) {
      const int64_t b = cp[q], e = cp[q + 1], j = jc[q];
      bool err = b < 0 || e < b || e > nnz || j < 0 || j >= ncols;
      if (q + 1 < nzc) err |= jc[q + 1] <= j;
      if (q == 0) err |= b != 0;
      if (q == nzc - 1) err |= e != nnz;
      bad += err;
      if (!err && q > 0 && b > 0 && b < nnz && cp[q - 1] < b) desc += ir[b] <= ir[b - 1];
    }
    block_add_counts<kValNT>(bad, desc, &cnt[0], &cnt[2]);
  }
}

__device__ __forceinline__ bool counts_valid(const unsigned long long* cnt) {
  return cnt[0] == 0 && cnt[1] == cnt[2];
}

__global__ void k_validate_flag(const unsigned long long* __restrict__ cnt, int flagbit, int* __restrict__ err) {
  if (threadIdx.x == 0 && !counts_valid(cnt)) atomicOr(err, 1 << flagbit);
}

// Launches the validation of X on s; cnt: 3 device counters, cleared before.
static cbx_status launch_validate(const cbx_dcsc* X, int32_t* rows32, unsigned long long* cnt, hipStream_t s) {
  auto blocks = [](int64_t n, int per) {
    return (unsigned)std::min<int64_t>(std::max<int64_t>((n + kValNT * per - 1) / (kValNT * per), 1), kValBlocks);
  };
  const unsigned eb = blocks(X->nnz, kValPer);
  k_validate<<<eb + blocks(X->nzc, 1), kValNT, 0, s>>>(X->cp, X->jc, X->ir, X->nzc, X->nnz, X->m, X->n, (int)eb, rows32,
                                                    cnt);
  CBX_HIP(hipGetLastError());
  return CBX_OK;
}

// 32-bit rows alone, for operands that need no validation.
__global__ void k_rows32(const int64_t* __restrict__ ir, int64_t nnz, int32_t* __restrict__ out) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < nnz) out[i] = (int32_t)ir[i];
}

// Columns by their products, largest class first: 0 beyond unit_split_nnz
// (large units possible), 1 the other unit-tier columns, 2..4 the sort tier's
// three workgroup sizes, 5 tiny, 6 empty.
struct FlopClasses {
  int64_t split, small, s4k, mid, tiny;  // lower bounds (exclusive) of classes 0 .. 4
  int64_t list_cap;                      // row-list region of a unit-tier column: min(flop, list_cap)
};
constexpr int kClasses = 7, kDigits = kClasses * 32;

// The column's class and, within it, 32 steps by size: the sort digit, small
// for large columns.
__device__ __forceinline__ int flop_digit(const FlopClasses& c, int64_t f) {
  auto octaves = [](int64_t f, int64_t lo) {  // half octaves above lo
    const int l = 63 - __clzll((unsigned long long)f), l0 = 63 - __clzll((unsigned long long)(lo | 1));
    return min(31, max(0, 2 * (l - l0) + (int)((f >> max(l - 1, 0)) & 1)));
  };
  int cls, sub = 0;
  if (f > c.split) cls = 0, sub = octaves(f, c.split);
  else if (f > c.small) cls = 1, sub = octaves(f, c.small);
  else if (f > c.s4k) cls = 2, sub = (int)(f >> 7);
  else if (f > c.mid) cls = 3, sub = (int)(f >> 6);
  else if (f > c.tiny) cls = 4, sub = (int)(f >> 5);
  else if (f > 0) cls = 5, sub = (int)(f >> 3);
  else cls = 6;
  return cls * 32 + 31 - min(31, sub);
}

// Device-side counters of one product, cleared together before it starts.
struct Counters {
  int err;
  int units[3];                     // small (bitmap), large, and small list units
  unsigned long long val[6];        // validation of A and of B
  unsigned int digits[kDigits];     // columns of each sort digit
  unsigned int cursor[kDigits];     // of them placed so far
  unsigned long long flops, tiny_flops, list_rows;  // totals: products, those of tiny columns, list regions
  unsigned long long tiny_at, list_at;              // of the latter two, handed out so far
  unsigned long long main_nnz;                      // outputs of the unit-tier columns
  unsigned long long dropped;                       // fused threshold: entries the staged tiny tier left out
  int runs;                                         // fused threshold: ranges appended
};

// What the host waits for, written by a kernel into pinned memory: after the
// setup, after the symbolic pass, at the end.
struct Report {
  int err, units[3];
  int64_t columns[kClasses];
  int64_t flops, tiny_flops, list_rows;
  int64_t nnz, nzc, main_nnz, dropped;
};

__global__ __launch_bounds__(256) void k_init(Counters* __restrict__ c, int32_t* __restrict__ colmap, int64_t n,
                                              int64_t* __restrict__ flop, int64_t* __restrict__ nnzcol, int64_t nzcB) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x, t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  for (int64_t i = t; i < (int64_t)(sizeof(Counters) / 4); i += stride) reinterpret_cast<uint32_t*>(c)[i] = 0;
  if (colmap)
    for (int64_t i = t; i < n; i += stride) colmap[i] = -1;
  for (int64_t i = t; i <= nzcB; i += stride) {
    flop[i] = 0;
    nnzcol[i] = 0;
  }
}

// colmap[jcA[p]] = p  (dense lookup replacing Dcsc::ConstructAux/FillColInds,
// dcsc.cpp:1042-1070 and :1361-1423)
__global__ void k_colmap(const int64_t* __restrict__ jc, int64_t nzc, const Counters* __restrict__ c,
                         int32_t* __restrict__ colmap) {
  if (c && !counts_valid(c->val)) return;
  int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p < nzc) colmap[jc[p]] = (int32_t)p;
}

// bpos[e] = stored-column position in A of B's row index irB[e] (-1 if A(:,k)
// is empty; the row itself where A stores every column, colmap null), and the
// columns' products flop_j (estimateFLOP, mtSpGEMM.h:1112-1130; flop cleared
// before).  One workgroup per 1024 consecutive entries: their A-column lengths
// are summed by a block scan, and every column takes the difference of two
// prefixes, so a hub column of 1e5 entries is shared by a hundred workgroups
// (a wave per column took 0.20 ms at R-MAT s19, this 0.04 with the positions).
constexpr int kFlopNT = 256, kFlopTile = 4 * kFlopNT;
__global__ __launch_bounds__(kFlopNT) void k_flops(const int64_t* __restrict__ cpB, const int64_t* __restrict__ irB,
                                                   int64_t nzcB, int64_t nnzB, const int32_t* __restrict__ colmap,
                                                   const int64_t* __restrict__ cpA, const Counters* __restrict__ c,
                                                   int32_t* __restrict__ bpos, int64_t* __restrict__ flop) {
  __shared__ int len[kFlopTile];
  __shared__ long long pre[kFlopTile + 1];
  __shared__ long long wsum[kFlopNT / kWave];
  if (c && !(counts_valid(c->val) && counts_valid(c->val + 3))) return;
  const int64_t t0 = blockIdx.x * (int64_t)kFlopTile;
  const int n = (int)min((int64_t)kFlopTile, nnzB - t0);
  // (each step's four loads in flight together)
  int64_t k[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) k[u] = irB[t0 + min(u * kFlopNT + (int)threadIdx.x, n - 1)];
#pragma unroll
  for (int u = 0; u < 4; ++u) pin(k[u]);
  int32_t p[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) p[u] = colmap ? colmap[k[u]] : (int32_t)k[u];
#pragma unroll
  for (int u = 0; u < 4; ++u) pin(p[u]);
  int64_t b[4], e[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int32_t q = max(p[u], 0);
    b[u] = cpA[q];
    e[u] = cpA[q + 1];
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    pin(b[u]);
    pin(e[u]);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = u * kFlopNT + threadIdx.x;
    if (i < n) bpos[t0 + i] = p[u];
    len[i] = i < n && p[u] >= 0 ? (int)(e[u] - b[u]) : 0;
  }
  __syncthreads();
  const int4 v = reinterpret_cast<const int4*>(len)[threadIdx.x];
  const long long s0 = v.x, s1 = s0 + v.y, s2 = s1 + v.z, s3 = s2 + v.w;
  long long total;
  const long long ex = block_excl_scan_ll<kFlopNT>(s3, wsum, total);
  const int i4 = threadIdx.x * 4;
  pre[i4] = ex;
  pre[i4 + 1] = ex + s0;
  pre[i4 + 2] = ex + s1;
  pre[i4 + 3] = ex + s2;
  if (threadIdx.x == kFlopNT - 1) pre[kFlopTile] = total;
  // the column of the tile's first entry: last c with cp[c] <= t0, 256 probes a step
  int64_t lo = 0, hi = nzcB;
  while (hi - lo > 1) {
    const int64_t step = (hi - lo + kFlopNT - 1) / kFlopNT;
    const int64_t at = lo + (int64_t)threadIdx.x * step;
    const int below = __syncthreads_count(at < hi && cpB[min(at, hi - 1)] <= t0);
    lo += (int64_t)(below - 1) * step;
    hi = min(hi, lo + step);
  }
  __syncthreads();
  for (int64_t q = lo + threadIdx.x; q < nzcB; q += kFlopNT) {
    const int64_t b = cpB[q], e = cpB[q + 1];
    if (b >= t0 + n) break;
    const int64_t from = max(b, t0), to = min(e, t0 + n);
    if (to <= from) continue;
    const long long f = pre[to - t0] - pre[from - t0];
    if (b >= t0 && e <= t0 + n) flop[q] = f;
    else if (f) atomicAdd((unsigned long long*)&flop[q], (unsigned long long)f);
  }
}

// Counts of the sort digits, and totals.  One workgroup per 1024 columns.
constexpr int kColTile = 1024;
__global__ __launch_bounds__(256) void k_count_digits(const int64_t* __restrict__ flop, int64_t nzcB,
                                                      const FlopClasses cls, Counters* __restrict__ c) {
  __shared__ unsigned int h[kDigits];
  for (int i = threadIdx.x; i < kDigits; i += 256) h[i] = 0;
  __syncthreads();
  long long all = 0, tiny = 0, list = 0;
#pragma unroll
  for (int u = 0; u < kColTile / 256; ++u) {
    const int64_t q = blockIdx.x * (int64_t)kColTile + u * 256 + threadIdx.x;
    const bool ok = q < nzcB;
    const int64_t f = ok ? flop[q] : 0;
    const int d = flop_digit(cls, f);
    const unsigned long long same = wave_match((uint32_t)d, 8, __ballot(ok));
    if (ok && __popcll(same & ((1ull << lane_id()) - 1ull)) == 0) atomicAdd(&h[d], (unsigned)__popcll(same));
    all += f;
    if (d / 32 == 5) tiny += f;
    if (d / 32 < 2) list += min(f, cls.list_cap);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kDigits; i += 256)
    if (h[i]) atomicAdd(&c->digits[i], h[i]);
  block_add_counts<256>(all, tiny, &c->flops, &c->tiny_flops);
  list = wave_sum_ll(list);
  if (lane_id() == 0 && list) atomicAdd(&c->list_rows, (unsigned long long)list);
}

// Columns in digit order (within a digit, tiles of 1024 columns stay together,
// nearly in column order): order and flop_s; the tiny columns' staging slots of
// flop_j entries (tiny_off, by position after the classes before) and the
// unit-tier columns' row-list regions (list_off, by position).  Two launches of
// one pass each; a full radix sort of (flop, column) took 0.45 ms at R-MAT s19
// and seven launches at 2^14 vertices.  The first workgroup reports the counts.
__global__ __launch_bounds__(256) void k_order_columns(const int64_t* __restrict__ flop, int64_t nzcB,
                                                       const FlopClasses cls, Counters* __restrict__ c,
                                                       int32_t* __restrict__ order, int64_t* __restrict__ flop_s,
                                                       int64_t* __restrict__ tiny_off, int64_t* __restrict__ list_off,
                                                       Report* __restrict__ rep) {
  constexpr int PT = kColTile / 256;
  __shared__ int base[256];  // first position of each digit
  __shared__ unsigned int h[kDigits], at[kDigits];
  __shared__ long long wsum[256 / kWave];
  __shared__ int isum[256 / kWave];
  __shared__ long long s_at[2];
  const int tid = threadIdx.x, lane = lane_id();
  const bool bad_a = !counts_valid(c->val), bad_b = !counts_valid(c->val + 3);
  if (blockIdx.x == 0 && tid == 0) {
    rep->err = (bad_a ? 16 : 0) | (bad_b ? 32 : 0);
    rep->flops = (int64_t)c->flops;
    rep->tiny_flops = (int64_t)c->tiny_flops;
    rep->list_rows = (int64_t)c->list_rows;
    for (int k = 0; k < kClasses; ++k) {
      int64_t n = 0;
      for (int i = 0; i < 32; ++i) n += c->digits[k * 32 + i];
      rep->columns[k] = n;
    }
  }
  if (bad_a || bad_b) return;
  int total;
  const int count = tid < kDigits ? (int)c->digits[tid] : 0;
  base[tid] = block_excl_scan<256>(count, isum, total);
  for (int i = tid; i < kDigits; i += 256) h[i] = 0;
  __syncthreads();
  int64_t f[PT];
  int d[PT];
  unsigned rank[PT];
  long long tiny = 0, list = 0;
#pragma unroll
  for (int u = 0; u < PT; ++u) {
    const int64_t q = blockIdx.x * (int64_t)kColTile + u * 256 + tid;
    const bool ok = q < nzcB;
    f[u] = ok ? flop[q] : 0;
    d[u] = flop_digit(cls, f[u]);
    const unsigned long long same = wave_match((uint32_t)d[u], 8, __ballot(ok));
    const int before = __popcll(same & ((1ull << lane) - 1ull));
    unsigned first = 0;
    if (ok && before == 0) first = atomicAdd(&h[d[u]], (unsigned)__popcll(same));
    first = (unsigned)__shfl((int)first, __ffsll((unsigned long long)same) - 1, kWave);
    rank[u] = first + before;
    if (d[u] / 32 == 5) tiny += f[u];
    if (ok && d[u] / 32 < 2) list += min(f[u], cls.list_cap);
  }
  __syncthreads();
  for (int i = tid; i < kDigits; i += 256) at[i] = h[i] ? atomicAdd(&c->cursor[i], h[i]) : 0;
  long long tiny_all, list_all;
  long long t_at = block_excl_scan_ll<256>(tiny, wsum, tiny_all);
  long long l_at = block_excl_scan_ll<256>(list, wsum, list_all);
  if (tid == 0) {
    s_at[0] = tiny_all ? (long long)atomicAdd(&c->tiny_at, (unsigned long long)tiny_all) : 0;
    s_at[1] = list_all ? (long long)atomicAdd(&c->list_at, (unsigned long long)list_all) : 0;
  }
  __syncthreads();
  t_at += s_at[0];
  l_at += s_at[1];
#pragma unroll
  for (int u = 0; u < PT; ++u) {
    const int64_t q = blockIdx.x * (int64_t)kColTile + u * 256 + tid;
    if (q >= nzcB) continue;
    const int pos = base[d[u]] + (int)(at[d[u]] + rank[u]);
    order[pos] = (int32_t)q;
    flop_s[pos] = f[u];
    if (d[u] / 32 == 5) {
      tiny_off[pos - base[5 * 32]] = t_at;
      t_at += f[u];
    }
    if (d[u] / 32 < 2) {
      list_off[pos] = l_at;
      l_at += min(f[u], cls.list_cap);
    }
  }
}

// Output offsets and the product's DCSC columns from the columns' sizes:
// sums of each 1024 columns, then (a scan of the sums in between where they
// are many and) offsets cpC, and the non-empty columns' starts and ids
// compacted into cp and jc.  The last workgroup reports the totals.
struct ColSum {
  long long nnz, cols;
};

__global__ __launch_bounds__(256) void k_col_sums(const int64_t* __restrict__ nnzcol, int64_t nzcB,
                                                  const int64_t* __restrict__ flop, int64_t main_above,
                                                  ColSum* __restrict__ sums, Counters* __restrict__ c) {
  __shared__ long long wsum[256 / kWave];
  long long nnz = 0, cols = 0, mine = 0;
#pragma unroll
  for (int u = 0; u < kColTile / 256; ++u) {
    const int64_t q = blockIdx.x * (int64_t)kColTile + u * 256 + threadIdx.x;
    const int64_t v = q < nzcB ? nnzcol[q] : 0;
    nnz += v;
    cols += v > 0;
    if (flop && v && flop[q] > main_above) mine += v;
  }
  nnz = block_sum_ll<256>(nnz, wsum);
  cols = block_sum_ll<256>(cols, wsum);
  mine = wave_sum_ll(mine);
  if (lane_id() == 0 && mine) atomicAdd(&c->main_nnz, (unsigned long long)mine);
  if (threadIdx.x == 0) sums[blockIdx.x] = ColSum{nnz, cols};
}

// sums[0..n) replaced by their exclusive prefixes (one workgroup).
__global__ __launch_bounds__(1024) void k_scan_sums(ColSum* __restrict__ sums, int64_t n) {
  __shared__ long long wsum[1024 / kWave];
  long long nnz = 0, cols = 0;
  for (int64_t i0 = 0; i0 < n; i0 += 1024) {
    const int64_t i = i0 + threadIdx.x;
    const ColSum v = i < n ? sums[i] : ColSum{0, 0};
    long long a, b;
    const long long ea = block_excl_scan_ll<1024>(v.nnz, wsum, a), eb = block_excl_scan_ll<1024>(v.cols, wsum, b);
    if (i < n) sums[i] = ColSum{nnz + ea, cols + eb};
    nnz += a;
    cols += b;
  }
}

__global__ __launch_bounds__(256) void k_col_offsets(const int64_t* __restrict__ nnzcol, int64_t nzcB,
                                                     const ColSum* __restrict__ sums, int scanned,
                                                     const int64_t* __restrict__ jcB, const Counters* __restrict__ c,
                                                     int64_t* __restrict__ cpC, int64_t* __restrict__ cp,
                                                     int64_t* __restrict__ jc, Report* __restrict__ rep) {
  constexpr int PT = kColTile / 256;
  __shared__ long long wsum[256 / kWave];
  const int tid = threadIdx.x;
  long long nnz0 = 0, cols0 = 0;  // before this workgroup's columns
  if (scanned) {
    nnz0 = sums[blockIdx.x].nnz;
    cols0 = sums[blockIdx.x].cols;
  } else {
    for (int i = tid; i < (int)blockIdx.x; i += 256) {
      nnz0 += sums[i].nnz;
      cols0 += sums[i].cols;
    }
    nnz0 = block_sum_ll<256>(nnz0, wsum);
    cols0 = block_sum_ll<256>(cols0, wsum);
  }
  const int64_t q0 = blockIdx.x * (int64_t)kColTile + tid * PT;
  int64_t v[PT];
  long long nnz = 0, cols = 0;
#pragma unroll
  for (int u = 0; u < PT; ++u) {
    v[u] = q0 + u < nzcB ? nnzcol[q0 + u] : 0;
    nnz += v[u];
    cols += v[u] > 0;
  }
  long long all_nnz, all_cols;
  long long at = nnz0 + block_excl_scan_ll<256>(nnz, wsum, all_nnz);
  long long col = cols0 + block_excl_scan_ll<256>(cols, wsum, all_cols);
#pragma unroll
  for (int u = 0; u < PT; ++u)
    if (q0 + u < nzcB) {
      cpC[q0 + u] = at;
      if (v[u] > 0 && cp) {
        cp[col] = at;
        jc[col] = jcB[q0 + u];
        ++col;
      }
      at += v[u];
    }
  if (blockIdx.x == gridDim.x - 1 && tid == 0) {
    const long long n = nnz0 + all_nnz, k = cols0 + all_cols;
    cpC[nzcB] = n;
    if (cp) cp[k] = n;
    rep->nnz = n;
    rep->nzc = k;
    rep->main_nnz = (int64_t)c->main_nnz;
    rep->dropped = (int64_t)c->dropped;
    rep->err = c->err;
    for (int i = 0; i < 3; ++i) rep->units[i] = c->units[i];
  }
}

__global__ void k_report_err(const int* __restrict__ err, Report* __restrict__ rep) {
  if (threadIdx.x == 0) rep->err = *err;
}

// Tile pointers: P[p*(S+1)+s] = number of entries of A's p-th stored column
// with row < s*TR.  One thread per stored column.
__global__ void k_ptable(const int64_t* __restrict__ cpA, int64_t nzcA, const int32_t* __restrict__ rowsA,
                         int S, int TR, int32_t* __restrict__ P) {
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p >= nzcA) return;
  const int64_t b = cpA[p];
  const int len = (int)(cpA[p + 1] - b);
  int32_t* out = P + p * (int64_t)(S + 1);
  int t = 0;
  for (int i = 0; i < len; ++i) {
    const int tile = rowsA[b + i] / TR;
    while (t <= tile) out[t++] = i;
  }
  while (t <= S) out[t++] = len;
}

// --------------------------------------------------------- symbolic: hash
// estimateNNZ_Hash restated for LDS (mtSpGEMM.h:861-927): insert each product's
// row into a linear-probing table, count first insertions.
template <int HMAX, int NT>
__global__ __launch_bounds__(NT) void k_sym_hash(const int32_t* __restrict__ order, int64_t first,
                                                 const int64_t* __restrict__ flop, const int64_t* __restrict__ cpB,
                                                 const int32_t* __restrict__ bpos, const int64_t* __restrict__ cpA,
                                                 const int32_t* __restrict__ rowsA, int64_t* __restrict__ nnzcol,
                                                 int* __restrict__ err) {
  __shared__ int32_t keys[HMAX];
  __shared__ long long wsum[NT / kWave];
  __shared__ FlatStage<uint8_t, NT, false> st;
  const int col = order[first + blockIdx.x];
  const int lg = min(ceil_log2_dev(max(2 * flop[col], 64ll)), ceil_log2_dev(HMAX));
  const int H = 1 << lg;
  for (int i = threadIdx.x; i < H; i += NT) keys[i] = -1;
  __syncthreads();
  flat_init(st);
  int cnt = 0, par = 0;
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  for (int64_t eb = b0; eb < b1; eb += NT) {
    int64_t base;
    int len;
    uint8_t dummy;
    load_seg<uint8_t, false>(eb + threadIdx.x, b1, bpos, cpA, Tiles{}, 0, 0, true, nullptr, base, len, dummy);
    const FlatSeg me = flat_stage<uint8_t, NT, false>(st, (int32_t)base, len, 0);
    flat_chunk<uint8_t, NT, false, 4>(st, me, par, [&](const int32_t(&idx)[4], uint8_t(&)[4], const bool(&ok)[4]) {
      int32_t rr[4];
      load_rows(rowsA, 0, idx, rr);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int32_t r = rr[u];
        if (!ok[u]) continue;
        uint32_t h = hash_slot(r, lg);
        int probe = 0;
        for (; probe < H; ++probe) {  // the table is at least twice the column's flops
          const int32_t old = atomicCAS(&keys[h], -1, r);
          if (old == -1) { ++cnt; break; }
          if (old == r) break;
          h = (h + 1) & (H - 1);
        }
        if (probe == H) atomicOr(err, 1);
      }
    });
  }
  const long long tot = block_sum_ll<NT>(cnt, wsum);
  if (threadIdx.x == 0) nnzcol[col] = tot;
}

// ------------------------------------------------------------ tiny tier
// Columns with at most 256 products (most columns of multigrid triple
// products, and the sparsest R-MAT columns): one wave per column.
//
// The products are gathered into registers, element e = u * 64 + lane in
// register u, their segments found by bit counts as in FlatStage.  Each then
// finds its row's slot in a per-wave hash table (linear probing, at most half
// full); the lanes whose products came first to their slots hold the distinct
// rows, which are compacted by ballots and sorted: up to 64 by counting the
// rows below each (broadcast reads of four), more by the digit passes of
// k_num_sort on one wave.  The row's rank replaces its key in the table, and
// every product accumulates at its slot's rank, so rows and values leave in
// order.  SYM only counts the distinct rows.
//
// A bitonic network over the 256 elements in registers took some 430
// cross-lane moves through LDS a column whatever its distinct rows: 4.0 ms for
// the two products of 16 Galerkin blocks (4.1e5 columns each of 216 and 64
// products, FP64); this takes 1.2 ms (1.7 with the loads of one register waited
// for before the next's are issued).  Bound by LDS latency at six waves per SIMD
// (27 KB for four waves).
constexpr int kTinyMax = 256;
constexpr int kTinyHash = 2 * kTinyMax;  // slots per wave at most
constexpr int kTinyWaves = 4;            // waves per workgroup at most (launch bound 256)
constexpr int kTinyDigit = 7;            // bits per digit pass: two 16-bit counters per lane

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class T, class Lds, bool SYM>
struct TinyLds {
  __align__(16) int32_t keys[kTinyHash];  // rows, then their ranks
  __align__(16) int32_t rows[kTinyMax + 4];
  uint16_t slot[kTinyMax];  // of each compacted row
  Lds vals[SYM ? 1 : kTinyMax];
  uint32_t hist[SYM ? 1 : kWave];
  unsigned long long starts[kTinyMax / 64];
  int32_t delta[kWave];
  T bval[SYM ? 1 : kWave];
};

// The products of one tiny column gathered into the wave's registers: rows
// and products of elements u * 64 + lane.  Returns their number
// (wave-uniform; above kTinyMax the rest is left out).
template <int K, class T, bool SYM, class L>
__device__ __forceinline__ int tiny_gather(L& ws, int64_t b0, int64_t b1, const int32_t* __restrict__ bpos,
                                           const T* __restrict__ valB, const int64_t* __restrict__ cpA,
                                           const int32_t* __restrict__ rowsA, const T* __restrict__ valA,
                                           int32_t (&key)[kTinyMax / kWave],
                                           typename Sem<K, T>::Acc (&val)[kTinyMax / kWave]) {
  using SR = Sem<K, T>;
  constexpr int kE = kTinyMax / kWave;
  const int lane = lane_id();
#pragma unroll
  for (int u = 0; u < kE; ++u) {
    key[u] = 0;
    val[u] = SR::ident();
  }
  int filled = 0;  // wave-uniform
  for (int64_t eb = b0; eb < b1; eb += kWave) {
    int64_t base;
    int len;
    T bv;
    load_seg<T, !SYM>(eb + lane, b1, bpos, cpA, Tiles{}, 0, 0, true, valB, base, len, bv);
    const unsigned long long some = __ballot(len > 0);
    if (!some) continue;
    const int incl = wave_incl_scan(len);
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    const int k = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(some >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)some, 0));
    const int start = filled + incl - len;
    if (lane < kE) ws.starts[lane] = 0ull;
    wave_lds_sync();
    if (len > 0) {
      ws.delta[k] = (int32_t)(base - start);
      if constexpr (!SYM) ws.bval[k] = bv;
      const int at = start - 1;  // one bit per segment after the first, before its first product
      if (k > 0 && at < kTinyMax)
        __hip_atomic_fetch_or(&ws.starts[at >> 6], 1ull << (at & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    wave_lds_sync();
    const int end = min(filled + total, kTinyMax);
    int before = 0;
    int32_t r[kE];
    T a[kE], b[kE];
#pragma unroll
    for (int u = 0; u < kE; ++u) {
      r[u] = 0;
      a[u] = b[u] = T{};
      const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)ws.starts[u]);
      const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(ws.starts[u] >> 32));
      // registers whose 64 elements miss this chunk's range stay as they are
      if ((u + 1) * kWave > filled && u * kWave < end) {
        const int s = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, (unsigned)before));
        // lanes outside repeat the chunk's first or last product
        const int32_t idx = min(max(u * kWave + lane, filled), end - 1) + ws.delta[s];
        r[u] = rowsA[idx];
        if constexpr (!SYM) {
          a[u] = valA[idx];
          b[u] = ws.bval[s];
        }
      }
      before += __popc(lo) + __popc(hi);
    }
#pragma unroll
    for (int u = 0; u < kE; ++u) {
      pin(r[u]);
      if constexpr (!SYM) pin(a[u]);
    }
#pragma unroll
    for (int u = 0; u < kE; ++u) {
      const int e = u * kWave + lane;
      if (e >= filled && e < end) {
        key[u] = r[u];
        if constexpr (!SYM) val[u] = SR::mul(a[u], b[u]);
      }
    }
    filled += total;
    wave_lds_sync();  // the chunk's segments have been read
  }
  return filled;
}

// Sorts rows[0..D) and slot[0..D) by row, D in (64, 256], with wave ballots:
// least significant digit first, over the bits in which the rows differ.
template <class L>
__device__ __forceinline__ void tiny_sort(L& ws, int D) {
  constexpr int kE = kTinyMax / kWave;
  const int lane = lane_id();
  uint32_t key[kE], slot[kE];
  const uint32_t first = (uint32_t)ws.rows[0];
  uint32_t diff = 0;
#pragma unroll
  for (int u = 0; u < kE; ++u) {
    const int e = u * kWave + lane;
    key[u] = (uint32_t)ws.rows[min(e, D - 1)];
    slot[u] = ws.slot[min(e, D - 1)];
    diff |= key[u] ^ first;
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) diff |= (uint32_t)__shfl_xor((int)diff, d, kWave);
  const int nbits = 32 - __clz((int)__builtin_amdgcn_readfirstlane((int)diff));  // at least 7: the rows are distinct
  const int npass = (nbits + kTinyDigit - 1) / kTinyDigit;
  const int width = (nbits + npass - 1) / npass;
  uint16_t* hist = reinterpret_cast<uint16_t*>(ws.hist);
  for (int p = 0, shift = 0; p < npass; ++p, shift += width) {
    ws.hist[lane] = 0;
    wave_lds_sync();
    int rank[kE];
#pragma unroll
    for (int u = 0; u < kE; ++u) {
      rank[u] = -1;
      if (u * kWave >= D) continue;  // uniform
      const bool valid = u * kWave + lane < D;
      const uint32_t d = (key[u] >> shift) & ((1u << width) - 1u);
      const unsigned long long same = wave_match(d, width, __ballot(valid));
      const int before = __popcll(same & ((1ull << lane) - 1ull));
      int seen = 0;
      if (valid) seen = hist[d];
      wave_lds_sync();
      if (valid && before == 0) hist[d] = (uint16_t)(seen + __popcll(same));
      wave_lds_sync();
      if (valid) rank[u] = seen + before;
    }
    const uint32_t pair = ws.hist[lane];
    const int c0 = (int)(pair & 0xffffu), c1 = (int)(pair >> 16);
    const int ex = wave_incl_scan(c0 + c1) - c0 - c1;
    ws.hist[lane] = (uint32_t)ex | (uint32_t)(ex + c0) << 16;
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < kE; ++u)
      if (rank[u] >= 0) {
        const int at = (int)hist[(key[u] >> shift) & ((1u << width) - 1u)] + rank[u];
        ws.rows[at] = (int32_t)key[u];
        ws.slot[at] = (uint16_t)slot[u];
      }
    wave_lds_sync();
    if (p + 1 < npass) {
#pragma unroll
      for (int u = 0; u < kE; ++u) {
        const int e = min(u * kWave + lane, D - 1);
        key[u] = (uint32_t)ws.rows[e];
        slot[u] = ws.slot[e];
      }
      wave_lds_sync();
    }
  }
}

// Six waves per SIMD, as its LDS allows, where the compiler would stop at 81
// VGPRs and five (FP64 min-plus, whose NaN rule is live to the end).
template <int K, class T, bool SYM>
struct TinyWavesPerSimd {
  static constexpr int value = K == kMinPlus && std::is_same<T, double>::value && !SYM ? 6 : 1;
};

template <int K, class T, bool SYM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TinyWavesPerSimd<K, T, SYM>::value))) void k_tiny(const int32_t* __restrict__ order, int64_t first, int64_t ncols,
                                              const int64_t* __restrict__ cpB, const int32_t* __restrict__ bpos,
                                              const T* __restrict__ valB, const int64_t* __restrict__ cpA,
                                              const int32_t* __restrict__ rowsA, const T* __restrict__ valA,
                                              int64_t* __restrict__ nnzcol, const int64_t* __restrict__ cpC,
                                              int64_t* __restrict__ irC, T* __restrict__ valC, int* __restrict__ err,
                                              const int64_t* __restrict__ stage_off = nullptr,
                                              const int64_t* __restrict__ stage_flop = nullptr, Filter<T> flt = {}) {
  using SR = Sem<K, T>;
  using Acc = typename SR::Acc;
  constexpr int kE = kTinyMax / kWave;
  constexpr int32_t kNone = 0x7fffffff, kEmpty = -1;
  __shared__ TinyLds<T, typename SR::Lds, SYM> s_ws[kTinyWaves];
  const int lane = lane_id(), w = wave_id_uniform();
  auto& ws = s_ws[w];
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x / kWave);
  for (int64_t i = (int64_t)blockIdx.x * (blockDim.x / kWave) + w; i < ncols; i += waves) {
    const int col = order[first + i];
    int32_t key[kE];
    Acc val[kE];
    int filled = tiny_gather<K, T, SYM>(ws, cpB[col], cpB[col + 1], bpos, valB, cpA, rowsA, valA, key, val);
    if (filled > kTinyMax) {  // the tier's bound keeps it below; guard anyway
      if (lane == 0) atomicOr(err, 4);
      filled = kTinyMax;
    }
    int lg = 6;  // 64 slots at least, and twice the products
    while ((1 << lg) < 2 * filled) ++lg;
    const int H = 1 << lg;
    for (int q = lane * 4; q < H; q += kWave * 4)
      *reinterpret_cast<int4*>(ws.keys + q) = int4{kEmpty, kEmpty, kEmpty, kEmpty};
    wave_lds_sync();
    // every product finds its row's slot; the first to come owns it
    int slot[kE];
    int D = 0;  // distinct rows
#pragma unroll
    for (int u = 0; u < kE; ++u) {
      if (u * kWave >= filled) continue;  // uniform
      bool owner = false;
      slot[u] = 0;
      if (u * kWave + lane < filled) {
        uint32_t h = hash_slot(key[u], lg);
        while (true) {
          const int32_t old = atomicCAS(&ws.keys[h], kEmpty, key[u]);
          owner = old == kEmpty;
          if (owner || old == key[u]) break;
          h = (h + 1) & (H - 1);
        }
        slot[u] = (int)h;
      }
      const unsigned long long om = __ballot(owner);
      if (!SYM && owner) {
        const int at = D + __popcll(om & ((1ull << lane) - 1ull));
        ws.rows[at] = key[u];
        ws.slot[at] = (uint16_t)slot[u];
      }
      D += __popcll(om);
    }
    if constexpr (SYM) {
      if (lane == 0) nnzcol[col] = D;
      wave_lds_sync();
      continue;
    } else {
      if (D <= kWave) {  // rank of every distinct row: the distinct rows below it
        if (lane < 4) ws.rows[D + lane] = kNone;  // padding for the four-wide reads
        wave_lds_sync();
        const int32_t mine = lane < D ? ws.rows[lane] : kNone;
        const int at = ws.slot[min(lane, max(D - 1, 0))];
        int rank = 0;
        for (int j = 0; j < D; j += 4) {
          const int4 q = *reinterpret_cast<const int4*>(ws.rows + j);
          rank += (q.x < mine) + (q.y < mine) + (q.z < mine) + (q.w < mine);
        }
        wave_lds_sync();
        if (lane < D) {
          ws.rows[rank] = mine;
          ws.keys[at] = rank;
        }
      } else {
        wave_lds_sync();
        tiny_sort(ws, D);
        for (int e = lane; e < D; e += kWave) ws.keys[ws.slot[e]] = e;
      }
      for (int e = lane; e < D; e += kWave) ws.vals[e] = SR::lident();
      wave_lds_sync();
#pragma unroll
      for (int u = 0; u < kE; ++u)
        if (u * kWave + lane < filled) SR::acc(&ws.vals[ws.keys[slot[u]]], val[u]);
      if constexpr (K != kPlusTimes && std::is_floating_point<T>::value) {
        // the semiring's add keeps a NaN that comes first (b < a ? b : a), the
        // accumulator one that is alone: rare, so product by product
        wave_lds_sync();
#pragma unroll
        for (int u = 0; u < kE; ++u) {
          unsigned long long nan = __ballot(u * kWave + lane < filled && val[u] != val[u]);
          while (nan) {
            const int l = __ffsll(nan) - 1;
            nan &= nan - 1;
            const int at = __builtin_amdgcn_readlane(slot[u], l);
            unsigned long long before = 0ull;  // products of the row before this one
#pragma unroll
            for (int w2 = 0; w2 <= u; ++w2) {
              const unsigned long long same = __ballot(w2 * kWave + lane < filled && slot[w2] == at);
              before |= w2 < u ? same : same & ((1ull << l) - 1ull);
            }
            if (!before && lane == 0) ws.vals[ws.keys[at]] = SR::lident();
          }
        }
      }
      // the column's allocation from the symbolic pass; or, staged (no symbolic
      // pass), its slot of flop_j entries in the staging buffer, and the count
      // is recorded for the copy into place
      int64_t have, out;
      if (stage_off) {
        out = stage_off[i];
        have = stage_flop[first + i];
        if (lane == 0) nnzcol[col] = D;
        if (lane == 0 && D > have) atomicOr(err, 8);
      } else {
        have = nnzcol[col];
        if (lane == 0 && D != have) atomicOr(err, 8);
        out = cpC[col];
      }
      wave_lds_sync();
      if (!flt.on) {
        for (int e = lane; e < D && e < have; e += kWave) {
          irC[out + e] = ws.rows[e];
          valC[out + e] = SR::lout(ws.vals[e]);
        }
      } else {  // the fused threshold: kept entries, in row order, at out
        int kept = 0;
        for (int e0 = 0; e0 < D; e0 += kWave) {
          const int e = e0 + lane;
          const T v = e < D ? SR::lout(ws.vals[e]) : T{};
          const bool keep = e < D && !(v < flt.thr);
          const unsigned long long km = __ballot(keep);
          const int at = kept + __popcll(km & ((1ull << lane) - 1ull));
          if (keep && at < have) {
            irC[out + at] = ws.rows[e];
            valC[out + at] = v;
          }
          kept += __popcll(km);
        }
        if (lane == 0) {
          if (stage_off) {
            nnzcol[col] = kept;
            if (D > kept) atomicAdd(flt.dropped, (unsigned long long)(D - kept));
          } else {
            filter_add_run(flt, out, kept, col, err);
          }
        }
      }
      wave_lds_sync();  // the next column reuses the wave's LDS
    }
  }
}

// Staged tiny columns into place: a wave copies the nnzcol[col] entries of 16
// columns from their staging slots to cpC[col], four columns' first 64 entries
// in flight together (one column per wave waited for its place, then for its
// entries: 0.60 ms for the two products of 16 Galerkin triples, now 0.40).
constexpr int kPlaceCols = 16;
template <class T>
__global__ __launch_bounds__(256) void k_tiny_place(
    const int32_t* __restrict__ order, int64_t first, int64_t ncols, const int64_t* __restrict__ stage_off,
    const int64_t* __restrict__ nnzcol, const int64_t* __restrict__ cpC, const int64_t* __restrict__ sir,
    const T* __restrict__ sval, int64_t* __restrict__ irC, T* __restrict__ valC, Filter<T> flt = {},
    int* __restrict__ err = nullptr) {
  constexpr int U = 4;
  const int64_t i0 = global_wave() * kPlaceCols;
  if (i0 >= ncols) return;
  const int lane = lane_id(), n = (int)min<int64_t>(ncols - i0, kPlaceCols);
  const int64_t mine = i0 + min(lane, n - 1);
  const int col = order[first + mine];
  const int64_t src = stage_off[mine], dst = cpC[col];
  const int cnt = lane < n ? (int)nnzcol[col] : 0;
  if (flt.on && lane < n) filter_add_run(flt, dst, cnt, col, err);  // staged entries are the kept ones
  for (int c = 0; c < n; c += U) {
    int64_t s[U], d[U], r[U];
    T v[U];
    int k[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s[u] = readlane_ll(src, c + u);
      d[u] = readlane_ll(dst, c + u);
      k[u] = __builtin_amdgcn_readlane(cnt, c + u);
      const int64_t e = lane < k[u] ? s[u] + lane : 0;
      r[u] = sir[e];
      v[u] = sval[e];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      pin(r[u]);
      pin(v[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (lane < k[u]) {
        irC[d[u] + lane] = r[u];
        valC[d[u] + lane] = v[u];
      }
      for (int e = kWave + lane; e < k[u]; e += kWave) {
        irC[d[u] + e] = sir[s[u] + e];
        valC[d[u] + e] = sval[s[u] + e];
      }
    }
  }
}

// -------------------------------------------------------- symbolic: dense
// Distinct-row count with an LDS bitmap of RBW*32 rows per pass; a pass
// covers G row tiles of the tile-pointer table.
template <int NT, int RBW>
__global__ __launch_bounds__(NT) void k_sym_dense(const int32_t* __restrict__ order, int64_t first,
                                                  const int64_t* __restrict__ cpB, const int32_t* __restrict__ bpos,
                                                  const int64_t* __restrict__ cpA, const int32_t* __restrict__ rowsA,
                                                  const int32_t* __restrict__ P, int S, int G, int TR,
                                                  int64_t* __restrict__ nnzcol) {
  __shared__ uint32_t bits[RBW];
  __shared__ long long wsum[NT / kWave];
  const int col = order[first + blockIdx.x];
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  long long cnt = 0;
  const int npass = (S + G - 1) / G;
  for (int sp = 0; sp < npass; ++sp) {
    for (int i = threadIdx.x; i < RBW; i += NT) bits[i] = 0u;
    __syncthreads();
    const int s_lo = sp * G, s_hi = min(S, s_lo + G);
    const int32_t row0 = s_lo * TR;
    for (int64_t eb = b0 + wave_id() * kWave; eb < b1; eb += NT) {
      const int64_t e = eb + lane_id();
      int64_t lo = 0;
      int len = 0;
      if (e < b1) {
        const int32_t p = bpos[e];
        if (p >= 0) {
          if (npass == 1) {
            lo = cpA[p];
            len = (int)(cpA[p + 1] - lo);
          } else {
            const int32_t* pp = P + (int64_t)p * (S + 1);
            const int a = pp[s_lo];
            lo = cpA[p] + a;
            len = pp[s_hi] - a;
          }
        }
      }
      wave_visit(lo, len, 0, [&](int64_t idx, int) {
        const int32_t r = rowsA[idx] - row0;
        const uint32_t bit = 1u << (r & 31);
        const uint32_t old = atomicOr(&bits[r >> 5], bit);
        if (!(old & bit)) ++cnt;
      });
    }
    __syncthreads();
  }
  const long long tot = block_sum_ll<NT>(cnt, wsum);
  if (threadIdx.x == 0) nnzcol[col] = tot;
}

// ---------------------------------------------------------- numeric: sort
// Columns with tiny_flop < flop_j <= 4 * NT products, one workgroup each:
// the heap / hash accumulation and sort of mtSpGEMM.h:311-440 as a radix sort
// of the products.  Every thread gathers four products into registers; their
// rows are sorted in LDS with the product's number as payload (least
// significant digit first, at most 7 bits a pass, over the bits in which the
// column's rows differ); the heads of equal rows, numbered by a block scan,
// give every product its rank, and the products then accumulate from the
// registers at vals[rank].  Rows and values leave in rank order, coalesced.
//
// A digit pass ranks 64 keys at a time by wave ballots: every wave counts its
// own 256 keys, so the pass needs one block scan over (digit, wave) and no
// atomics.  At R-MAT s19 ef16 (int64) the columns of 1025 to 4096 products
// take 1.9 ms and the smaller ones 0.32 ms; a hash table with LDS compaction
// and a bitonic sort took 17.3 ms (one 119 KB workgroup per CU, 78 barriers a
// sort) and 1.2 ms.  Bound by VALU (the ballots) and LDS; 60 KB at 1024
// threads: two workgroups per CU, all 32 waves.  The workgroup has a quarter
// of the tier's product bound in threads, so that none idles: bounds of 1024,
// 2048 and 4096 products.
template <int K, class T, int NT>
__global__ __launch_bounds__(NT) void k_num_sort(const int32_t* __restrict__ order, int64_t first,
                                                 const int64_t* __restrict__ nnzcol, const int64_t* __restrict__ cpB,
                                                 const int32_t* __restrict__ bpos, const T* __restrict__ valB,
                                                 const int64_t* __restrict__ cpA, const int32_t* __restrict__ rowsA,
                                                 const T* __restrict__ valA, const int64_t* __restrict__ cpC,
                                                 int64_t* __restrict__ irC, T* __restrict__ valC,
                                                 int* __restrict__ err, Filter<T> flt = {}) {
  using SR = Sem<K, T>;
  using Acc = typename SR::Acc;
  constexpr int U = 4, CAP = U * NT, NW = NT / kWave;
  constexpr int kDigit = 7;  // bits per pass at most: 128 * NW 16-bit counters, two per thread
  constexpr int kRow = (1 << kDigit) + 2;  // a wave's counters, padded so that equal digits differ in bank
  static_assert((1 << kDigit) * NW == 2 * NT, "one pair of counters per thread");
  union Window {
    FlatStage<T, NT, true> st;  // while the products are gathered
    typename SR::Lds vals[CAP];  // once their ranks are known
  };
  __shared__ __align__(16) uint32_t keys[CAP];
  __shared__ __align__(8) uint16_t pay[CAP];  // product numbers, then the products' ranks
  __shared__ __align__(8) uint16_t hist[kRow * NW];
  __shared__ __align__(16) unsigned char window_mem[sizeof(Window)];
  __shared__ long long wsum[NW];
  __shared__ int isum[NW];
  Window& win = *reinterpret_cast<Window*>(window_mem);
  const int tid = threadIdx.x, lane = lane_id(), w = wave_id_uniform();
  // where position p of the sorted order is kept: a pass's stores come 4096 /
  // 128 positions apart where a segment's rows are dense, one bank without it
  auto place = [](int p) { return p ^ ((p >> 6) & 63); };
  auto clear_hist = [&]() {
    for (int i = tid; i < kRow * NW / 2; i += NT) reinterpret_cast<uint32_t*>(hist)[i] = 0;
  };
  const int col = order[first + blockIdx.x];
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  // products (u * NW + w) * 64 + lane of the column
  uint32_t key[U], num[U];
  Acc prod[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    key[u] = 0;
    num[u] = (uint32_t)((u * NW + w) * kWave + lane);
    prod[u] = SR::ident();
  }
  int total = 0, par = 0;
  flat_init(win.st);
  for (int64_t eb = b0; eb < b1; eb += NT) {
    int64_t base;
    int len;
    T bv;
    load_seg<T, true>(eb + tid, b1, bpos, cpA, Tiles{}, 0, 0, true, valB, base, len, bv);
    const FlatSeg me = flat_stage<T, NT, true>(win.st, (int32_t)base, len, bv, total);
    if (me.total == 0 || total >= CAP) {  // (uniform)
      total += me.total;
      __syncthreads();  // every wave has read the counts before the next chunk's are written
      continue;
    }
    const FlatTile ft = flat_tile(win.st, me, 0, 0, par);
    par ^= 1;
    const int end = min(total + me.total, CAP);
    int32_t idx[U], r[U];
    T a[U], bvs[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int wd = u * NW + w;  // at most 63: the tile's first half
      const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)ft.w0, wd);
      const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(ft.w0 >> 32), wd);
      const unsigned kb = (unsigned)__builtin_amdgcn_readlane(ft.p0, wd);
      const int k = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, kb));
      // products of other chunks repeat this one's first or last
      idx[u] = min(max((int)num[u], total), end - 1) + win.st.delta[k];
      bvs[u] = win.st.bval[k];
    }
    load_entries(rowsA, valA, 0, idx, bvs, r, a);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if ((int)num[u] >= total && (int)num[u] < end) {
        key[u] = (uint32_t)r[u];
        prod[u] = SR::mul(a[u], bvs[u]);
      }
    total += me.total;
  }
  if (total > CAP) {  // the tier's bound keeps it below; guard anyway (uniform)
    if (tid == 0) atomicOr(err, 2);
    total = CAP;
  }
  // the bits in which the rows differ from the column's first
  if (tid == 0) isum[0] = (int)key[0];
  __syncthreads();
  const uint32_t key0 = (uint32_t)isum[0];
  uint32_t diff = 0;
#pragma unroll
  for (int u = 0; u < U; ++u)
    if ((int)num[u] < total) diff |= key[u] ^ key0;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) diff |= (uint32_t)__shfl_xor((int)diff, d, kWave);
  __syncthreads();
  if (lane == 0) isum[w] = (int)diff;
  clear_hist();
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) diff |= (uint32_t)isum[i];
  const int nbits = 32 - __clz((int)diff);  // 0 when every row is the same
  const int npass = max(1, (nbits + kDigit - 1) / kDigit);
  const int width = (nbits + npass - 1) / npass;
  const uint32_t dmask = (1u << width) - 1u;
  for (int p = 0, shift = 0; p < npass; ++p, shift += width) {
    // in the first pass a wave's keys are those it gathered, later the sorted positions [256 w, 256 w + 256)
    int rank[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool valid = (p == 0 ? (int)num[u] : (w * U + u) * kWave + lane) < total;
      const uint32_t d = (key[u] >> shift) & dmask;
      const unsigned long long same = wave_match(d, width, __ballot(valid));
      const int before = __popcll(same & ((1ull << lane) - 1ull));
      uint16_t* h = &hist[w * kRow + d];
      int seen = 0;
      if (valid) seen = *h;
      wave_lds_sync();
      if (valid && before == 0) *h = (uint16_t)(seen + __popcll(same));
      wave_lds_sync();
      rank[u] = valid ? seen + before : -1;
    }
    __syncthreads();
    {
      // counters 2 tid and 2 tid + 1 in (digit, wave) order
      uint16_t* h = &hist[2 * tid % NW * kRow + 2 * tid / NW];
      const int c0 = h[0], c1 = h[kRow];
      int all;
      const int ex = block_excl_scan<NT>(c0 + c1, isum, all);
      h[0] = (uint16_t)ex;
      h[kRow] = (uint16_t)(ex + c0);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (rank[u] >= 0) {
        const int at = place((int)hist[w * kRow + ((key[u] >> shift) & dmask)] + rank[u]);
        keys[at] = key[u];
        pay[at] = (uint16_t)num[u];
      }
    __syncthreads();
    if (p + 1 < npass) {
      clear_hist();
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = place((w * U + u) * kWave + lane);
        key[u] = keys[e];  // (past the end: never counted)
        num[u] = pay[e];
      }
      __syncthreads();
    }
  }
  // heads of equal rows among the thread's four sorted positions, and their numbers
  uint32_t prev = tid > 0 ? keys[place(tid * U - 1)] : 0u;
  bool head[U];
  int heads = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int e = tid * U + u;
    key[u] = keys[place(e)];
    num[u] = pay[place(e)];
    head[u] = e < total && (e == 0 || key[u] != prev);
    prev = key[u];
    heads += head[u];
  }
  int cnt;
  int rk = block_excl_scan<NT>(heads, isum, cnt) - 1;  // its barriers: every position has been read
  const int64_t nz = nnzcol[col];
  if (cnt != nz && tid == 0) atomicOr(err, 8);
  cnt = (int)min((int64_t)cnt, nz);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (tid * U + u >= total) continue;
    rk += head[u];
    if (head[u]) keys[rk] = key[u];  // the output rows
    pay[num[u]] = (uint16_t)rk;
  }
  for (int i = tid; i < cnt; i += NT) win.vals[i] = SR::lident();
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u)
    if ((u * NW + w) * kWave + lane < total) {
      const int q = pay[(u * NW + w) * kWave + lane];
      if (q < cnt) SR::acc(&win.vals[q], prod[u]);
    }
  __syncthreads();
  const int64_t out = cpC[col];
  if (!flt.on) {
    for (int i = tid; i < cnt; i += NT) {
      irC[out + i] = (int64_t)keys[i];
      valC[out + i] = SR::lout(win.vals[i]);
    }
    return;
  }
  auto item = [&](int i, T& v) {  // the fused threshold
    v = SR::lout(win.vals[i]);
    return true;
  };
  emit_filtered<T, NT>(cnt, cnt, item, [&](int i) { return (int64_t)keys[i]; }, out, irC, valC, flt, col, isum, err);
}

// --------------------------------------------------------- numeric: dense
// Row-tiled dense accumulation: TR rows per tile, TR = 32*NT so that each
// thread owns one 32-bit word of the presence bitmap during emission.
template <int K, class T, int NT>
__global__ __launch_bounds__(NT) void k_num_dense(const int32_t* __restrict__ order, int64_t first,
                                                  const int64_t* __restrict__ cpB, const int32_t* __restrict__ bpos,
                                                  const T* __restrict__ valB, const int64_t* __restrict__ cpA,
                                                  const int32_t* __restrict__ rowsA, const T* __restrict__ valA,
                                                  const int32_t* __restrict__ P, int S,
                                                  const int64_t* __restrict__ cpC, int64_t* __restrict__ irC,
                                                  T* __restrict__ valC, int* __restrict__ err) {
  using SR = Sem<K, T>;
  using Acc = typename SR::Acc;
  constexpr int TR = 32 * NT;
  __shared__ typename SR::Lds acc[TR];
  __shared__ uint32_t bits[NT];
  __shared__ int wsum[NT / kWave];
  const int col = order[first + blockIdx.x];
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  int64_t out = cpC[col];
  const int64_t out_end = cpC[col + 1];
  for (int i = threadIdx.x; i < TR; i += NT) acc[i] = SR::lident();
  bits[threadIdx.x] = 0u;
  __syncthreads();
  for (int s = 0; s < S; ++s) {
    const int32_t row0 = s * TR;
    for (int64_t eb = b0 + wave_id() * kWave; eb < b1; eb += NT) {
      const int64_t e = eb + lane_id();
      int64_t lo = 0;
      int len = 0;
      T bv{};
      if (e < b1) {
        const int32_t p = bpos[e];
        if (p >= 0) {
          const int32_t* pp = P + (int64_t)p * (S + 1) + s;
          const int a = pp[0];
          lo = cpA[p] + a;
          len = pp[1] - a;
          bv = valB[e];
        }
      }
      wave_visit(lo, len, bv, [&](int64_t idx, T b) {
        const int32_t r = rowsA[idx] - row0;
        SR::acc(&acc[r], SR::mul(valA[idx], b));
        atomicOr(&bits[r >> 5], 1u << (r & 31));
      });
    }
    __syncthreads();
    uint32_t w = bits[threadIdx.x];
    int tot;
    const int ex = block_excl_scan<NT>(__popc(w), wsum, tot);
    int64_t o = out + ex;
    while (w) {
      const int b = __ffs(w) - 1;
      w &= w - 1;
      const int r = threadIdx.x * 32 + b;
      if (o < out_end) {  // symbolic and numeric agree; guard anyway
        irC[o] = (int64_t)row0 + r;
        valC[o] = SR::lout(acc[r]);
      } else {
        atomicOr(err, 4);
      }
      acc[r] = SR::lident();
      ++o;
    }
    bits[threadIdx.x] = 0u;
    out += tot;
    __syncthreads();
  }
}

// Symbolic pass of the unit tier: one workgroup per column.  Units are cut
// over passes of 256 blocks (2^20 rows); within a pass the presence bitmap is
// built IBLK blocks at a time (each sub-pass gathers only the products in its
// rows, through the tile table P), so the LDS bitmap stays small enough for
// several workgroups per CU.  Writes nnz_j and the column's units.
//
// With `lists`, the column's sorted output rows in blocks of at most
// kListBlockMax outputs are also written, as 12-bit offsets within their
// 4096-row blocks, at their output positions in the column's region
// of min(flop_j, region_cap) entries from lists[list_off[slot]] on (slot = the workgroup), and its
// per-block counts into bcnt16[slot * S ..].  The small units of a pass whose
// rows fit the region are then cut by output count alone over runs of such
// blocks: those wider than rblk_l blocks go to units_s, whose numeric pass
// takes ranks from the list instead of a bitmap.
//
// Eight waves per SIMD: the pass is latency-bound on its gathers, so the
// kernel asks for 64 VGPRs at most (it takes 55, and 60 with seven waves if
// left alone) and keeps its LDS under 40 KB (the unit staging lives in the
// bitmap, idle while a pass is cut), four workgroups per CU.  At R-MAT s20 it
// takes 30.9 ms; before the products were flattened by bitmaps, 55.7, and 64
// with the 80 VGPRs, 47 KB and six waves of then.
template <int NT, int U, int IBLK>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_sym_units(
    const int32_t* __restrict__ order, int64_t first,
                                                  const int64_t* __restrict__ cpB, const int32_t* __restrict__ bpos,
                                                  const int64_t* __restrict__ cpA, const int32_t* __restrict__ rowsA,
                                                  const Tiles P, int S, int kmax_l, int rblk_l,
                                                  int kmax_h, int rblk_h, int64_t heavy_thr,
                                                  int64_t* __restrict__ nnzcol, Unit* __restrict__ units_l,
                                                  int* __restrict__ n_l, int cap_l, Unit* __restrict__ units_h,
                                                  int* __restrict__ n_h, int cap_h, uint32_t* __restrict__ rmap,
                                                  int64_t rm_cols, int* __restrict__ err,
                                                  uint16_t* __restrict__ lists = nullptr,
                                                  const int64_t* __restrict__ list_off = nullptr,
                                                  const int64_t* __restrict__ flop = nullptr, int64_t region_cap = 0,
                                                  uint16_t* __restrict__ bcnt16 = nullptr,
                                                  Unit* __restrict__ units_s = nullptr, int* __restrict__ n_s = nullptr,
                                                  int cap_s = 0) {
  constexpr int BPP = 256;             // blocks per cutting pass (2^20 rows)
  constexpr int BMW = IBLK * kBRW;     // bitmap words of one sub-pass
  static_assert(BPP % IBLK == 0, "sub-passes tile the cutting pass");
  static_assert(IBLK <= kWave, "a wave scans the block counts of a sub-pass");
  __shared__ __align__(16) uint32_t bits[BMW];
  __shared__ int bpre[BPP];           // block counts, then their inclusive prefix
  __shared__ FlatStage<uint8_t, NT, false> st;
  __shared__ int s_nu, s_slot, s_ns, s_sslot;
  // the units of a pass, staged while it is cut: in the bitmap, which every
  // thread has finished reading (barrier) and the next pass clears only after
  // the end-of-pass barrier
  static_assert(sizeof(uint32_t) * BMW >= 2 * BPP * sizeof(Unit), "the bitmap holds a pass's units");
  Unit* su = reinterpret_cast<Unit*>(bits);
  __shared__ unsigned long long s_dense[BPP / kWave];  // blocks of the pass above kListBlockMax outputs
  Unit* su2 = su + BPP;  // list units of a pass
  const int col = order[first + blockIdx.x];
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  const int npass = (S + BPP - 1) / BPP;
  const bool whole = S <= IBLK;  // one sub-pass covers every row: no tile look-ups
  int64_t list_base = 0, region = 0;
  if (lists) {
    list_base = list_off[blockIdx.x];
    region = min(flop[col], region_cap);
  }
  int64_t colcnt = 0;
  int par = 0;
  flat_init(st);
  int unit_off = 0;  // meaningful in thread 0 only
  for (int sp = 0; sp < npass; ++sp) {
    const int t_lo = sp * BPP, t_hi = min(S, t_lo + BPP), nblk = t_hi - t_lo;
    bool listok = lists != nullptr;  // every row of this pass written so far (uniform)
    int64_t run = 0;                 // this pass's rows before the current sub-pass (uniform)
    for (int i_lo = t_lo; i_lo < t_hi; i_lo += IBLK) {
      const int i_hi = min(t_hi, i_lo + IBLK), inb = i_hi - i_lo;
      const int32_t row0 = i_lo * kBR;
      for (int i = threadIdx.x * 4; i < inb * kBRW; i += NT * 4) *reinterpret_cast<uint4*>(bits + i) = uint4{0, 0, 0, 0};
      // (the staging barrier below orders the clear before any insertion)
      for (int64_t eb = b0; eb < b1; eb += NT) {
        int64_t base;
        int len;
        uint8_t dummy;
        load_seg<uint8_t, false>(eb + threadIdx.x, b1, bpos, cpA, P, i_lo, i_hi, whole, nullptr, base, len,
                                 dummy);
        const FlatSeg me = flat_stage<uint8_t, NT, false>(st, (int32_t)base, len, 0);
        flat_chunk<uint8_t, NT, false, U>(st, me, par, [&](const int32_t(&idx)[U], uint8_t(&)[U], const bool(&ok)[U]) {
          int32_t r[U];
          load_rows(rowsA, row0, idx, r);
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (ok[u]) atomicOr(&bits[r[u] >> 5], 1u << (r[u] & 31));
        });
      }
      __syncthreads();
      // the column's row map (its presence bitmap, S blocks of kBRW words)
      // for the numeric pass, which then need not rebuild it; kept for the
      // first rm_cols columns of the launch (the only ones that can form
      // large units)
      if (rmap && blockIdx.x < rm_cols) {
        uint32_t* dst = rmap + (int64_t)blockIdx.x * S * kBRW + (int64_t)i_lo * kBRW;
        for (int i = threadIdx.x; i < inb * kBRW; i += NT) dst[i] = bits[i];
      }
      // per-block counts: one wave per block, two words per lane
      for (int b = wave_id_uniform(); b < inb; b += NT / kWave) {
        const uint2 x = reinterpret_cast<const uint2*>(bits + b * kBRW)[lane_id()];
        const int c = __builtin_amdgcn_readlane(wave_incl_scan(__popc(x.x) + __popc(x.y)), kWave - 1);
        if (lane_id() == 0) {
          bpre[i_lo - t_lo + b] = c;
          if (lists) bcnt16[(int64_t)blockIdx.x * S + i_lo + b] = (uint16_t)c;
        }
      }
      __syncthreads();  // the counts are read, and the next sub-pass clears the bitmap
      if (lists) {
        // the sub-pass's rows in order, one wave per block as for the counts
        // (two words, 64 rows, per lane): every wave scans the sub-pass's
        // block counts (IBLK <= 64, one per lane) for the block offsets and
        // the total, and its lanes place their rows by a wave scan, so the
        // stores of a wave cover one contiguous range
        const int bc = lane_id() < inb ? bpre[i_lo - t_lo + lane_id()] : 0;
        const int bincl = wave_incl_scan(bc);
        const int sub_total = __shfl(bincl, kWave - 1, kWave);
        const int64_t have = colcnt + run;
        listok = listok && have + sub_total <= region;
        if (listok) {
          for (int b = wave_id_uniform(); b < inb; b += NT / kWave) {
            const int nb = __builtin_amdgcn_readlane(bc, b);
            if (nb == 0 || nb > kListBlockMax) continue;  // dense block: its units use the bitmap
            const int boff = __builtin_amdgcn_readlane(bincl, b) - nb;
            uint2 x = reinterpret_cast<const uint2*>(bits + b * kBRW)[lane_id()];
            const int c = __popc(x.x) + __popc(x.y);
            uint16_t* dst = lists + list_base + have + boff + (wave_incl_scan(c) - c);
            int row = lane_id() * 64;
            while (x.x) {
              *dst++ = (uint16_t)(row + __builtin_ctz(x.x));
              x.x &= x.x - 1;
            }
            row += 32;
            while (x.y) {
              *dst++ = (uint16_t)(row + __builtin_ctz(x.y));
              x.y &= x.y - 1;
            }
          }
        }
        run += sub_total;
        __syncthreads();  // the bitmap is read before the next sub-pass clears it
      }
    }
    if (wave_id() == 0) {  // inclusive prefix over blocks, and the mask of the blocks without a list
      int carry = 0;
      for (int b0i = 0; b0i < nblk; b0i += kWave) {
        const int b = b0i + lane_id();
        const int v = b < nblk ? bpre[b] : 0;
        const int inc = wave_incl_scan(v) + carry;
        if (b < nblk) bpre[b] = inc;
        carry = __shfl(inc, kWave - 1, kWave);
        const unsigned long long dense = __ballot(b < nblk && v > kListBlockMax);
        if (lane_id() == 0) s_dense[b0i / kWave] = dense;
      }
    }
    __syncthreads();
    const int pass_total = bpre[nblk - 1];
    if (threadIdx.x == 0) {
      // greedy cut into units of at most kmax outputs (a unit of one block may
      // have more, up to kBR: it is direct, its rows fit the value window); a
      // small-unit pass with its list written is cut by count alone
      const bool heavy = pass_total > heavy_thr;
      const bool by_list = !heavy && listok;
      const int kmax = heavy ? kmax_h : kmax_l, rblk = heavy ? rblk_h : rblk_l;
      // first block at or after `from` whose rows were not listed (nblk if none)
      auto next_dense = [&](int from) {
        for (int q = from / kWave; q * kWave < nblk; ++q) {
          unsigned long long msk = s_dense[q];
          if (q == from / kWave) msk &= ~0ull << (from % kWave);
          if (msk) return min(nblk, q * kWave + __ffsll(msk) - 1);
        }
        return nblk;
      };
      int start = 0, before = 0, nu = 0, ns = 0;
      while (start < nblk) {
        const int lim = before + kmax;
        // a unit wider than rblk blocks takes its ranks from the list, so it
        // stops before the next block whose rows were not listed
        const int endmax = by_list ? min(nblk, max(start + rblk, next_dense(start))) : min(nblk, start + rblk);
        int lo = start, hi = endmax - 1;  // last b in [start, endmax) with bpre[b] <= lim
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (bpre[mid] <= lim) lo = mid;
          else hi = mid - 1;
        }
        // a unit whose first blocks alone fill half the value window stops
        // at the window's rows, so the numeric pass handles it in one sweep
        const int dl = max(kmax / kBR, 1);
        if (lo - start + 1 > dl && bpre[start + dl - 1] - before >= kmax / 2) lo = start + dl - 1;
        const int c = bpre[lo] - before;
        if (c > 0) {
          Unit& u = (by_list && lo + 1 - start > rblk) ? su2[ns++] : su[nu++];
          u.col = col;
          u.blk_lo = t_lo + start;
          u.blk_hi = t_lo + lo + 1;
          u.cnt = c;
          u.off = unit_off;
          u.slot = (int32_t)blockIdx.x;
          unit_off += c;
        }
        before = bpre[lo];
        start = lo + 1;
      }
      s_nu = nu;
      s_ns = ns;
      int* cnt = heavy ? n_h : n_l;
      s_slot = nu ? atomicAdd(cnt, nu) : 0;
      if (s_slot + nu > (heavy ? cap_h : cap_l)) atomicOr(err, 32);
      s_sslot = ns ? atomicAdd(n_s, ns) : 0;
      if (ns && s_sslot + ns > cap_s) atomicOr(err, 32);
    }
    __syncthreads();
    {
      const bool heavy = pass_total > heavy_thr;
      Unit* dst = heavy ? units_h : units_l;
      const int cap = heavy ? cap_h : cap_l;
      for (int i = threadIdx.x; i < s_nu; i += NT)
        if (s_slot + i < cap) dst[s_slot + i] = su[i];
      for (int i = threadIdx.x; i < s_ns; i += NT)
        if (s_sslot + i < cap_s) units_s[s_sslot + i] = su2[i];
    }
    colcnt += pass_total;
    __syncthreads();
  }
  if (threadIdx.x == 0) nnzcol[col] = colcnt;
}

// Banded form of the same symbolic pass, in two kernels.  k_sym_band runs one
// workgroup per (column, band of IBLK row blocks) with the band as the slow
// grid dimension, so the workgroups in flight at any moment gather only the
// A entries of one band of rows (IBLK * 4096 rows: about nnz(A) * IBLK / S
// entries, which the L2 caches can hold), where the per-column pass sweeps
// every band of a few columns.  It builds the band's presence bitmap, keeps
// the row-map slice, and writes the band's per-block counts.  k_sym_cut then
// cuts every column into units from its block counts, as k_sym_units does.
template <int NT, int U, int IBLK>
__global__ __launch_bounds__(NT) void k_sym_band(const int32_t* __restrict__ order, int64_t first,
                                                 const int64_t* __restrict__ cpB, const int32_t* __restrict__ bpos,
                                                 const int64_t* __restrict__ cpA, const int32_t* __restrict__ rowsA,
                                                 const Tiles P, int S, int32_t* __restrict__ bcnt,
                                                 uint32_t* __restrict__ rmap, int64_t rm_cols) {
  constexpr int BMW = IBLK * kBRW;  // bitmap words of one band
  __shared__ uint32_t bits[BMW];
  __shared__ FlatStage<uint8_t, NT, false> st;
  const int64_t slot = blockIdx.x;  // the column's position in the launch
  const int col = order[first + slot];
  const int i_lo = (int)blockIdx.y * IBLK, i_hi = min(S, i_lo + IBLK), inb = i_hi - i_lo;
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  const int32_t row0 = i_lo * kBR;
  const bool whole = S <= IBLK;  // one band covers every row: no tile look-ups
  for (int i = threadIdx.x; i < inb * kBRW; i += NT) bits[i] = 0u;
  // (the staging barrier below orders the clear before any insertion)
  int par = 0;
  flat_init(st);
  for (int64_t eb = b0; eb < b1; eb += NT) {
    int64_t base;
    int len;
    uint8_t dummy;
    load_seg<uint8_t, false>(eb + threadIdx.x, b1, bpos, cpA, P, i_lo, i_hi, whole, nullptr, base, len, dummy);
    const FlatSeg me = flat_stage<uint8_t, NT, false>(st, (int32_t)base, len, 0);
    flat_chunk<uint8_t, NT, false, U>(st, me, par, [&](const int32_t(&idx)[U], uint8_t(&)[U], const bool(&ok)[U]) {
      int32_t r[U];
      load_rows(rowsA, row0, idx, r);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ok[u]) atomicOr(&bits[r[u] >> 5], 1u << (r[u] & 31));
    });
  }
  __syncthreads();
  if (rmap && slot < rm_cols) {
    uint32_t* dst = rmap + slot * S * kBRW + (int64_t)i_lo * kBRW;
    for (int i = threadIdx.x; i < inb * kBRW; i += NT) dst[i] = bits[i];
  }
  for (int b = wave_id(); b < inb; b += NT / kWave) {  // one wave per block, two words per lane
    const uint32_t* wv = bits + b * kBRW;
    int c = __popc(wv[lane_id()]) + __popc(wv[lane_id() + kWave]);
    c = (int)wave_sum_ll(c);
    if (lane_id() == 0) bcnt[slot * S + i_lo + b] = c;
  }
}

// Unit cutting of the banded symbolic pass: one workgroup of 256 threads per
// column, over passes of 256 blocks, with the greedy rule of k_sym_units.
__global__ __launch_bounds__(256) void k_sym_cut(const int32_t* __restrict__ order, int64_t first,
                                                 const int32_t* __restrict__ bcnt, int S, int kmax_l, int rblk_l,
                                                 int kmax_h, int rblk_h, int64_t heavy_thr,
                                                 int64_t* __restrict__ nnzcol, Unit* __restrict__ units_l,
                                                 int* __restrict__ n_l, int cap_l, Unit* __restrict__ units_h,
                                                 int* __restrict__ n_h, int cap_h, int* __restrict__ err) {
  constexpr int BPP = 256;
  __shared__ int bpre[BPP];
  __shared__ Unit su[BPP];
  __shared__ long long wsum[256 / kWave];
  __shared__ int s_nu, s_slot;
  const int64_t slot = blockIdx.x;
  const int col = order[first + slot];
  const int npass = (S + BPP - 1) / BPP;
  int64_t colcnt = 0;
  int unit_off = 0;  // meaningful in thread 0 only
  for (int sp = 0; sp < npass; ++sp) {
    const int t_lo = sp * BPP, nblk = min(S, t_lo + BPP) - t_lo;
    const int c = (int)threadIdx.x < nblk ? bcnt[slot * S + t_lo + threadIdx.x] : 0;
    long long total;
    const long long ex = block_excl_scan_ll<256>(c, wsum, total);
    bpre[threadIdx.x] = (int)(ex + c);  // inclusive prefix over the pass's blocks
    __syncthreads();
    const int pass_total = (int)total;
    if (threadIdx.x == 0) {
      const bool heavy = pass_total > heavy_thr;
      const int kmax = heavy ? kmax_h : kmax_l, rblk = heavy ? rblk_h : rblk_l;
      int start = 0, before = 0, nu = 0;
      while (start < nblk) {
        const int lim = before + kmax;
        const int endmax = min(nblk, start + rblk);
        int lo = start, hi = endmax - 1;  // last b in [start, endmax) with bpre[b] <= lim
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (bpre[mid] <= lim) lo = mid;
          else hi = mid - 1;
        }
        const int dl = max(kmax / kBR, 1);
        if (lo - start + 1 > dl && bpre[start + dl - 1] - before >= kmax / 2) lo = start + dl - 1;
        const int cu = bpre[lo] - before;
        if (cu > 0) {
          su[nu].col = col;
          su[nu].blk_lo = t_lo + start;
          su[nu].blk_hi = t_lo + lo + 1;
          su[nu].cnt = cu;
          su[nu].off = unit_off;
          su[nu].slot = (int32_t)slot;
          unit_off += cu;
          ++nu;
        }
        before = bpre[lo];
        start = lo + 1;
      }
      s_nu = nu;
      int* cnt = heavy ? n_h : n_l;
      s_slot = nu ? atomicAdd(cnt, nu) : 0;
      if (s_slot + nu > (heavy ? cap_h : cap_l)) atomicOr(err, 32);
    }
    __syncthreads();
    {
      const bool heavy = pass_total > heavy_thr;
      Unit* dst = heavy ? units_h : units_l;
      const int cap = heavy ? cap_h : cap_l;
      for (int i = threadIdx.x; i < s_nu; i += 256)
        if (s_slot + i < cap) dst[s_slot + i] = su[i];
    }
    colcnt += pass_total;
    __syncthreads();
  }
  if (threadIdx.x == 0) nnzcol[col] = colcnt;
}

// A unit's accumulators: vals[row] for the DR rows of a direct unit (at most
// DR / kBR blocks), or vals[rank] with the rows of its KMAX outputs at most
// behind them (16 bits each: a unit spans at most 16 blocks).  Every product
// leaves its row at its rank as it accumulates, so rows are emitted like
// values; rebuilding them from the bitmap's words, as many steps as the
// fullest of 64 words had outputs, took as long as a third of the unit.
template <class Lds, int KMAX, int DR>
struct UnitWindow {
  static constexpr size_t bytes =
      sizeof(Lds) * DR > (sizeof(Lds) + 2) * KMAX ? sizeof(Lds) * DR : (sizeof(Lds) + 2) * KMAX;
  __align__(16) unsigned char mem[bytes];
  __device__ __forceinline__ Lds* vals() { return reinterpret_cast<Lds*>(mem); }
  __device__ __forceinline__ uint16_t* rows() { return reinterpret_cast<uint16_t*>(mem + sizeof(Lds) * KMAX); }
};

// pre[w] = outputs of the unit below bitmap word w, four words per thread and
// step; returns their number.  Contains barriers.
template <int NT, int NW32>
__device__ __forceinline__ int unit_prefix(const uint32_t* bits, uint16_t* pre, int nw32, int* isum) {
  static_assert(NW32 % 4 == 0 && NW32 <= 4 * NT, "one step");
  const int w = threadIdx.x * 4;
  uint4 q{0, 0, 0, 0};
  if (w < nw32) q = *reinterpret_cast<const uint4*>(bits + w);
  const int c0 = __popc(q.x), c1 = c0 + __popc(q.y), c2 = c1 + __popc(q.z), c3 = c2 + __popc(q.w);
  int total;
  const int ex = block_excl_scan<NT>(c3, isum, total);
  if (w < nw32) {
    const uint2 p{(uint32_t)ex | (uint32_t)(ex + c0) << 16, (uint32_t)(ex + c1) | (uint32_t)(ex + c2) << 16};
    *reinterpret_cast<uint2*>(pre + w) = p;
  }
  __syncthreads();
  return total;
}

// Emission of a unit's cnt outputs at `out`, rows ascending: from rows and
// vals in rank order, or (direct) from the rows present in the window, a wave
// per 64 rows.
template <int K, class T, int NT, int KMAX, int DR, class R>
__device__ __forceinline__ void unit_emit(bool direct, int nw32, int cnt, const uint32_t* bits, const uint16_t* pre,
                                          UnitWindow<typename Sem<K, T>::Lds, KMAX, DR>& win, int32_t row0,
                                          int64_t out, R* __restrict__ irC, T* __restrict__ valC,
                                          const Filter<T>& flt, int col, int* isum, int* err) {
  using SR = Sem<K, T>;
  constexpr int NW = NT / kWave;
  auto* vals = win.vals();
  const uint16_t* rows = win.rows();
  if (sizeof(R) == 8 && flt.on) {
    auto in_window = [&](int i, T& v) {
      v = SR::lout(vals[i]);
      return ((bits[i >> 5] >> (i & 31)) & 1u) != 0;
    };
    auto at_rank = [&](int i, T& v) {
      v = SR::lout(vals[i]);
      return true;
    };
    if (direct)
      emit_filtered<T, NT>(nw32 * 32, cnt, in_window, [&](int i) { return (int64_t)row0 + i; }, out, (int64_t*)irC, valC, flt,
                           col, isum, err);
    else
      emit_filtered<T, NT>(cnt, cnt, at_rank, [&](int i) { return (int64_t)row0 + rows[i]; }, out, (int64_t*)irC, valC, flt, col,
                           isum, err);
    return;
  }
  if (direct) {
    for (int q = wave_id_uniform(); q < nw32 / 2; q += NW) {
      const uint32_t lo = __builtin_amdgcn_readfirstlane(bits[2 * q]);
      const uint32_t hi = __builtin_amdgcn_readfirstlane(bits[2 * q + 1]);
      const uint32_t p = __builtin_amdgcn_readfirstlane((int)pre[2 * q]);
      const int at = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, p));
      const int r = q * 64 + lane_id();
      if (((lane_id() < 32 ? lo : hi) >> (lane_id() & 31) & 1u) && at < cnt) {
        irC[out + at] = (R)(row0 + r);
        valC[out + at] = SR::lout(vals[r]);
      }
    }
    return;
  }
  for (int i = threadIdx.x; i < cnt; i += NT) {
    irC[out + i] = (R)(row0 + rows[i]);
    valC[out + i] = SR::lout(vals[i]);
  }
}

// Numeric pass of the unit tier: one workgroup per unit.  Sweep 1 sets the
// unit's presence bitmap, a block scan turns it into per-word ranks, sweep 2
// accumulates every product at its row's rank.  When the column's B entries
// fit one chunk, the first CR rounds of products (row, product value) stay in
// registers between the sweeps, so sweep 2 re-reads nothing for them.
// Waves per SIMD the small-unit kernel asks for, as many as its LDS allows:
// eight for a value window of at most 16 KB (4-byte accumulators; 64 VGPRs),
// else six (three 512-thread workgroups of 53 KB; 80 VGPRs).  Left alone, the
// compiler takes 84 to 86 for 8-byte values, and a third workgroup stays out.
template <class Lds, int NT, int DR>
struct UnitWaves {
  static constexpr int value = NT != 512 ? 1 : sizeof(Lds) * DR <= 16384 ? 8 : 6;
};

template <int K, class T, int NT, int U, int KMAX, int DR, int RBLK, int CR>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(
    UnitWaves<typename Sem<K, T>::Lds, NT, DR>::value))) void k_num_units(const Unit* __restrict__ units,
                                                                            const int64_t* __restrict__ cpB,
                                                  const int32_t* __restrict__ bpos, const T* __restrict__ valB,
                                                  const int64_t* __restrict__ cpA, const int32_t* __restrict__ rowsA,
                                                  const T* __restrict__ valA, const Tiles P, int S,
                                                  const int64_t* __restrict__ cpC, int64_t* __restrict__ irC,
                                                  T* __restrict__ valC, int* __restrict__ err, Filter<T> flt = {}, int xg = 0) {
  using SR = Sem<K, T>;
  using Acc = typename SR::Acc;
  constexpr int NW32 = RBLK * kBRW;   // bitmap words
  __shared__ UnitWindow<typename SR::Lds, KMAX, DR> win;
  __shared__ __align__(16) uint32_t bits[NW32];
  __shared__ __align__(8) uint16_t pre[NW32];
  __shared__ FlatStage<T, NT, true> st;
  __shared__ int isum[NT / kWave];
  auto* vals = win.vals();
  uint16_t* rows = win.rows();
  const Unit un = units[xcd_unit((int)blockIdx.x, (int)gridDim.x, xg)];
  const int col = un.col;
  const int t_lo = un.blk_lo, t_hi = un.blk_hi;
  const int32_t row0 = t_lo * kBR;
  const int cnt = un.cnt;
  const int64_t out = cpC[col] + un.off;
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  // A unit whose rows fit the value window (dense output) accumulates at
  // vals[row - row0] in a single sweep; the others count first and
  // accumulate at the rank in a second sweep.
  const bool direct = (t_hi - t_lo) * kBR <= DR;
  const bool single_chunk = !direct && (b1 - b0) <= NT;
  if ((!direct && cnt > KMAX) || t_hi - t_lo > RBLK) {  // units are cut to fit; guard anyway
    if (threadIdx.x == 0) atomicOr(err, 64);
    return;
  }
  const int ninit = direct ? (t_hi - t_lo) * kBR : cnt;
  flat_init(st);
  for (int i = threadIdx.x; i < ninit; i += NT) vals[i] = SR::lident();
  const int nw32 = (t_hi - t_lo) * kBRW;
  for (int i = threadIdx.x; i < nw32; i += NT) bits[i] = 0u;

  auto set_bits = [&](const int32_t(&idx)[U], T(&)[U], const bool(&ok)[U]) {
    int32_t r[U];
    load_rows(rowsA, row0, idx, r);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (ok[u]) atomicOr(&bits[r[u] >> 5], 1u << (r[u] & 31));
  };
  auto rank_of = [&](int32_t r) {
    const int w = r >> 5;
    return (int)pre[w] + __popc(__builtin_amdgcn_ubfe(bits[w], 0, r & 31));
  };
  auto ranks_of = [&](const int32_t(&r)[U], int(&rank)[U]) {  // all the LDS reads in flight together
#pragma unroll
    for (int u = 0; u < U; ++u) rank[u] = rank_of(r[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) pin(rank[u]);
  };
  auto accumulate = [&](const int32_t(&idx)[U], T(&bvs)[U], const bool(&ok)[U]) {
    int32_t r[U];
    T a[U];
    load_entries(rowsA, valA, row0, idx, bvs, r, a);
    int rank[U];
    ranks_of(r, rank);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (ok[u] && rank[u] < cnt) {
        SR::acc(&vals[rank[u]], SR::mul(a[u], bvs[u]));
        rows[rank[u]] = (uint16_t)r[u];
      }
  };

  int32_t crow[CR][U];
  Acc cprod[CR][U];
  int par = 0;
  FlatSeg me{};
  FlatTile ft{};
  bool cached = false;  // the only chunk is one tile: its first CR rounds stay in registers
  unsigned cok = 0;     // which of them are products
  auto acc_direct = [&](const int32_t(&idx)[U], T(&bvs)[U], const bool(&ok)[U]) {
    int32_t r[U];
    T a[U];
    load_entries(rowsA, valA, row0, idx, bvs, r, a);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (ok[u]) {
        atomicOr(&bits[r[u] >> 5], 1u << (r[u] & 31));
        SR::acc(&vals[r[u]], SR::mul(a[u], bvs[u]));
      }
  };
  // sweep 1 (the staging barrier orders the initialisation before any insertion)
  for (int64_t eb = b0; eb < b1; eb += NT) {
    int64_t base;
    int len;
    T bv;
    load_seg<T, true>(eb + threadIdx.x, b1, bpos, cpA, P, t_lo, t_hi, false, valB, base, len, bv);
    me = flat_stage<T, NT, true>(st, (int32_t)base, len, bv);
    cached = single_chunk && me.total <= kTileProducts;
    if (cached) {
      ft = flat_tile(st, me, 0, 0, par);
      par ^= 1;
#pragma unroll
      for (int rr = 0; rr < CR; ++rr) {
#pragma unroll
        for (int u = 0; u < U; ++u) crow[rr][u] = 0;
        if (rr * U * (NT / kWave) + wave_id_uniform() >= flat_words(ft, me.total)) continue;
        int32_t idx[U];
        T bvs[U], a[U];
        bool ok[U];
        flat_round<T, NT, true, U>(st, ft, me.total, rr, idx, bvs, ok);
        load_entries(rowsA, valA, row0, idx, bvs, crow[rr], a);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          cprod[rr][u] = SR::mul(a[u], bvs[u]);
          if (ok[u]) {
            cok |= 1u << (rr * U + u);
            atomicOr(&bits[crow[rr][u] >> 5], 1u << (crow[rr][u] & 31));
          }
        }
      }
      flat_visit<T, NT, true, U>(st, ft, me.total, set_bits, CR);
    } else if (direct) {
      flat_chunk<T, NT, true, U>(st, me, par, acc_direct);
    } else {
      flat_chunk<T, NT, true, U>(st, me, par, set_bits);
    }
  }
  __syncthreads();
  const int total = unit_prefix<NT, NW32>(bits, pre, nw32, isum);
  if (threadIdx.x == 0 && total != cnt) atomicOr(err, 128);
  if (direct) {  // values already sit at their rows
    unit_emit<K, T, NT, KMAX, DR>(true, nw32, cnt, bits, pre, win, row0, out, irC, valC, flt, col, isum, err);
    return;
  }
  // sweep 2: accumulate values at their ranks
  if (cached) {
#pragma unroll
    for (int rr = 0; rr < CR; ++rr) {
      int rank[U];
      ranks_of(crow[rr], rank);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if ((cok >> (rr * U + u) & 1u) && rank[u] < cnt) {
          SR::acc(&vals[rank[u]], cprod[rr][u]);
          rows[rank[u]] = (uint16_t)crow[rr][u];
        }
    }
    flat_visit<T, NT, true, U>(st, ft, me.total, accumulate, CR);
  } else {
    for (int64_t eb = b0; eb < b1; eb += NT) {
      int64_t base;
      int len;
      T bv;
      load_seg<T, true>(eb + threadIdx.x, b1, bpos, cpA, P, t_lo, t_hi, false, valB, base, len, bv);
      me = flat_stage<T, NT, true>(st, (int32_t)base, len, bv);
      flat_chunk<T, NT, true, U>(st, me, par, accumulate);
    }
  }
  __syncthreads();
  unit_emit<K, T, NT, KMAX, DR>(false, nw32, cnt, bits, pre, win, row0, out, irC, valC, flt, col, isum, err);
}

// Numeric pass of the unit tier with the symbolic pass's row map: the unit's
// presence bitmap is loaded (coalesced) instead of rebuilt, ranks come from
// its prefix popcounts, and one sweep gathers every product once and
// accumulates it at its rank (at its row for a unit whose rows fit the value
// window).
template <int K, class T, int NT, int U, int KMAX, int DR, int RBLK>
__global__ __launch_bounds__(NT) void k_num_units_rm(const Unit* __restrict__ units, const uint32_t* __restrict__ rmap,
                                                     const int64_t* __restrict__ cpB, const int32_t* __restrict__ bpos,
                                                     const T* __restrict__ valB, const int64_t* __restrict__ cpA,
                                                     const int32_t* __restrict__ rowsA, const T* __restrict__ valA,
                                                     const Tiles P, int S, int64_t rm_cols,
                                                     const int64_t* __restrict__ cpC, int64_t* __restrict__ irC,
                                                     T* __restrict__ valC, int* __restrict__ err,
                                                     Filter<T> flt = {}, int xg = 0) {
  using SR = Sem<K, T>;
  using Acc = typename SR::Acc;
  constexpr int NW32 = RBLK * kBRW;
  __shared__ UnitWindow<typename SR::Lds, KMAX, DR> win;
  __shared__ __align__(16) uint32_t bits[NW32];
  __shared__ __align__(8) uint16_t pre[NW32];
  __shared__ FlatStage<T, NT, true> st;
  __shared__ int isum[NT / kWave];
  auto* vals = win.vals();
  uint16_t* rows = win.rows();
  const Unit un = units[xcd_unit((int)blockIdx.x, (int)gridDim.x, xg)];
  const int col = un.col;
  const int t_lo = un.blk_lo, t_hi = un.blk_hi;
  const int32_t row0 = t_lo * kBR;
  const int cnt = un.cnt;
  const int64_t out = cpC[col] + un.off;
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  const bool direct = (t_hi - t_lo) * kBR <= DR;
  if ((!direct && cnt > KMAX) || t_hi - t_lo > RBLK || t_lo < 0 || t_hi > S || un.slot < 0 || un.slot >= rm_cols) {
    if (threadIdx.x == 0) atomicOr(err, 64);
    return;
  }
  const int ninit = direct ? (t_hi - t_lo) * kBR : cnt;
  flat_init(st);
  for (int i = threadIdx.x; i < ninit; i += NT) vals[i] = SR::lident();
  const int nw32 = (t_hi - t_lo) * kBRW;
  const uint32_t* src = rmap + (int64_t)un.slot * S * kBRW + (int64_t)t_lo * kBRW;
  for (int i = threadIdx.x; i < nw32; i += NT) bits[i] = src[i];
  __syncthreads();
  const int total = unit_prefix<NT, NW32>(bits, pre, nw32, isum);
  if (threadIdx.x == 0 && total != cnt) atomicOr(err, 128);
  auto rank_of = [&](int32_t r) {
    const int w = r >> 5;
    return (int)pre[w] + __popc(__builtin_amdgcn_ubfe(bits[w], 0, r & 31));
  };
  auto ranks_of = [&](const int32_t(&r)[U], int(&rank)[U]) {  // all the LDS reads in flight together
#pragma unroll
    for (int u = 0; u < U; ++u) rank[u] = rank_of(r[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) pin(rank[u]);
  };
  auto accumulate = [&](const int32_t(&idx)[U], T(&bvs)[U], const bool(&ok)[U]) {
    int32_t r[U];
    T a[U];
    load_entries(rowsA, valA, row0, idx, bvs, r, a);
    int q[U];
    if (direct) {
#pragma unroll
      for (int u = 0; u < U; ++u) q[u] = r[u];
    } else {
      ranks_of(r, q);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (ok[u] && q[u] < (direct ? ninit : cnt)) {
        SR::acc(&vals[q[u]], SR::mul(a[u], bvs[u]));
        if (!direct) rows[q[u]] = (uint16_t)r[u];
      }
  };
  int par = 0;
  for (int64_t eb = b0; eb < b1; eb += NT) {
    int64_t base;
    int len;
    T bv;
    load_seg<T, true>(eb + threadIdx.x, b1, bpos, cpA, P, t_lo, t_hi, false, valB, base, len, bv);
    const FlatSeg me = flat_stage<T, NT, true>(st, (int32_t)base, len, bv);
    flat_chunk<T, NT, true, U>(st, me, par, accumulate);
  }
  __syncthreads();
  unit_emit<K, T, NT, KMAX, DR>(direct, nw32, cnt, bits, pre, win, row0, out, irC, valC, flt, col, isum, err);
}

// Numeric pass of the list units: at most KMAX outputs of one column over
// any number of the row blocks of one 256-block pass.  Their ranks come from
// the column's sorted row list that the symbolic pass wrote (12-bit offsets
// grouped by block, with per-block counts), so one sweep gathers every
// product once: a product's rank is its block's first list position plus a
// binary search among that block's offsets.  Units this sparse would need a
// bitmap of up to 256 blocks (128 KB), or many narrow units that each
// re-read the B column and gather one- or two-entry A segments.
template <int K, class T, int NT, int U, int KMAX>
__global__ __launch_bounds__(NT) void k_num_list(const Unit* __restrict__ units, const uint16_t* __restrict__ lists,
                                                 const int64_t* __restrict__ list_off,
                                                 const uint16_t* __restrict__ bcnt16, const int64_t* __restrict__ cpB,
                                                 const int32_t* __restrict__ bpos, const T* __restrict__ valB,
                                                 const int64_t* __restrict__ cpA, const int32_t* __restrict__ rowsA,
                                                 const T* __restrict__ valA, const Tiles P, int S,
                                                 const int64_t* __restrict__ cpC, int64_t* __restrict__ irC,
                                                 T* __restrict__ valC, int* __restrict__ err, Filter<T> flt = {}, int xg = 0) {
  using SR = Sem<K, T>;
  using Acc = typename SR::Acc;
  constexpr int BPP = 256;  // blocks of one symbolic cutting pass
  static_assert(NT > BPP, "one block count per thread, plus the total");
  __shared__ typename SR::Lds vals[KMAX];
  __shared__ uint16_t lst[KMAX];
  __shared__ int s_full[NT / kWave];  // each wave's blocks: none with 16 outputs, some with 16, some with 64
  __shared__ int dir[BPP + 1];  // list position of each block's first row; dir[nb] = cnt
  __shared__ FlatStage<T, NT, true> st;
  __shared__ long long wsum[NT / kWave];
  const Unit un = units[xcd_unit((int)blockIdx.x, (int)gridDim.x, xg)];
  const int col = un.col;
  const int t_lo = un.blk_lo, t_hi = un.blk_hi, nb = t_hi - t_lo;
  const int32_t row0 = t_lo * kBR;
  const int cnt = un.cnt;
  const int64_t out = cpC[col] + un.off;
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  if (cnt > KMAX || nb <= 0 || nb > BPP) {  // units are cut to fit; guard anyway
    if (threadIdx.x == 0) atomicOr(err, 64);
    return;
  }
  flat_init(st);
  const uint16_t* src = lists + list_off[un.slot] + un.off;
  for (int i = threadIdx.x; i < cnt; i += NT) {
    lst[i] = src[i];
    vals[i] = SR::lident();
  }
  {
    const int c = threadIdx.x < nb ? (int)bcnt16[(int64_t)un.slot * S + t_lo + threadIdx.x] : 0;
    long long tot;
    const int ex = (int)block_excl_scan_ll<NT>(c, wsum, tot);  // barriers: lst and vals are ready after it
    if (tot != cnt) {  // the counts and the unit disagree (uniform): positions would leave the list
      if (threadIdx.x == 0) atomicOr(err, 128);
      return;
    }
    if (threadIdx.x <= nb) dir[threadIdx.x] = ex;
    const unsigned long long wide = __ballot(c >= 16), wider = __ballot(c >= 64);
    if (lane_id() == 0) s_full[wave_id()] = wider ? 2 : wide ? 1 : 0;
  }
  __syncthreads();
  int top = 8;  // the search's first step: half the power of two above the fullest block's count
#pragma unroll
  for (int i = 0; i < NT / kWave; ++i) top = max(top, s_full[i] == 2 ? 128 : s_full[i] == 1 ? 32 : 8);
  auto accumulate = [&](const int32_t(&idx)[U], T(&bvs)[U], const bool(&ok)[U]) {
    int32_t r[U];
    T a[U];
    load_entries(rowsA, valA, row0, idx, bvs, r, a);
    // first position in the row's block with an offset not below the row's:
    // all U searches step together, with as many steps as the unit's fullest
    // block needs
    int pos[U], end[U], off[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int b = r[u] >> 12;  // kBR = 4096 rows per block
      off[u] = r[u] & (kBR - 1);
      pos[u] = dir[b];
      end[u] = dir[b + 1];
    }
    for (int step = top; step > 0; step >>= 1) {
      int v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = (int)lst[min(pos[u] + step, end[u]) - 1];
#pragma unroll
      for (int u = 0; u < U; ++u) pin(v[u]);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (pos[u] + step <= end[u] && v[u] < off[u]) pos[u] += step;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!ok[u]) continue;
      if (pos[u] < end[u] && lst[pos[u]] == off[u]) SR::acc(&vals[pos[u]], SR::mul(a[u], bvs[u]));
      else atomicOr(err, 4);  // symbolic and numeric agree; guard anyway
    }
  };
  int par = 0;
  for (int64_t eb = b0; eb < b1; eb += NT) {
    int64_t base;
    int len;
    T bv;
    load_seg<T, true>(eb + threadIdx.x, b1, bpos, cpA, P, t_lo, t_hi, false, valB, base, len, bv);
    const FlatSeg me = flat_stage<T, NT, true>(st, (int32_t)base, len, bv);
    flat_chunk<T, NT, true, U>(st, me, par, accumulate);
  }
  __syncthreads();
  auto row_of = [&](int i) {  // the block holding list position i: largest b with dir[b] <= i
    int lo = 0, hi = nb;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (dir[mid] <= i) lo = mid;
      else hi = mid;
    }
    return (int64_t)row0 + (int64_t)lo * kBR + lst[i];
  };
  if (!flt.on) {
    for (int i = threadIdx.x; i < cnt; i += NT) {
      irC[out + i] = row_of(i);
      valC[out + i] = SR::lout(vals[i]);
    }
    return;
  }
  auto item = [&](int i, T& v) {
    v = SR::lout(vals[i]);
    return true;
  };
  emit_filtered<T, NT>(cnt, cnt, item, row_of, out, irC, valC, flt, col, s_full, err);
}

// Predictor features per stored column of B (one wave per column); see
// cbx_spgemm_features in cbx.h for the list.
__global__ void k_features(const int64_t* __restrict__ cpB, int64_t nzcB, const int32_t* __restrict__ bpos,
                           const int64_t* __restrict__ cpA, const int32_t* __restrict__ rowsA, int64_t m,
                           float* __restrict__ feats) {
  const int64_t col = global_wave();
  if (col >= nzcB) return;
  const int lane = lane_id();
  long long f = 0, mx = 0, lo = m, hi = -1;
  for (int64_t e = cpB[col] + lane; e < cpB[col + 1]; e += kWave) {
    const int32_t p = bpos[e];
    if (p < 0) continue;
    const int64_t a0 = cpA[p], a1 = cpA[p + 1];
    if (a1 == a0) continue;
    const long long len = a1 - a0;
    f += len;
    mx = len > mx ? len : mx;
    const long long r0 = rowsA[a0], r1 = rowsA[a1 - 1];
    lo = r0 < lo ? r0 : lo;
    hi = r1 > hi ? r1 : hi;
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    f += __shfl_xor(f, d, kWave);
    const long long m2 = __shfl_xor(mx, d, kWave);
    mx = m2 > mx ? m2 : mx;
    const long long l2 = __shfl_xor(lo, d, kWave);
    lo = l2 < lo ? l2 : lo;
    const long long h2 = __shfl_xor(hi, d, kWave);
    hi = h2 > hi ? h2 : hi;
  }
  if (lane != 0) return;
  const double b = (double)(cpB[col + 1] - cpB[col]);
  const double span = f > 0 ? (double)(hi - lo + 1) : 0.0;
  const double est = span > 0 ? span * (1.0 - exp(-(double)f / span)) : 0.0;
  float* o = feats + col * CBX_MLP_FEATURES;
  o[0] = (float)log2(1.0 + b);
  o[1] = (float)log2(1.0 + (double)f);
  o[2] = (float)log2(1.0 + (double)mx);
  o[3] = (float)log2(1.0 + (double)f / (b > 0 ? b : 1.0));
  o[4] = (float)(span / (double)(m > 0 ? m : 1));
  o[5] = (float)log2(1.0 + est);
}

// ============================================================ learned tier
// Single pass: units are cut from predicted column sizes; a unit counts its
// outputs from its bitmap, takes room for them from a running total, writes
// them there (32-bit rows) and moves on.  Once all sizes are known a copy puts
// every unit's outputs at its place.
//
// The copy (24 B per output more than writing in place) buys units that wait
// for nobody.  With their places taken from a look-back over the units before
// them, units retired in order: a unit that waits keeps its workgroup's LDS,
// and a hub's dense blocks, of up to 1e5 products, held up the 768 units in
// flight again and again.  At 2^17 vertices, edge factor 16, that kernel took
// 13.2 ms with its VALU 18 % busy.
struct UnitL {
  int32_t col;
  int32_t blk_lo;
  int32_t blk_hi;
};

// Row histogram of A over kBR-row blocks (the prior that spreads a
// predicted column size over the blocks).
__global__ void k_row_hist(const int32_t* __restrict__ rowsA, int64_t nnzA, int S, unsigned long long* __restrict__ hist) {
  extern __shared__ unsigned int lh[];
  for (int b = threadIdx.x; b < S; b += blockDim.x) lh[b] = 0;
  __syncthreads();
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nnzA; i += (int64_t)gridDim.x * blockDim.x)
    atomicAdd(&lh[rowsA[i] / kBR], 1u);
  __syncthreads();
  for (int b = threadIdx.x; b < S; b += blockDim.x)
    if (lh[b]) atomicAdd(&hist[b], (unsigned long long)lh[b]);
}

// Lowest and highest output row block a column can touch (from the first and
// last row of every contributing A column).  One wave per column.
__global__ void k_col_blocks(const int64_t* __restrict__ cpB, int64_t nzcB, const int32_t* __restrict__ bpos,
                             const int64_t* __restrict__ cpA, const int32_t* __restrict__ rowsA,
                             int32_t* __restrict__ blo, int32_t* __restrict__ bhi) {
  const int64_t col = global_wave();
  if (col >= nzcB) return;
  int lo = 0x7fffffff, hi = -1;
  for (int64_t e = cpB[col] + lane_id(); e < cpB[col + 1]; e += kWave) {
    const int32_t p = bpos[e];
    if (p < 0) continue;
    const int64_t a0 = cpA[p], a1 = cpA[p + 1];
    if (a1 == a0) continue;
    lo = min(lo, rowsA[a0] / kBR);
    hi = max(hi, rowsA[a1 - 1] / kBR);
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    lo = min(lo, __shfl_xor(lo, d, kWave));
    hi = max(hi, __shfl_xor(hi, d, kWave));
  }
  if (lane_id() == 0) {
    blo[col] = lo;
    bhi[col] = hi;
  }
}

// Greedy cut of a column into units from expected block counts.  Block b of
// column j is expected to hold flop_j * w[b] products (w = A's row
// histogram) and, its 4096 rows each being hit at rate
// lambda = flop_j * w[b] / 4096, g_b = 4096 (1 - e^-lambda) distinct rows
// (saturating for dense columns, proportional to w for sparse ones); the
// predicted column size is spread over the blocks in proportion to g_b.  A
// block expected to hold at least direct_flop products forms a unit of its
// own (its rows fit the value window: one sweep, no counting sweep).  Other
// units close when their expected outputs would pass `target`, their
// expected products would pass `fcap`, or their span would pass rblk blocks.
// Capping the products keeps the units' work even.  Pass 1 counts (out == null),
// pass 2 writes at `base`.
__device__ __forceinline__ float distinct_rows(float flop, float wb) {
  return (float)kBR * (1.f - __expf(-flop * wb * (1.f / (float)kBR)));
}

__device__ __forceinline__ int cut_units(int col, float pred, float flop, int lo, int hi,
                                         const float* __restrict__ w, float target, float fcap, int rblk,
                                         float direct_flop, UnitL* out) {
  float gsum = 0.f;
  for (int b = lo; b <= hi; ++b) gsum += distinct_rows(flop, w[b]);
  const float scale = gsum > 0.f ? pred / gsum : 0.f;
  int n = 0, start = lo;
  float acc = 0.f, accf = 0.f;
  for (int b = lo; b <= hi; ++b) {
    const float e = scale * distinct_rows(flop, w[b]), ef = flop * w[b];
    if (ef >= direct_flop) {  // a block of its own, one sweep
      if (b > start) {
        if (out) out[n] = UnitL{col, start, b};
        ++n;
      }
      if (out) out[n] = UnitL{col, b, b + 1};
      ++n;
      start = b + 1;
      acc = 0.f;
      accf = 0.f;
      continue;
    }
    if (b > start && (acc + e > target || accf + ef > fcap || b - start >= rblk)) {
      if (out) out[n] = UnitL{col, start, b};
      ++n;
      start = b;
      acc = 0.f;
      accf = 0.f;
    }
    acc += e;
    accf += ef;
  }
  if (start <= hi) {
    if (out) out[n] = UnitL{col, start, hi + 1};
    ++n;
  }
  return n;
}

__global__ void k_learned_units(const int64_t* __restrict__ flop, int64_t nzcB, int64_t small_max,
                                const float* __restrict__ logpred, const int32_t* __restrict__ blo,
                                const int32_t* __restrict__ bhi, const float* __restrict__ w, float target,
                                float heavy_pred, float fcap, int rblk, float direct_flop, int64_t m,
                                const int64_t* __restrict__ ubase, int64_t* __restrict__ ucount,
                                UnitL* __restrict__ units, float* __restrict__ pred_nnz,
                                uint8_t* __restrict__ heavy_flag) {
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j >= nzcB) return;
  if (!units) heavy_flag[j] = 0;
  if (flop[j] <= small_max || bhi[j] < 0) {
    if (!units) {
      ucount[j] = 0;
      pred_nnz[j] = 0.f;
    }
    return;
  }
  float pred = exp2f(logpred[j]) - 1.f;
  const float cap = (float)min<int64_t>(flop[j], m);
  pred = fminf(fmaxf(pred, 1.f), cap);
  if (pred > heavy_pred) {  // predicted heavy: exact symbolic and the large two-phase units
    if (!units) {
      heavy_flag[j] = 1;
      ucount[j] = 0;
      pred_nnz[j] = 0.f;
    }
    return;
  }
  if (!units) {
    ucount[j] = cut_units((int)j, pred, (float)flop[j], blo[j], bhi[j], w, target, fcap, rblk, direct_flop, nullptr);
    pred_nnz[j] = pred;
  } else {
    cut_units((int)j, pred, (float)flop[j], blo[j], bhi[j], w, target, fcap, rblk, direct_flop, units + ubase[j]);
  }
}

// What the learned units write: sizes and places in the staging arrays, and
// the arrays with the running total of what is taken.
template <class T>
struct LearnedStage {
  int64_t* cnt;
  int64_t* at;
  unsigned long long* taken;
  int64_t cap;
  int32_t* rows;
  T* vals;
};

// One workgroup per unit, units first + blockIdx.x.
template <int K, class T, int NT, int U, int KMAX, int DR, int RBLK, int CR>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(
    UnitWaves<typename Sem<K, T>::Lds, NT, DR>::value))) void k_num_learned(
    const UnitL* __restrict__ units, int64_t first, const int64_t* __restrict__ cpB,
    const int32_t* __restrict__ bpos, const T* __restrict__ valB, const int64_t* __restrict__ cpA,
    const int32_t* __restrict__ rowsA, const T* __restrict__ valA, const Tiles P, int S,
    const LearnedStage<T> out, unsigned long long* __restrict__ col_total, int* __restrict__ ovf_units,
    int* __restrict__ err) {
  using SR = Sem<K, T>;
  using Acc = typename SR::Acc;
  constexpr int NW32 = RBLK * kBRW;
  __shared__ UnitWindow<typename SR::Lds, KMAX, DR> win;
  __shared__ __align__(16) uint32_t bits[NW32];
  __shared__ __align__(8) uint16_t pre[NW32];
  __shared__ FlatStage<T, NT, true> st;
  __shared__ int isum[NT / kWave];
  __shared__ long long s_at;
  auto* vals = win.vals();
  uint16_t* rows = win.rows();
  const int64_t t = first + blockIdx.x;
  const UnitL un = units[t];
  const int col = un.col, t_lo = un.blk_lo, t_hi = un.blk_hi;
  const int32_t row0 = t_lo * kBR;
  const int64_t b0 = cpB[col], b1 = cpB[col + 1];
  const bool single_chunk = (b1 - b0) <= NT;
  const int nw32 = min(t_hi - t_lo, RBLK) * kBRW;
  for (int i = threadIdx.x; i < nw32; i += NT) bits[i] = 0u;

  auto set_bits = [&](const int32_t(&idx)[U], T(&)[U], const bool(&ok)[U]) {
    int32_t r[U];
    load_rows(rowsA, row0, idx, r);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (ok[u]) atomicOr(&bits[r[u] >> 5], 1u << (r[u] & 31));
  };
  auto rank_of = [&](int32_t r) {
    const int w = r >> 5;
    return (int)pre[w] + __popc(__builtin_amdgcn_ubfe(bits[w], 0, r & 31));
  };
  auto ranks_of = [&](const int32_t(&r)[U], int(&rank)[U]) {  // all the LDS reads in flight together
#pragma unroll
    for (int u = 0; u < U; ++u) rank[u] = rank_of(r[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) pin(rank[u]);
  };
  int q0 = 0;  // first rank of the current value window
  auto accumulate = [&](const int32_t(&idx)[U], T(&bvs)[U], const bool(&ok)[U]) {
    int32_t r[U];
    T a[U];
    load_entries(rowsA, valA, row0, idx, bvs, r, a);
    int q[U];
    ranks_of(r, q);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (ok[u] && q[u] >= q0 && q[u] < q0 + KMAX) {
        SR::acc(&vals[q[u] - q0], SR::mul(a[u], bvs[u]));
        rows[q[u] - q0] = (uint16_t)r[u];
      }
  };

  int32_t crow[CR][U];
  Acc cprod[CR][U];
  int par = 0;
  FlatSeg me{};
  FlatTile ft{};
  bool cached = false;  // the only chunk is one tile: its first CR rounds stay in registers
  unsigned cok = 0;     // which of them are products
  flat_init(st);
  const bool valid = (t_hi - t_lo) <= RBLK;
  if (!valid && threadIdx.x == 0) atomicOr(err, 64);
  // A unit whose rows fit the value window accumulates at its rows in a
  // single sweep (its size, known after that sweep, never exceeds the window)
  const bool direct = valid && (t_hi - t_lo) * kBR <= DR;
  // the first window (the staging barrier orders it and the bitmap before any insertion)
  for (int i = threadIdx.x; i < (direct ? (t_hi - t_lo) * kBR : KMAX); i += NT) vals[i] = SR::lident();
  if (direct) {
    auto acc_direct = [&](const int32_t(&idx)[U], T(&bvs)[U], const bool(&ok)[U]) {
      int32_t r[U];
      T a[U];
      load_entries(rowsA, valA, row0, idx, bvs, r, a);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ok[u]) {
          atomicOr(&bits[r[u] >> 5], 1u << (r[u] & 31));
          SR::acc(&vals[r[u]], SR::mul(a[u], bvs[u]));
        }
    };
    for (int64_t eb = b0; eb < b1; eb += NT) {
      int64_t base;
      int len;
      T bv;
      load_seg<T, true>(eb + threadIdx.x, b1, bpos, cpA, P, t_lo, t_hi, false, valB, base, len, bv);
      me = flat_stage<T, NT, true>(st, (int32_t)base, len, bv);
      flat_chunk<T, NT, true, U>(st, me, par, acc_direct);
    }
  } else {
    for (int64_t eb = b0; eb < b1; eb += NT) {
      int64_t base;
      int len;
      T bv;
      load_seg<T, true>(eb + threadIdx.x, b1, bpos, cpA, P, t_lo, t_hi, false, valB, base, len, bv);
      if (!valid) len = 0;
      me = flat_stage<T, NT, true>(st, (int32_t)base, len, bv);
      cached = single_chunk && me.total <= kTileProducts;
      if (!cached) {
        flat_chunk<T, NT, true, U>(st, me, par, set_bits);
        continue;
      }
      ft = flat_tile(st, me, 0, 0, par);
      par ^= 1;
#pragma unroll
      for (int rr = 0; rr < CR; ++rr) {
#pragma unroll
        for (int u = 0; u < U; ++u) crow[rr][u] = 0;
        if (rr * U * (NT / kWave) + wave_id_uniform() >= flat_words(ft, me.total)) continue;
        int32_t idx[U];
        T bvs[U], a[U];
        bool ok[U];
        flat_round<T, NT, true, U>(st, ft, me.total, rr, idx, bvs, ok);
        load_entries(rowsA, valA, row0, idx, bvs, crow[rr], a);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          cprod[rr][u] = SR::mul(a[u], bvs[u]);
          if (ok[u]) {
            cok |= 1u << (rr * U + u);
            atomicOr(&bits[crow[rr][u] >> 5], 1u << (crow[rr][u] & 31));
          }
        }
      }
      flat_visit<T, NT, true, U>(st, ft, me.total, set_bits, CR);
    }
  }
  __syncthreads();
  const int cnt = unit_prefix<NT, NW32>(bits, pre, nw32, isum);
  if (threadIdx.x == 0) {
    const long long at = (long long)atomicAdd(out.taken, (unsigned long long)cnt);
    s_at = at;
    out.cnt[t] = cnt;
    out.at[t] = at;
    if (cnt) atomicAdd(&col_total[col], (unsigned long long)cnt);
    if (cnt > (direct ? DR : KMAX)) atomicAdd(ovf_units, 1);
    if (at + cnt > out.cap) atomicOr(err, 512);
  }
  if (direct) {
    __syncthreads();  // s_at
    if (s_at + cnt <= out.cap)
      unit_emit<K, T, NT, KMAX, DR, int32_t>(true, nw32, cnt, bits, pre, win, row0, s_at, out.rows, out.vals,
                                             Filter<T>{}, col, isum, err);
    return;
  }
  // values, in windows of KMAX ranks (one window unless the unit overflowed)
  for (q0 = 0; q0 < cnt; q0 += KMAX) {
    const int wn = min(KMAX, cnt - q0);
    if (q0) {
      __syncthreads();  // the previous window has been written
      for (int i = threadIdx.x; i < wn; i += NT) vals[i] = SR::lident();
      __syncthreads();
    }
    if (cached) {
#pragma unroll
      for (int rr = 0; rr < CR; ++rr) {
        int q[U];
        ranks_of(crow[rr], q);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if ((cok >> (rr * U + u) & 1u) && q[u] >= q0 && q[u] < q0 + KMAX) {
            SR::acc(&vals[q[u] - q0], cprod[rr][u]);
            rows[q[u] - q0] = (uint16_t)crow[rr][u];
          }
      }
      flat_visit<T, NT, true, U>(st, ft, me.total, accumulate, CR);
    } else {
      for (int64_t eb = b0; eb < b1; eb += NT) {
        int64_t base;
        int len;
        T bv;
        load_seg<T, true>(eb + threadIdx.x, b1, bpos, cpA, P, t_lo, t_hi, false, valB, base, len, bv);
        if (!valid) len = 0;
        me = flat_stage<T, NT, true>(st, (int32_t)base, len, bv);
        flat_chunk<T, NT, true, U>(st, me, par, accumulate);
      }
    }
    __syncthreads();
    const int64_t at = s_at;
    if (at + cnt <= out.cap)
      for (int i = threadIdx.x; i < wn; i += NT) {
        out.rows[at + q0 + i] = row0 + rows[i];
        out.vals[at + q0 + i] = SR::lout(vals[i]);
      }
  }
}

// A learned unit's outputs from the staging arrays into place: after the units
// before it (upto, the scan of the sizes) and the exactly sized columns before
// its own (hcs).  One workgroup per unit.
template <class T>
__global__ __launch_bounds__(256) void k_learned_place(const UnitL* __restrict__ units, int64_t first,
                                                       const LearnedStage<T> in, const int64_t* __restrict__ upto,
                                                       const int64_t* __restrict__ hcs, int64_t* __restrict__ irC,
                                                       T* __restrict__ valC) {
  const int64_t t = first + blockIdx.x;
  const int64_t n = in.cnt[t], src = in.at[t], dst = upto[t] + hcs[units[t].col];
  for (int64_t i = threadIdx.x; i < n; i += 256) {
    irC[dst + i] = in.rows[src + i];
    valC[dst + i] = in.vals[src + i];
  }
}

// Tile pointers (Tiles): thread per stored A column and run of kTileRun tiles,
// so a wave's stores cover 64 consecutive columns of one tile.  Each pointer
// is searched for from the previous one.
constexpr int kTileRun = 32;
__global__ __launch_bounds__(256) void k_tiles(const int64_t* __restrict__ cpA, int64_t nzcA,
                                               const int32_t* __restrict__ rowsA, int S, int32_t* __restrict__ at) {
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p >= nzcA) return;
  const int32_t end = (int32_t)cpA[p + 1];
  int32_t lo = (int32_t)cpA[p];
  const int t0 = (int)blockIdx.y * kTileRun, t1 = min(S + 1, t0 + kTileRun);
  for (int t = t0; t < t1; ++t) {
    lo = first_from([&](int32_t i) { return rowsA[i]; }, lo, end, (int64_t)t * kBR);
    at[t * nzcA + p] = lo;
  }
}

// w[b] = hist[b] / nnzA
__global__ void k_hist_to_w(const unsigned long long* __restrict__ hist, int S, double inv, float* __restrict__ w) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < S) w[b] = (float)((double)hist[b] * inv);
}

__global__ void k_add_col_totals(int64_t* __restrict__ nnzcol, const unsigned long long* __restrict__ col_total,
                                 int64_t n) {
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j < n) nnzcol[j] += (int64_t)col_total[j];
}

// logpred[j] = log2(1 + est[j]): an estimated column size in the network's output form.
__global__ void k_log2p1(const float* __restrict__ est, int64_t n, float* __restrict__ logpred) {
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j < n) logpred[j] = log2f(1.0f + fmaxf(est[j], 0.0f));
}

__global__ void k_sum_f32(const float* __restrict__ v, int64_t n, double* __restrict__ out) {
  double a = 0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    a += v[i];
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) a += __shfl_xor(a, d, kWave);
  if (lane_id() == 0) atomicAdd(out, a);
}

// ------------------------------------------------------------------ driver
namespace {

// Row maps of the symbolic pass (from the caching allocator): returned to
// the cache once the stream's unit kernels that read them are done.
struct RowMap {
  uint32_t* p = nullptr;
  hipStream_t s = nullptr;
  ~RowMap() {
    if (!p) return;
    (void)hipStreamSynchronize(s);
    dev_free(p);
  }
};

template <class X>
cbx_status dalloc(ScratchSet& ws, size_t count, X** out) {
  if (ws.take(out, count)) return CBX_OK;
  *out = nullptr;
  return CBX_ERR_NOMEM;
}

// Whether `bytes` fit a share of the free memory (the library's idle blocks
// included).  Up to 64 MB do without asking the driver, which costs more than
// a small product's kernels.
bool fits(double bytes, double share) {
  if (bytes <= 64.0 * (1 << 20) && share > 0.0) return true;
  size_t freeb = 0, totb = 0;
  return hipMemGetInfo(&freeb, &totb) == hipSuccess && bytes <= share * (double)(freeb + cache_idle_bytes());
}

#define CBX_TRY(x)                 \
  do {                             \
    cbx_status st_ = (x);          \
    if (st_ != CBX_OK) return st_; \
  } while (0)

inline unsigned nblk(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Unit order for the numeric pass: by first row block, so that the units in
// flight at any moment gather the A entries of a narrow band of rows (a few
// hundred KB of A), which the XCDs' L2 caches can hold, instead of every row
// range of a few heavy columns.  Units are independent (their output offsets
// are known), so the order changes nothing but the cache footprint.
__global__ void k_unit_keys(const Unit* __restrict__ u, int n, int32_t* __restrict__ key, int32_t* __restrict__ idx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    key[i] = u[i].blk_lo;
    idx[i] = i;
  }
}

__global__ void k_unit_permute(const Unit* __restrict__ src, const int32_t* __restrict__ idx, int n,
                               Unit* __restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}

__global__ void k_gather_flop(const int32_t* __restrict__ cols, int64_t n, const int64_t* __restrict__ flop,
                              int64_t* __restrict__ key) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) key[i] = flop[cols[i]];
}

// Reorders cols[0..n) by descending flop (into *out), so a
// per-column launch over them starts its longest columns first, as the
// two-phase path's flop-sorted order does.
cbx_status sort_cols_by_flop(const int32_t* cols, int64_t n, const int64_t* flop, ScratchSet& ws, int32_t** out) {
  hipStream_t s = ws.s;
  int64_t *k1, *k2;
  uint8_t* t;
  CBX_TRY(dalloc(ws, n, &k1));
  CBX_TRY(dalloc(ws, n, &k2));
  CBX_TRY(dalloc(ws, n, out));
  size_t tb = 0;
  CBX_HIP(hipcub::DeviceRadixSort::SortPairsDescending(nullptr, tb, k1, k2, cols, *out, (int)n, 0, 64, s));
  CBX_TRY(dalloc(ws, std::max<size_t>(tb, 16), &t));
  k_gather_flop<<<nblk(n, 256), 256, 0, s>>>(cols, n, flop, k1);
  CBX_HIP(hipcub::DeviceRadixSort::SortPairsDescending(t, tb, k1, k2, cols, *out, (int)n, 0, 64, s));
  CBX_HIP(hipGetLastError());
  return CBX_OK;
}

// A copy of units[0, n) sorted by blk_lo (stable), in *out.
cbx_status sort_units_by_block(const Unit* units, int n, int S, ScratchSet& ws, Unit** out) {
  hipStream_t s = ws.s;
  int32_t *k1, *k2, *i1, *i2;
  uint8_t* t;
  CBX_TRY(dalloc(ws, n, &k1));
  CBX_TRY(dalloc(ws, n, &k2));
  CBX_TRY(dalloc(ws, n, &i1));
  CBX_TRY(dalloc(ws, n, &i2));
  CBX_TRY(dalloc(ws, n, out));
  int bits = 1;
  while ((1 << bits) <= S) ++bits;
  size_t tb = 0;
  CBX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, k1, k2, i1, i2, n, 0, bits, s));
  CBX_TRY(dalloc(ws, std::max<size_t>(tb, 16), &t));
  k_unit_keys<<<nblk(n, 256), 256, 0, s>>>(units, n, k1, i1);
  CBX_HIP(hipcub::DeviceRadixSort::SortPairs(t, tb, k1, k2, i1, i2, n, 0, bits, s));
  k_unit_permute<<<nblk(n, 256), 256, 0, s>>>(units, i2, n, *out);
  CBX_HIP(hipGetLastError());
  return CBX_OK;
}

// Timings from a call's events (on: the caller asked for statistics).
struct Timer {
  hipEvent_t* ev;
  bool on;
  void mark(int i, hipStream_t s) {
    if (on) (void)hipEventRecord(ev[i], s);
  }
  double ms(int a, int b) {
    float f = 0;
    if (on) (void)hipEventElapsedTime(&f, ev[a], ev[b]);
    return f;
  }
};

constexpr int kHashNT = 256;
constexpr int kDenseNT = 512;                 // dense numeric threads
constexpr int kDenseTR = 32 * kDenseNT;       // rows per numeric tile (16384)
constexpr int kSymNT = 512;
constexpr int kSymRBW = 32768;                // bitmap words per symbolic pass (2^20 rows)
// unit tier
constexpr int kSymUnitNT = 512, kSymUnitIBLK = 64;  // 32 KB bitmap (38 KB in all): four workgroups per CU
constexpr int kSymBandNT = 256;                     // banded symbolic pass
// Light units: at most 16 blocks (64K rows) and 3264 outputs, whose 8-byte
// accumulators and 16-bit rows share the 32 KB of a direct unit's 4096 rows:
// 53 KB of LDS with the bitmap and its prefix, three workgroups per CU.
// Heavy units: 13056 outputs or 16384 direct rows, 128 KB.
constexpr int kLightNT = 512, kLightK = 3264, kLightDR = 4096, kLightRB = 16;
constexpr int kHeavyNT = 1024, kHeavyK = 13056, kHeavyDR = 16384, kHeavyRB = 16;
static_assert(kLightDR >= kBR && kHeavyDR >= kBR, "a unit of one block is direct, whatever its outputs");
// learned units: the light units' workgroup shape and window, cut to
// target * 3264 predicted outputs.  One round of products stays in registers
// between the sweeps: two spill at the 80 registers of three workgroups per CU
// (R-MAT s17, int64: 4.5 ms in k_num_learned, 3.7 with one).
constexpr int kLearnNT = 512, kLearnK = kLightK, kLearnRB = kLightRB, kLearnCR = 1;
// Expected products from which a block forms a unit of its own, accumulated in
// one sweep (half of it measured 3.9 ms).
constexpr int kLearnDirect = 8 * kLearnNT;
constexpr int kLearnFlopCap = 131072;  // expected products per learned unit
constexpr int64_t kLearnChunk = 1 << 21;  // workgroups per learned launch
// Tiny tier launch: `waves` columns (one wave each) per workgroup, grid-stride
// beyond 256K columns in flight.
inline unsigned tiny_grid(int64_t ncols, int waves) {
  return (unsigned)std::min<int64_t>((ncols + waves - 1) / waves, (int64_t)262144 / waves);
}

// The tiny tier in the configured workgroup shape.
template <int K, class T, bool SYM>
void launch_tiny(const SpgemmConfig& cfg, const int32_t* order, int64_t first, int64_t ncols, const int64_t* cpB,
                 const int32_t* bpos, const T* valB, const int64_t* cpA, const int32_t* rowsA, const T* valA,
                 int64_t* nnzcol, const int64_t* cpC, int64_t* irC, T* valC, int* err, const int64_t* stage_off,
                 const int64_t* stage_flop, hipStream_t s, const Filter<T>& flt = {}) {
  const dim3 g(tiny_grid(ncols, cfg.tiny_wg_waves)), b(kWave * cfg.tiny_wg_waves);
  k_tiny<K, T, SYM><<<g, b, 0, s>>>(order, first, ncols, cpB, bpos, valB, cpA, rowsA, valA, nnzcol, cpC, irC, valC, err,
                                    stage_off, stage_flop, flt);
}

// Row lists of the small units (k_sym_units); lists == nullptr: none.
struct UnitLists {
  uint16_t* lists = nullptr;
  int64_t* off = nullptr;         // first entry, per symbolic slot
  const int64_t* flop = nullptr;  // per column; a region holds min(flop, region_cap)
  int64_t region_cap = 0;
  uint16_t* bcnt = nullptr;
  Unit* units = nullptr;
  int* n = nullptr;
  int cap = 0;
};

// Region sizes of the symbolic slots order[0..n): a column's outputs in the
// small-unit passes are at most min(flop_j, unit_split_nnz, m).
__global__ void k_list_regions(const int32_t* __restrict__ order, const int64_t* __restrict__ flop, int64_t n,
                               int64_t cap, int64_t* __restrict__ sz) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) {
    const int64_t f = flop[order[i]];
    sz[i] = f < cap ? f : cap;
  } else if (i == n) {
    sz[i] = 0;
  }
}

// Row lists of `rows` entries, block counts and list-unit array for n symbolic
// slots with region starts `off`, when they fit a fifth of the free memory;
// otherwise ul.lists stays null.
static void alloc_unit_lists(int64_t* off, const int64_t* flop, int64_t n, int64_t rows, int S, int64_t cap_units,
                             int64_t region_cap, int* counter, ScratchSet& ws, UnitLists& ul) {
  ul = UnitLists{};
  const double bytes = 2.0 * (double)rows + 2.0 * (double)n * S + (double)sizeof(Unit) * cap_units;
  uint16_t *lists = nullptr, *bcnt = nullptr;
  Unit* units = nullptr;
  if (fits(bytes, 0.2) && dalloc(ws, std::max<int64_t>(rows, 1), &lists) == CBX_OK &&
      dalloc(ws, n * (int64_t)S, &bcnt) == CBX_OK && dalloc(ws, cap_units, &units) == CBX_OK) {
    ul.lists = lists;
    ul.off = off;
    ul.flop = flop;
    ul.region_cap = region_cap;
    ul.bcnt = bcnt;
    ul.units = units;
    ul.n = counter;
    ul.cap = (int)cap_units;
  }
  (void)hipGetLastError();
}

// The unit tier's symbolic pass: per column (sym_band 0, optionally with the
// small units' row lists) or banded (the band height in row blocks, 16 or 64;
// bcnt_buf receives the block counts).
cbx_status launch_sym_units(const SpgemmConfig& cfg, const int32_t* order, int64_t ncols, const cbx_dcsc* A,
                            const cbx_dcsc* B, const int32_t* bpos, const int32_t* rowsA, const Tiles& P, int S,
                            int64_t* nnzcol, Unit* units_l, int* n_l, int cap_l, Unit* units_h, int* n_h, int cap_h,
                            uint32_t* rmap, int64_t rm_cols, int* err, int kmax_h, ScratchSet& ws,
                            const UnitLists& ul = {}) {
  hipStream_t s = ws.s;
  if (cfg.sym_band == 0) {
    k_sym_units<kSymUnitNT, 4, kSymUnitIBLK><<<(unsigned)ncols, kSymUnitNT, 0, s>>>(
        order, 0, B->cp, bpos, A->cp, rowsA, P, S, kLightK, kLightRB, kmax_h, kHeavyRB, cfg.unit_split_nnz, nnzcol,
        units_l, n_l, cap_l, units_h, n_h, cap_h, rmap, rm_cols, err, ul.lists, ul.off, ul.flop,
        ul.region_cap, ul.bcnt, ul.units, ul.n, ul.cap);
    return CBX_OK;
  }
  int32_t* bcnt;
  CBX_TRY(dalloc(ws, (size_t)ncols * S, &bcnt));
  const int band = cfg.sym_band;
  const dim3 g((unsigned)ncols, (unsigned)((S + band - 1) / band));  // band-major dispatch order
  if (band == 16)
    k_sym_band<kSymBandNT, 4, 16><<<g, kSymBandNT, 0, s>>>(order, 0, B->cp, bpos, A->cp, rowsA, P, S, bcnt, rmap,
                                                          rm_cols);
  else
    k_sym_band<kSymBandNT, 4, 64><<<g, kSymBandNT, 0, s>>>(order, 0, B->cp, bpos, A->cp, rowsA, P, S, bcnt, rmap,
                                                          rm_cols);
  k_sym_cut<<<(unsigned)ncols, 256, 0, s>>>(order, 0, bcnt, S, kLightK, kLightRB, kmax_h, kHeavyRB,
                                            cfg.unit_split_nnz, nnzcol, units_l, n_l, cap_l, units_h, n_h, cap_h, err);
  return CBX_OK;
}

}  // namespace

struct LearnedInfo {
  int64_t nnzC = 0, units = 0, overflow_units = 0, hash_total = 0, heavy_units = 0;
  int64_t exact_total = 0;  // outputs of the predicted-heavy columns (computed exactly)
  double pred_sum = 0;
  float kernel_ms = 0;  // the single-pass numeric kernel alone
  bool over_capacity = false;
};

// Learned single pass for the unit-tier columns (see the learned tier above).
// On entry nnzcol holds the exact sizes of the sort- and tiny-tier columns (0 for the
// rest).  On success C->ir / C->val are allocated and the unit-tier outputs
// written, nnzcol holds every column's size and cpC its exclusive scan.
template <int K, class T>
static cbx_status learned_numeric(const cbx_dcsc* A, const cbx_dcsc* B, const SpgemmConfig& cfg, hipStream_t s,
                                  const int32_t* rowsA, const int32_t* bpos, const int64_t* flop, const Tiles& P,
                                  int S, int64_t* nnzcol, int64_t* cpC, cbx_dcsc* C, int* err, hipEvent_t* kev,
                                  LearnedInfo& info) {
  const int64_t nzcB = B->nzc, m = A->m;
  ScratchSet ws(s);
  size_t tmp_bytes = 0;  // scans over up to nzcB + 1 columns
  CBX_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, nnzcol, cpC, (int)(nzcB + 1), s));
  tmp_bytes = std::max<size_t>(tmp_bytes, 16);
  void* tmp;
  CBX_TRY(dalloc(ws, tmp_bytes, (uint8_t**)&tmp));
  UnitLists ul;
  uint8_t* heavy_flag;
  int32_t* hcols;
  int64_t* nh_dev;
  int* hucnt;
  Unit *units_l = nullptr, *units_h = nullptr;
  float *feats, *logpred, *w, *pred_nnz;
  unsigned long long *hist, *col_total;
  int32_t *blo, *bhi;
  int64_t *ucount, *ubase, *hcs;
  int* ovf;
  double* dsum;
  UnitL* units;
  CBX_TRY(dalloc(ws, nzcB * CBX_MLP_FEATURES, &feats));
  CBX_TRY(dalloc(ws, nzcB, &logpred));
  CBX_TRY(dalloc(ws, S, &hist));
  CBX_TRY(dalloc(ws, S, &w));
  CBX_TRY(dalloc(ws, nzcB, &blo));
  CBX_TRY(dalloc(ws, nzcB, &bhi));
  CBX_TRY(dalloc(ws, nzcB + 1, &ucount));
  CBX_TRY(dalloc(ws, nzcB + 1, &ubase));
  CBX_TRY(dalloc(ws, nzcB, &pred_nnz));
  CBX_TRY(dalloc(ws, nzcB + 1, &hcs));
  CBX_TRY(dalloc(ws, 2, &dsum));
  CBX_TRY(dalloc(ws, 2, &ovf));
  CBX_TRY(dalloc(ws, nzcB, &col_total));
  CBX_TRY(dalloc(ws, nzcB, &heavy_flag));
  CBX_TRY(dalloc(ws, nzcB, &hcols));
  CBX_TRY(dalloc(ws, 1, &nh_dev));
  CBX_TRY(dalloc(ws, 3, &hucnt));
  // prediction: the network on the columns' features, or (without it) the
  // min-hash estimates of estimateNNZ_sampling
  if (cfg.sampling_rounds > 0) {
    float *samp, *est;
    CBX_TRY(dalloc(ws, sampling_scratch_floats(A, cfg.sampling_rounds), &samp));
    CBX_TRY(dalloc(ws, nzcB, &est));
    CBX_TRY(sampling_estimate_launch(A, B, cfg.sampling_rounds, rowsA, bpos, samp, est, s));
    k_log2p1<<<nblk(nzcB, 256), 256, 0, s>>>(est, nzcB, logpred);
  } else {
    k_features<<<wave_grid(nzcB), 256, 0, s>>>(B->cp, nzcB, bpos, A->cp, rowsA, m, feats);
    mlp_infer_launch(cfg.predictor, feats, nzcB, logpred, s);
  }
  // block prior and per-column block range
  CBX_HIP(hipMemsetAsync(hist, 0, sizeof(unsigned long long) * S, s));
  k_row_hist<<<256, 256, sizeof(unsigned int) * S, s>>>(rowsA, A->nnz, S, hist);
  k_hist_to_w<<<nblk(S, 256), 256, 0, s>>>(hist, S, 1.0 / (double)std::max<int64_t>(A->nnz, 1), w);
  k_col_blocks<<<wave_grid(nzcB), 256, 0, s>>>(B->cp, nzcB, bpos, A->cp, rowsA, blo, bhi);
  // units in column order: count, scan, write
  const float target = cfg.learned_target * (float)kLearnK;
  const float heavy_pred = (float)cfg.heavy_nnz;
  const float fcap = (float)kLearnFlopCap;
  const float direct_flop = (float)kLearnDirect;
  k_learned_units<<<nblk(nzcB, 256), 256, 0, s>>>(flop, nzcB, cfg.small_flop_max, logpred, blo, bhi, w, target,
                                                  heavy_pred, fcap, kLearnRB, direct_flop, m, nullptr, ucount,
                                                  nullptr, pred_nnz, heavy_flag);
  CBX_HIP(hipMemsetAsync(ucount + nzcB, 0, sizeof(int64_t), s));
  CBX_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, ucount, ubase, (int)(nzcB + 1), s));
  // columns predicted heavy: exact sizes from the symbolic unit pass (their
  // units then go through the two-phase unit kernels), so the single pass
  // covers the many light columns and its outputs are placed around the heavy columns'
  // sizes up front, like the sort tier's
  int64_t hash_only = 0;
  {
    size_t need = 0, need2 = 0;
    CBX_HIP(hipcub::DeviceReduce::Sum(nullptr, need, nnzcol, nh_dev, (int)nzcB, s));
    CBX_HIP(hipcub::DeviceSelect::Flagged(nullptr, need2, hipcub::CountingInputIterator<int32_t>(0), heavy_flag,
                                          hcols, nh_dev, (int)nzcB, s));
    need = std::max(need, need2);
    void* t2 = tmp;
    if (need > tmp_bytes) CBX_TRY(dalloc(ws, need, (uint8_t**)&t2));
    const size_t tb = std::max(need, tmp_bytes);
    size_t tb1 = tb, tb2 = tb;
    CBX_HIP(hipcub::DeviceReduce::Sum(t2, tb1, nnzcol, nh_dev, (int)nzcB, s));
    CBX_HIP(hipMemcpyAsync(&hash_only, nh_dev, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    CBX_HIP(hipcub::DeviceSelect::Flagged(t2, tb2, hipcub::CountingInputIterator<int32_t>(0), heavy_flag, hcols,
                                          nh_dev, (int)nzcB, s));
    CBX_HIP(hipStreamSynchronize(s));  // hash_only
  }
  int64_t nheavy = 0;
  CBX_HIP(hipMemcpyAsync(&nheavy, nh_dev, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  int64_t cap_l = 0, cap_h = 0;
  // row maps of the exact columns, as in the two-phase path: their large
  // units then load them instead of a counting sweep (when they fit the
  // share of free memory; from the caching allocator)
  RowMap rm;
  rm.s = s;
  int64_t rm_cols = 0;
  if (nheavy > 1) {  // longest columns first
    int32_t* hs = nullptr;
    CBX_TRY(sort_cols_by_flop(hcols, nheavy, flop, ws, &hs));
    hcols = hs;
  }
  if (nheavy) {
    cap_l = std::max<int64_t>(1, std::min<int64_t>(nheavy * (int64_t)S, 1ll << 30));
    cap_h = cap_l;
    CBX_TRY(dalloc(ws, cap_l, &units_l));
    CBX_TRY(dalloc(ws, cap_h, &units_h));
    CBX_HIP(hipMemsetAsync(hucnt, 0, 3 * sizeof(int), s));
    if (cfg.row_map_share > 0.0f) {
      const int64_t rm_words = nheavy * (int64_t)S * kBRW;
      if (fits(4.0 * (double)rm_words, cfg.row_map_share) &&
          dev_alloc((void**)&rm.p, sizeof(uint32_t) * rm_words) == CBX_OK)
        rm_cols = nheavy;
      (void)hipGetLastError();
    }
    // the small units' row lists, as in the two-phase path
    if (cfg.unit_lists && cfg.sym_band == 0) {
      const int64_t region = std::min<int64_t>(cfg.unit_split_nnz, m);
      int64_t *lsz, *loff;
      CBX_TRY(dalloc(ws, nheavy + 1, &lsz));
      CBX_TRY(dalloc(ws, nheavy + 1, &loff));
      k_list_regions<<<nblk(nheavy + 1, 256), 256, 0, s>>>(hcols, flop, nheavy, region, lsz);
      CBX_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, lsz, loff, (int)(nheavy + 1), s));
      int64_t rows = 0;
      CBX_HIP(hipMemcpyAsync(&rows, loff + nheavy, sizeof(int64_t), hipMemcpyDeviceToHost, s));
      CBX_HIP(hipStreamSynchronize(s));
      alloc_unit_lists(loff, flop, nheavy, rows, S, cap_l, region, hucnt + 2, ws, ul);
    }
    CBX_TRY(launch_sym_units(cfg, hcols, nheavy, A, B, bpos, rowsA, P, S, nnzcol, units_l, hucnt, (int)cap_l, units_h,
                             hucnt + 1, (int)cap_h, rm.p, rm_cols, err, kHeavyK, ws, ul));
    CBX_HIP(hipGetLastError());
  }
  CBX_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, nnzcol, hcs, (int)(nzcB + 1), s));
  CBX_HIP(hipMemsetAsync(dsum, 0, sizeof(double), s));
  k_sum_f32<<<256, 256, 0, s>>>(pred_nnz, nzcB, dsum);
  int64_t nunits = 0, hash_total = 0;
  double pred_sum = 0;
  CBX_HIP(hipMemcpyAsync(&nunits, ubase + nzcB, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipMemcpyAsync(&hash_total, hcs + nzcB, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipMemcpyAsync(&pred_sum, dsum, sizeof(double), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  info.units = nunits;
  info.pred_sum = pred_sum;
  info.hash_total = hash_only;
  info.exact_total = hash_total - hash_only;
  CBX_TRY(dalloc(ws, std::max<int64_t>(nunits, 1), &units));
  if (nunits)
    k_learned_units<<<nblk(nzcB, 256), 256, 0, s>>>(flop, nzcB, cfg.small_flop_max, logpred, blo, bhi, w, target,
                                                    heavy_pred, fcap, kLearnRB, direct_flop, m, ubase, nullptr,
                                                    units, nullptr, nullptr);
  // staging capacity from the predictions; where it does not fit beside the
  // output (the exactly sized columns and the predictions), the exact two-phase
  // path computes the product, before anything is done twice
  LearnedStage<T> stage;
  stage.cap = (int64_t)(pred_sum * (1.0 + cfg.capacity_margin)) + (1 << 20);
  const double staged = (double)stage.cap * (double)(sizeof(int32_t) + sizeof(T));
  const double output = ((double)hash_total + pred_sum) * (double)(sizeof(int64_t) + sizeof(T));
  if (rm.p && !fits(staged + output, 1.0)) {  // without the row maps the large units count in a sweep
    dev_free(rm.p);                           // (the stream is idle)
    rm.p = nullptr;
  }
  if (!fits(staged + output, 1.0)) {
    info.over_capacity = true;
    return CBX_OK;
  }
  int64_t* upto;
  if (dalloc(ws, nunits + 1, &stage.cnt) != CBX_OK || dalloc(ws, nunits + 1, &stage.at) != CBX_OK ||
      dalloc(ws, nunits + 1, &upto) != CBX_OK || dalloc(ws, 1, &stage.taken) != CBX_OK ||
      dalloc(ws, stage.cap, &stage.rows) != CBX_OK || dalloc(ws, stage.cap, &stage.vals) != CBX_OK) {
    info.over_capacity = true;
    return CBX_OK;
  }
  CBX_HIP(hipMemsetAsync(stage.cnt + nunits, 0, sizeof(int64_t), s));
  CBX_HIP(hipMemsetAsync(stage.taken, 0, sizeof(unsigned long long), s));
  CBX_HIP(hipMemsetAsync(ovf, 0, sizeof(int) * 2, s));
  CBX_HIP(hipMemsetAsync(col_total, 0, sizeof(unsigned long long) * nzcB, s));
  (void)hipEventRecord(kev[0], s);
  // launches of at most 2^21 workgroups (a dispatch holds fewer than 2^32 work-items)
  for (int64_t done = 0; done < nunits; done += kLearnChunk) {
    const int64_t nb = std::min<int64_t>(kLearnChunk, nunits - done);
    k_num_learned<K, T, kLearnNT, 4, kLearnK, kLightDR, kLearnRB, kLearnCR><<<(unsigned)nb, kLearnNT, 0, s>>>(
        units, done, B->cp, bpos, (const T*)B->val, A->cp, rowsA, (const T*)A->val, P, S, stage, col_total, ovf, err);
  }
  (void)hipEventRecord(kev[1], s);
  CBX_HIP(hipGetLastError());
  k_add_col_totals<<<nblk(nzcB, 256), 256, 0, s>>>(nnzcol, col_total, nzcB);
  CBX_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, nnzcol, cpC, (int)(nzcB + 1), s));
  int herr = 0, hovf = 0;
  CBX_HIP(hipMemcpyAsync(&info.nnzC, cpC + nzcB, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipMemcpyAsync(&herr, err, sizeof(int), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipMemcpyAsync(&hovf, ovf, sizeof(int), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  info.overflow_units = hovf;
  (void)hipEventElapsedTime(&info.kernel_ms, kev[0], kev[1]);
  info.over_capacity = (herr & 512) != 0;
  if (herr & ~512 || info.over_capacity) {
    if (herr & ~512) return set_error(CBX_ERR_HIP, "cbx_spgemm: learned pass inconsistency (flag %d)", herr);
    return CBX_OK;
  }
  auto alloc_out = [&]() { return dev_alloc_entries(&C->ir, &C->val, info.nnzC, sizeof(T)); };
  cbx_status ast = alloc_out();
  if (ast != CBX_OK && rm.p) {  // give the row maps back; the large units then count in a sweep
    dev_free(rm.p);             // (the stream is idle)
    rm.p = nullptr;
    release_cache();
    ast = alloc_out();
  }
  if (ast != CBX_OK) {  // the exact path has the staging arrays' room too
    if (ast != CBX_ERR_NOMEM) return ast;
    info.over_capacity = true;
    return CBX_OK;
  }
  (void)hipEventRecord(kev[2], s);  // the copy into place, and the numeric pass of the heavy columns
  if (nunits) {
    size_t need = 0;
    CBX_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, need, stage.cnt, upto, (int)(nunits + 1), s));
    void* t4 = tmp;
    if (need > tmp_bytes) CBX_TRY(dalloc(ws, need, (uint8_t**)&t4));
    need = std::max(need, tmp_bytes);
    CBX_HIP(hipcub::DeviceScan::ExclusiveSum(t4, need, stage.cnt, upto, (int)(nunits + 1), s));
    for (int64_t done = 0; done < nunits; done += kLearnChunk)
      k_learned_place<T><<<(unsigned)std::min<int64_t>(kLearnChunk, nunits - done), 256, 0, s>>>(
          units, done, stage, upto, hcs, C->ir, (T*)C->val);
    CBX_HIP(hipGetLastError());
  }
  if (!nheavy) {
    (void)hipEventRecord(kev[1], s);
    CBX_HIP(hipStreamSynchronize(s));
    float place_ms = 0;
    (void)hipEventElapsedTime(&place_ms, kev[2], kev[1]);
    info.kernel_ms += place_ms;
    return CBX_OK;
  }
  // the heavy columns' values, at the offsets the scan above fixed
  int hu[3] = {0, 0, 0};  // small (bitmap), large, and small list units
  CBX_HIP(hipMemcpy(hu, hucnt, sizeof(hu), hipMemcpyDeviceToHost));
  CBX_RETURN_IF(hu[0] > cap_l || hu[1] > cap_h || hu[2] > cap_l, CBX_ERR_HIP, "cbx_spgemm: unit list overflow");
  CBX_RETURN_IF((int64_t)hu[0] * kLightNT >= (1ll << 32) || (int64_t)hu[1] * kHeavyNT >= (1ll << 32) ||
                    (int64_t)hu[2] * kLightNT >= (1ll << 32),
                CBX_ERR_LIMIT, "cbx_spgemm: too many units for a single launch");
  info.heavy_units = hu[0] + hu[1] + hu[2];
  if (cfg.unit_order == 1) {
    if (hu[0] > 1) CBX_TRY(sort_units_by_block(units_l, hu[0], S, ws, &units_l));
    if (hu[1] > 1) CBX_TRY(sort_units_by_block(units_h, hu[1], S, ws, &units_h));
    if (hu[2] > 1) CBX_TRY(sort_units_by_block(ul.units, hu[2], S, ws, &ul.units));
  }
  if (hu[1] && rm.p)
    k_num_units_rm<K, T, kHeavyNT, 4, kHeavyK, kHeavyDR, kHeavyRB><<<(unsigned)hu[1], kHeavyNT, 0, s>>>(
        units_h, rm.p, B->cp, bpos, (const T*)B->val, A->cp, rowsA, (const T*)A->val, P, S, rm_cols, cpC, C->ir,
        (T*)C->val, err, Filter<T>{}, cfg.unit_xcd_group);
  else if (hu[1])
    k_num_units<K, T, kHeavyNT, 4, kHeavyK, kHeavyDR, kHeavyRB, 4><<<(unsigned)hu[1], kHeavyNT, 0, s>>>(
        units_h, B->cp, bpos, (const T*)B->val, A->cp, rowsA, (const T*)A->val, P, S, cpC, C->ir, (T*)C->val, err,
        Filter<T>{}, cfg.unit_xcd_group);
  if (hu[0])
    k_num_units<K, T, kLightNT, 4, kLightK, kLightDR, kLightRB, 2><<<(unsigned)hu[0], kLightNT, 0, s>>>(
        units_l, B->cp, bpos, (const T*)B->val, A->cp, rowsA, (const T*)A->val, P, S, cpC, C->ir, (T*)C->val, err,
        Filter<T>{}, cfg.unit_xcd_group);
  if (hu[2])
    k_num_list<K, T, kLightNT, 4, kLightK><<<(unsigned)hu[2], kLightNT, 0, s>>>(
        ul.units, ul.lists, ul.off, ul.bcnt, B->cp, bpos, (const T*)B->val, A->cp, rowsA, (const T*)A->val, P, S, cpC,
        C->ir, (T*)C->val, err, Filter<T>{}, cfg.unit_xcd_group);
  CBX_HIP(hipGetLastError());
  (void)hipEventRecord(kev[1], s);
  CBX_HIP(hipMemcpyAsync(&herr, err, sizeof(int), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  float heavy_ms = 0;
  (void)hipEventElapsedTime(&heavy_ms, kev[2], kev[1]);
  info.kernel_ms += heavy_ms;
  if (herr) return set_error(CBX_ERR_HIP, "cbx_spgemm: learned pass, large columns inconsistent (flag %d)", herr);
  return CBX_OK;
}

// Gather of the fused threshold's runs: run k (in start order) moves its kept
// entries from its start in the unfiltered layout to dst[k], one wave per run.
template <class T>
__global__ __launch_bounds__(256) void k_run_copy(const int32_t* __restrict__ idx, const int64_t* __restrict__ src,
                                                  const int32_t* __restrict__ kept, const int64_t* __restrict__ dst,
                                                  const int64_t* __restrict__ ir, const T* __restrict__ val,
                                                  int nrun, int64_t* __restrict__ ir2, T* __restrict__ val2) {
  const int k = (int)global_wave();
  if (k >= nrun) return;
  const int i = idx[k];
  const int64_t a = src[i], d = dst[k];
  const int n = kept[i];
  constexpr int U = 8;  // entries of a lane in flight together
  for (int e0 = lane_id(); e0 < n; e0 += kWave * U) {
    int64_t r[U];
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = min(e0 + u * kWave, n - 1);
      r[u] = ir[a + e];
      v[u] = val[a + e];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      pin(r[u]);
      pin(v[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + u * kWave;
      if (e < n) {
        ir2[d + e] = r[u];
        val2[d + e] = v[u];
      }
    }
  }
}

__global__ void k_run_sizes(const int32_t* __restrict__ idx, const int32_t* __restrict__ kept,
                            const int32_t* __restrict__ col, int n, int64_t* __restrict__ kept_sorted,
                            unsigned long long* __restrict__ colkept) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = idx[k];
  kept_sorted[k] = kept[i];
  atomicAdd(&colkept[col[i]], (unsigned long long)kept[i]);
}

__global__ void k_iota32(int32_t* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

// The product after a fused threshold: the runs the numeric kernels appended
// (sorted by start, which is column then row order in the unfiltered layout)
// gathered into new arrays; nnzcol becomes the kept counts.  C keeps its other fields.
template <class T>
static cbx_status filter_compact(const Filter<T>& flt, int64_t nzcB, int64_t* nnzcol, cbx_dcsc* C, ScratchSet& ws) {
  hipStream_t s = ws.s;
  int nrun = 0;
  CBX_HIP(hipMemcpyAsync(&nrun, flt.run_count, sizeof(int), hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  CBX_RETURN_IF(nrun > flt.run_cap, CBX_ERR_HIP, "cbx_spgemm: run list overflow (%d > %d)", nrun, flt.run_cap);
  int64_t *k2, *ks, *dst;
  int32_t *i1, *i2;
  uint8_t* t;
  const int nr = std::max(nrun, 1);
  CBX_TRY(dalloc(ws, nr, &k2));
  CBX_TRY(dalloc(ws, nr, &i1));
  CBX_TRY(dalloc(ws, nr, &i2));
  CBX_TRY(dalloc(ws, nr + 1, &ks));
  CBX_TRY(dalloc(ws, nr + 1, &dst));
  size_t tb = 0, tb2 = 0;
  CBX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, flt.run_src, k2, i1, i2, nr, 0, 64, s));
  CBX_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb2, ks, dst, nr + 1, s));
  tb = std::max(tb, tb2);
  CBX_TRY(dalloc(ws, std::max<size_t>(tb, 16), &t));
  CBX_HIP(hipMemsetAsync(nnzcol, 0, sizeof(int64_t) * (nzcB + 1), s));
  int64_t total = 0;
  if (nrun) {
    k_iota32<<<nblk(nrun, 256), 256, 0, s>>>(i1, nrun);
    size_t tb1 = tb;
    CBX_HIP(hipcub::DeviceRadixSort::SortPairs(t, tb1, flt.run_src, k2, i1, i2, nrun, 0, 64, s));
    k_run_sizes<<<nblk(nrun, 256), 256, 0, s>>>(i2, flt.run_kept, flt.run_col, nrun, ks,
                                                (unsigned long long*)nnzcol);
    CBX_HIP(hipMemsetAsync(ks + nrun, 0, sizeof(int64_t), s));
    size_t tb3 = tb;
    CBX_HIP(hipcub::DeviceScan::ExclusiveSum(t, tb3, ks, dst, nrun + 1, s));
    CBX_HIP(hipMemcpyAsync(&total, dst + nrun, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    CBX_HIP(hipStreamSynchronize(s));
  }
  int64_t* ir2 = nullptr;
  void* val2 = nullptr;
  if (dev_alloc_entries(&ir2, &val2, total, sizeof(T)) != CBX_OK)
    return set_error(CBX_ERR_NOMEM, "cbx_spgemm: allocation of the thresholded product failed");
  if (nrun) k_run_copy<T><<<wave_grid(nrun), 256, 0, s>>>(i2, flt.run_src, flt.run_kept, dst, C->ir, (const T*)C->val,
                                                         (int)nrun, ir2, (T*)val2);
  CBX_HIP(hipGetLastError());
  CBX_HIP(hipStreamSynchronize(s));
  dev_free(C->ir);
  dev_free(C->val);
  C->ir = ir2;
  C->val = val2;
  C->nnz = total;
  return CBX_OK;
}

template <int K, class T>
static cbx_status spgemm_typed_once(const cbx_dcsc* A, const cbx_dcsc* B, cbx_spgemm_mode mode,
                                    const SpgemmConfig& cfg, cbx_dcsc* C, cbx_spgemm_stats* stats, hipStream_t s,
                                    int64_t* symbolic_out, bool* lists_used) {
  const int64_t m = A->m, n = B->n;
  const int64_t nzcA = A->nzc, nzcB = B->nzc, nnzA = A->nnz, nnzB = B->nnz;

  std::memset(C, 0, sizeof(*C));
  C->m = m;
  C->n = n;
  C->dtype = A->dtype;
  C->location = CBX_DEVICE;
  if (stats) std::memset(stats, 0, sizeof(*stats));

  if (nnzA == 0 || nnzB == 0 || nzcA == 0 || nzcB == 0) {  // mtSpGEMM.h:224-227
    if (symbolic_out) {
      if (nzcB) CBX_HIP(hipMemsetAsync(symbolic_out, 0, sizeof(int64_t) * nzcB, s));
      CBX_HIP(hipStreamSynchronize(s));
      return CBX_OK;
    }
    CBX_TRY(dev_alloc((void**)&C->cp, sizeof(int64_t)));
    CBX_HIP(hipMemsetAsync(C->cp, 0, sizeof(int64_t), s));
    CBX_HIP(hipStreamSynchronize(s));
    return CBX_OK;
  }

  // places in A's entries and stored columns are 32-bit numbers in the kernels (tile pointers, segment bases, bpos)
  CBX_RETURN_IF(nnzA >= (1ll << 31) || nzcA >= (1ll << 31), CBX_ERR_LIMIT,
                "cbx_spgemm: the left operand must hold fewer than 2^31 nonzeros");

  // Three waits for the device per product: after the setup (the tiers' sizes),
  // after the symbolic pass (the output's), at the end.  Kernels report into
  // the slot's pinned page; counters are cleared together, and all scratch is
  // taken from one set and returned after the last wait.
  SlotHold slot;
  CBX_RETURN_IF(!slot.p, CBX_ERR_NOMEM, "cbx_spgemm: no pinned host memory");
  volatile Report* rep = (volatile Report*)slot.p->host;
  Report* rep_dev = (Report*)slot.p->host;
  ScratchSet ws(s);
  Timer tm{slot.p->ev, stats != nullptr};
  tm.mark(0, s);

  // Unit tier needs the tile-pointer table at kBR-row granularity; it is used
  // when that table stays modest, otherwise the streaming dense tier runs.
  const int S4 = (int)((m + kBR - 1) / kBR);
  const bool use_units = m <= (1ll << 24) && (double)nzcA * (S4 + 1) * 4.0 <= 8.0e9;
  const int TR = kDenseTR;
  const int S16 = (int)((m + TR - 1) / TR);
  const int S = use_units ? S4 : S16;
  const int G = kSymRBW * 32 / TR;  // tiles per symbolic pass of the streaming tier

  int32_t *colmap = nullptr, *rowsA = nullptr, *bpos, *order_s, *P = nullptr;
  Counters* ctr;
  int64_t *stage_off, *stage_ir = nullptr;  // staged tiny tier (see the symbolic pass)
  T* stage_val = nullptr;
  bool tiny_staged = false;
  int64_t *flop, *flop_s, *nnzcol, *cpC, *list_off;
  ColSum* sums;
  const int64_t ctiles = (nzcB + kColTile - 1) / kColTile;
  CBX_TRY(dalloc(ws, 1, &ctr));
  if (nzcA != A->n) CBX_TRY(dalloc(ws, A->n, &colmap));
  if (!cfg.rows_a) CBX_TRY(dalloc(ws, nnzA, &rowsA));
  CBX_TRY(dalloc(ws, nnzB, &bpos));
  CBX_TRY(dalloc(ws, nzcB + 1, &flop));
  CBX_TRY(dalloc(ws, nzcB, &flop_s));
  CBX_TRY(dalloc(ws, nzcB, &order_s));
  CBX_TRY(dalloc(ws, nzcB + 1, &nnzcol));
  CBX_TRY(dalloc(ws, nzcB + 1, &cpC));
  CBX_TRY(dalloc(ws, nzcB, &stage_off));
  CBX_TRY(dalloc(ws, nzcB, &list_off));
  CBX_TRY(dalloc(ws, ctiles, &sums));
  int* err = &ctr->err;
  int* ucnt = ctr->units;

  const T* valA = (const T*)A->val;
  const T* valB = (const T*)B->val;
  // the fused threshold (two-phase, unit or sort tiers; the streaming tier has no filtered emission)
  Filter<T> flt;
  flt.on = cfg.filter && mode == CBX_SPGEMM_TWO_PHASE && use_units && symbolic_out == nullptr;
  flt.thr = (T)cfg.filter_thr;
  flt.dropped = &ctr->dropped;
  flt.run_count = &ctr->runs;

  // --- setup: both operands validated before any indexed access (kernels that
  // index through them do nothing where the counts say they are malformed),
  // column map, 32-bit rows, B->A positions, products and order of the columns
  k_init<<<(unsigned)std::min<int64_t>(1024, nblk(std::max<int64_t>({colmap ? A->n : 1, nzcB + 1, 1024}), 256)), 256, 0,
           s>>>(ctr, colmap, A->n, flop, nnzcol, nzcB);
  if (cfg.rows_a) rowsA = const_cast<int32_t*>(cfg.rows_a);
  else if (cfg.trusted_a) k_rows32<<<nblk(nnzA, 256), 256, 0, s>>>(A->ir, nnzA, rowsA);
  else CBX_TRY(launch_validate(A, rowsA, ctr->val, s));
  const bool same = A->cp == B->cp && A->jc == B->jc && A->ir == B->ir && nzcA == nzcB && nnzA == nnzB &&
                    A->m == B->m && A->n == B->n;  // A*A: one look will do
  if (!cfg.trusted_b && !(same && !cfg.trusted_a)) CBX_TRY(launch_validate(B, nullptr, ctr->val + 3, s));
  if (colmap) k_colmap<<<nblk(nzcA, 256), 256, 0, s>>>(A->jc, nzcA, ctr, colmap);
  k_flops<<<nblk(nnzB, kFlopTile), kFlopNT, 0, s>>>(B->cp, B->ir, nzcB, nnzB, colmap, A->cp, ctr, bpos, flop);
  FlopClasses cls;
  cls.split = cfg.unit_split_nnz;
  cls.small = cfg.small_flop_max;
  cls.s4k = 2048;
  cls.mid = cfg.hash_mid_flop;
  cls.tiny = cfg.tiny_flop;
  cls.list_cap = std::min<int64_t>(cfg.unit_split_nnz, m);
  k_count_digits<<<(unsigned)ctiles, 256, 0, s>>>(flop, nzcB, cls, ctr);
  k_order_columns<<<(unsigned)ctiles, 256, 0, s>>>(flop, nzcB, cls, ctr, order_s, flop_s, stage_off, list_off, rep_dev);
  CBX_HIP(hipGetLastError());
  CBX_HIP(hipStreamSynchronize(s));
  if (rep->err)
    return set_error(CBX_ERR_INVALID,
                     "cbx_spgemm: %s is not a valid DCSC (cp/jc/ir out of range, or rows not strictly "
                     "increasing within a column)", (rep->err & 16) ? "A" : "B");
  // tiers in the order of order_s: units, sort tier (1024, 512, 256 threads), tiny (one wave)
  const int64_t n_heavy_max = rep->columns[0];  // columns whose flops (an upper bound of nnz) exceed unit_split_nnz
  const int64_t n_dense = n_heavy_max + rep->columns[1];
  const int64_t n_s4k = rep->columns[2], n_h8 = n_s4k + rep->columns[3], n_h2 = rep->columns[4];
  const int64_t n_h256 = rep->columns[5];
  const int64_t hb[3] = {n_dense, n_dense + n_h8, n_dense + n_h8 + n_h2};  // tier ends
  const int64_t total_flop = rep->flops, tiny_slots = rep->tiny_flops, list_rows = rep->list_rows;
  // one workgroup per column (sort tier, symbolic units): a dispatch holds
  // fewer than 2^32 work-items
  CBX_RETURN_IF(n_dense * 1024 >= (1ll << 32) || n_h8 * 1024 >= (1ll << 32) || n_h2 * kHashNT >= (1ll << 32),
                CBX_ERR_LIMIT, "cbx_spgemm: too many columns in one tier for a single launch");
  // tile pointers only when some column is beyond the sort tier (the table is
  // nzc(A) x m/4096 entries, large for tall packed batches of small columns)
  if (n_dense) {
    CBX_TRY(dalloc(ws, (size_t)nzcA * (S + 1), &P));
    if (use_units)
      k_tiles<<<dim3(nblk(nzcA, 256), nblk(S + 1, kTileRun)), 256, 0, s>>>(A->cp, nzcA, rowsA, S, P);
    else
      k_ptable<<<nblk(nzcA, 256), 256, 0, s>>>(A->cp, nzcA, rowsA, S, TR, P);
  }
  const Tiles tiles{P, nzcA};
  tm.mark(1, s);

  // sizes of the output's columns to offsets and its DCSC columns, and the report
  auto finish_columns = [&]() -> cbx_status {
    k_col_sums<<<(unsigned)ctiles, 256, 0, s>>>(nnzcol, nzcB, n_dense ? flop : nullptr, cfg.small_flop_max, sums, ctr);
    const int scanned = ctiles > 1024;
    if (scanned) k_scan_sums<<<1, 1024, 0, s>>>(sums, ctiles);
    k_col_offsets<<<(unsigned)ctiles, 256, 0, s>>>(nnzcol, nzcB, sums, scanned, B->jc, ctr, cpC, C->cp, C->jc, rep_dev);
    CBX_HIP(hipGetLastError());
    return CBX_OK;
  };
  auto alloc_columns = [&]() -> cbx_status {
    CBX_TRY(dev_alloc((void**)&C->cp, sizeof(int64_t) * (nzcB + 1)));
    CBX_TRY(dev_alloc((void**)&C->jc, sizeof(int64_t) * std::max<int64_t>(nzcB, 1)));
    return CBX_OK;
  };

  auto launch_sym_small = [&]() {
    if (n_h8)
      k_sym_hash<8192, kHashNT><<<(unsigned)n_h8, kHashNT, 0, s>>>(order_s, hb[0], flop, B->cp, bpos, A->cp, rowsA,
                                                                 nnzcol, err);
    if (n_h2)
      k_sym_hash<2048, kHashNT><<<(unsigned)n_h2, kHashNT, 0, s>>>(order_s, hb[1], flop, B->cp, bpos, A->cp, rowsA,
                                                                 nnzcol, err);
  };

  // --- learned single pass (unit-tier columns), with the exact sort-tier
  //     symbolic for the small columns
  bool learned = mode == CBX_SPGEMM_LEARNED && use_units && n_dense > 0 &&
                 (cfg.predictor != nullptr || cfg.sampling_rounds > 0);
  bool learned_done = false;
  LearnedInfo linfo;
  int64_t nnzC = 0, nnz_main = 0, nzcC = 0;
  int hu[3] = {0, 0, 0};  // small (bitmap), large, and small list units
  if (learned) {
    launch_sym_small();
    if (n_h256)
      launch_tiny<K, T, true>(cfg, order_s, hb[2], n_h256, B->cp, bpos, valB, A->cp, rowsA, valA, nnzcol, nullptr,
                              nullptr, nullptr, err, nullptr, nullptr, s);
    tm.mark(2, s);
    tm.mark(3, s);
    CBX_TRY((learned_numeric<K, T>(A, B, cfg, s, rowsA, bpos, flop, tiles, S, nnzcol, cpC, C, err, slot.p->ev + 6,
                                   linfo)));
    if (linfo.over_capacity) {  // predictions too small overall: redo exactly
      dev_free(C->ir);
      dev_free(C->val);
      C->ir = nullptr;
      C->val = nullptr;
      CBX_HIP(hipMemsetAsync(nnzcol, 0, sizeof(int64_t) * (nzcB + 1), s));
      CBX_HIP(hipMemsetAsync(err, 0, sizeof(int), s));
    } else {
      learned_done = true;
      nnzC = linfo.nnzC;
      nnz_main = linfo.nnzC - linfo.hash_total;
      C->nnz = nnzC;
      CBX_TRY(alloc_columns());
      CBX_TRY(finish_columns());
      tm.mark(4, s);
    }
  }
  int64_t nnz_unfiltered = 0;
  if (!learned_done) {
  // --- symbolic
  Unit *units_l = nullptr, *units_h = nullptr;
  UnitLists ul;
  int64_t cap_l = 0, cap_h = 0;
  // row maps (presence bitmaps, 512 B per 4096 rows) of the columns that can
  // form large units (flop above unit_split_nnz; they lead the flop order),
  // when they fit a share of the free memory: the large units then load them
  // instead of rebuilding them in a counting sweep.  From the caching
  // allocator, so repeated products reuse the block.  (cfg.row_map_share of
  // the free memory at most; 0 turns them off.)
  RowMap rm;
  rm.s = s;
  uint32_t*& rmap = rm.p;
  const int64_t rm_cols = std::min<int64_t>(n_heavy_max, n_dense);
  if (use_units && rm_cols > 0 && cfg.row_map_share > 0.0f) {
    const int64_t rm_words = rm_cols * (int64_t)S * kBRW;
    if (fits(4.0 * (double)rm_words, cfg.row_map_share) &&
        dev_alloc((void**)&rmap, sizeof(uint32_t) * rm_words) != CBX_OK)
      rmap = nullptr;
    (void)hipGetLastError();
  }
  if (use_units && n_dense) {
    cap_l = std::max<int64_t>(1, std::min<int64_t>(n_dense * (int64_t)S, 1ll << 30));
    cap_h = std::max<int64_t>(1, std::min<int64_t>(n_heavy_max * (int64_t)S, 1ll << 30));
    CBX_TRY(dalloc(ws, cap_l, &units_l));
    CBX_TRY(dalloc(ws, cap_h, &units_h));
    // the small units' row lists (per-column symbolic form only): one region
    // of min(flop_j, unit_split_nnz, m) 2-byte entries per column, plus the
    // per-block counts, when they fit a fifth of the free memory
    if (cfg.unit_lists && cfg.sym_band == 0 && symbolic_out == nullptr) {
      alloc_unit_lists(list_off, flop, n_dense, list_rows, S, cap_l, cls.list_cap, ucnt + 2, ws, ul);
      if (ul.lists && lists_used) *lists_used = true;
    }
    CBX_TRY(launch_sym_units(cfg, order_s, n_dense, A, B, bpos, rowsA, tiles, S, nnzcol, units_l, ucnt, (int)cap_l,
                             units_h, ucnt + 1, (int)cap_h, rmap, rm_cols, err, kHeavyK, ws, ul));
  } else if (n_dense) {
    k_sym_dense<kSymNT, kSymRBW><<<(unsigned)n_dense, kSymNT, 0, s>>>(order_s, 0, B->cp, bpos, A->cp, rowsA, P, S, G,
                                                                       TR, nnzcol);
  }
  launch_sym_small();
  // tiny tier: its numeric kernel runs now into a staging buffer (a slot of
  // flop_j entries per column) and records the exact counts; after the
  // output scan the entries are copied into place.  One gather and sort per
  // column instead of two (symbolic + numeric), when the slots fit a
  // quarter of the free memory.
  if (n_h256) {
    // a symbolic-only call (symbolic_out) stages nothing: it counts rows
    // without reading values, so it runs for operands of any value type
    if (symbolic_out == nullptr && fits((double)tiny_slots * (sizeof(int64_t) + sizeof(T)), 0.25) &&
        dalloc(ws, std::max<int64_t>(tiny_slots, 1), &stage_ir) == CBX_OK &&
        dalloc(ws, std::max<int64_t>(tiny_slots, 1), &stage_val) == CBX_OK)
      tiny_staged = true;
    (void)hipGetLastError();
    if (tiny_staged)
      launch_tiny<K, T, false>(cfg, order_s, hb[2], n_h256, B->cp, bpos, valB, A->cp, rowsA, valA, nnzcol, nullptr,
                               stage_ir, stage_val, err, stage_off, flop_s, s, flt);
    else
      launch_tiny<K, T, true>(cfg, order_s, hb[2], n_h256, B->cp, bpos, valB, A->cp, rowsA, valA, nnzcol, nullptr,
                              nullptr, nullptr, err, nullptr, nullptr, s);
  }
  if (!symbolic_out) CBX_TRY(alloc_columns());
  CBX_TRY(finish_columns());
  tm.mark(2, s);
  if (symbolic_out) CBX_HIP(hipMemcpyAsync(symbolic_out, nnzcol, sizeof(int64_t) * nzcB, hipMemcpyDeviceToDevice, s));
  CBX_HIP(hipStreamSynchronize(s));
  if (rep->err) {
    const int e = rep->err;
    cbx_dcsc_free(C);
    return set_error(CBX_ERR_HIP, "cbx_spgemm: symbolic pass failed (flag %d)", e);
  }
  if (symbolic_out) return CBX_OK;
  nnzC = rep->nnz;
  nzcC = rep->nzc;
  nnz_main = rep->main_nnz;
  for (int i = 0; i < 3; ++i) hu[i] = rep->units[i];
  nnz_unfiltered = nnzC;
  if (flt.on) {
    nnz_unfiltered += rep->dropped;
    // one run per unit and per sort- or tiny-tier column at most
    const int64_t cap = (int64_t)hu[0] + hu[1] + hu[2] + nzcB + 16;
    CBX_RETURN_IF(cap >= (1ll << 31), CBX_ERR_LIMIT, "cbx_spgemm: too many output ranges for the fused threshold");
    CBX_TRY(dalloc(ws, cap, &flt.run_src));
    CBX_TRY(dalloc(ws, cap, &flt.run_kept));
    CBX_TRY(dalloc(ws, cap, &flt.run_col));
    flt.run_cap = (int)cap;
  }

  // --- output allocation (cached: repeated products reuse the arrays)
  auto alloc_out = [&]() { return dev_alloc_entries(&C->ir, &C->val, nnzC, sizeof(T)); };
  cbx_status ast = alloc_out();
  if (ast != CBX_OK && rmap) {  // give the row maps back and use the two-sweep numeric pass
    CBX_HIP(hipStreamSynchronize(s));
    dev_free(rmap);
    rmap = nullptr;
    release_cache();
    ast = alloc_out();
  }
  CBX_TRY(ast);
  C->nnz = nnzC;
  tm.mark(3, s);

  // --- numeric
  CBX_RETURN_IF((int64_t)hu[0] * kLightNT >= (1ll << 32) || (int64_t)hu[1] * kHeavyNT >= (1ll << 32) ||
                    (int64_t)hu[2] * kLightNT >= (1ll << 32),
                CBX_ERR_LIMIT, "cbx_spgemm: too many units for a single launch");
  if (use_units && cfg.unit_order == 1) {
    if (hu[0] > 1) CBX_TRY(sort_units_by_block(units_l, hu[0], S, ws, &units_l));
    if (hu[1] > 1) CBX_TRY(sort_units_by_block(units_h, hu[1], S, ws, &units_h));
    if (hu[2] > 1) CBX_TRY(sort_units_by_block(ul.units, hu[2], S, ws, &ul.units));
  }
  if (use_units) {
    // large units: one sweep over the row map when it was kept (their
    // products exceed what the two-sweep kernel holds in registers); small
    // units keep the two-sweep kernel, whose second sweep mostly replays
    // registers
    if (hu[1] && rmap)
      k_num_units_rm<K, T, kHeavyNT, 4, kHeavyK, kHeavyDR, kHeavyRB><<<(unsigned)hu[1], kHeavyNT, 0, s>>>(
          units_h, rmap, B->cp, bpos, valB, A->cp, rowsA, valA, tiles, S, rm_cols, cpC, C->ir, (T*)C->val, err, flt,
          cfg.unit_xcd_group);
    else if (hu[1])
      k_num_units<K, T, kHeavyNT, 4, kHeavyK, kHeavyDR, kHeavyRB, 4><<<(unsigned)hu[1], kHeavyNT, 0, s>>>(
          units_h, B->cp, bpos, valB, A->cp, rowsA, valA, tiles, S, cpC, C->ir, (T*)C->val, err, flt,
          cfg.unit_xcd_group);
    if (hu[0])
      k_num_units<K, T, kLightNT, 4, kLightK, kLightDR, kLightRB, 2><<<(unsigned)hu[0], kLightNT, 0, s>>>(
          units_l, B->cp, bpos, valB, A->cp, rowsA, valA, tiles, S, cpC, C->ir, (T*)C->val, err, flt,
          cfg.unit_xcd_group);
    if (hu[2])
      k_num_list<K, T, kLightNT, 4, kLightK><<<(unsigned)hu[2], kLightNT, 0, s>>>(
          ul.units, ul.lists, ul.off, ul.bcnt, B->cp, bpos, valB, A->cp, rowsA, valA, tiles, S, cpC, C->ir, (T*)C->val,
          err, flt, cfg.unit_xcd_group);
  } else if (n_dense) {
    k_num_dense<K, T, kDenseNT><<<(unsigned)n_dense, kDenseNT, 0, s>>>(order_s, 0, B->cp, bpos, valB, A->cp, rowsA,
                                                                     valA, P, S, cpC, C->ir, (T*)C->val, err);
  }
  tm.mark(4, s);
  }  // !learned_done
  // sort-tier columns by the products that a workgroup holds (four per thread)
  if (n_s4k)
    k_num_sort<K, T, 1024><<<(unsigned)n_s4k, 1024, 0, s>>>(order_s, hb[0], nnzcol, B->cp, bpos, valB, A->cp, rowsA,
                                                            valA, cpC, C->ir, (T*)C->val, err, flt);
  if (n_h8 - n_s4k)
    k_num_sort<K, T, 512><<<(unsigned)(n_h8 - n_s4k), 512, 0, s>>>(order_s, hb[0] + n_s4k, nnzcol, B->cp, bpos, valB,
                                                                  A->cp, rowsA, valA, cpC, C->ir, (T*)C->val, err,
                                                                  flt);
  if (n_h2)
    k_num_sort<K, T, 256><<<(unsigned)n_h2, 256, 0, s>>>(order_s, hb[1], nnzcol, B->cp, bpos, valB, A->cp, rowsA, valA,
                                                        cpC, C->ir, (T*)C->val, err, flt);
  if (n_h256 && tiny_staged)
    k_tiny_place<T><<<wave_grid((n_h256 + kPlaceCols - 1) / kPlaceCols), 256, 0, s>>>(order_s, hb[2], n_h256, stage_off, nnzcol, cpC, stage_ir,
                                                       stage_val, C->ir, (T*)C->val, flt, err);
  else if (n_h256)
    launch_tiny<K, T, false>(cfg, order_s, hb[2], n_h256, B->cp, bpos, valB, A->cp, rowsA, valA, nnzcol, cpC, C->ir,
                             (T*)C->val, err, nullptr, nullptr, s, flt);
  CBX_HIP(hipGetLastError());

  if (flt.on) {  // the fused threshold's runs into the final arrays
    k_report_err<<<1, 64, 0, s>>>(err, rep_dev);
    CBX_HIP(hipStreamSynchronize(s));
    if (!rep->err) CBX_TRY(filter_compact<T>(flt, nzcB, nnzcol, C, ws));
    if (!rep->err) CBX_TRY(finish_columns());  // (reports err as it is then)
    nnzC = C->nnz;
  } else {
    k_report_err<<<1, 64, 0, s>>>(err, rep_dev);
  }
  tm.mark(5, s);
  CBX_HIP(hipStreamSynchronize(s));
  if (learned_done || flt.on) nzcC = rep->nzc;
  C->nzc = nzcC;
  if (rep->err) {
    const int e = rep->err;
    cbx_dcsc_free(C);
    return set_error(CBX_ERR_HIP, "cbx_spgemm: numeric pass inconsistency (flag %d)", e);
  }
  if (stats) {
    stats->flops = total_flop;
    stats->nnz = nnzC;
    stats->nnz_before_filter = learned_done ? nnzC : nnz_unfiltered;
    stats->nzc = nzcC;
    stats->ms_setup = tm.ms(0, 1);
    stats->ms_symbolic = tm.ms(1, 2);
    stats->ms_alloc = tm.ms(2, 3);
    stats->ms_numeric = tm.ms(3, 5);
    stats->ms_main_kernel = learned_done ? linfo.kernel_ms : tm.ms(3, 4);
    stats->ms_total = tm.ms(0, 5);
    stats->units_light = learned_done ? linfo.units : hu[0] + hu[2];
    stats->units_heavy = learned_done ? linfo.heavy_units : hu[1];
    stats->nnz_main = nnz_main;
    stats->overflow_cols = linfo.overflow_units;
    stats->predicted_nnz = (int64_t)linfo.pred_sum;
    stats->actual_nnz_predicted = learned_done ? linfo.nnzC - linfo.hash_total - linfo.exact_total : 0;
    stats->learned_fallback = learned && !learned_done;
  }
  return CBX_OK;
}

// A product whose small units took row lists and then found no room for its
// output runs again without the lists (its list units cannot run without
// them, and the lists are released when the first attempt returns).
template <int K, class T>
static cbx_status spgemm_typed(const cbx_dcsc* A, const cbx_dcsc* B, cbx_spgemm_mode mode, const SpgemmConfig& cfg,
                               cbx_dcsc* C, cbx_spgemm_stats* stats, hipStream_t s,
                               int64_t* symbolic_out = nullptr) {
  bool lists_used = false;
  cbx_status st = spgemm_typed_once<K, T>(A, B, mode, cfg, C, stats, s, symbolic_out, &lists_used);
  if (st != CBX_OK) cbx_dcsc_free(C);
  if (st != CBX_ERR_NOMEM || !lists_used) return st;
  (void)hipStreamSynchronize(s);
  release_cache();
  SpgemmConfig plain = cfg;
  plain.unit_lists = 0;
  st = spgemm_typed_once<K, T>(A, B, mode, plain, C, stats, s, symbolic_out, nullptr);
  if (st != CBX_OK) cbx_dcsc_free(C);
  return st;
}

// The operands as the features and the sampling estimator read them: validated
// (invalid: an error naming `who`), with A's rows as 32 bits and B's entries'
// positions in A.
static cbx_status index_operands(const cbx_dcsc* A, const cbx_dcsc* B, const char* who, ScratchSet& ws,
                                 int32_t** rowsA, int32_t** bpos) {
  hipStream_t s = ws.s;
  SlotHold slot;
  CBX_RETURN_IF(!slot.p, CBX_ERR_NOMEM, "%s: no pinned host memory", who);
  Report* rep = (Report*)slot.p->host;
  int32_t* colmap = nullptr;
  int64_t *flop, *nnzcol;
  Counters* ctr;
  CBX_TRY(dalloc(ws, 1, &ctr));
  if (A->nzc != A->n) CBX_TRY(dalloc(ws, A->n, &colmap));
  CBX_TRY(dalloc(ws, std::max<int64_t>(A->nnz, 1), rowsA));
  CBX_TRY(dalloc(ws, std::max<int64_t>(B->nnz, 1), bpos));
  CBX_TRY(dalloc(ws, B->nzc + 1, &flop));
  CBX_TRY(dalloc(ws, B->nzc + 1, &nnzcol));
  k_init<<<256, 256, 0, s>>>(ctr, colmap, A->n, flop, nnzcol, B->nzc);
  CBX_TRY(launch_validate(A, *rowsA, ctr->val, s));
  CBX_TRY(launch_validate(B, nullptr, ctr->val + 3, s));
  k_validate_flag<<<1, 64, 0, s>>>(ctr->val, 4, &ctr->err);
  k_validate_flag<<<1, 64, 0, s>>>(ctr->val + 3, 5, &ctr->err);
  k_report_err<<<1, 64, 0, s>>>(&ctr->err, rep);
  CBX_HIP(hipStreamSynchronize(s));
  if (((volatile Report*)rep)->err) return set_error(CBX_ERR_INVALID, "%s: operand is not a valid DCSC", who);
  if (colmap && A->nzc) k_colmap<<<nblk(A->nzc, 256), 256, 0, s>>>(A->jc, A->nzc, nullptr, colmap);
  if (B->nnz && A->nzc)
    k_flops<<<nblk(B->nnz, kFlopTile), kFlopNT, 0, s>>>(B->cp, B->ir, B->nzc, B->nnz, colmap, A->cp, nullptr, *bpos,
                                                       flop);
  else if (B->nnz)
    k_fill_i32<<<nblk(B->nnz, 256), 256, 0, s>>>(*bpos, B->nnz, -1);
  CBX_HIP(hipGetLastError());
  return CBX_OK;
}

cbx_status spgemm_features(const cbx_dcsc* A, const cbx_dcsc* B, float* feats, hipStream_t s) {
  if (B->nzc == 0) return CBX_OK;
  ScratchSet ws(s);
  int32_t *rowsA, *bpos;
  CBX_TRY(index_operands(A, B, "cbx_spgemm_features", ws, &rowsA, &bpos));
  k_features<<<wave_grid(B->nzc), 256, 0, s>>>(B->cp, B->nzc, bpos, A->cp, rowsA, A->m, feats);
  CBX_HIP(hipGetLastError());
  CBX_HIP(hipStreamSynchronize(s));
  return CBX_OK;
}

cbx_status spgemm_estimate_sampling(const cbx_dcsc* A, const cbx_dcsc* B, int rounds, float* est, double* total,
                                    hipStream_t s) {
  const int64_t nzcB = B->nzc;
  if (total) *total = 0.0;
  if (nzcB == 0) return CBX_OK;
  ScratchSet ws(s);
  int32_t *rowsA, *bpos;
  float *samp, *e;
  double* dsum;
  CBX_TRY(index_operands(A, B, "cbx_spgemm_estimate_sampling", ws, &rowsA, &bpos));
  CBX_TRY(dalloc(ws, sampling_scratch_floats(A, rounds), &samp));
  CBX_TRY(dalloc(ws, 1, &dsum));
  e = est;
  if (!e) CBX_TRY(dalloc(ws, nzcB, &e));
  CBX_TRY(sampling_estimate_launch(A, B, rounds, rowsA, bpos, samp, e, s));
  if (total) {
    CBX_HIP(hipMemsetAsync(dsum, 0, sizeof(double), s));
    k_sum_f32<<<256, 256, 0, s>>>(e, nzcB, dsum);
    CBX_HIP(hipMemcpyAsync(total, dsum, sizeof(double), hipMemcpyDeviceToHost, s));
  }
  CBX_HIP(hipGetLastError());
  CBX_HIP(hipStreamSynchronize(s));
  return CBX_OK;
}

cbx_status spgemm_flops(const cbx_dcsc* A, const cbx_dcsc* B, int64_t* flop_host, hipStream_t s) {
  const int64_t nzcA = A->nzc, nzcB = B->nzc, nnzB = B->nnz;
  if (nzcB == 0) return CBX_OK;
  ScratchSet ws(s);
  int32_t *colmap = nullptr, *bpos;
  int64_t *flop, *nnzcol;
  Counters* ctr;
  CBX_TRY(dalloc(ws, 1, &ctr));
  if (nzcA != A->n) CBX_TRY(dalloc(ws, A->n, &colmap));
  CBX_TRY(dalloc(ws, std::max<int64_t>(nnzB, 1), &bpos));
  CBX_TRY(dalloc(ws, nzcB + 1, &flop));
  CBX_TRY(dalloc(ws, nzcB + 1, &nnzcol));
  k_init<<<256, 256, 0, s>>>(ctr, colmap, A->n, flop, nnzcol, nzcB);
  // a malformed operand has no products here; the product itself reports it
  CBX_TRY(launch_validate(A, nullptr, ctr->val, s));
  CBX_TRY(launch_validate(B, nullptr, ctr->val + 3, s));
  if (colmap && nzcA) k_colmap<<<nblk(nzcA, 256), 256, 0, s>>>(A->jc, nzcA, ctr, colmap);
  if (nnzB && nzcA)
    k_flops<<<nblk(nnzB, kFlopTile), kFlopNT, 0, s>>>(B->cp, B->ir, nzcB, nnzB, colmap, A->cp, ctr, bpos, flop);
  CBX_HIP(hipGetLastError());
  CBX_HIP(hipMemcpyAsync(flop_host, flop, sizeof(int64_t) * nzcB, hipMemcpyDeviceToHost, s));
  CBX_HIP(hipStreamSynchronize(s));
  return CBX_OK;
}

// The symbolic pass alone for operands of any value type: with symbolic_out
// set, spgemm_typed runs only structure kernels (the unit, hash and tiny
// tiers' counting forms, no staged tiny numeric), so no value is read and the
// instantiation's value type is immaterial.
cbx_status spgemm_symbolic(const cbx_dcsc* A, const cbx_dcsc* B, int64_t* nnz, hipStream_t s) {
  cbx_dcsc C;
  SpgemmConfig cfg = current_config();
  return spgemm_typed<kPlusTimes, int64_t>(A, B, CBX_SPGEMM_TWO_PHASE, cfg, &C, nullptr, s, nnz);
}

cbx_status spgemm_dispatch(const cbx_dcsc* A, const cbx_dcsc* B, cbx_semiring sr, cbx_spgemm_mode mode,
                           const SpgemmConfig& cfg, cbx_dcsc* C, cbx_spgemm_stats* stats, hipStream_t s) {
  switch (sr) {
    case CBX_SR_PLUS_TIMES:
      switch (A->dtype) {
        case CBX_I64: return spgemm_typed<kPlusTimes, int64_t>(A, B, mode, cfg, C, stats, s);
        case CBX_F64: return spgemm_typed<kPlusTimes, double>(A, B, mode, cfg, C, stats, s);
        case CBX_F32: return spgemm_typed<kPlusTimes, float>(A, B, mode, cfg, C, stats, s);
        case CBX_BOOL: return spgemm_typed<kPlusTimes, uint8_t>(A, B, mode, cfg, C, stats, s);
      }
      break;
    case CBX_SR_MIN_PLUS:
      switch (A->dtype) {
        case CBX_I64: return spgemm_typed<kMinPlus, int64_t>(A, B, mode, cfg, C, stats, s);
        case CBX_F64: return spgemm_typed<kMinPlus, double>(A, B, mode, cfg, C, stats, s);
        case CBX_F32: return spgemm_typed<kMinPlus, float>(A, B, mode, cfg, C, stats, s);
      }
      break;
    case CBX_SR_SELECT_MAX:
      switch (A->dtype) {
        case CBX_I64: return spgemm_typed<kSelectMax, int64_t>(A, B, mode, cfg, C, stats, s);
        case CBX_F64: return spgemm_typed<kSelectMax, double>(A, B, mode, cfg, C, stats, s);
        case CBX_F32: return spgemm_typed<kSelectMax, float>(A, B, mode, cfg, C, stats, s);
      }
      break;
  }
  return set_error(CBX_ERR_UNSUPPORTED, "cbx_spgemm: semiring %d with dtype %d is not provided", (int)sr,
                   (int)A->dtype);
}

}  // namespace cbx
