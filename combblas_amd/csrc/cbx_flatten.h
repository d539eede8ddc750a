// Block-level flattening of segment products (shared by SpGEMM, SpMV and BFS).
//
// A chunk holds at most one segment per thread: consecutive entries (an A
// column restricted to some rows, a run, a vertex's neighbours), paired with a
// multiplier.
#pragma once

#include "cbx_device.h"

namespace cbx {

// ------------------------------------------------------------- bit-flattened
// Flattening by a bitmap of segment starts.  Product x of a chunk lies in
// segment k(x) = the number of segments (after the first) that start at or
// before x: with one bit per segment at position start - 1, that is the number
// of bits below x, which a lane gets from the word that its wave's 64 products
// share (held in two scalar registers) with two mbcnt instructions, the bits
// of earlier words included.  Its A entry is x + delta[k].
//
// Per product this is about ten VALU instructions and two LDS reads (delta and
// the multiplier), and the lanes of a wave read consecutive entries of A.  A
// binary search for every four products took about 30, with nine
// dependent LDS reads, and lanes four entries apart: the symbolic pass ran
// with the VALU 81 % busy and the small units' kernel 56 %.
//
// A chunk's products are visited in tiles of kTileWords * 64.
constexpr int kTileWords = 2 * kWave;  // two words per lane
constexpr int kTileProducts = kTileWords * 64;

template <class T, int NT, bool VAL>
struct FlatStage {
  unsigned long long starts[2][kTileWords];  // alternate from tile to tile
  int32_t delta[NT];
  T bval[VAL ? NT : 1];
  int wcount[NT / kWave], wlen[NT / kWave];  // segments and products of each wave
};

// A thread's segment of the staged chunk, and the chunk's product count.
struct FlatSeg {
  int k;      // its number among the non-empty ones; -1: empty
  int start;  // its first product
  int total;  // products of the chunk (uniform)
};

// One tile as every wave holds it: lane i has words i and 64 + i and the
// number of segments started before each.
struct FlatTile {
  unsigned long long w0, w1;
  int p0, p1;
  int base;  // first product of the tile
  int next;  // segments (after the first) started up to the tile's end (uniform)
};

// Clears the bitmaps: once per workgroup, before its first chunk.
template <class T, int NT, bool VAL>
__device__ __forceinline__ void flat_init(FlatStage<T, NT, VAL>& st) {
  for (int i = threadIdx.x; i < 2 * kTileWords; i += NT) (&st.starts[0][0])[i] = 0ull;
}

// Stages one chunk, at most one segment per thread; its products are numbered
// from x0 on (0 where flat_chunk visits them).  One barrier; the caller's
// earlier writes to LDS are visible after it, and the previous chunk must have
// been visited by each wave when it calls.
template <class T, int NT, bool VAL>
__device__ __forceinline__ FlatSeg flat_stage(FlatStage<T, NT, VAL>& st, int32_t base, int len, T bv, int x0 = 0) {
  constexpr int NW = NT / kWave;
  const int lane = lane_id(), w = wave_id_uniform();
  const unsigned long long some = __ballot(len > 0);
  const int incl = wave_incl_scan(len);
  if (lane == kWave - 1) {
    st.wcount[w] = __popcll(some);
    st.wlen[w] = incl;
  }
  __syncthreads();
  const int wc = wave_incl_scan(lane < NW ? st.wcount[lane] : 0);
  const int wl = wave_incl_scan(lane < NW ? st.wlen[lane] : 0);
  const int c0 = w ? __builtin_amdgcn_readlane(wc, w - 1) : 0;
  const int l0 = w ? __builtin_amdgcn_readlane(wl, w - 1) : 0;
  FlatSeg me;
  me.total = __builtin_amdgcn_readlane(wl, NW - 1);
  me.start = x0 + l0 + incl - len;
  me.k = -1;
  if (len > 0) {
    me.k = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(some >> 32),
                                          __builtin_amdgcn_mbcnt_lo((unsigned)some, (unsigned)c0));
    st.delta[me.k] = base - me.start;
    if constexpr (VAL) st.bval[me.k] = bv;
  }
  return me;
}

// Tile number t of the staged chunk; `before` is the previous tile's `next` (0
// for the first), `par` alternates from tile to tile over the workgroup's whole
// life, starting anywhere.  Contains barriers.
template <class T, int NT, bool VAL>
__device__ __forceinline__ FlatTile flat_tile(FlatStage<T, NT, VAL>& st, const FlatSeg& me, int t, int before,
                                              int par) {
  if (t) __syncthreads();  // the bitmap that the previous tile's waves cleared
  FlatTile ft;
  ft.base = t * kTileProducts;
  const int at = me.start - 1 - ft.base;
  if (me.k > 0 && at >= 0 && at < kTileProducts)
    __hip_atomic_fetch_or(&st.starts[par][at >> 6], 1ull << (at & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  __syncthreads();
  ft.w0 = st.starts[par][lane_id()];
  ft.w1 = st.starts[par][kWave + lane_id()];
  // every wave has read the other bitmap (before the barrier above): clear it
  for (int i = threadIdx.x; i < kTileWords; i += NT) st.starts[par ^ 1][i] = 0ull;
  const int c0 = __popcll(ft.w0), c1 = __popcll(ft.w1);
  const int i0 = wave_incl_scan(c0), i1 = wave_incl_scan(c1);
  const int half = before + __builtin_amdgcn_readlane(i0, kWave - 1);
  ft.p0 = before + i0 - c0;
  ft.p1 = half + i1 - c1;
  ft.next = half + __builtin_amdgcn_readlane(i1, kWave - 1);
  return ft;
}

// A-entry index and multiplier of this lane's product in words
// (round * U + u) * NW + wave, u < U, and whether there is one: past the end
// the lane has the chunk's last product again, ok false, so that the caller
// loads what the indices name without a branch (a branch around each load
// would wait for it before the next is issued).  The round's first word must
// hold products; rounds do not straddle the tile's halves.  No barriers.
template <class T, int NT, bool VAL, int U>
__device__ __forceinline__ void flat_round(const FlatStage<T, NT, VAL>& st, const FlatTile& ft, int total, int round,
                                           int32_t (&idx)[U], T (&bvs)[U], bool (&ok)[U]) {
  constexpr int NW = NT / kWave;
  static_assert(kWave % (U * NW) == 0 || U * NW == kWave, "a round lies in one half of the tile");
  const int j0 = round * U * NW + wave_id_uniform();
  const bool low = j0 < kWave;  // uniform
  const unsigned wl = low ? (unsigned)ft.w0 : (unsigned)ft.w1;
  const unsigned wh = low ? (unsigned)(ft.w0 >> 32) : (unsigned)(ft.w1 >> 32);
  const int pp = low ? ft.p0 : ft.p1;
  const int end = min(total - ft.base, kTileProducts);
  int k[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = (j0 + u * NW) & (kWave - 1);  // scalar
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)wl, j);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)wh, j);
    const unsigned kb = (unsigned)__builtin_amdgcn_readlane(pp, j);
    k[u] = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, kb));
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int x = (j0 + u * NW) * kWave + lane_id();
    ok[u] = x < end;
    idx[u] = ft.base + min(x, end - 1) + st.delta[k[u]];
    if constexpr (VAL) bvs[u] = st.bval[k[u]];
    else bvs[u] = T{};
  }
}

// The words of the tile that hold products.
__device__ __forceinline__ int flat_words(const FlatTile& ft, int total) {
  return (min(total - ft.base, kTileProducts) + 63) >> 6;
}

// f(idx, bvs, ok) for every round of the tile from first_round on.
template <class T, int NT, bool VAL, int U, class F>
__device__ __forceinline__ void flat_visit(const FlatStage<T, NT, VAL>& st, const FlatTile& ft, int total, F&& f,
                                           int first_round = 0) {
  constexpr int NW = NT / kWave;
  const int words = flat_words(ft, total) - wave_id_uniform();
  for (int r = first_round; r * U * NW < words; ++r) {
    int32_t idx[U];
    T bvs[U];
    bool ok[U];
    flat_round<T, NT, VAL, U>(st, ft, total, r, idx, bvs, ok);
    f(idx, bvs, ok);
  }
}

// Every product of a staged chunk; `par` is carried from chunk to chunk.
template <class T, int NT, bool VAL, int U, class F>
__device__ __forceinline__ void flat_chunk(FlatStage<T, NT, VAL>& st, const FlatSeg& me, int& par, F&& f) {
  if (me.total == 0) __syncthreads();  // every wave has read the counts before the next chunk's are written
  int before = 0;
  for (int t = 0; t * kTileProducts < me.total; ++t) {
    const FlatTile ft = flat_tile(st, me, t, before, par);
    par ^= 1;
    before = ft.next;
    flat_visit<T, NT, VAL, U>(st, ft, me.total, f);
  }
}

}  // namespace cbx
