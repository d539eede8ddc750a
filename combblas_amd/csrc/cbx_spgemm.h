// Internal interface of the SpGEMM driver.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "cbx_internal.h"

namespace cbx {

// Tunables of the SpGEMM driver.
struct SpgemmConfig {
  // Columns with flop_j <= small_flop_max are formed by one workgroup (sort
  // tier), the rest by row-range units.  At most 4096 (four products per thread
  // of the largest workgroup; the counting hash table of 8192 slots is kept at
  // most half full).
  int64_t small_flop_max = 4096;
  // Sort tier sizes: flop_j in (hash_mid_flop, small_flop_max] are counted in
  // the 8192-slot table and sorted by 512 threads (1024 beyond 2048 products),
  // (tiny_flop, hash_mid_flop] in the 2048-slot table by 256; columns with
  // flop_j <= tiny_flop (<= 256) take one wave each (the tiny tier).
  int64_t hash_mid_flop = 1024;
  int64_t tiny_flop = 256;
  // Learned mode: columns predicted to exceed heavy_nnz outputs are computed
  // exactly (symbolic, then two-phase units).
  int64_t heavy_nnz = 65536;
  // Unit tier: columns whose exact output exceeds unit_split_nnz use the
  // large units.
  int64_t unit_split_nnz = 131072;
  // Learned mode: device parameters of the nnz predictor (null = not loaded),
  // unit size target as a fraction of the value window, and the headroom of
  // the output capacity over the predicted total.
  const float* predictor = nullptr;
  // Learned mode without the network: with sampling_rounds > 0 the column
  // sizes come from the min-hash estimator of estimateNNZ_sampling
  // (sampling_estimate_launch) instead of the predictor.
  int sampling_rounds = 0;
  float learned_target = 0.75f;
  // Operands the library produced itself (a transpose, an earlier product)
  // are valid by construction and skip the device validation pass.
  bool trusted_a = false, trusted_b = false;
  // A's rows as 32-bit, where the caller has them (and has checked A): A.ir is
  // not read then.
  const int32_t* rows_a = nullptr;
  float capacity_margin = 0.15f;
  // Two-phase mode: share of the free memory the large units' row maps may take (0: none).
  float row_map_share = 0.25f;
  // Workgroup shape of the tiny tier: columns (one wave each) per workgroup.
  int tiny_wg_waves = 4;
  // Exactly sized (two-phase) units in the symbolic pass's order (0) or
  // sorted by first row block (1).
  int unit_order = 1;
  // Symbolic pass of the unit tier: per column (0) or in bands of 16 / 64
  // row blocks dispatched band by band.
  int sym_band = 0;
  // Fused threshold (set by the MCL expansion, two-phase mode only): the
  // product keeps only entries with !(v < filter_thr).
  bool filter = false;
  double filter_thr = 0.0;
  // cbx_mcl_expand may fuse its hard threshold into two-phase products.
  bool mcl_fuse = true;
  // Two-phase, per-column symbolic form: the symbolic pass writes the sorted
  // rows of the small-unit columns, whose units are then cut by output count
  // over any number of row blocks (k_num_list).
  int unit_lists = 1;
  // Numeric unit launches: runs of this many consecutive (row-block sorted)
  // units per XCD (0: the hardware's round-robin order).
  int unit_xcd_group = 0;
};

// The process-wide tunables (cbx_spgemm_set_config) with the installed
// predictor: the starting configuration of every product.
SpgemmConfig current_config();

// Per-column min-hash estimates of nnz(C(:,j)) (cbx_sampling.hip): `scratch`
// holds sampling_scratch_floats(A, rounds) floats; rowsA (int32 rows of A)
// and bpos (B's rows as A stored-column positions) come from the product's
// setup; est gets nzc(B) floats.  rounds in [2, 8].
size_t sampling_scratch_floats(const cbx_dcsc* A, int rounds);
cbx_status sampling_estimate_launch(const cbx_dcsc* A, const cbx_dcsc* B, int rounds, const int32_t* rowsA,
                                    const int32_t* bpos, float* scratch, float* est, hipStream_t s);
int sampling_rounds_setting();

// Launches the predictor's inference kernel (cbx_mlp.hip).
void mlp_infer_launch(const float* params, const float* X, int64_t n, float* out, hipStream_t s);
const float* predictor_params();

// Cached device allocations for arrays handed to callers (see cbx_runtime.hip).
cbx_status dev_alloc(void** p, size_t bytes, bool exact = false);  // exact: a new block is not rounded up
// A matrix's ir and val; where one does not fit beside the other's surplus, both
// at their own sizes.  Both null on failure.
cbx_status dev_alloc_entries(int64_t** ir, void** val, int64_t nnz, size_t value_size);
void dev_free(void* p);
void release_cache();
size_t cache_idle_bytes();  // bytes of the current device held by the cache and free for reuse

// The scratch blocks of one call, from the caching allocator above, released
// together once the stream's kernels are done (at the latest when the set goes
// out of scope).  Requests of up to 64 KB are carved (256-byte aligned) from
// 1 MB chunks.  The stream-ordered pool is not used: its frees took 10-20 us of
// host time each (blocks of a few megabytes 2-4 ms), some thirty a product,
// and growing it by gigabytes up to 1.5 s.
struct ScratchSet {
  static constexpr size_t kSmall = (size_t)64 << 10, kChunk = (size_t)1 << 20;
  hipStream_t s;
  std::vector<void*> blocks;
  uint8_t* chunk = nullptr;
  size_t chunk_used = 0;
  explicit ScratchSet(hipStream_t st) : s(st) {}
  ScratchSet(const ScratchSet&) = delete;
  ScratchSet& operator=(const ScratchSet&) = delete;
  bool take_bytes(void** p, size_t bytes) {
    bytes = bytes < 256 ? 256 : (bytes + 255) & ~(size_t)255;
    if (bytes <= kSmall) {
      if (!chunk || chunk_used + bytes > kChunk) {
        void* c = nullptr;
        if (dev_alloc(&c, kChunk) != CBX_OK) return false;
        blocks.push_back(c);
        chunk = (uint8_t*)c;
        chunk_used = 0;
      }
      *p = chunk + chunk_used;
      chunk_used += bytes;
      return true;
    }
    if (dev_alloc(p, bytes) != CBX_OK) return false;
    blocks.push_back(*p);
    return true;
  }
  template <class X>
  bool take(X** p, size_t count) {
    void* q = nullptr;
    const bool ok = take_bytes(&q, count * sizeof(X));
    *p = (X*)q;
    return ok;
  }
  void release() {
    if (!blocks.empty()) (void)hipStreamSynchronize(s);  // the stream's kernels may still read them
    for (void* b : blocks) dev_free(b);
    blocks.clear();
    chunk = nullptr;
    chunk_used = 0;
  }
  ~ScratchSet() { release(); }
};

// What one call at a time holds beside device memory: a page of pinned host
// memory that its kernels report into, and events for its timings.  Kept in a
// list of idle ones, as many as calls ran at once on a device, and given back
// by cbx_release_cached_memory.
struct CallSlot {
  static constexpr int kEvents = 9;
  int device = 0;
  void* host = nullptr;  // 4096 bytes
  hipEvent_t ev[kEvents] = {};
};
CallSlot* slot_acquire();  // null: no memory
void slot_release(CallSlot* slot);
struct SlotHold {
  CallSlot* p;
  SlotHold() : p(slot_acquire()) {}
  ~SlotHold() {
    if (p) slot_release(p);
  }
  SlotHold(const SlotHold&) = delete;
  SlotHold& operator=(const SlotHold&) = delete;
};

// Shared front-door helpers (cbx_runtime.hip).
size_t dtype_size(cbx_dtype t);
cbx_status init_device_once();
cbx_status check_dcsc(const cbx_dcsc* X, const char* name, cbx_location loc);

// flop_j of every stored column of B (estimateFLOP), copied to host memory.
cbx_status spgemm_flops(const cbx_dcsc* A, const cbx_dcsc* B, int64_t* flop_host, hipStream_t s);
cbx_status spgemm_features(const cbx_dcsc* A, const cbx_dcsc* B, float* feats, hipStream_t s);
cbx_status spgemm_symbolic(const cbx_dcsc* A, const cbx_dcsc* B, int64_t* nnz, hipStream_t s);
cbx_status spgemm_estimate_sampling(const cbx_dcsc* A, const cbx_dcsc* B, int rounds, float* est, double* total,
                                    hipStream_t s);

// Structural check of a device DCSC (the rules of cbx_dcsc_check) with
// caller-provided counters: the launch clears cnt[0..3) and runs the check on
// s; the result call waits for s and reads them.
void dcsc_check_launch(const cbx_dcsc* X, unsigned long long* cnt, hipStream_t s);
cbx_status dcsc_check_result(const unsigned long long* cnt, hipStream_t s);
// The check's kernel alone, on counters that are 0 (cnt[0] violations; it
// passes with none and cnt[1] == cnt[2], the descents ir[e+1] <= ir[e] and
// those at column starts); colmap, if given, receives the place of each column
// that breaks no rule.
void dcsc_check_structure_launch(const cbx_dcsc* X, unsigned long long* cnt, int32_t* colmap, hipStream_t s);

// One member of a concatenation, and where its entries, columns, rows and
// column ids start in it.
struct PackSeg {
  const int64_t *cp, *jc, *ir;
  const void* val;
  int64_t row_off, col_off, nz_off, c_off;
  int64_t m, n, nnz, nzc;    // the member's own shape and sizes (for its bounds)
  int64_t nz_base, col_base; // of a column range of a matrix: its first entry (cp counts from there) and column id
};

// Writes the members' concatenation to out.cp / jc / val and their rows to
// out.ir and rows32, where these are not null (out.nnz, nzc, dtype set), and
// checks every member against its own bounds by the product's rules: the
// concatenation needs no other check.  CBX_ERR_INVALID if one is malformed.
cbx_status pack_members(const PackSeg* segs, int64_t count, const cbx_dcsc& out, int32_t* rows32, hipStream_t s);

cbx_status spgemm_dispatch(const cbx_dcsc* A, const cbx_dcsc* B, cbx_semiring sr, cbx_spgemm_mode mode,
                           const SpgemmConfig& cfg, cbx_dcsc* C, cbx_spgemm_stats* stats, hipStream_t s);

}  // namespace cbx
