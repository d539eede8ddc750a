"""The caching allocator's block sizes and lists, and products at the limit of
the card's memory."""
from __future__ import annotations

import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

import combblas_amd as cb
from combblas_amd import predictor

CSRC = Path(__file__).resolve().parents[1] / "combblas_amd" / "csrc"
GB = 1 << 30


def test_block_sizes(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(r"""
#include <cstdio>
#include "cbx_blocks.h"
int main() {
  size_t last = 0;
  for (int e = 8; e < 39; ++e)
    for (size_t k = 0; k < 64; ++k) {
      const size_t bytes = ((size_t)1 << e) + (k << e) / 64 + k % 3, got = cbx::block_bytes(bytes);
      const bool ok = got >= bytes && (got - bytes) * 8 <= bytes + 8 * 256 && got - bytes < (size_t)1 << 30 &&
                      got >= last && got % 256 == 0;
      if (!ok) return std::printf("%zu -> %zu\n", bytes, got), 1;
      last = got;
    }
  // sizes a few percent apart share a block
  return cbx::block_bytes((size_t)20 << 20) == cbx::block_bytes(((size_t)20 << 20) - (1 << 19)) ? 0 : 2;
}
""")
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_idle_blocks_stay_on_their_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(r"""
#include <cstdio>
#include "cbx_blocks.h"
#define CHECK(x) do { if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), 1; } while (0)
int main() {
  char mem[4];
  cbx::BlockLists b;
  b.add(mem, 0, 1000);
  b.add(mem + 1, 1, 5 << 20);
  b.add(mem + 2, 0, 5 << 20);
  CHECK(!b.take(0, 1000));  // in use
  CHECK(b.give_back(mem) && b.give_back(mem + 1) && b.give_back(mem + 2));
  CHECK(!b.give_back(mem) && !b.give_back(mem + 3));
  CHECK(b.idle_bytes(0) == 1000 + (5 << 20) && b.idle_bytes(1) == 5 << 20 && b.idle_bytes(2) == 0);
  CHECK(!b.take(1, 6 << 20) && !b.take(2, 1000));
  CHECK(b.take(1, 4 << 20) == mem + 1 && !b.take(1, 4 << 20));  // device 0 has another
  CHECK(!b.take(0, 3 << 20) || !"more than a quarter and 1 MB larger");
  CHECK(b.take(0, 1000) == mem && b.take(0, 5 << 20) == mem + 2 && b.idle_bytes(0) == 0);
  b.give_back(mem);
  b.give_back(mem + 1);
  int n = 0;
  b.release([&](void* p) { n += p == mem || p == mem + 1; });
  CHECK(n == 2 && !b.take(0, 1000) && b.idle_bytes(1) == 0 && b.give_back(mem + 2));
  return 0;
}
""")
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def _free():
    free, total = C.c_size_t(), C.c_size_t()
    assert cb.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def leave(free):
    """Blocks that leave about `free` bytes of device memory (of sizes that the allocator does not round)."""
    held = []
    for size in (64 * GB, GB, GB // 16):
        while _free() - size >= free:
            held.append(cb.DeviceArray(size, np.uint8))
    return held


def _outer():
    """Operands of a full 40,000 x 27,200 product: ir and val of 8.1 GiB, 9 each when rounded up."""
    m, n = 40_000, 27_200
    A = cb.Dcsc.from_coo(m, 1, np.arange(m), np.zeros(m, np.int64), np.arange(m) % 9 + 1).to_device()
    return A, cb.Dcsc.from_coo(1, n, np.zeros(n, np.int64), np.arange(n), np.arange(n) % 5 + 1).to_device()


@pytest.mark.gpu
def test_output_that_fits_without_its_surplus():
    A, B = _outer()
    base = cb.get_config()
    held = []
    try:
        cb.set_config(unit_lists=0)  # (a product that fails with row lists runs again without them)
        C_, _ = cb.spgemm(A, B)
        sums = C_.column_checksums(1)
        C_.release()
        cb.release_cached_memory()
        # 9 GiB and 8.1 do not fit, twice 8.1 and the scratch of some 20 MB do
        held = leave(16 * GB + 3 * GB // 4)
        C_, _ = cb.spgemm(A, B)
        assert C_.nnz == A.m * B.n and np.array_equal(C_.column_checksums(1), sums)
        C_.release()
    finally:
        cb.set_config(**base)
        for h in held:
            h.release()
        cb.release_cached_memory()


@pytest.mark.gpu
def test_product_that_does_not_fit_leaves_nothing():
    A, B = _outer()
    C_, _ = cb.spgemm(A, B)  # (what the runtime itself takes for the kernels)
    C_.release()
    held = []
    try:
        cb.release_cached_memory()
        before = _free()
        held = leave(15 * GB)  # room for the row lists, but in no attempt for the output
        out = cb.cbx_dcsc()
        st = cb.lib().cbx_spgemm(C.byref(A.s), C.byref(B.s), 0, 0, C.byref(out), None, None)
        assert st == cb.ERR_NOMEM
        assert not (out.cp or out.jc or out.ir or out.val)
    finally:
        for h in held:
            h.release()
        cb.release_cached_memory()
    assert _free() >= before - GB // 4  # (none of the output's arrays)


@pytest.mark.gpu
def test_learned_pass_is_not_begun_where_its_staging_area_does_not_fit():
    """Beside the output, that is: the pass would be done and then done again."""
    A = cb.gen_rmat(18, 16).to_device()
    base = cb.get_config()
    held = []
    cb.set_predictor(predictor.load())
    try:
        cb.set_config(learned_target=2.0)  # a pass then has units to re-run, and counts them
        C_, st = cb.spgemm(A, A, mode="learned")
        assert st["overflow_cols"] > 0 and st["learned_fallback"] == 0
        staging = 12 * st["predicted_nnz"]
        assert staging > 10 * GB
        sums = C_.column_checksums(1)
        C_.release()
        cb.release_cached_memory()
        before = _free()
        C_, _ = cb.spgemm(A, A)
        C_.release()
        used = before - _free()  # by the two-phase product
        cb.release_cached_memory()
        held = leave(used + 2 * GB)
        C_, st = cb.spgemm(A, A, mode="learned")
        assert st["learned_fallback"] == 1 and st["overflow_cols"] == 0
        assert np.array_equal(C_.column_checksums(1), sums)
        C_.release()
    finally:
        cb.set_predictor(None)
        cb.set_config(**base)
        for h in held:
            h.release()
        cb.release_cached_memory()
