"""Index arithmetic of the kernels (csrc/cbx_index.h) at the end of its 32-bit
range, compiled for the host."""
from __future__ import annotations

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "combblas_amd" / "csrc"


def _run(tmp_path, body: str) -> None:
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include <cstdio>\n#include <cstdlib>\n#include <initializer_list>\n#include "cbx_index.h"\n'
                   '#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\\n", __LINE__, #x); std::exit(1); } } '
                   'while (0)\n' + body)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-fwrapv", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


def test_search_up_to_the_last_index(tmp_path):
    """A column whose entries end at 2^31 - 1: no probe leaves it, and every answer is the linear search's."""
    _run(tmp_path, r"""
int main() {
  const int32_t last = 0x7fffffff;
  for (int32_t len : {1, 2, 3, 64, 4097, 20000}) {
    for (int32_t end : {last, last - 1, last - 5000, len}) {
      for (int32_t gap : {1, 3, 4096}) {  // row of entry k: gap * k
        const int32_t begin = end - len;
        auto row = [&](int32_t i) {
          CHECK(i >= begin && i < end);
          return (int64_t)gap * (i - begin);
        };
        int32_t lo = begin;
        for (int t = 0; t <= 20; ++t) {
          const int64_t key = (int64_t)t * 4096;
          lo = cbx::first_from(row, lo, end, key);
          int64_t want = (key + gap - 1) / gap;
          if (want > len) want = len;
          CHECK(lo == begin + want);
        }
      }
    }
  }
}
""")


def test_entries_of_a_piece_at_the_last_index(tmp_path):
    """Pieces of 1024 entries of ranges that end at 2^31 - 1: every index lies in its piece."""
    _run(tmp_path, r"""
int main() {
  const int32_t last = 0x7fffffff;
  for (int32_t len : {1, 1023, 1024, 1025, 5000}) {
    for (int32_t end : {last, last - 1, last - 1024, len}) {
      for (int32_t first = end - len; end - first > 0; first += 1024) {
        for (int32_t off = 0; off < 1024; ++off) {
          bool ok;
          const int32_t e = cbx::entry_from(first, end, off, ok);
          CHECK(ok == ((int64_t)first + off < end));
          CHECK(e == (ok ? first + off : end - 1));
        }
        if (end - first <= 1024) break;
      }
    }
  }
}
""")
