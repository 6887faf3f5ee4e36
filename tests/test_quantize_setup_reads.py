"""CPU check of the addresses the quantize set-up reads.

``FqTileRows::load`` (quant_ops_amd/csrc/flatquant_tile.h) copies L or R into
registers as whole 16-byte chunks and one element of the tail per thread. Here
the same function runs on the host, for every thread of a workgroup, on
matrices whose element i holds i (modulo 2^15) and which are followed by a
pattern that no element holds: a register with the pattern in it was read past
the matrix. The smallest matrix, 2 x 2, is 8 bytes and has no whole chunk.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SOURCE = r"""
#include <cstdio>
#include <cstring>
#include "flatquant_tile.h"

int main() {
  constexpr int kNt = 64, kCh = 128;   // 64 threads cover 256 x 256
  static _Float16 buf[256 * 256 + 64] __attribute__((aligned(16)));
  int bad = 0;
  for (int n = 2; n <= 256; ++n) {
    const int elems = n * n;
    for (int i = 0; i < elems + 64; ++i) {
      const uint16_t v = i < elems ? (uint16_t)(i & 0x7FFF) : (uint16_t)0xFFFF;
      std::memcpy(buf + i, &v, 2);
    }
    for (int tid = 0; tid < kNt; ++tid) {
      static qo::FqTileRows<_Float16, kCh> rows;
      std::memset(&rows, 0, sizeof rows);
      rows.load(buf, elems, tid, kNt);
      uint16_t got[8 * kCh + 1];
      std::memcpy(got, rows.v, sizeof rows.v);
      std::memcpy(got + 8 * kCh, &rows.tail, 2);
      bool past = false, whole = true;
      for (uint16_t g : got) past |= g == 0xFFFF;
      for (int c = tid; c < elems / 8; c += kNt)   // this thread's chunks arrived
        for (int j = 0; j < 8; ++j) whole &= got[8 * ((c - tid) / kNt) + j] == ((8 * c + j) & 0x7FFF);
      if (elems / 8 * 8 + tid < elems) whole &= got[8 * kCh] == ((elems / 8 * 8 + tid) & 0x7FFF);
      if (past || !whole) {
        if (bad++ == 0) std::printf("n=%d thread %d: %s\n", n, tid, past ? "read past the matrix" : "wrong elements");
      }
    }
  }
  std::printf("bad=%d\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc absent")
def test_set_up_reads_stay_inside_l_and_r(tmp_path):
    src, exe = tmp_path / "reads.hip", tmp_path / "reads"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-O1", "-w",
                    f"-I{ROOT}/include", f"-I{ROOT}/quant_ops_amd/csrc", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert out.returncode == 0, out.stdout
