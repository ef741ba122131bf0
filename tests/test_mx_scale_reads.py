"""Where the MXFP4 prefill kernel reads its weights' block scales in LDS (mx_last_rows, mx_scale_src,
mx_scale_back of hh_mfma.hpp), for every wave of every row tile, lane, stage and block: inside the
16 bytes loaded for the row (its last dword may pass into the next row's where the block lies past
the row's end), and, for a block of the row, the byte that holds it. Whole waves past the last row
included. Host code only."""
import os
import subprocess

from hydra_amd import build

SOURCE = r"""
#include "hh_mfma.hpp"
#include <algorithm>
#include <cstdio>
using namespace hh;
int main() {
  // (rows, columns): one row tile and less, ragged last tiles, rows of odd and even dwords of scales
  const int shapes[][2] = {{64, 64}, {64, 2880}, {128, 64}, {320, 192}, {640, 192}, {2880, 64},
                           {2880, 2880}, {5760, 2880}, {2048, 1024}, {576, 1088}};
  long bad = 0;
  for (auto &sh : shapes) {
    const int out = sh[0], K = sh[1], nsb = K / 32, n = (K + 127) / 128;
    for (int rw = 0; rw < (out + 255) / 256 * 256; rw += 64)
      for (int s = 0; s < n; ++s)
        for (int r = 0; r < 64; ++r)
          for (int g = 0; g < 4; ++g) {
            const int s3 = s % 3, sc0 = 4 * (s - s3), row = rw + r, srow = std::min(row, out - 1);
            const int src = mx_scale_src(srow, out, nsb, sc0);
            const int back = mx_last_rows(rw, out) ? mx_scale_back(row, out, nsb, sc0) : 0;
            const int byte = ((row * nsb) & 3) + back + 4 * s3 + g;   // of the row's 16 bytes
            bool ok = src >= 0 && src + 16 <= out * nsb && byte >= 0 && byte < 20;
            if (row < out && 4 * s + g < nsb) ok = ok && byte < 16 && src + byte == row * nsb + 4 * s + g;
            if (!ok && bad++ < 5) std::printf("rows %d cols %d row %d stage %d group %d: byte %d\n", out, K, row, s, g, byte);
          }
  }
  return bad != 0;
}
"""


def test_scale_reads_stay_in_the_loaded_bytes(tmp_path):
    src, exe = tmp_path / "reads.hip", tmp_path / "reads"
    src.write_text(SOURCE)
    r = subprocess.run([build.hipcc(), "--offload-host-only", "-O2", "-std=c++17", "-w", "-I", build.CSRC,
                        "-I", os.path.join(build.ROOT, "include"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
