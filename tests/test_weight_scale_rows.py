"""The row of weight scales a wave of a tile reads, for every wave of every column tile (compiled for the host; no GPU needed): inside the
matrix of scales, the columns' own row where the wave has columns, and taken by the kernel that reads it through a plain pointer."""
import os
import subprocess

from modular_amd import build

PROGRAM = """
#include <initializer_list>

#include "scale_rows.h"
int main() {
  for (int N = 1; N <= 1500; ++N)
    for (int tile : {128, 192, 256})
      for (int wave : {32, 64, 96, 128})
        for (int n0 = 0; n0 < N; n0 += tile)
          for (int n = n0; n < n0 + tile; n += wave) {
            const int row = maxfp8::weight_scale_row(n, N);
            if (row < 0 || row >= (N + 127) / 128 || (n < N && row != n / 128)) return 1;
          }
  return maxfp8::weight_scale_row(2147483392, 2147483136) == 16777211 ? 0 : 2;
}
"""


def test_rows_of_the_scales_are_the_operands(tmp_path):
    source, program = tmp_path / "rows.cpp", tmp_path / "rows"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", f"-I{build.CSRC}", str(source), "-o", str(program)], check=True)
    assert subprocess.run([str(program)]).returncode == 0
    with open(os.path.join(build.CSRC, "gemm_tiled.hip")) as f:
        body = f.read().split("__device__ __forceinline__ void tile_body(")[1].split("\n}\n")[0]
    assert "bs_row = bs_ptr + (int64_t)weight_scale_row(n0 + wn * WN, p.N) * p.b_scales_ld" in body
