"""What mfma_tiles.hpp relies on and no result shows: the code that the compiler makes of it (CPU: hipcc compiles for gfx950 without one)."""
import os
import re
import subprocess

import pytest

from vllmini_amd import build

PROBE = """
#include "mfma_tiles.hpp"
template <int MI, int NI, int D>
__global__ __launch_bounds__(256, 2) void tiles_kernel(const void* x, const void* w, const float* b, float* y, long ldx, int M, int N, int K) {
  float bias[NI];
  vmi_tiles::tiles_product<vmi_tiles::Half, MI, NI, D>(
      x, ldx, w, M, N, K, [&](int, int s, int SL) { for (int n = 0; n < NI; ++n) bias[n] = b[min(s + n, SL - 1)]; },
      [&](const auto& acc, int m, int s, int SL) {
        for (int n = 0; n < NI; ++n)
          for (int i = 0; i < MI; ++i)
            if (m + 16 * i < M && s + n < SL)
              for (int r = 0; r < 4; ++r) y[(m + 16 * i) * (long)N + (s + n) * 16 + r] = acc[n][i][r] + bias[n];
      });
}
"""
SHAPES = [(2, 1, 2), (2, 1, 4), (4, 2, 4), (6, 2, 2), (8, 3, 4)]      # rows / 16, columns / 64, chunks in flight


@pytest.mark.parametrize("strategy", ["", "max-ilp", "iterative-ilp", "iterative-minreg"])
def test_requests_of_a_tile_go_out_in_the_order_that_its_waits_count(strategy, tmp_path):
    """A wave lets a barrier pass when all but so many of its last requests are there: chunk by chunk the ones into LDS, then the weights', whatever the compiler's scheduler prefers."""
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE + "".join(f"template __global__ void tiles_kernel<{a}, {b}, {c}>(const void*, const void*, const float*, float*, long, int, int, int);\n" for a, b, c in SHAPES))
    cmd = [build._hipcc(), *build._flags("fma"), "-I", build.CSRC, *(["-mllvm", f"-amdgpu-sched-strategy={strategy}"] if strategy else []), "--cuda-device-only", "-S", str(src), "-o", str(out)]
    done = subprocess.run(cmd, capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    seen = {}
    for text in re.split(r"\n(?=_Z\w+:)", out.read_text()):
        name = re.match(r"_Z\d+tiles_kernelILi(\d+)ELi(\d+)ELi(\d+)E", text)
        if name:
            marks = ("B" if m.startswith("s_barrier") else "X" if " lds" in m else "W" for m in map(str.strip, text.split("\n")) if re.match(r"s_barrier|buffer_load", m))
            seen[tuple(map(int, name.groups()))] = "".join(marks).split("B")
    assert sorted(seen) == SHAPES
    for (mi, ni, d), parts in seen.items():
        chunk = "X" * (mi // 2) + "W" * (2 * ni)
        assert parts[0] == chunk * (d - 1), (mi, ni, d, parts[0])
        assert parts[1:] == [chunk] * (d + 1) + [""] * (d - 1), (mi, ni, d, parts)
