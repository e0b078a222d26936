"""What mfma_tiles.hpp relies on and no result shows: the code that the compiler makes of it (CPU: hipcc compiles for gfx950 without one)."""
import os
import re
import struct
import subprocess

import msgpack
import pytest

from tests import tile_cases
from vllmini_amd import build

PROBE = """
#include "mfma_tiles.hpp"
using namespace vmi_tiles;
template <int MI, int NI, int D>
__global__ __launch_bounds__(256, 2) void tiles_kernel(const void* x, const void* w, const _Float16* b, const u32x4* r, _Float16* y, long ldx, int M, int N, int K) {
  constexpr int PIECES = 8 * NI, MINE = MI / 2 * NI;
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  h4 bias[NI];
  u32x4 res[MINE];
  tiles_product<Half, MI, NI, D>(
      x, ldx, w, M, N, K,
      [&](const Where& at) {
#pragma unroll
        for (int n = 0; n < NI; ++n) bias[n] = *reinterpret_cast<const h4*>(b + min(at.s0 + at.wave * NI + n, at.SL - 1) * 16 + 4 * at.kc);
#pragma unroll
        for (int k = 0; k < MINE; ++k) {
          const int u = (int)threadIdx.x + 256 * (k % NI), row = u / PIECES, piece = u - row * PIECES;
          res[k] = r[(min(at.m0 + 32 * (k / NI) + row, M - 1) * (long)N + min(at.s0 * 16 + 8 * piece, N - 8)) / 8];
        }
      },
      [&](const f32x4(&acc)[NI][MI], const Where& at) {
        lines_out<u32x2, MI, NI, false>(
            at,
            [&](int n, int i) {
              h4 o;
#pragma unroll
              for (int e = 0; e < 4; ++e) o[e] = (_Float16)(acc[n][i][e] + (float)bias[n][e]);
              return __builtin_bit_cast(u32x2, o);
            },
            [&](int row, int piece, const u32x4& v, int k) {
              put_piece(at.m0 + row < M && at.s0 * 16 + 8 * piece < N, y + (at.m0 + row) * (long)N + at.s0 * 16 + 8 * piece, v + res[k], true);
            });
      });
}
"""
SHAPES = [(2, 1, 2), (2, 1, 4), (4, 2, 4), (6, 2, 2), (8, 3, 4)]      # rows / 16, columns / 64, chunks in flight


@pytest.mark.parametrize("strategy", ["", "max-ilp", "iterative-ilp", "iterative-minreg"])
def test_requests_of_a_tile_go_out_in_the_order_that_its_waits_count(strategy, tmp_path):
    """A wave lets a barrier pass when all but so many of its last requests are there: chunk by chunk the ones into LDS, then the weights', whatever the compiler's scheduler prefers.  With
    what ships around the walk: a bias and residuals that are asked for early (which only make a wait longer), results that leave as lines behind one barrier and one more for every 32 rows."""
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE + "".join(f"template __global__ void tiles_kernel<{a}, {b}, {c}>(const void*, const void*, const _Float16*, const u32x4*, _Float16*, long, int, int, int);\n" for a, b, c in SHAPES))
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
        assert parts[1:] == [chunk] * (d + 1) + [""] * (d - 1 + 1 + mi // 2), (mi, ni, d, parts)


def _code_objects(path):
    """The gfx950 code objects of a library built here."""
    data, at = open(path, "rb").read(), 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        p = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24: p + 24 + n]:
                yield data[at + offset: at + offset + size]
            p += 24 + n
        at += 24


def _kernels(obj):
    """Its kernels as the metadata note lists them."""
    sections, (step, n) = struct.unpack_from("<Q", obj, 0x28)[0], struct.unpack_from("<HH", obj, 0x3A)
    for i in range(n):
        kind, offset, size = (struct.unpack_from(f, obj, sections + i * step + a)[0] for f, a in (("<I", 4), ("<Q", 24), ("<Q", 32)))
        if kind == 7:      # SHT_NOTE; its records: sizes of name and content, type
            while size > 0:
                a, b, t = struct.unpack_from("<III", obj, offset)
                if t == 32:
                    return msgpack.unpackb(obj[offset + 12 + (a + 3) // 4 * 4:][:b])["amdhsa.kernels"]
                used = 12 + (a + 3) // 4 * 4 + (b + 3) // 4 * 4
                offset, size = offset + used, size - used
    return []


@pytest.mark.parametrize("lib,kinds", [(build.LAYER_LIB_PATH, 3), (build.HYBRID_LIB_PATH, 5)])
def test_every_tile_keeps_its_registers_and_its_scalars(lib, kinds, tmp_path):
    """What the cost of a tile is fitted to: no instance of a tile keeps values in scratch memory, and none asks for weights lane by lane because an offset is no scalar."""
    objdump = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(build._hipcc()))), "llvm", "bin", "llvm-objdump")
    seen = 0
    for obj in _code_objects(lib):
        tiles = {k[".name"]: k for k in _kernels(obj) if "tiles_kernelILi" in k[".name"]}
        if not tiles:
            continue
        (tmp_path / "code").write_bytes(obj)
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", str(tmp_path / "code")], capture_output=True, text=True, check=True).stdout
        code = {m.group(1): part for part in re.split(r"\n(?=[0-9a-f]{16} <)", text) if (m := re.match(r"[0-9a-f]{16} <(\w+)>:", part))}
        for name, k in tiles.items():
            assert k[".private_segment_fixed_size"] == k[".vgpr_spill_count"] == k[".sgpr_spill_count"] == 0, name
            walk = code[name][: code[name].rfind("s_barrier")]
            assert "s_barrier" in walk and "execnz" not in walk and "scratch_" not in walk, name
        seen += len(tiles)
    assert seen == len(tile_cases.tiles()) * kinds      # (a launch of each for every kind of end)


def test_a_size_reaches_every_tile_with_every_number_of_chunks_left():
    """What the tests on the card run over; a tile that no size reaches has no business in the list."""
    sizes = {place: tile_cases.size_for(*place) for place in tile_cases.places()}
    assert all(sizes.values()), [p for p, s in sizes.items() if s is None]
    assert len(set(sizes.values())) == len(sizes) == sum(d for _, _, d in tile_cases.tiles())
    assert all(tile_cases.size_for(i, d, (2, 3, 8, 16, 32)) for i, (_, _, d) in enumerate(tile_cases.tiles()))
