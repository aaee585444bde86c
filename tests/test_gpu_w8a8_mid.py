"""The int8 GEMM tiles below 256 x 256: which one a problem takes, and GPU parity at their edges.

The rule is compiled for the host and checked without a GPU.  The sums are
exact integers, so every form is compared for equality with the oracle.
"""

from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch

import oracle
from qpu_xla_amd import _lib
from qpu_xla_amd.kernels import gemm_int8

def dev(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


CSRC = Path(__file__).resolve().parent.parent / "qpu-xla-triton_amd" / "csrc"
CUS = 256
# In the order of MidTile: "groups" split K inside the workgroup, "short" has K stages of 64 bytes.
TILES = ("128x128 short", "128x128", "128x128 groups", "128x64 groups", "32x32 groups", "64x32 groups", "64x64 groups",
         "64x64")
SHIM = r"""
#include "qxt_w8a8_tiles.h"
extern "C" int tile(long m, long n, long k, int packed, long cus) {
    return static_cast<int>(qxt::w8a8_mid_tile(m, n, k, packed, cus));
}
"""

# (m, n, k), then the tile over [N, K] and over packed weights on 256 CUs.
CASES = [
    (5, 72, 16, "64x64", "64x64"),               # one short stage
    (64, 64, 256, "64x64", "64x64"),
    (65, 132, 272, "64x64", "64x64"),            # three stages, the last one short
    (65, 132, 528, "64x64 groups", "64x64 groups"),  # three stages of the first group, two of the second
    (300, 3200, 976, "64x64 groups", "64x64 groups"),  # more stages than are in flight
    (300, 6000, 80, "64x64", "64x64"),           # past one tile per CU
    (300, 6004, 656, "64x64", "64x64"),
    (500, 4092, 400, "64x64", "64x64"),
    (500, 4092, 528, "64x64", "128x64 groups"),  # two stages or three per group
    (500, 4092, 1552, "128x64 groups", "128x64 groups"),  # seven: two turns of the ring and one
    (500, 4092, 2064, "128x64 groups", "128x64 groups"),
    (1000, 2600, 208, "64x64", "64x64"),
    (990, 2604, 1040, "64x64", "64x64"),
    (1000, 2604, 2064, "128x128 groups", "64x64"),
    (1000, 3600, 1552, "128x128 groups", "64x64"),  # short K: a nearly full chip of them
    (1000, 3140, 3088, "128x128 groups", "128x128 groups"),
    (1100, 4004, 3088, "128x128", "128x128"),
    (1500, 4004, 336, "128x128", "128x128 short"),
    (1500, 5500, 336, "128x128 short", "128x128 short"),  # one round of three to a CU
    (1400, 2900, 336, "64x64", "64x64"),         # 253 tiles of 128 x 128, a short K
    (1400, 3000, 336, "64x64", "64x64"),         # 264: just past one per CU
    # 32 x 32 tiles, eight groups of one wave
    (5, 72, 1024, "32x32 groups", "32x32 groups"),   # one stage each
    (33, 36, 1040, "32x32 groups", "32x32 groups"),  # a second, short stage of the first group
    (17, 4100, 1168, "32x32 groups", "32x32 groups"),
    (17, 4100, 3088, "32x32 groups", "32x32 groups"),  # four stages: one more than are in flight
    (32, 8192, 1168, "32x32 groups", "32x32 groups"),  # the last size of the rule: 256 tiles
    (7, 20, 14352, "32x32 groups", "32x32 groups"),
    # 64 x 32 tiles, four groups of two waves
    (64, 8192, 1024, "64x32 groups", "64x32 groups"),  # two stages each
    (65, 4096, 1552, "64x32 groups", "64x32 groups"),  # the second row of tiles holds one row
    (230, 2044, 2064, "64x32 groups", "64x32 groups"),
    # just past both rules, and below their K
    (32, 8196, 1040, "64x64 groups", "64x64 groups"),
    (40, 260, 1008, "64x64 groups", "64x64 groups"),
]


@pytest.fixture(scope="module")
def tile_of(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("clang++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    folder = tmp_path_factory.mktemp("w8a8_tiles")
    (folder / "tile.cpp").write_text(SHIM)
    subprocess.run([compiler, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", str(CSRC),
                    str(folder / "tile.cpp"), "-o", str(folder / "tile.so")], check=True)
    library = ctypes.CDLL(str(folder / "tile.so"))
    return lambda m, n, k, packed: TILES[library.tile(ctypes.c_long(m), ctypes.c_long(n), ctypes.c_long(k), int(packed),
                                                      ctypes.c_long(CUS))]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:3])))
def test_cases_take_the_tiles_that_they_are_for(tile_of, case) -> None:
    assert (tile_of(*case[:3], False), tile_of(*case[:3], True)) == case[3:]


@pytest.mark.parametrize("m,k,n,packed,tile", [
    # Measured on MI355X: 128 x 128 tiles in two groups / these, us.
    (512, 512, 5632, False, "64x64"),            # 8.6 / 7.0
    (512, 512, 5632, True, "64x64"),
    (192, 512, 14336, True, "64x64"),
    (768, 4096, 4096, True, "64x64"),            # 47.2 / 38.7
    (200, 14336, 14336, True, "128x128 groups"),  # 147 / 161 with 64 x 64
    (1536, 512, 5632, False, "128x128 short"),   # 20.3 with stages of 128 bytes / 16.3
    (1536, 2048, 5632, False, "128x128 short"),
    (512, 14336, 4096, False, "128x64 groups"),
    (256, 4096, 14336, False, "128x128 groups"),
    (48, 4096, 14336, False, "64x64 groups"),
    (8, 14336, 4096, False, "32x32 groups"),
])
def test_measured_problems_take_the_faster_tile(tile_of, m: int, k: int, n: int, packed: bool, tile: str) -> None:
    assert tile_of(m, n, k, packed) == tile


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("m,n,k", [case[:3] for case in CASES])
def test_mid_size_gemm_tiles_exact(m: int, n: int, k: int, packed: bool) -> None:
    rng = np.random.default_rng(m * 7 + n + k)
    a = rng.integers(-127, 128, size=(m, k), dtype=np.int8)
    w = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    sa = rng.uniform(0.001, 0.1, m).astype(np.float32)
    sw = rng.uniform(0.001, 0.1, n).astype(np.float32)
    bias = rng.standard_normal(n, dtype=np.float32)
    ad, sad, swd, bd = dev(a), dev(sa), dev(sw), dev(bias)
    wd = gemm_int8.pack_int8_quads(dev(w)).t().contiguous() if packed else dev(w)
    ldw = wd.stride(0) * wd.element_size()
    layout = _lib.WEIGHT_K4N if packed else _lib.WEIGHT_NK
    rows = np.unique(np.concatenate([np.arange(min(m, 6)), np.arange(60, min(m, 70)), np.arange(max(0, m - 70), m, 5),
                                     np.array([m - 1])]))
    acc = oracle.int8_gemm_i32(a[rows], w)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    out = torch.full((m, n + 4), -5, dtype=torch.int32, device="cuda")
    _lib.call("qxt_w8a8_gemm_i32", _p(ad), k, _p(wd), ldw, _p(out), (n + 4) * 4, m, n, k, layout, stream)
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[rows, :n], acc)
    np.testing.assert_array_equal(got[:, n:], -5)
    for b, bt in ((None, None), (bias, bd)):
        y = torch.full((m, n + 4), -5.0, device="cuda")
        _lib.call("qxt_w8a8_gemm_dequantize", _p(ad), k, _p(wd), ldw, _p(sad), _p(swd), _p(bt), _p(y), (n + 4) * 4,
                  m, n, k, layout, stream)
        got = y.cpu().numpy()
        np.testing.assert_array_equal(got[rows, :n], oracle.dequantize_epilogue(acc, sa[rows], sw, b))
        np.testing.assert_array_equal(got[:, n:], -5.0)
