"""GPU parity for the int8 GEMM's 32 x 32 and 64 x 32 tiles, at the edges of their tiles, stages and groups.

The sums are exact integers, so every form is compared for equality with the oracle.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import oracle
from qpu_xla_amd import _lib
from qpu_xla_amd.kernels import gemm_int8

pytestmark = pytest.mark.gpu


def dev(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("m,n,k", [
    # 32 x 32 tiles, eight groups of one wave
    (5, 72, 1024),       # one stage each
    (33, 36, 1040),      # a second, short stage of the first group; the others have none
    (17, 4100, 3088),    # four stages: one more than are in flight
    (32, 8192, 1168),    # the last size of the rule: 256 tiles on 256 CUs
    (7, 20, 14352),
    # 64 x 32 tiles, four groups of two waves
    (64, 8192, 1024),    # two stages each
    (65, 4096, 1552),    # the second row of tiles holds one row
    (230, 2044, 2064),
    # just past both rules, and below their K
    (32, 8196, 1040),
    (40, 260, 1008),
])
def test_narrow_gemm_tiles_exact(m: int, n: int, k: int, packed: bool) -> None:
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
