"""Per-row int8 quantiser with 1024-thread workgroups (few rows longer than 4096) against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from qpu_xla_amd.kernels.quantize import quantize_rows_int8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra_rows", [0, 1])
def test_both_sides_of_the_row_limit(extra_rows: int) -> None:
    check(2 * torch.cuda.get_device_properties(0).multi_processor_count + extra_rows, 4100, 4112)


@pytest.mark.parametrize(
    "rows,cols,pad",
    [(1, 4096, 4096), (3, 4100, 4128), (1, 8192, 8192), (5, 8196, 8224), (2, 12292, 12292), (48, 14336, 14336),
     (3, 16384, 16400), (2, 16388, 16388)],
)
def test_edges_of_the_row_lengths(rows: int, cols: int, pad: int) -> None:
    check(rows, cols, pad)


def check(rows: int, cols: int, pad: int) -> None:
    rng = np.random.default_rng(rows * 100003 + cols)
    x = rng.standard_normal((rows, cols), dtype=np.float32)
    x[0, -1] = -11.0  # the maximum in the last lane's chunk
    x[-1] *= np.float32(1e-3)  # floor active on the last row
    q, s = quantize_rows_int8(torch.from_numpy(x).to("cuda"), padded_columns=pad)
    want_q, want_s = oracle.quantize_rows_int8(x)
    np.testing.assert_array_equal(s.cpu().numpy(), want_s)
    np.testing.assert_array_equal(q.cpu().numpy()[:, :cols], want_q)
    np.testing.assert_array_equal(q.cpu().numpy()[:, cols:], 0)
