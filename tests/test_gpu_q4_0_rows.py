"""GPU parity for the Q4_0 kernels over 16-row matrix-core tiles, at the edges of their tiles and rules.

Every case is compared bit for bit with the oracle: the integer dots are
exact and the fp32 terms are scaled and added in the oracle's order.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from qpu_xla_amd.kernels import ggml_q4_0 as q4

pytestmark = pytest.mark.gpu


def dev(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _operands(seed: int, rows: int, blocks: int, outputs: int):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, blocks * 32), dtype=np.float32)
    w = (rng.standard_normal((outputs, blocks * 32), dtype=np.float32) * np.float32(0.02)).astype(np.float32)
    return oracle.quantize_q8_0_blocks(x), oracle.quantize_q4_0_blocks(w)


@pytest.mark.parametrize("scale_dtype", [torch.int16, torch.int32])
@pytest.mark.parametrize("rows,blocks,outputs", [
    (16, 1, 64),     # one block of one tile
    (17, 15, 65),    # a row, a block short of a group, and a column past the tile
    (31, 16, 63),    # exactly one group of blocks
    (16, 17, 130),   # a group and a block
    (48, 33, 16),    # a staged round and a block; one wave's columns
    (77, 176, 200),  # a short prompt over long rows
    (41, 64, 11009),   # past two waves per SIMD: 32-row tiles, ragged rows and columns
    (33, 81, 11008),   # the same over a K that is no whole group
    (41, 63, 11009),   # the same grid over shorter rows: the 64 x 64 tiles
])
def test_split_plane_short_tiles_bit_exact(rows: int, blocks: int, outputs: int, scale_dtype) -> None:
    act, wt = _operands(rows * 1000 + blocks, rows, blocks, outputs)
    wscales, wquants = q4.pack_ggml_q4_0_tiled_weights(dev(wt))
    ascales, aquants = q4.split_ggml_q8_0_blocks(dev(act))
    ascales = (ascales.to(torch.int32) & 0xFFFF).to(scale_dtype) if scale_dtype == torch.int32 else ascales
    out = q4.ggml_q4_0_q8_0_tiled_linear(aquants, ascales.contiguous(), wquants, wscales).cpu().numpy()
    some = np.unique(np.concatenate([np.arange(min(outputs, 130)), np.arange(max(0, outputs - 130), outputs)]))
    np.testing.assert_array_equal(out[:, some], oracle.q4_0_q8_0_reference(act, wt[some]))


def test_split_plane_32_row_tiles_redo_a_tile_with_a_non_finite_scale() -> None:
    # One infinite weight scale: its workgroup's tile is computed again in the exact form.
    act, wt = _operands(7, 41, 64, 11009)
    wt[5000, 3, :2] = np.array([0x00, 0x7C], dtype=np.uint8)
    wscales, wquants = q4.pack_ggml_q4_0_tiled_weights(dev(wt))
    ascales, aquants = q4.split_ggml_q8_0_blocks(dev(act))
    out = q4.ggml_q4_0_q8_0_tiled_linear(aquants, ascales, wquants, wscales).cpu().numpy()
    some = np.arange(4960, 5060)
    with np.errstate(invalid="ignore"):
        np.testing.assert_array_equal(out[:, some], oracle.q4_0_q8_0_reference(act, wt[some]))
