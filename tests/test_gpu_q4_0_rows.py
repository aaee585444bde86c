"""GPU parity for the Q4_0 kernels over 16-row matrix-core tiles, at the edges of their tiles and rules,
and for what those rules leave to the other kernels.

Every case is compared bit for bit with the oracle: the integer dots are
exact and the fp32 terms are scaled and added in the oracle's order.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from qpu_xla_amd import _lib
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


def _check_linear(layout: str, rows: int, blocks: int, n: int, wcol0: int, ncols: int, act=None, wt=None) -> None:
    if act is None:
        act, wt = _operands(rows * 100003 + blocks * 17 + n, rows, blocks, n)
    out = torch.full((rows, ncols + 9), -77.0, device="cuda")
    weight = q4.pack_ggml_q4_0_lane_weights(dev(wt)) if layout == "lanes" else dev(wt)
    linear = q4.ggml_q4_0_q8_0_lane_linear if layout == "lanes" else q4.ggml_q4_0_q8_0_linear
    linear(dev(act), weight, out, weight_column_start=wcol0, output_column_start=5, column_count=ncols)
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:, :5], -77.0)
    np.testing.assert_array_equal(got[:, 5 + ncols:], -77.0)
    some = np.unique(np.concatenate([np.arange(min(ncols, 96)), np.arange(max(0, ncols - 96), ncols)]))
    np.testing.assert_array_equal(got[:, 5 + some], oracle.q4_0_q8_0_reference(act, wt[wcol0 + some]))


@pytest.mark.parametrize("layout", ["lanes", "native"])
@pytest.mark.parametrize("rows,blocks,n,wcol0,ncols", [
    (2, 8, 33, 0, 33),        # one unit, ragged columns
    (3, 16, 40, 7, 20),       # one half-unit chunk of four lanes, a column range
    (4, 24, 17, 1, 16),       # one unit past a chunk
    (5, 40, 100, 0, 100),     # two rows per lane, or two row groups
    (6, 32, 6000, 0, 6000),   # more tiles than CUs: every row in one group
    (8, 64, 5632, 3, 5629),
    (9, 72, 300, 0, 300),     # units no power of two
    (12, 48, 4200, 0, 4200),  # three rows per lane
    (15, 136, 2048, 0, 2048),
    (13, 56, 8300, 0, 8300),  # four rows per lane, whole-unit chunks
    (5, 128, 9000, 2, 8990),  # several tiles per workgroup
    (10, 264, 4112, 0, 4112),  # several chunks per wave
    (15, 344, 4112, 16, 4096),  # rows in groups (LDS)
    (4, 520, 4112, 0, 4112),  # three chunks per wave, four rows
])
def test_row_tile_linear_bit_exact(layout: str, rows: int, blocks: int, n: int, wcol0: int, ncols: int) -> None:
    _check_linear(layout, rows, blocks, n, wcol0, ncols)


@pytest.mark.parametrize("layout", ["lanes", "native"])
def test_row_tile_linear_non_finite_and_extreme_scales_bit_exact(layout: str) -> None:
    # dw enters as dw / 16 times 16 dots: subnormal, largest, infinite and NaN fp16 scales.
    act, wt = _operands(11, 6, 24, 64)
    bits = np.array([0x0001, 0x03FF, 0x0400, 0x7BFF, 0xFBFF, 0x7C00, 0xFC00, 0x7E00, 0x0000, 0x8000], dtype=np.uint16)
    wt.reshape(-1, 18)[:: 7, :2] = np.resize(bits, (wt.reshape(-1, 18)[:: 7].shape[0],)).view(np.uint8).reshape(-1, 2)
    act.reshape(-1, 34)[:: 5, :2] = np.resize(bits, (act.reshape(-1, 34)[:: 5].shape[0],)).view(np.uint8).reshape(-1, 2)
    with np.errstate(all="ignore"):
        _check_linear(layout, 6, 24, 64, 0, 64, act, wt)


def test_row_tile_linear_unaligned_activation_takes_the_general_kernel() -> None:
    act, wt = _operands(12, 5, 64, 80)
    raw = torch.zeros(act.size + 2, dtype=torch.uint8, device="cuda")
    raw[2:] = dev(act).flatten()
    shifted = raw[2:].view(act.shape)  # two bytes past a word
    assert shifted.data_ptr() % 4 == 2
    out = q4.ggml_q4_0_q8_0_linear(shifted, dev(wt)).cpu().numpy()
    np.testing.assert_array_equal(out, oracle.q4_0_q8_0_reference(act, wt))


@pytest.mark.parametrize("count", [2, 4, 7])  # kernel arguments up to four tasks, device tables past that
@pytest.mark.parametrize("layouts", ["lanes", "native", "mixed"])
def test_row_tile_batch_mixed_rows_lengths_and_activations_bit_exact(count: int, layouts: str) -> None:
    rng = np.random.default_rng(count * 10 + len(layouts))
    shapes = [(4, 64, 700), (1, 8, 16), (3, 176, 130), (2, 264, 50), (4, 40, 1), (2, 16, 4100), (1, 128, 33)][:count]
    tasks, expected = [], []
    for i, (rows, blocks, n) in enumerate(shapes):
        x = rng.standard_normal((rows, blocks * 32), dtype=np.float32)
        w = (rng.standard_normal((n, blocks * 32), dtype=np.float32) * np.float32(0.02)).astype(np.float32)
        act, wt = oracle.quantize_q8_0_blocks(x), oracle.quantize_q4_0_blocks(w)
        lanes = layouts == "lanes" or (layouts == "mixed" and i % 2 == 0)
        task = {"weight": q4.pack_ggml_q4_0_lane_weights(dev(wt)) if lanes else dev(wt),
                "destination": torch.full((rows, n + 3), -77.0, device="cuda"), "output_column_start": 2}
        task["x" if i % 3 != 1 else "activation"] = dev(x) if i % 3 != 1 else dev(act)
        tasks.append(task)
        expected.append(oracle.q4_0_q8_0_reference(act, wt))
    with q4.Q4_0LinearBatch(tasks) as batch:
        for _ in range(2):
            batch.launch()
        torch.cuda.synchronize()
        for task, want in zip(tasks, expected):
            got = task["destination"].cpu().numpy()
            np.testing.assert_array_equal(got[:, 2:-1], want)
            np.testing.assert_array_equal(got[:, [0, 1, -1]], -77.0)


def test_row_tile_batch_captured_and_replayed_reads_the_rows_of_each_replay() -> None:
    act, wt = _operands(13, 4, 64, 300)
    x = torch.zeros((4, 2048), device="cuda")
    out = torch.zeros((4, 300), device="cuda")
    with q4.Q4_0LinearBatch([{"x": x, "weight": dev(wt), "destination": out}]) as batch:
        batch.launch()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            batch.launch()
        rng = np.random.default_rng(14)
        for _ in range(3):
            rows = rng.standard_normal((4, 2048), dtype=np.float32)
            x.copy_(torch.from_numpy(rows))
            graph.replay()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(
                out.cpu().numpy(), oracle.q4_0_q8_0_reference(oracle.quantize_q8_0_blocks(rows), wt))


@pytest.mark.parametrize("layout", ["lanes", "native"])
@pytest.mark.parametrize("rows,blocks,n,wcol0,ncols", [
    (16, 64, 70, 0, 70),       # a whole group of sixteen rows, or several smaller ones
    (17, 24, 300, 5, 290),     # one row past a group
    (33, 40, 4200, 0, 4200),   # groups of sixteen rows over more tiles than CUs
    (100, 128, 256, 0, 256),
    (40, 176, 2048, 0, 2048),  # past K = 4096: one workgroup's LDS a CU
    (24, 344, 4100, 0, 4100),  # groups of eight rows (LDS)
    (300, 64, 100, 0, 100),
    (64, 64, 5632, 0, 5632),   # the last row count here, the prefill tiles past it
    (96, 64, 5632, 0, 5632),
    (24, 64, 32000, 0, 32000),  # lanes only from here: more column tiles than a round of them
    (70, 448, 256, 16, 240),    # a K past two groups' LDS
    (16, 448, 64, 0, 64),       # the four-row kernels
    (33, 8, 11008, 0, 11008),
    (259, 16, 2000, 1, 1990),
])
def test_short_prompts_on_row_tiles_bit_exact(layout: str, rows: int, blocks: int, n: int, wcol0: int, ncols: int) -> None:
    _check_linear(layout, rows, blocks, n, wcol0, ncols)


def _check_batch(shapes, source: str, layouts: str, offset: int = 0) -> None:
    """One batch of (rows, blocks, columns) tasks; `offset` bytes before every native activation."""
    rng = np.random.default_rng(len(shapes) * 1000 + len(source) + len(layouts))
    tasks, checks = [], []
    for i, (rows, blocks, n) in enumerate(shapes):
        act, wt = _operands(int(rng.integers(1 << 30)), rows, blocks, n)
        lanes = layouts == "lanes" or (layouts == "mixed" and i % 2 == 0)
        task = {"weight": q4.pack_ggml_q4_0_lane_weights(dev(wt)) if lanes else dev(wt),
                "destination": torch.full((rows, n + 3), -77.0, device="cuda"), "output_column_start": 2}
        if source == "fp32" or (source == "mixed" and i % 2 == 0):
            x = rng.standard_normal((rows, blocks * 32), dtype=np.float32)
            act = oracle.quantize_q8_0_blocks(x)
            task["x"] = dev(x)
        else:
            raw = torch.zeros(act.size + offset, dtype=torch.uint8, device="cuda")
            raw[offset:] = dev(act).flatten()
            task["activation"] = raw[offset:].view(act.shape)
        tasks.append(task)
        checks.append((act, wt))
    with q4.Q4_0LinearBatch(tasks) as batch:
        for _ in range(2):
            batch.launch()
        torch.cuda.synchronize()
        for task, (act, wt) in zip(tasks, checks):
            got = task["destination"].cpu().numpy()
            n = wt.shape[0]
            some = np.unique(np.concatenate([np.arange(min(n, 200)), np.arange(0, n, 67), np.arange(max(0, n - 200), n)]))
            np.testing.assert_array_equal(got[:, 2 + some], oracle.q4_0_q8_0_reference(act, wt[some]))
            np.testing.assert_array_equal(got[:, [0, 1, -1]], -77.0)


@pytest.mark.parametrize("source", ["fp32", "native", "mixed"])
@pytest.mark.parametrize("layouts", ["lanes", "native", "mixed"])
@pytest.mark.parametrize("shapes", [
    # A long K beside short ones that fill the chip: several column tiles of a workgroup side by side.
    [(4, 64, 5000), (2, 512, 40)],                                      # kernel arguments
    [(2, 16, 4001), (3, 32, 3000), (4, 256, 130), (1, 64, 333), (2, 264, 50), (4, 16, 9)],  # device tables
    [(3, 32, 9000), (2, 96, 2100), (4, 448, 17), (2, 32, 15)],          # waves past the last group
])
def test_row_tile_batch_of_short_and_long_k_bit_exact(shapes, layouts: str, source: str) -> None:
    _check_batch(shapes, source, layouts)


@pytest.mark.parametrize("shapes", [
    [(2, 64, 700), (4, 40, 130)],                                   # kernel arguments
    [(3, 32, 9000), (2, 96, 2100), (4, 448, 17), (2, 32, 15), (1, 8, 40)],  # device tables, tiles side by side
    [(2, 128, 300)] * 5,
])
def test_small_batch_of_mixed_activations_is_one_launch(shapes) -> None:
    # fp32 rows beside native ones are quantised in the workgroups: no pre-pass, no buffer that launches share.
    with _lib.launch_timing() as timing:
        _check_batch(shapes, "mixed", "mixed")
    names = [name for name, _ in timing.records if "pack" not in name]
    assert names == ["q4_0_batch_kernel"] * 2


@pytest.mark.parametrize("layout,rows,blocks,n,wcol0,ncols", [
    # Four-row matrix-core tiles at every unit count per column, past the row tiles' column counts.
    ("lanes", 4, 8, 2104, 4, 2100),
    ("lanes", 4, 16, 2100, 0, 2100),
    ("lanes", 4, 32, 2077, 0, 2077),
    ("lanes", 5, 8, 8300, 0, 8300),      # a second row group of one row
    ("lanes", 7, 64, 9000, 0, 9000),
    ("lanes", 6, 128, 6000, 3, 5990),
    ("native", 4, 8, 8300, 0, 8300),
    ("native", 4, 16, 8305, 5, 8300),
    ("native", 4, 32, 8300, 0, 8300),
    ("native", 6, 128, 4200, 0, 4200),
    # v_dot4 tiles over lanes, and blocks over lanes of a wave: a second round of row tiles, few columns of a long K.
    ("lanes", 2, 176, 4200, 0, 4200),
    ("lanes", 3, 144, 4200, 1, 4190),
    ("lanes", 4, 176, 4300, 0, 4300),
    ("lanes", 12, 344, 200, 0, 200),
    ("native", 8, 176, 256, 0, 256),
    ("native", 10, 448, 4608, 0, 4608),
])
def test_linears_left_to_the_other_kernels_bit_exact(layout: str, rows: int, blocks: int, n: int, wcol0: int,
                                                     ncols: int) -> None:
    _check_linear(layout, rows, blocks, n, wcol0, ncols)


@pytest.mark.parametrize("layouts", ["lanes", "native", "mixed"])
@pytest.mark.parametrize("source", ["fp32", "native", "mixed"])
@pytest.mark.parametrize("shapes", [
    [(4, 8, 17000), (2, 8, 17000), (3, 8, 500)],    # chunks mostly empty, in kernel arguments
    [(4, 8, 9000)] * 4 + [(2, 16, 500), (3, 8, 33)],  # and in device tables
    [(4, 776, 40), (2, 64, 300)],                   # K past the row tiles' LDS
    [(2, 776, 33), (3, 8, 100), (4, 64, 70), (1, 16, 5), (4, 784, 16)],
])
def test_multi_row_batches_left_to_the_v_dot4_kernel_bit_exact(shapes, source: str, layouts: str) -> None:
    _check_batch(shapes, source, layouts)


@pytest.mark.parametrize("shapes", [[(4, 64, 700), (1, 8, 16), (3, 176, 130)], [(2, 40, 200)] * 5])
def test_multi_row_batch_of_activations_two_bytes_off_a_word_bit_exact(shapes) -> None:
    _check_batch(shapes, "native", "mixed", offset=2)
