"""The rules and the launch plan of the 16-row tiles, compiled for the host and checked without a GPU.

A batch has one LDS size and one workgroup size, so tasks of a short K share
the chip with the needs of the longest: the plan has to keep the waves of
their workgroups at work.  The kernel's split of a workgroup's columns and
chunks over its waves is restated here and checked to cover each exactly once.
"""

from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "qpu-xla-triton_amd" / "csrc"
CUS = 256
LDS = 160 * 1024
FIGURES = ("waves", "lds", "groups", "steps", "columns")

SHIM = r"""
#include "qxt_q4_0_rows_plan.h"
extern "C" int plan(const int *chunks, const long *tiles, int n, int cus, double units, int fp32, long *out) {
    qxt::RowsTiles t;
    for (int i = 0; i < n; ++i) t[chunks[i]] += tiles[i];
    const qxt::RowsPlan p = qxt::rows_batch_plan(t, cus);
    out[0] = p.waves, out[1] = static_cast<long>(p.lds), out[2] = p.groups, out[3] = p.steps;
    for (int i = 0; i < n; ++i) out[4 + i] = p.columns(chunks[i]);
    return qxt::rows_batch_preferred(t, units, fp32, cus);
}
extern "C" int linear_takes(int lanes, int rows, int blocks, long tiles, long cus) {
    return rows < 16 ? qxt::rows_linear_takes(lanes, rows, blocks, tiles, cus)
                     : qxt::rows_lanes_prefill_takes(rows, blocks, tiles, cus);
}
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("clang++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    folder = tmp_path_factory.mktemp("rows_plan")
    (folder / "plan.cpp").write_text(SHIM)
    subprocess.run([compiler, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", str(CSRC),
                    str(folder / "plan.cpp"), "-o", str(folder / "plan.so")], check=True)
    return ctypes.CDLL(str(folder / "plan.so"))


def _plan(library, shapes, fp32=False):
    """Plan of tasks (K, N): (figures, preferred), columns per workgroup by chunks of K."""
    tiles: dict[int, int] = {}
    for k, n in shapes:
        chunks = -(-k // 1024)
        tiles[chunks] = tiles.get(chunks, 0) + -(-n // 16)
    chunks = sorted(tiles)
    out = (ctypes.c_long * (4 + len(chunks)))()
    preferred = library.plan((ctypes.c_int * len(chunks))(*chunks), (ctypes.c_long * len(chunks))(*[tiles[c] for c in chunks]),
                             len(chunks), CUS, ctypes.c_double(sum(k // 256 * n for k, n in shapes)), int(fp32), out)
    plan = dict(zip(FIGURES, out[:4]))
    plan["columns"] = dict(zip(chunks, out[4:]))
    return plan, tiles, bool(preferred)


def _layer(hidden, ffn, kv=256):
    return [(hidden, hidden), (hidden, kv), (hidden, kv), (hidden, hidden), (hidden, ffn), (hidden, ffn), (ffn, hidden)]


@pytest.mark.parametrize("hidden,ffn", [(512, 8192), (512, 16384), (1024, 8192), (2048, 16384), (4096, 14336),
                                        (2048, 5632), (4096, 11008), (1024, 4096), (2816, 1024)])
@pytest.mark.parametrize("layers", [6, 20])
def test_whole_steps_keep_the_waves_of_every_k_at_work(library, hidden: int, ffn: int, layers: int) -> None:
    plan, tiles, _ = _plan(library, _layer(hidden, ffn) * layers)
    waves = plan["waves"]
    per_cu = max(1, min(12 // waves, LDS // plan["lds"]))
    for chunks, count in tiles.items():
        passes = -(-chunks // waves)
        groups = max(1, waves // chunks) if plan["groups"] else 1
        working = chunks / passes if passes > 1 else groups * chunks
        # Most of the work waits for eight waves on a CU; the few tiles of a longer K may take five.
        share = count * chunks / sum(n * c for c, n in tiles.items())
        assert per_cu * working >= (7 if share > 0.4 else 5), (plan, chunks, per_cu, working)


@pytest.mark.parametrize("shapes", [
    [(2048, 256)], [(2048, 5632), (2048, 5632)], [(512, 1000), (24576, 100)], [(1024, 33000), (8192, 2049)],
    [(256, 40000), (512, 9000), (3072, 5000), (11008, 4096), (16384, 300)], [(4096, 4096 * 30), (11008, 4096 * 8)],
    _layer(2048, 16384) * 3, _layer(1280, 3072) * 2, [(512, 100), (4096, 128)],
])
def test_every_tile_and_chunk_belongs_to_one_wave(library, shapes) -> None:
    plan, tiles, _ = _plan(library, shapes)
    waves = plan["waves"]
    assert 1 <= waves <= 8 and plan["lds"] <= LDS
    for k, n in shapes:
        chunks = -(-k // 1024)
        assert -(-chunks // waves) <= 4
        columns = min(plan["columns"][chunks], -(-n // 16) * 16)
        assert columns % 16 == 0
        # The kernel has groups wherever the plan asks for them, and sums of every group behind the chunks.
        groups = max(1, waves // chunks) if plan["groups"] else 1
        span = min(waves, chunks) if plan["groups"] else waves
        assert plan["lds"] >= chunks * 6656 + groups * 256
        for base in {0, (n - 1) // columns * columns}:
            tile_count = -(-min(columns, n - base) // 16)
            passes = -(-chunks // waves)
            done = {}
            for step in range(-(-tile_count // groups) * passes):
                for wave in range(waves):
                    group, place = (wave // span, wave % span) if plan["groups"] else (0, wave)
                    tile, chunk = groups * (step // passes) + group, step % passes * span + place
                    if group < groups and tile < tile_count and chunk < chunks:
                        done[tile, chunk] = done.get((tile, chunk), 0) + 1
            assert done == {(t, c): 1 for t in range(tile_count) for c in range(chunks)}


def test_small_grids_of_a_longer_k_take_it_in_one_pass(library) -> None:
    plan, _, _ = _plan(library, [(512, 100), (4096, 128)])
    assert plan["waves"] == 4 and not plan["groups"] and set(plan["columns"].values()) == {16}


@pytest.mark.parametrize("shapes,fp32,preferred", [
    ([(256, 32000)] * 8 + [(2048, 2048)] * 8, False, False),   # chunks mostly empty
    ([(256, 32000)] * 8 + [(2048, 2048)] * 8, True, False),
    ([(256, 512), (512, 512)], False, True),                    # the same, few tiles
    ([(256, 17000), (256, 17000), (256, 500)], True, False),
    ([(256, 9000)] * 4 + [(512, 500), (256, 33)], False, False),
    ([(1024, 4096), (24576, 128)], False, False),               # passes over a very long K, little else
    ([(1024, 4096), (24576, 128)], True, True),                 # quantised here
    ([(1024, 32000), (24576, 2048)], False, True),
    (_layer(512, 8192) * 6, True, True),
    (_layer(4096, 11008) * 4, True, True),
])
def test_which_batches_take_the_row_tiles(library, shapes, fp32: bool, preferred: bool) -> None:
    assert _plan(library, shapes, fp32)[2] is preferred


@pytest.mark.parametrize("layout,rows,k,n,taken", [
    # Measured on MI355X: the other kernels / the row tiles, us.
    ("lanes", 2, 4608, 32000, False),   # 21.3 / 45.3
    ("lanes", 2, 5632, 11008, False),   # 12.9 / 21.3
    ("lanes", 2, 5632, 4608, False),    # 8.7 / 13.1
    ("lanes", 2, 11008, 1024, False),
    ("lanes", 2, 2048, 8192, True),
    ("lanes", 2, 16384, 8192, True),    # 39.2 / 26.3
    ("lanes", 3, 4608, 4608, False),    # 8.4 / 12.0
    ("lanes", 3, 8192, 8192, True),     # 19.1 / 15.1
    ("lanes", 4, 5632, 4608, False),
    ("lanes", 4, 5120, 16384, True),    # 28.5 / 20.8
    ("lanes", 4, 4096, 4096, False),
    ("lanes", 4, 2304, 6000, True),
    ("lanes", 8, 2048, 16384, False),   # 8.8 / 9.8
    ("lanes", 8, 14336, 256, False),    # 9.6 / 11.3
    ("lanes", 8, 4096, 11008, True),
    ("lanes", 9, 256, 32000, True),
    ("lanes", 15, 256, 32000, False),
    ("native", 3, 5632, 2048, False),
    ("native", 4, 11008, 4608, False),  # 14.7 / 18.0
    ("native", 4, 14336, 4608, False),  # 15.7 / 23.4
    ("native", 4, 11008, 4096, True),
    ("native", 5, 6144, 64, False),     # 3.9 / 6.9
    ("native", 8, 4096, 256, False),    # 3.8 / 5.1
    ("native", 8, 5632, 256, False),    # 4.9 / 6.1
    ("native", 8, 11008, 4096, True),
    ("native", 9, 14336, 4608, False),  # 35.3 / 42.4
    ("native", 12, 4096, 4096, True),
    # The linears that the GPU tests hold for the other kernels.
    ("lanes", 4, 256, 2100, False),
    ("lanes", 4, 512, 2100, False),
    ("lanes", 4, 1024, 2077, False),
    ("lanes", 5, 256, 8300, False),
    ("lanes", 7, 2048, 9000, False),
    ("lanes", 6, 4096, 5990, False),
    ("native", 4, 256, 8300, False),
    ("native", 4, 512, 8300, False),
    ("native", 4, 1024, 8300, False),
    ("native", 6, 4096, 4200, False),
    ("lanes", 2, 5632, 4200, False),
    ("lanes", 3, 4608, 4190, False),
    ("lanes", 4, 5632, 4300, False),
    ("lanes", 12, 11008, 200, False),
    ("native", 10, 14336, 4608, False),
    # Lane weights have no prefill tiles to lose to.
    ("lanes", 16, 2048, 32000, True),
    ("lanes", 24, 2048, 32000, True),
    ("lanes", 512, 2048, 5632, True),
    ("lanes", 16, 14336, 64, False),    # 9.3 / 11.2
    ("lanes", 64, 256, 11008, False),   # 7.6 / 9.9
    ("lanes", 64, 14336, 1024, True),
])
def test_which_linears_take_the_row_tiles(library, layout: str, rows: int, k: int, n: int, taken: bool) -> None:
    got = library.linear_takes(int(layout == "lanes"), rows, k // 32, ctypes.c_long(-(-n // 16)), ctypes.c_long(CUS))
    assert bool(got) is taken
