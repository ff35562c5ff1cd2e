"""The rule that picks the several-row GEMM's kernel (no GPU: the query only
plans): every shape that the operators accept gets a grid that covers it and
that a launch can have."""
from __future__ import annotations

import pytest

import llmrs_hip as lh

MAX_GRID_Y = 65535
MAX_ROWS = 65535 * 128  # the operators' limit


@pytest.mark.parametrize("weight", ["q4h", "q4f", "q8h"])
@pytest.mark.parametrize("n", [1, 32, 64, 65, 128, 192, 200, 320, 4096, 28672])
@pytest.mark.parametrize("m", [161, 2048, 65535 * 64, 65535 * 64 + 1, 65535 * 96, MAX_ROWS])
def test_tile_grid_covers_and_fits(weight, n, m):
    for epi in ("store", "resid") + (("silu",) if n % 64 == 0 else ()):
        name, (gx, gy) = lh.probe_gemm_plan(weight, epi, m, n, 32)
        bm, bn = map(int, name.rsplit("_", 1)[1].split("x"))
        assert gx * bn >= n > (gx - 1) * bn and gy * bm >= m > (gy - 1) * bm, name
        assert gy <= MAX_GRID_Y, f"{name}: grid of {gy} token tiles"


@pytest.mark.parametrize("value", ["0", "00", "1", ""])
def test_prompt_switch_leaves_the_rule(value, monkeypatch):
    """LLMRS_PREFILL_SKINNY is about prompts: the operators' and the batches'
    rule does not read it."""
    shapes = [(m, n, k) for m in (2, 16, 77, 160) for n, k in ((4096, 4096), (28672, 4096), (512, 512))]
    want = [lh.probe_gemm_plan("q4h", "store", *s) for s in shapes]
    assert any(name.startswith("sgemm") for name, _ in want)
    monkeypatch.setenv("LLMRS_PREFILL_SKINNY", value)
    assert [lh.probe_gemm_plan("q4h", "store", *s) for s in shapes] == want
