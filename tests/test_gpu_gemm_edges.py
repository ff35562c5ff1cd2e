"""The several-row GEMMs at the edges of their tiles and of the rule that picks
one, against the oracle's block loop, bit for bit (matmul_transposed with a
quantised weight; cpu.rs:90-110): whole and ragged row and token tiles, one to
many rounds of blocks with every remainder, and one row beyond each range."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32

# Shapes (m, n, k) through the operator, which picks the kernel (which one each
# kernel's own edges are tested with: test_gemm_variants below).  Few rows: ragged
# 16-row and 16-token tiles, k = 384 (12 blocks, half a stage at the end), one to
# many rounds, the last row count the skinny GEMM takes (160) and the one after
SKINNY = [(2, 16, 128), (15, 33, 128), (16, 64, 256), (17, 100, 384), (31, 1, 640), (33, 4112, 2176),
          (64, 8200, 512), (65, 130, 4224), (160, 72, 1024), (161, 72, 1024)]

# more rows, or K not of whole runs of 128: ragged tokens and rows, K of less than a
# stage (4 or 8 blocks), of whole stages and of every kind of remainder
TILES = [(130, 200, 32), (165, 100, 224), (161, 65, 256), (200, 33, 288), (1000, 4090, 416), (2047, 4095, 288),
         (96, 6144, 1024), (100, 28672, 128)]
# few rows of wide weights
WIDE = [(2, 32770, 128), (16, 32000, 384), (23, 28700, 640), (32, 28672, 256), (48, 28700, 1152), (64, 16400, 896)]


@pytest.mark.parametrize("wtype", ["q4_0", "q4_ref", "q8_0"])
@pytest.mark.parametrize("m,n,k", SKINNY + TILES + WIDE)
def test_gemm_edges_bit_exact(hip, orc, rng, wtype, m, n, k):
    a = rng.normal(0, 1, (m, k)).astype(F32)
    a[0, :32] = 0.0
    if wtype == "q8_0":
        qs, sc = hip.synth_q8(20260021, m + n + k, n, k, 2e-4, 3.5e-4)
        w = hip.Tensor.from_q8_0(qs, sc, n, k)
        want = orc.matmul_transposed_q8w(a, qs, sc, n)
    else:
        if wtype == "q4_ref":
            qs, sc = orc.quantize_q4(rng.uniform(-1, 1, (n, k)).astype(F32))
        else:
            qs, sc = hip.synth_q4(20260022, m + n + k, n, k, 0.003, 0.006)
        w = hip.Tensor.from_q4(qs, sc, n, k)
        want = orc.matmul_transposed_q4(a, qs, sc, n)
    got = hip.HipBackend().matmul_transposed(hip.Tensor.from_numpy(a), w).data()
    assert np.array_equal(got.view(np.uint32), np.asarray(want, F32).reshape(m, n).view(np.uint32))


def same_bits(got, want, what):
    """Equal in every bit, any NaN equal to any other."""
    got, want = np.asarray(got, F32), np.asarray(want, F32)
    bad = (got.view(np.uint32) != want.view(np.uint32)) & ~(np.isnan(got) & np.isnan(want))
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.size} differ, first {got[bad][0]!r} for {want[bad][0]!r}"


def check_variant(hip, orc, epi, variant, a, w, y, res, order):
    """One launch of a GEMM kernel against the oracle's products y [m, n] of
    the same rows: stored, added to `res`, or as the SwiGLU product (runs of 32
    gate rows, then their up rows) with its Q8_0 codes."""
    ta = hip.Tensor.from_numpy(a)
    if epi == "store":
        same_bits(hip.probe_gemm(ta, w, epi, variant), y, variant)
    elif epi == "resid":
        with np.errstate(all="ignore"):
            same_bits(hip.probe_gemm(ta, w, epi, variant, hip.Tensor.from_numpy(res)), y + res, variant)
    else:
        m, n = y.shape
        runs = y.reshape(m, n // 64, 2, 32)
        want = orc.silu_mul(runs[:, :, 0].reshape(m, n // 2), runs[:, :, 1].reshape(m, n // 2)).reshape(m, n // 2)
        got, q, d = hip.probe_gemm(ta, w, epi, variant, order=order)
        same_bits(got, want, variant)
        for t in range(m):
            oq, od = orc.quantize_row_q8_0(want[t])
            some = ~np.isnan(want[t]).reshape(-1, 32).all(1)  # a block of nothing but NaN has no scale
            assert np.array_equal(q[t].reshape(-1, 32)[some], oq.reshape(-1, 32)[some]), f"{variant}: codes of row {t}"
            same_bits(d[t][some], od[some], f"{variant}: scales of row {t}")


Q4_VARIANTS = [(v, e) for v in ("r1", "r2", "r4", "w1", "w2", "w3", "128x128", "64x128", "64x64")
               for e in ("store", "resid", "silu") if e != "silu" or v not in ("r1", "r2", "64x64")]


@pytest.mark.parametrize("wtype", ["q4_0", "q4_ref"])
@pytest.mark.parametrize("variant,epi", Q4_VARIANTS, ids=["-".join(v) for v in Q4_VARIANTS])
def test_gemm_near_overflow(hip, orc, rng, wtype, variant, epi):
    """Rows whose terms and sums lie from far below the largest float to beyond
    it: what the block loop keeps finite stays finite, and what overflows there
    overflows the same way, whatever factor a kernel carries its codes with."""
    m, n, k = 70, 256, 640
    a = (rng.normal(0, 1, (m, k)) * 10.0 ** rng.uniform(34.0, 37.5, (m, 1))).astype(F32)
    a[3, 70], a[4, 300], a[5, 64:96] = np.inf, np.nan, -np.inf  # scales that are not finite, a NaN that has no code
    qs = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    sc = rng.uniform(0.1, 1.0, (n, k // 32)).astype(F32)
    if wtype == "q4_0":
        sc = sc.astype(np.float16).astype(F32)
    elif epi == "silu":
        sc.reshape(n // 64, 2, 32, -1)[:, 1] *= F32(1e-37)  # up rows that bring the product back into range
    with np.errstate(all="ignore"):
        y = np.asarray(orc.matmul_transposed_q4(a, qs, sc, n), F32).reshape(m, n)
    assert np.any(np.isfinite(y) & (np.abs(y) > 2.0 ** 124)) and np.any(np.isinf(y))
    res = (rng.normal(0, 1, (m, n)) * 1e37).astype(F32)
    check_variant(hip, orc, epi, variant, a, hip.Tensor.from_q4(qs, sc, n, k), y, res, order=1)


VARIANTS = [(w, v, e) for w in ("q4_0", "q4_ref", "q8_0") for v, e in Q4_VARIANTS if w != "q8_0" or v != "w3"]
# ragged rows and tokens for every tile: one stage of 4 blocks alone (all of a wide
# kernel's loads partial, fewer stages than buffers), 12 and 36 blocks (half a stage
# at the end), 68 (a round of the split kernels and 4 blocks); for the tiles also 3
# and 33 blocks, less than a stage and an odd remainder
SHAPES = [(7, 100, 128), (37, 130, 384), (53, 330, 1152), (70, 257, 2176)]
TILE_SHAPES = [(37, 130, 96), (140, 257, 1056)]


@pytest.mark.parametrize("wtype,variant,epi", VARIANTS, ids=["-".join(v) for v in VARIANTS])
def test_gemm_variants(hip, orc, rng, wtype, variant, epi):
    """Every kernel of the several-row GEMMs at the edges of its own tiles, each
    with every epilogue and weight type, whatever the rule picks."""
    for m, n, k in SHAPES + (TILE_SHAPES if "x" in variant else []):
        n = (n + 63) // 64 * 64 if epi == "silu" else n
        a = rng.normal(0, 1, (m, k)).astype(F32)
        a[0, :32] = 0.0
        if wtype == "q8_0":
            qs, sc = hip.synth_q8(20260023, m + n + k, n, k, 2e-4, 3.5e-4)
            w, y = hip.Tensor.from_q8_0(qs, sc, n, k), orc.matmul_transposed_q8w(a, qs, sc, n)
        else:
            if wtype == "q4_ref":
                qs, sc = orc.quantize_q4(rng.uniform(-1, 1, (n, k)).astype(F32))
            else:
                qs, sc = hip.synth_q4(20260024, m + n + k, n, k, 0.003, 0.006)
            w, y = hip.Tensor.from_q4(qs, sc, n, k), orc.matmul_transposed_q4(a, qs, sc, n)
        res = rng.normal(0, 1, (m, n)).astype(F32)
        for order in (0, 1) if epi == "silu" and n % 256 == 0 else (0,):
            check_variant(hip, orc, epi, variant, a, w, np.asarray(y, F32).reshape(m, n), res, order)


def test_gemm_probe_refuses(hip):
    """What a kernel cannot run is refused before any launch."""
    w = {n: hip.Tensor.from_q4(*hip.synth_q4(1, n, n, 96, 0.003, 0.006), n, 96) for n in (64, 65)}
    a, a1 = (hip.Tensor.from_numpy(np.zeros((4, k), F32)) for k in (96, 128))
    for args in [(a, w[64], "store", "r1"),      # K not of whole runs of 128
                 (a, w[65], "silu", "64x128"),   # rows not in runs of 64
                 (a1, w[64], "store", "64x64"),  # another K
                 (a, w[64], "store", "32x32"), (a, w[64], "silu", "64x64"), (a, w[64], "resid", "64x64")]:
        with pytest.raises(hip.LlmrsError):
            hip.probe_gemm(*args)
