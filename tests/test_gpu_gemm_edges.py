"""The several-row GEMMs at the edges of their tiles and of the rule that picks
one, against the oracle's block loop, bit for bit (matmul_transposed with a
quantised weight; cpu.rs:90-110): whole and ragged row and token tiles, one to
many rounds of blocks with every remainder, and one row beyond each range."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32

# (m, n, k): the skinny GEMM's 16-row and 16-token tiles, its steps of 8 blocks
# (k = 384: 12 blocks), its rounds of 64, 32 and 16 blocks, 1, 2 and 4 row
# tiles per workgroup, and its last row (160) and the one after
SKINNY = [(2, 16, 128), (15, 33, 128), (16, 64, 256), (17, 100, 384), (31, 1, 640), (33, 4112, 2176),
          (64, 8200, 512), (65, 130, 4224), (160, 72, 1024), (161, 72, 1024)]

# the tile GEMM: 64 x 64, 64 x 128 and 128 x 128 tiles with ragged tokens and
# rows, K of less than a stage (4 or 8 blocks), of whole stages and of every
# kind of remainder
TILES = [(130, 200, 32), (165, 100, 224), (161, 65, 256), (200, 33, 288), (1000, 4090, 416), (2047, 4095, 288),
         (96, 6144, 1024), (100, 28672, 128)]
# the skinny GEMM's wide kernels: one, two and three token tiles with ragged
# last ones, rows past a 64-row set, less than a stage of eight blocks, half
# stages at the end, fewer stages than buffers and more
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
