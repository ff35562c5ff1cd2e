"""Host transfers at the edges of their paths: downloads through the pinned
buffer (up to 1 MiB) and beyond it, and prompts whose ids travel in a launch's
arguments (up to 512) or by a copy - every value exactly as it was."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 65537, (1 << 18) - 1, 1 << 18, (1 << 18) + 1])
def test_download_sizes(hip, rng, n):
    a = rng.normal(0, 1, n).astype(np.float32)
    hip.init()
    t = hip.Tensor.from_numpy(a)
    for _ in range(2):
        assert np.array_equal(t.data(), a)


@pytest.mark.parametrize("n", [1, 511, 512, 513, 700])
def test_prompt_ids_arrive(hip, rng, n):
    from llmrs_hip import synthetic as sy
    spec = sy.tiny(prompt=n, decode=4)
    m = hip.HipModel(spec.config())
    sy.load_model(m, sy.make_weights(spec))
    for _ in range(2):
        ids = rng.integers(0, spec.vocab, n).astype(np.int32)
        m.begin(ids)
        m.decode_steps(2)
        assert np.array_equal(m.tokens(n), ids)
        assert m.produced() == (3, False)
