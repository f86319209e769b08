"""Queries on their way to a search on the GPU."""

import numpy as np
import pytest
import torch

from quickstart_streaming_agents_amd.ops import dispatch as D
from quickstart_streaming_agents_amd.vector.index import VectorIndex

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [32, 61, 1536])
@pytest.mark.parametrize("scale", [1.0, 1e-18, 3e17, 2e19])
def test_norms_are_rounded_once(dim, scale):
    """Against unit vectors a score is a normalized number: half a place of f32
    around its value, nought where the norm is beyond what floats hold."""
    g = np.random.default_rng(dim)
    q = (g.standard_normal((7, dim)) * scale).astype(np.float32)
    got = D.topk_cosine_host(q, torch.eye(dim, device="cuda:0"), 5)
    score, at = got[0].view(np.float32).astype(np.float64), got[1]
    x = q.astype(np.float64)
    norm = np.sqrt((x * x).sum(1, keepdims=True))
    if scale == 2e19:
        norm[:] = np.inf
    want = np.take_along_axis(x / np.maximum(norm, 1e-12), at, 1)
    assert (np.abs(score - want) <= 2.0 ** -24 * (1 + 1e-6) * np.abs(want)
            + 2.0 ** -150).all()


@pytest.mark.parametrize("queries", [np.zeros(8, np.float32), np.float32(1.0),
                                     [0.5] * 8])
def test_queries_that_are_not_rows(queries):
    """The error that numpy raises for their norms, on either device."""
    index = VectorIndex()
    index.add("a", "", np.ones(8, np.float32))
    for device in ("cpu", "cuda:0"):
        with pytest.raises(np.exceptions.AxisError):
            index.search_batch_gpu(queries, 1, device=device)
