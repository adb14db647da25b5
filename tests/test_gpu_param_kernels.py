"""Kernels behind the reference's per-parameter calls, at the sizes where their tilings can go wrong."""
import numpy as np
import pytest
import torch

import templar_amd.compress as tc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need an MI355X"
    return torch.device("cuda:0")


@pytest.mark.parametrize("h,w", [(1, 1), (1, 17), (1, 50), (1, 64), (2, 2), (7, 1), (16, 16), (16, 17), (17, 16), (15, 48),
                                 (31, 64), (33, 5), (48, 33), (49, 32), (60, 50), (63, 63), (64, 49), (64, 64)])
@pytest.mark.parametrize("Y,X", [(1, 1), (3, 5), (37, 41)])
def test_dense_transform_at_tile_edges(dev, h, w, Y, X):
    rng = np.random.default_rng(h * 100 + w)
    x = rng.standard_normal((Y * h, X * w)).astype(np.float32)
    bh, bw = rng.standard_normal((h, h)).astype(np.float32), rng.standard_normal((w, w)).astype(np.float32)
    chunks = x.reshape(Y, h, X, w).transpose(0, 2, 1, 3)
    x64 = chunks.astype(np.float64)
    want = bh.T.astype(np.float64) @ x64 @ bw.astype(np.float64)
    # h terms, then w terms, every product and sum rounded once: (h + w) 2^-24 of the sum of magnitudes, doubled
    bound = (h + w + 2) * 2.0 ** -23 * (np.abs(bh.T) @ np.abs(x64) @ np.abs(bw))
    rows = lambda a: a.transpose(0, 2, 1, 3).reshape(Y * h, X * w)  # noqa: E731
    for in_chunked, out_chunked in ((False, True), (True, False), (True, True), (False, False)):
        src = torch.from_numpy(np.ascontiguousarray(chunks) if in_chunked else x).to(dev)
        got = tc.ChunkingTransformer._dense(src, Y * h, X * w, h, w, torch.from_numpy(bh).to(dev),
                                            torch.from_numpy(bw).to(dev), in_chunked, out_chunked).cpu().numpy()
        ref, tol = (want, bound) if out_chunked else (rows(want), rows(bound))
        assert (np.abs(got - ref) <= tol).all(), (in_chunked, out_chunked)
