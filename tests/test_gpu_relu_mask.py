"""ReLU pass bits of ``forward_epilogue`` over every lane layout of a row.

A set bit is a value the ReLU passes, which leaves it non-zero (or NaN) in the
output, so the expected words come from the output itself, exactly.  Widths:
one, two and four columns a lane, rows of a power of two of lanes and others,
one and two mask words; sample counts around a wave tile and a small batch
that is spread over more workgroups than its tables alone would ask for.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import ple_oracle as po
from piecewiselinearembeddings_optimized_amd import workloads

pytestmark = pytest.mark.gpu

WIDTHS = (1, 2, 3, 4, 6, 8, 10, 12, 15, 16, 20, 24, 28, 31, 32, 33, 34, 36, 40, 48, 52, 60, 62, 63, 64)


@pytest.mark.parametrize("d", WIDTHS)
@pytest.mark.parametrize("n,f", [(1, 3), (67, 5), (1500, 9)])
def test_pass_bits_match_output(n, f, d):
    assert torch.cuda.is_available(), "HIP device required"
    import piecewiselinearembeddings_optimized_amd  # noqa: F401  (registers the ops)

    rng = np.random.default_rng(1000 * d + n)
    bins = [np.sort(rng.standard_normal(2 + 7 * (j % 4))).astype(np.float32) for j in range(f)]
    edges, inv_w, n_bins = workloads.pad_bins(bins)
    bmax = edges.shape[1] - 1
    x = rng.standard_normal((n, f)).astype(np.float32)
    x[rng.random((n, f)) < 0.02] = np.nan
    w = rng.uniform(-1, 1, (f, bmax, d)).astype(np.float32)
    bias = rng.uniform(-1, 1, (f, d)).astype(np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
    out, idx, mask = torch.ops.rtdl_num_embeddings_cuda.forward_epilogue(
        t(x), t(edges), t(inv_w), t(n_bins), t(w), t(bias), None, None, True, True, torch.float32)
    np.testing.assert_array_equal(idx.cpu().numpy().astype(np.int64), po.bin_indices(x, edges, n_bins))
    o = out.cpu().numpy()
    np.testing.assert_array_equal(mask.cpu().numpy(), po.pack_pass_bits((o != 0) | np.isnan(o)))
