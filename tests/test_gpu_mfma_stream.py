"""The matrix-core backward's two load policies give the same bits.

Large gradients are read past the caches, smaller ones with plain loads; the
knob forces either on shapes that cover every instantiation (dtype, bin tiles,
row width), one chunk and several, and odd feature counts.
"""

from __future__ import annotations

import pytest
import torch

from piecewiselinearembeddings_optimized_amd import capi
from tests.test_gpu_wide_tables import QT, _inputs, wide_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", ["bf16", "f16"])
@pytest.mark.parametrize("d", [8, 16, 24, 32])
@pytest.mark.parametrize("bmax", [1, 32, 33, 64, 65, 96])
def test_streamed_gradient_gives_the_same_bits(bmax, d, quant, tune):
    assert torch.cuda.is_available(), "HIP device required"
    import piecewiselinearembeddings_optimized_amd  # noqa: F401  (registers the ops)

    ops = torch.ops.rtdl_num_embeddings_cuda
    qt = QT[quant]
    chunks = set()
    for n, f in ((200, 5), (1500, 33), (300, 257)):
        pl = capi.backward_plan(n, f, bmax, d, grad_dtype=qt)
        assert pl["matrix_cores"] == 1
        chunks.add(pl["chunks"] > 1)
        x, e, iw, nb, wt, _ = _inputs(wide_case(n, f, bmax, d, seed=bmax + d))
        _, idx = ops.forward(x, e, iw, nb, wt, qt)
        g = torch.randn((n, f, d), device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(n)).to(qt)
        results = []
        for policy in (1, 2):
            tune("BWD_STREAM", policy)
            results.append(ops.backward_with_bias(g, x, e, iw, nb, wt, idx, qt, True, True, True))
        assert all(torch.equal(a, b) for a, b in zip(*results))
    assert chunks == {False, True}
