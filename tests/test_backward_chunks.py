"""Sample chunks of the backward where the feature groups do not divide the CUs.

The planner rounds the chunk count down, so that every workgroup has a place
from the start, and gives all sub-tiles of the sorted path one size, smaller
than a full one.  On the CPU: the plans over a range of sizes.  On the GPU:
the gradients at such sizes against the quantisation-aware float64 oracle at
the fp32 bar (``|err| <= 1e-6 + 1e-5 * sum|terms|``), bitwise on a repeat.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from piecewiselinearembeddings_optimized_amd import capi

CUS = 256       # the planner's assumption without a device
LDS = 160 * 1024

# (N, F, max bins, d): 1 to 10 chunks of partial sub-tiles, last ones of a
# few samples, one, two and four features a group
SHAPES = [(2500, 300, 10, 8), (1500, 600, 9, 15), (2049, 260, 40, 48), (3075, 101, 30, 32), (5130, 51, 64, 24)]
MFMA_SHAPES = [(2100, 200, 40, 24), (1100, 300, 20, 16), (1030, 170, 70, 8)]


def _places(pl, n, f, d):
    """Workgroups of a plan, and how many are resident at once."""
    groups = -(-f // pl["features_per_group"]) * pl["windows"]
    one = pl["matrix_cores"] or pl["threads"] == 512
    return groups * pl["chunks"], CUS * (1 if one else min(2, LDS // pl["lds_bytes"]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_chunks_fit_the_first_round(dtype):
    if torch.cuda.is_available():
        pytest.skip("the plans depend on the device's CUs")
    seen = 0
    for f in (1, 3, 33, 50, 75, 100, 129, 170, 260, 300, 600, 1024):
        for n in (1, 255, 1024, 1025, 5000, 30001, 262144):
            for bins, d in ((20, 8), (48, 15), (48, 24), (90, 32), (128, 64)):
                pl = capi.backward_plan(n, f, bins, d, grad_dtype=dtype)
                if not (pl["sorted"] or pl["matrix_cores"]):
                    continue
                used, places = _places(pl, n, f, d)
                assert used <= places or pl["chunks"] == 1, (n, f, bins, d, pl)
                seen += pl["chunks"] > 1
    assert seen > 50


def _gradients(shape, quant, c_oracle):
    import piecewiselinearembeddings_optimized_amd  # noqa: F401  (registers the ops)
    from tests.test_gpu_wide_tables import QT, _check_backward, _inputs, wide_case

    ops = torch.ops.rtdl_num_embeddings_cuda
    n, f, bins, d = shape
    w = wide_case(n, f, bins, d, seed=sum(shape))
    x, e, iw, nb, wt, bt = _inputs(w)
    g_h = torch.from_numpy(np.random.default_rng(n).standard_normal((n, f, d), dtype=np.float32)).to(QT[quant])
    g = g_h.to("cuda:0")
    if quant == "f32":
        _, idx = ops.forward_with_bias(x, e, iw, nb, wt, bt, QT[quant])
    else:
        _, idx = ops.forward(x, e, iw, nb, wt, QT[quant])
    first = ops.backward_with_bias(g, x, e, iw, nb, wt, idx, QT[quant], True, True, True)
    again = ops.backward_with_bias(g, x, e, iw, nb, wt, idx, QT[quant], True, True, True)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    _check_backward(w, g_h.float().numpy(), *first, c_oracle, quant=quant)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_sorted_backward(shape, c_oracle):
    _gradients(shape, "f32", c_oracle)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", MFMA_SHAPES, ids=["x".join(map(str, s)) for s in MFMA_SHAPES])
def test_matrix_core_backward(shape, c_oracle):
    n, f, bins, d = shape
    assert capi.backward_plan(n, f, bins, d, grad_dtype=torch.bfloat16)["matrix_cores"] == 1
    _gradients(shape, "bf16", c_oracle)
