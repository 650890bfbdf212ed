"""Performance cases of the piecewise-linear embedding framework.

What a user's program has this package do, over the sizes it does it at:
training steps and inference of ``CudaPiecewiseLinearEmbeddings`` (both
versions, with and without ReLU, with and without autocast), the operator pair
that programs with a layer of their own call, and the dense encoding of
``CudaPiecewiseLinearEncoding``.

A case is a dict of plain values:

``path``     "train" (module, forward and backward), "infer" (module, forward
             without gradients), "pair" (forward and backward operators) or
             "encode" (dense encoding, forward and backward)
``n`` ``f`` ``bins`` ``d``   samples, features, bins asked for per feature,
             embedding width (0 for "encode")
``data``     the features' distribution, which also decides how many of the
             asked bins survive: "normal" (all), "mixed" (thirds of lognormal,
             uniform and Poisson features: ragged bins, down to a few),
             "narrow" (90% of a feature's samples within a few bins)
``edges``    share of the samples that lie on a bin edge, in hundredths
             (quantile edges are values of the data, so repeated values hit
             them); a fifth as many lie outside the edges
``version`` ``relu``         the module's version and activation
``dtype``    "f32", or the 16-bit type of the autocast region (module) or of
             the output and its gradient (pair)
``dx``       whether x needs a gradient (an embedding on raw inputs needs none)
"""

from __future__ import annotations

import math

import torch

from piecewiselinearembeddings_optimized_amd import (
    CudaPiecewiseLinearEmbeddings,
    CudaPiecewiseLinearEncoding,
    bin_tables,
    compute_bins,
)

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BIN_ROWS = 10_000      # rows of the data that the bins are computed from

# caps of a drawn case: below the largest listed ones also where its width or
# option costs more per element
MAX_PAIRS = 3_000_000
MAX_ELEMENTS = 64_000_000


def _case(name, path, n, f, bins, d, *, data="normal", edges=0, version="A", relu=False, dtype="f32", dx=False):
    return {"name": name, "path": path, "n": n, "f": f, "bins": bins, "d": d, "data": data, "edges": edges,
            "version": version, "relu": relu, "dtype": dtype, "dx": dx}


def listed():
    return [
        # the smallest training step (a toy table, a smoke test): latency and launches
        _case("train_tiny", "train", 256, 8, 48, 24),
        # a serving call of a small request
        _case("infer_small", "infer", 64, 20, 48, 16, version="B", relu=True, data="mixed", edges=5),
        # scoring a table in bulk
        _case("infer_bulk", "infer", 65536, 128, 48, 32, version="B", edges=5),
        # an ordinary tabular model's training batch: 1024 rows, some dozens of
        # features, the ragged bins that real columns give
        _case("train_batch", "train", 1024, 50, 48, 24, version="B", relu=True, data="mixed", edges=5),
        # a large-batch training step of the version B module, the benchmark's headline
        _case("train_headline", "train", 65536, 128, 48, 32, version="B", edges=5),
        # the same sizes through the operators, with the bias and all gradients
        _case("pair_headline", "pair", 65536, 128, 48, 32, edges=5, dx=True),
        # wide rows, ragged bins up to 128, version A with its activation
        _case("train_ragged", "train", 16384, 64, 128, 64, relu=True, data="mixed", edges=5),
        # many samples in few of many bins (heavy contention), narrow rows
        _case("pair_contention", "pair", 262144, 32, 256, 16, data="narrow", dx=True),
        # a thousand features in bfloat16
        _case("pair_wide_bf16", "pair", 8192, 1024, 96, 24, data="mixed", dtype="bf16", dx=True),
        # a training step under bfloat16 autocast: 32-bit output and gradient,
        # the embedding rounded to 16 bits inside
        _case("train_autocast", "train", 16384, 100, 64, 32, version="B", relu=True, data="mixed", dtype="bf16"),
        # odd sizes throughout (the width too), with the gradient of x: stacked
        # under a learned transform
        _case("train_odd", "train", 10007, 37, 100, 15, relu=True, data="mixed", edges=5, dx=True),
        # the dense encoding under a learned layer
        _case("encode_dense", "encode", 16384, 128, 48, 0, edges=5, dx=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["train", "train", "train", "infer", "infer", "pair", "pair", "encode"])
    n, f, bins = _log(rng, 64, 262144), _log(rng, 4, 1024), _log(rng, 4, 256)
    d = 0 if path == "encode" else rng.choice([8, 10, 12, 15, 16, 20, 24, 24, 32, 32, 40, 48, 64])
    if rng.random() < 0.5:      # whole batches as often as odd ones
        n = max(64, n // 64 * 64)
    row = f * (bins if path == "encode" else d)
    n = max(1, min(n, MAX_PAIRS // f, MAX_ELEMENTS // row))
    dtype = "f32"
    if path in ("train", "infer", "pair") and rng.random() < 0.35:
        dtype = rng.choice(["bf16", "bf16", "f16"])
    module = path in ("train", "infer")
    return {"path": path, "n": n, "f": f, "bins": bins, "d": d, "data": rng.choice(["normal", "mixed", "mixed", "narrow"]),
            "edges": rng.choice([0, 5]), "version": rng.choice(["A", "B"]) if module else "A",
            "relu": module and rng.random() < 0.5, "dtype": dtype,
            "dx": path in ("pair", "encode") or (path == "train" and rng.random() < 0.3)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _columns(case, rows, gen, centres):
    f, kind = case["f"], case["data"]
    x = torch.randn(rows, f, device=DEVICE, generator=gen)
    if kind == "mixed":
        a, b = f // 3, 2 * f // 3
        x[:, :a] = x[:, :a].exp()
        x[:, a:b] = torch.rand(rows, b - a, device=DEVICE, generator=gen) * 10 - 5
        x[:, b:] = torch.poisson(torch.full((rows, f - b), 3.0, device=DEVICE), generator=gen)
    elif kind == "narrow" and centres is not None:
        tight = torch.rand(rows, f, device=DEVICE, generator=gen) < 0.9
        x = torch.where(tight, centres + 0.05 * x, x)
    return x


def _inputs(case, seed):
    """Bins from a sample of the data, as a list of edge tensors on the host, and one batch."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    n, f = case["n"], case["f"]
    centres = torch.rand(f, device=DEVICE, generator=gen) * 3 - 1.5
    bins = [e.cpu() for e in compute_bins(_columns(case, BIN_ROWS, gen, None), case["bins"])]
    x = _columns(case, n, gen, centres)
    if case["edges"]:
        edges, _, n_bins = bin_tables(bins, device=DEVICE)
        lo, hi = edges[:, 0], edges.gather(1, n_bins.long()[:, None])[:, 0]
        pick = torch.rand(n, f, device=DEVICE, generator=gen)
        which = (torch.rand(n, f, device=DEVICE, generator=gen) * (n_bins + 1)).long()
        which = torch.minimum(which, n_bins.long())
        on = edges.gather(1, which.T).T
        beyond = 3 * (hi - lo) * torch.rand(n, f, device=DEVICE, generator=gen)
        out = torch.where(torch.rand(n, f, device=DEVICE, generator=gen) < 0.5, lo - beyond, hi + beyond)
        share = case["edges"] / 100
        x = torch.where(pick < share, on, torch.where(pick < 1.2 * share, out, x))
    return bins, x.contiguous(), gen


def _uniform(shape, bound, gen):
    return (torch.rand(shape, device=DEVICE, generator=gen) * 2 - 1) * bound


def prepare(case, seed):
    bins, x, gen = _inputs(case, seed)
    n, f, d, dtype = case["n"], case["f"], case["d"], DTYPES[case["dtype"]]
    state = {"case": case, "x": x}
    if case["path"] == "encode":
        m = CudaPiecewiseLinearEncoding(bins).to(DEVICE)
        state.update(module=m, x=x.requires_grad_(case["dx"]),
                     g=torch.randn(n, m.get_output_shape()[0], device=DEVICE, generator=gen))
        return state
    if case["path"] == "pair":
        edges, inv_widths, n_bins = bin_tables(bins, device=DEVICE)
        bound = edges.shape[1] ** -0.5
        state.update(edges=edges, inv_widths=inv_widths, n_bins=n_bins,
                     weight=_uniform((f, edges.shape[1] - 1, d), bound, gen), bias=_uniform((f, d), bound, gen),
                     g=torch.randn(n, f, d, device=DEVICE, generator=gen).to(dtype))
        return state
    m = CudaPiecewiseLinearEmbeddings(bins, d, activation=case["relu"], version=case["version"]).to(DEVICE)
    with torch.no_grad():   # weights as training leaves them (version B starts from zeros)
        for p in m.parameters():
            p.copy_(_uniform(p.shape, m.max_n_bins ** -0.5, gen))
    state["module"] = m
    if case["path"] == "train":
        state["x"] = x.requires_grad_(case["dx"])
        state["wrt"] = ([state["x"]] if case["dx"] else []) + list(m.parameters())
        state["g"] = torch.randn(n, f, d, device=DEVICE, generator=gen)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

_ops = torch.ops.rtdl_num_embeddings_cuda


def _module_out(state):
    dtype = DTYPES[state["case"]["dtype"]]
    if dtype == torch.float32:
        return state["module"](state["x"])
    with torch.autocast("cuda", dtype=dtype):
        return state["module"](state["x"])


def run(state):
    case = state["case"]
    if case["path"] == "infer":
        with torch.no_grad():
            return _module_out(state)
    if case["path"] == "train":
        out = _module_out(state)
        return [out, *torch.autograd.grad(out, state["wrt"], state["g"])]
    if case["path"] == "encode":
        out = state["module"](state["x"])
        return [out, *torch.autograd.grad(out, [state["x"]], state["g"])]
    x, g, weight = state["x"], state["g"], state["weight"]
    tables = state["edges"], state["inv_widths"], state["n_bins"]
    if case["dtype"] == "f32":
        out, idx = _ops.forward_with_bias(x, *tables, weight, state["bias"], torch.float32)
        return [out, idx, *_ops.backward_with_bias(g, x, *tables, weight, idx, torch.float32, True, True, True)]
    out, idx = _ops.forward(x, *tables, weight, DTYPES[case["dtype"]])
    return [out, idx, *_ops.backward(g, x, *tables, weight, idx, True, True)]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how close outputs have to be
# ---------------------------------------------------------------------------

def work(case):
    n, f, b, d, path = case["n"], case["f"], case["bins"], case["d"], case["path"]
    if path == "encode":
        # (the backward reads the gradient's one or two elements per pair, a
        # 32-byte sector at least)
        return {"bytes": 4 * n * f + 4 * n * f * b + 32 * n * f + 4 * n * f + 4 * f * (2 * b + 2), "flops": 4 * n * f}
    half = 2 if path == "pair" and case["dtype"] != "f32" else 4
    tables = 4 * f * (2 * b + 2) + 4 * f * b * d + 8 * f * d
    size = 4 * n * f + half * n * f * d + tables
    flops = 2 * n * f * d
    if path == "pair":
        size += n * f                                           # the bin indices, an output
    if path != "infer":
        size += half * n * f * d + 4 * f * b * d + 8 * f * d    # gradient in, parameter gradients out
        flops += 3 * n * f * d
        if case["dx"]:
            size += 4 * n * f
            flops += 2 * n * f * d
    return {"bytes": size, "flops": flops}


def tolerance(case):
    # 32-bit sums over the samples in another order: the outputs are 3e-8 to
    # 2.5e-7 off their 64-bit values
    if case["dtype"] == "f32":
        return {"rel": 1e-6, "max": 1e-4}
    # 16-bit outputs are 2e-3 off by their own rounding
    if case["path"] == "pair":
        return {"rel": 7e-3, "max": 2e-2}
    # the embedding rounded to 16 bits inside a 32-bit module: a value may
    # round to its neighbour (and pass or not pass the ReLU then)
    return {"rel": 1e-3, "max": 0.2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def exact(case, seed):
    state = prepare(case, seed)
    bins = [e.to(DEVICE) for e in _inputs(case, seed)[0]]
    x, n = state["x"].detach(), case["n"]
    if case["path"] == "encode":
        out = torch.zeros_like(state["g"], dtype=torch.float64)
        dx = torch.zeros(n, case["f"], dtype=torch.float64, device=DEVICE)
        at = 0
        for f, e in enumerate(bins):
            k, frac, iw, left = _locate(x[:, f].contiguous(), e)
            cols = torch.arange(e.numel() - 1, device=DEVICE)
            out[:, at:at + len(cols)] = torch.where(cols < k[:, None], 1.0, 0.0)
            out[torch.arange(n, device=DEVICE), at + k] = frac
            g = state["g"][:, at:at + len(cols)].double()
            pick = g.gather(1, k[:, None])[:, 0] * iw[k]
            low = (k - 1).clamp_min(0)
            dx[:, f] = pick + torch.where(left, g.gather(1, low[:, None])[:, 0] * iw[low], 0.0)
            at += len(cols)
        return [out, dx]

    qt = DTYPES[case["dtype"]]
    q = (lambda t: t.double()) if qt == torch.float32 else (lambda t: t.float().to(qt).double())
    pair, train, relu = case["path"] == "pair", case["path"] == "train", case["relu"]
    if pair:
        weight, bias, w0, b0 = state["weight"], state["bias"] if qt == torch.float32 else None, None, None
    else:
        m = state["module"]
        weight, bias = m.linear.weight.detach(), m.linear.bias
        w0, b0 = (None, None) if m.linear0 is None else (m.linear0.weight.detach(), m.linear0.bias.detach())
    nf, bmax, d = weight.shape
    zeros = lambda *s: torch.zeros(*s, dtype=torch.float64, device=DEVICE)  # noqa: E731
    out, dw, db = zeros(n, nf, d), zeros(nf, bmax, d), zeros(nf, d)
    dx, dw0, db0 = zeros(n, nf), zeros(nf, d), zeros(nf, d)
    for f, e in enumerate(bins):
        nb = e.numel() - 1
        slots = torch.arange(nb, device=DEVICE)
        slots[-1] = bmax - 1                                   # the last bin's weights are in the last slot
        w = q(weight[f, slots])
        k, frac, iw, left = _locate(x[:, f].contiguous(), e)
        if qt != torch.float32:
            e32 = e.float()
            frac = q((x[:, f] - e32[k]) * torch.reciprocal(e32[1:] - e32[:-1])[k])
        prefix = torch.cat([zeros(1, d), w.cumsum(0)[:-1]])
        v = prefix[k] + frac[:, None] * w[k]
        if relu or qt != torch.float32:
            # what is rounded to 16 bits or passes the ReLU is decided on the
            # 32-bit value: the prefix summed in bin order, one fma
            p32 = torch.zeros(nb, d, device=DEVICE)
            for i in range(1, nb):
                p32[i] = p32[i - 1] + w[i - 1].float()
            frac32 = frac if qt != torch.float32 else ((x[:, f] - e[k]) * torch.reciprocal(e[1:] - e[:-1])[k]).double()
            v32 = (p32[k].double() + frac32[:, None] * w[k]).float()
            if qt != torch.float32:
                v32 = v32.to(qt).float()
                v = v32.double() if not pair else v
        if bias is not None:
            v = v + bias[f].detach().double()
        if relu:
            passed = (v32 + bias[f].detach() if bias is not None else v32) > 0
            v = torch.where(passed, v, 0.0)
        if w0 is not None:
            v = v + b0[f].double() + w0[f].double() * x[:, f, None].double()
        out[:, f] = v
        if not (pair or train):
            continue
        g = state["g"][:, f].double()
        gp = torch.where(passed, g, 0.0) if relu else g
        gq = q(gp)
        bucket = zeros(nb, d).index_add_(0, k, gq)
        weighted = zeros(nb, d).index_add_(0, k, gq * frac[:, None])
        dw[f, slots] = weighted + bucket.sum(0) - bucket.cumsum(0)
        db[f] = gp.sum(0)
        low = (k - 1).clamp_min(0)
        dx[:, f] = (gq * w[k]).sum(1) * iw[k] + torch.where(left, (gq * w[low]).sum(1) * iw[low], 0.0)
        if w0 is not None:
            dw0[f] = (g * x[:, f, None].double()).sum(0)
            db0[f] = g.sum(0)
            dx[:, f] += (g * w0[f].double()).sum(1)
    if pair:
        return [out, None, dx, dw, db] if bias is not None else [out, None, dx, dw]
    if not train:
        return out
    by_name = {"linear.weight": dw, "linear.bias": db, "linear0.weight": dw0, "linear0.bias": db0}
    return [out, *([dx] if case["dx"] else []), *(by_name[k] for k, _ in m.named_parameters())]


def _locate(x, e):
    """Bin, fraction in it, inverse widths of the bins, and whether x is on the bin's left edge and not the first."""
    k = (torch.searchsorted(e, x, right=True) - 1).clamp(0, e.numel() - 2)
    e64 = e.double()
    iw = 1.0 / (e64[1:] - e64[:-1])
    return k, (x.double() - e64[k]) * iw[k], iw, (k > 0) & (x == e[k])
