"""The autograd formulas under compiled autograd and saved-tensor hooks.

Meta tensors: the formulas run without a GPU.
"""

import pytest
import torch

import piecewiselinearembeddings_optimized_amd  # noqa: F401

_ops = torch.ops.rtdl_num_embeddings_cuda
N, F, B, D = 6, 3, 4, 5


def _meta(*shape, **kw):
    return torch.empty(*shape, device="meta", **kw)


def _call(op):
    """An operator's output, and the tensors a gradient is taken of."""
    x, edges, iw, nb = _meta(N, F), _meta(F, B + 1), _meta(F, B), _meta(F, dtype=torch.int32)
    weight, bias = _meta(F, B, D), _meta(F, D)
    wrt = [x.requires_grad_()] + ([] if op == "encode" else [weight.requires_grad_()])
    if op == "forward":
        out = _ops.forward(x, edges, iw, nb, weight, torch.float32)[0]
    elif op == "forward_with_bias":
        out = _ops.forward_with_bias(x, edges, iw, nb, weight, bias.requires_grad_(), torch.float32)[0]
        wrt.append(bias)
    elif op == "forward_epilogue":
        out = _ops.forward_epilogue(x, edges, iw, nb, weight, bias.requires_grad_(), None, None, True, True,
                                    torch.float32)[0]
        wrt.append(bias)
    else:
        out = _ops.encode(x, edges, iw, nb, _meta(F, dtype=torch.int32), F * B)
    return out, wrt


OPS = ["forward", "forward_with_bias", "forward_epilogue", "encode"]


@pytest.mark.parametrize("op", OPS)
def test_compiled_autograd(op):
    from torch._dynamo import compiled_autograd

    out, wrt = _call(op)
    graphs = []
    with compiled_autograd._enable(lambda gm: graphs.append(gm) or gm):
        out.sum().backward()
    assert len(graphs) == 1
    assert [t.grad.shape for t in wrt] == [t.shape for t in wrt]


def _one_graph_compiler(graphs):
    """A compiler that takes whole graphs only, and notes the operator calls of each."""
    from torch._dynamo.backends.common import aot_autograd

    def compile_graph(gm, _example_inputs):
        graphs.append([(str(n.target), [a for a in n.args if not isinstance(a, torch.fx.Node)])
                       for n in gm.graph.nodes if "rtdl_num_embeddings_cuda" in str(n.target)])
        return gm.forward

    torch._dynamo.reset()
    return torch.compile(backend=aot_autograd(fw_compiler=compile_graph), fullgraph=True)


@pytest.mark.parametrize("op", OPS)
def test_compiled_autograd_is_one_graph(op):
    from torch._dynamo import compiled_autograd

    graphs = []
    compiler = _one_graph_compiler(graphs)
    out, wrt = _call(op)
    with compiled_autograd._enable(compiler):
        out.sum().backward()
    backward = "encode_backward" if op == "encode" else op.replace("forward", "backward")
    assert [[name for name, _ in g] for g in graphs] == [[f"rtdl_num_embeddings_cuda.{backward}.default"]]
    assert [t.grad.shape for t in wrt] == [t.shape for t in wrt]


def test_compiled_autograd_keeps_a_graph_per_option():
    """The flags and the dtype a node saved are constants of its graph."""
    from torch._dynamo import compiled_autograd

    graphs = []
    compiler = _one_graph_compiler(graphs)

    def step(quant, relu, grad_bias):
        x, edges, iw, nb = _meta(N, F), _meta(F, B + 1), _meta(F, B), _meta(F, dtype=torch.int32)
        weight, bias = _meta(F, B, D, requires_grad=True), _meta(F, D, requires_grad=grad_bias)
        out = _ops.forward_epilogue(x, edges, iw, nb, weight, bias, None, None, relu, True, quant)[0]
        known = len(graphs)
        with compiled_autograd._enable(compiler):
            out.sum().backward()
        return [args for g in graphs[known:] for _, args in g]

    for quant, relu, grad_bias in [(torch.float32, True, True), (torch.bfloat16, True, True),
                                   (torch.bfloat16, False, True), (torch.bfloat16, False, False)]:
        assert step(quant, relu, grad_bias) == [[None, relu, quant, False, True, grad_bias, False, False]]
    assert step(torch.bfloat16, True, True) == []     # the second one's graph


@pytest.mark.parametrize("op", OPS)
def test_saved_tensor_hooks(op):
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
        out, wrt = _call(op)
    assert packed
    assert [g.shape for g in torch.autograd.grad(out, wrt, _meta(*out.shape))] == [t.shape for t in wrt]


@pytest.mark.parametrize("op", OPS[:3])
def test_integer_outputs_need_no_gradient(op):
    x, edges, iw, nb = _meta(N, F), _meta(F, B + 1), _meta(F, B), _meta(F, dtype=torch.int32)
    weight, bias = _meta(F, B, D, requires_grad=True), _meta(F, D)
    args = {"forward": (torch.float32,), "forward_with_bias": (bias, torch.float32),
            "forward_epilogue": (bias, None, None, True, True, torch.float32)}[op]
    out, *whole = getattr(_ops, op)(x, edges, iw, nb, weight, *args)
    assert out.requires_grad and not any(t.requires_grad for t in whole)
