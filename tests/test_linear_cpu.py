"""``ops.linear`` off the GPU: torch's Linear, bit for bit and with its errors, and the rule
that sends a call to the kernel on one; the drafter's modules under torch's compilers,
tracers and module swaps."""

import copy

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from flashmap_amd import _native, drafter, ops


def test_cpu_calls_are_torchs():
    x, w, b = torch.randn(3, 64), torch.randn(8, 64), torch.randn(8)
    assert torch.equal(ops.linear(x, w, b), F.linear(x, w, b))
    xb, wb = x.bfloat16(), w.bfloat16()
    assert torch.equal(ops.linear(xb, wb), F.linear(xb, wb))
    assert torch.equal(ops.linear(x[0], w), F.linear(x[0], w))
    assert ops.linear(torch.empty(0, 64), w).shape == (0, 8)
    assert torch.equal(ops.linear(x, w[0]), F.linear(x, w[0]))  # a vector for a weight
    assert ops.linear(x.to("meta"), w.to("meta")).shape == (3, 8)
    with pytest.raises(RuntimeError):
        ops.linear(x[:, :32], w)


@pytest.mark.parametrize("rows,n,k,takes", [(16, 2048, 2048, True), (16, 8192, 2048, True), (16, 2048, 4096, True),
                                            (16, 2048, 8192, False), (16, 32000, 2048, False),
                                            (16, 4096, 4096, True), (16, 4097, 2080, False), (16, 6144, 3072, False),
                                            (1, 8192, 4096, False), (32, 4096, 2048, True),
                                            (17, 4096, 2048, True), (17, 6144, 2048, False), (33, 64, 64, False),
                                            (4, 64, 48, False), (4, 0, 64, False)])
def test_rule(rows, n, k, takes):
    assert ops._linear_streams(rows, n, k) is takes


def _modules():
    cfg = dict(hidden_size=64, num_attention_heads=2, intermediate_size=96, cond_dim=32, time_embed_dim=32)
    return {"gelu": (drafter.FlashMapMLP(drafter.drafter_config(**cfg)), torch.randn(3, 64)),
            "swiglu": (drafter.FlashMapMLP(drafter.drafter_config(mlp_type="swiglu", **cfg)), torch.randn(3, 64)),
            "time": (drafter.FlashMapTimeEmbedding(drafter.drafter_config(**cfg)), torch.rand(3))}


@pytest.mark.parametrize("which", ["gelu", "swiglu", "time"])
def test_modules_trace_and_compile(which, monkeypatch):
    """One graph with torch's own Linears in it, whatever follows the module; sizes stay
    symbolic; and the guard of the kernel's calls is not part of it."""
    module, x = _modules()[which]
    want = module(x)
    monkeypatch.setattr(ops, "_eager_here", lambda *a: pytest.fail("a guard in a traced call"))
    traced = torch.fx.symbolic_trace(module)
    assert sum(n.op == "call_module" for n in traced.graph.nodes) == 2
    assert torch.equal(traced(x), want)
    torch._dynamo.reset()
    assert torch.equal(torch.compile(module, fullgraph=True, backend="eager")(x), want)
    assert torch.equal(torch.jit.trace(module, x)(x), want)
    rows = torch.export.Dim("rows", min=2, max=4096)
    exported = torch.export.export(module, (x,), dynamic_shapes=({0: rows},)).module()
    many = x.repeat(50, *[1] * (x.dim() - 1))
    assert torch.allclose(exported(many), module(many), atol=1e-6)


def test_time_embedding_scripts():
    module, x = _modules()["time"]
    assert torch.equal(torch.jit.script(module)(x), module(x))


def test_projections_are_torchs_linears():
    """Swaps by exact type (dynamic quantization among them) reach every projection."""
    model = drafter.FlashMapDraftModel(hidden_size=64, num_attention_heads=2, intermediate_size=96, cond_dim=32,
                                       time_embed_dim=32, target_hidden_size=64, num_hidden_layers=1,
                                       target_layer_ids=[1])
    assert {type(m) for m in model.modules() if isinstance(m, nn.Linear)} == {nn.Linear}
    for which in ("gelu", "swiglu"):
        module, x = _modules()[which]
        swapped = torch.ao.quantization.quantize_dynamic(copy.deepcopy(module), {nn.Linear})
        assert not any(type(m) is nn.Linear for m in swapped.modules())
        assert swapped(x).shape == module(x).shape


def test_what_was_put_around_a_projection_runs():
    class Doubled(nn.Linear):
        def forward(self, x):
            return 2 * super().forward(x)

    plain = nn.Linear(64, 8)
    assert drafter._bare(plain)
    hooked = copy.deepcopy(plain)
    hooked.register_forward_hook(lambda *a: None)
    before = copy.deepcopy(plain)
    before.register_forward_pre_hook(lambda *a: None)
    back = copy.deepcopy(plain)
    back.register_full_backward_hook(lambda *a: None)
    replaced = copy.deepcopy(plain)
    replaced.forward = lambda x: x
    normed = torch.nn.utils.parametrizations.weight_norm(copy.deepcopy(plain))
    for module in (hooked, before, back, replaced, normed, Doubled(64, 8)):
        assert not drafter._bare(module)
    handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
    try:
        assert not drafter._bare(plain)
    finally:
        handle.remove()
    assert drafter._bare(plain)
    assert torch.equal(drafter._project(replaced, torch.ones(2)), torch.ones(2))


def test_entry_refuses_what_it_cannot_launch():
    """The C entry's own checks, which return before anything is launched."""
    at = 4096  # an aligned address that no check follows
    for rows, n, k in ((33, 16, 64), (16, 16, 48), (16, (1 << 26) + 1, 64)):
        with pytest.raises(_native.NativeError, match="at most"):
            ops.call("fm_linear_rows", at, k, at, k, None, at, n, rows, n, k, None)
    with pytest.raises(_native.NativeError, match="aligned"):
        ops.call("fm_linear_rows", at + 2, 64, at, 64, None, at, 16, 16, 16, 64, None)
