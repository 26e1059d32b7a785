"""The few-row projection kernel (fm_linear_rows) against float64: every row count of its
two row blocks' edges, output widths that end inside a 16-row tile and on both sides of the
8 / 16 wavefront rule, reductions that leave some wavefronts without a step or with a
partial group; strided weights; and what keeps a call on torch's Linear."""

import pytest
import torch
import torch.nn.functional as F

from _inputs import gen
from flashmap_amd import drafter, ops

pytestmark = pytest.mark.gpu


@pytest.fixture
def launches(monkeypatch):
    """The native calls made, by name."""
    made, call = [], ops.call
    monkeypatch.setattr(ops, "call", lambda name, *args: (made.append(name), call(name, *args))[1])
    return made


def _bound(x, w, bias, ref):
    """Per element: the sum of k products in fp32 in any order (k 2^-24 of the absolute
    sum, twice for the bias and the partials' order) and the rounding to bf16 (2^-8)."""
    total = x.double().abs() @ w.double().abs().T + (0 if bias is None else bias.double().abs())
    return 2 * x.shape[-1] * 2.0 ** -24 * total + 2.0 ** -8 * ref.abs()


@pytest.mark.parametrize("rows,n,k", [(1, 1, 32), (16, 100, 64), (15, 17, 1376), (16, 4097, 2048), (16, 8192, 2048),
                                      (16, 2048, 4096), (16, 4096, 4096), (17, 2048, 2048), (32, 4096, 1056), (31, 33, 544)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_linear_rows(dev, launches, rows, n, k, with_bias):
    print(f"linear rows={rows} n={n} k={k}", flush=True)
    g = gen(rows + n + k)
    x = torch.randn(rows, k, generator=g).bfloat16()
    wide = (torch.randn(n, k + 8, generator=g) / k ** 0.5).bfloat16()
    bias = torch.randn(n, generator=g).bfloat16() if with_bias else None
    assert ops._linear_streams(rows, n, k)
    for w in (wide[:, :k].contiguous(), wide[:, :k]):
        wd = w.to(dev) if w.is_contiguous() else wide.to(dev)[:, :k]
        got = ops.linear(x.to(dev), wd, None if bias is None else bias.to(dev)).cpu()
        ref = x.double() @ w.double().T + (0 if bias is None else bias.double())
        assert launches == ["fm_linear_rows"], "the kernel and not the library"
        launches.clear()
        assert got.shape == (rows, n) and got.dtype == torch.bfloat16
        assert ((got.double() - ref).abs() <= _bound(x, w, bias, ref)).all()


def test_two_row_blocks_of_eight_wavefronts(dev):
    """The C entry's widest form (32 rows, more than a tile of columns per CU), which the rule
    above leaves to the library."""
    rows, n, k = 32, 8200, 96
    g = gen(4)
    x, w = torch.randn(rows, k, generator=g).bfloat16(), torch.randn(n, k, generator=g).bfloat16()
    assert not ops._linear_streams(rows, n, k)
    xd, wd, out = x.to(dev), w.to(dev), torch.empty(rows, n, dtype=torch.bfloat16, device=dev)
    ops.call("fm_linear_rows", xd.data_ptr(), k, wd.data_ptr(), k, None, out.data_ptr(), n, rows, n, k,
             torch.cuda.current_stream().cuda_stream)
    ref = x.double() @ w.double().T
    assert ((out.cpu().double() - ref).abs() <= _bound(x, w, None, ref)).all()


def test_leading_dimensions_and_fallbacks(dev, launches):
    g = gen(3)
    x = torch.randn(2, 5, 64, generator=g).bfloat16().to(dev)
    w = torch.randn(48, 64, generator=g).bfloat16().to(dev)
    got = ops.linear(x, w)
    assert got.shape == (2, 5, 48)
    assert torch.equal(got.view(10, 48), ops.linear(x.view(10, 64), w))
    assert ops.linear(x[0, 0], w).shape == (48,)
    assert launches == ["fm_linear_rows"] * 3
    launches.clear()
    # gradients, other types and strided rows go to torch, with its results
    wp = w.clone().requires_grad_(True)
    ops.linear(x, wp).float().sum().backward()
    ref = w.clone().requires_grad_(True)
    F.linear(x, ref).float().sum().backward()
    assert torch.equal(wp.grad, ref.grad)
    assert torch.equal(ops.linear(x.float(), w.float()), F.linear(x.float(), w.float()))
    strided = torch.randn(10, 128, generator=g).bfloat16().to(dev)[:, ::2]
    assert torch.equal(ops.linear(strided, w), F.linear(strided, w))
    off = torch.randn(10 * 64 + 1, generator=g).bfloat16().to(dev)[1:].view(10, 64)  # not 16-byte aligned
    assert torch.equal(ops.linear(off, w), F.linear(off, w))
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w).dtype == torch.float16
    with torch.no_grad():
        mapped = torch.func.vmap(lambda row: ops.linear(row, w))(x.view(10, 64))
    assert torch.equal(mapped, torch.func.vmap(lambda row: F.linear(row, w))(x.view(10, 64)))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        tangent = torch.autograd.forward_ad.unpack_dual(ops.linear(dual, w)).tangent
    assert torch.equal(tangent, F.linear(torch.ones_like(x), w))
    with pytest.raises(RuntimeError):
        ops.linear(x[..., :32], w)
    with pytest.raises(RuntimeError):
        ops.linear(x[0, 0, 0], w)
    assert launches == []


def test_modules_take_the_kernel_and_keep_their_hooks(dev, launches):
    torch.manual_seed(5)
    cfg = drafter.drafter_config(hidden_size=64, num_attention_heads=2, intermediate_size=96)
    mlp = drafter.FlashMapMLP(cfg).bfloat16().to(dev)
    x = torch.randn(16, 64, device=dev).bfloat16()
    with torch.no_grad():
        want = F.linear(F.gelu(F.linear(x, mlp.fc1.weight, mlp.fc1.bias)), mlp.fc2.weight, mlp.fc2.bias)
        got = mlp(x)
        assert launches == ["fm_linear_rows"] * 2
        # two bf16 roundings (2^-8 each) between sums in another order
        assert float((got.double() - want.double()).norm() / want.double().norm()) < 2 ** -7
        launches.clear()
        torch._dynamo.reset()
        assert torch.equal(torch.compile(mlp, fullgraph=True, backend="eager")(x), want)
        assert torch.equal(torch.jit.trace(mlp, x, check_trace=False)(x), want)
        assert launches == []
        plain = drafter.FlashMapMLP(cfg).bfloat16().to(dev)
        plain.load_state_dict(mlp.state_dict())
        weight = plain.fc1.weight.detach()
        del plain.fc1.weight
        plain.fc1.weight = weight  # no parameter any more
        launches.clear()
        assert plain(x).shape == want.shape and launches == ["fm_linear_rows"]  # fc2's
        launches.clear()
        seen = []
        mlp.fc1.register_forward_hook(lambda m, args, out: seen.append(out))
        hooked = mlp(x)
        assert len(seen) == 1 and launches == ["fm_linear_rows"]  # fc2's
        assert torch.equal(hooked, ops.linear(F.gelu(seen[0]), mlp.fc2.weight, mlp.fc2.bias))
    launches.clear()
    mlp(x).float().sum().backward()
    assert mlp.fc1.weight.grad is not None and launches == []
