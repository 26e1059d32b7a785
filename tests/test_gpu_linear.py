"""The few-row projection kernel (fm_linear_rows) against float64: every row count of its
two row blocks' edges, output widths that end inside a 16-row tile and on both sides of the
8 / 16 wavefront rule, reductions that leave some wavefronts without a step or with a
partial group; strided weights; and what keeps a call on torch's Linear."""

import pytest
import torch
import torch.nn.functional as F

from _inputs import gen
from flashmap_amd import ops

pytestmark = pytest.mark.gpu


def _bound(x, w, bias, ref):
    """Per element: the sum of k products in fp32 in any order (k 2^-24 of the absolute
    sum, twice for the bias and the partials' order) and the rounding to bf16 (2^-8)."""
    total = x.double().abs() @ w.double().abs().T + (0 if bias is None else bias.double().abs())
    return 2 * x.shape[-1] * 2.0 ** -24 * total + 2.0 ** -8 * ref.abs()


@pytest.mark.parametrize("rows,n,k", [(1, 1, 32), (16, 100, 64), (15, 17, 1376), (16, 4097, 2048), (16, 8192, 2048),
                                      (16, 2048, 4096), (17, 2048, 2048), (32, 4096, 1056), (31, 33, 544)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_linear_rows(dev, rows, n, k, with_bias):
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
        assert got.shape == (rows, n) and got.dtype == torch.bfloat16
        assert ((got.double() - ref).abs() <= _bound(x, w, bias, ref)).all()


def test_leading_dimensions_and_fallbacks(dev):
    g = gen(3)
    x = torch.randn(2, 5, 64, generator=g).bfloat16().to(dev)
    w = torch.randn(48, 64, generator=g).bfloat16().to(dev)
    got = ops.linear(x, w)
    assert got.shape == (2, 5, 48)
    assert torch.equal(got.view(10, 48), ops.linear(x.view(10, 64), w))
    # gradients, other types and strided rows go to torch, with its results
    wp = w.clone().requires_grad_(True)
    ops.linear(x, wp).float().sum().backward()
    ref = w.clone().requires_grad_(True)
    F.linear(x, ref).float().sum().backward()
    assert torch.equal(wp.grad, ref.grad)
    assert torch.equal(ops.linear(x.float(), w.float()), F.linear(x.float(), w.float()))
    strided = torch.randn(10, 128, generator=g).bfloat16().to(dev)[:, ::2]
    assert torch.equal(ops.linear(strided, w), F.linear(strided, w))
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w).dtype == torch.float16
    with torch.no_grad():
        mapped = torch.func.vmap(lambda row: ops.linear(row, w))(x.view(10, 64))
    assert torch.equal(mapped, torch.func.vmap(lambda row: F.linear(row, w))(x.view(10, 64)))
    with pytest.raises(RuntimeError):
        ops.linear(x[..., :32], w)
