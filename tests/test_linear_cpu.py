"""``ops.linear`` off the GPU: torch's Linear, bit for bit and with its errors, and the rule
that sends a call to the kernel on one."""

import pytest
import torch
import torch.nn.functional as F

from flashmap_amd import ops


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
                                            (17, 4096, 2048, True), (17, 6144, 2048, False), (33, 64, 64, False),
                                            (4, 64, 48, False), (4, 0, 64, False)])
def test_rule(rows, n, k, takes):
    assert ops._linear_streams(rows, n, k) is takes
