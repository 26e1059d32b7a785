"""The several-jump draft's state kernels (fm_state_embed_rows, fm_state_update;
flashmap/vllm/model.py:944-956 and 1031-1036) against the same formulas in float64 on
the CPU: the posterior softmax(evidence * state) and the state rounded to bf16, every
element within one bf16 ulp of the correctly rounded float64 value (and almost all equal
to it); the updated state ((1 - end) state + (end - start) softmax(logits)) / (1 - start)
within 1e-5 relative of the float64 value (the sum of up to 151936 exponentials in
float32). Row widths with a tail (not a multiple
of 4), the 151936-token vocabulary, strided rows, and the wrappers' checks."""

import pytest
import torch

from _inputs import gen
from flashmap_amd import ops

pytestmark = pytest.mark.gpu


def _bf16_ulps(got, want64):
    """|got - want| in units of the bf16 ulp at want (float64 reference)."""
    w = want64.float()
    ulp = torch.where(w == 0, torch.full_like(w, 2.0 ** -133),
                      2.0 ** (torch.floor(torch.log2(w.abs().clamp_min(1e-38))) - 7))
    return ((got.double() - want64).abs() / ulp.double())


def _state(rows, vocab, g, scale=3.0):
    return (scale * torch.randn(rows, vocab, generator=g)).float()


def _rows(x, dev):
    """x on the device in rows padded to a multiple of 4 values (the kernels' layout)."""
    buf = torch.zeros(x.shape[0], -(-x.shape[1] // 4) * 4, dtype=x.dtype, device=dev)
    return buf[:, :x.shape[1]].copy_(x)


@pytest.mark.parametrize("rows,vocab,evidence", [(3, 200, 0.0), (17, 1003, 1.7), (64, 4096, 0.4),
                                                 (16, 151936, 2.5)])
def test_state_embed_rows(dev, rows, vocab, evidence):
    print(f"state_embed_rows rows={rows} vocab={vocab} evidence={evidence}", flush=True)
    g = gen(rows + vocab)
    state = _state(rows, vocab, g)
    got = ops.state_embed_rows(_rows(state, dev), evidence).cpu()
    post64 = torch.softmax(state.double() * evidence, dim=-1)
    ulps = _bf16_ulps(got[:rows], post64)
    exact = float((got[:rows].double() == post64.bfloat16().double()).float().mean())
    print(f"  posterior: max {float(ulps.max()):.3f} bf16 ulps, {exact:.4f} equal to the rounded float64", flush=True)
    assert float(ulps.max()) <= 1.0 and exact >= 0.99
    assert torch.equal(got[rows:], state.bfloat16()), "the state rows are the state rounded to bf16"
    assert torch.allclose(got[:rows].double().sum(-1), torch.ones(rows, dtype=torch.float64), atol=0.02)
    alone = ops.state_embed_rows(_rows(state, dev), evidence, posterior=False).cpu()
    assert torch.equal(alone, state.bfloat16()), "posterior=False: the state rows alone"


@pytest.mark.parametrize("rows,vocab,start,end", [(3, 200, 0.0, 0.5), (17, 1003, 0.25, 0.75),
                                                  (64, 4096, 0.5, 1.0), (16, 151936, 0.1, 0.6)])
def test_state_update(dev, rows, vocab, start, end):
    print(f"state_update rows={rows} vocab={vocab} start={start} end={end}", flush=True)
    g = gen(7 * rows + vocab)
    state = torch.softmax(_state(rows, vocab, g), dim=-1)  # a distribution, as between jumps
    logits = (2 * torch.randn(rows, vocab, generator=g)).bfloat16()
    s_dev = _rows(state, dev)
    out = ops.state_update(s_dev, logits.to(dev), start, end)
    assert out.data_ptr() == s_dev.data_ptr(), "in place"
    want = ((1.0 - end) * state.double() + (end - start) * torch.softmax(logits.double(), -1)) / (1.0 - start)
    rel = ((out.cpu().double() - want).abs() / want.abs().clamp_min(1e-30))
    print(f"  max relative error {float(rel.max()):.3e}", flush=True)
    # float32 with the sum of up to 151936 exponentials in another order: ~1e-6 typical
    assert float(rel.max()) <= 1e-5
    assert torch.allclose(out.cpu().double().sum(-1), torch.ones(rows, dtype=torch.float64), atol=1e-4)


@pytest.mark.parametrize("evidence", [1e3, 1e5, 1e6, -1e3])
def test_posterior_at_large_evidence(dev, evidence):
    """Products of up to 5e6, whose float32 rounding is up to a quarter: the posterior is that
    of the exact products all the same, and adds up to 1."""
    rows, vocab = 70, 5003
    g = gen(int(abs(evidence)))
    state = torch.randn(rows, vocab, generator=g)
    peak = 4.5 if evidence > 0 else -4.5
    state[:, 17] = peak + 0.1 * torch.rand(rows, generator=g)
    state[:, 4999] = state[:, 17] - torch.rand(rows, generator=g) * 2 / evidence  # within two of it
    got = ops.state_embed_rows(_rows(state, dev), evidence).cpu()[:rows].double()
    want = torch.softmax(state.double() * evidence, dim=-1)
    # an exponent's one float32 rounding and the exponential's are below 1e-4 of the value at
    # exponents of -100 and more; then bf16's half ulp, 2^-8 of the value at most
    seen = want > 1e-40
    assert float(((got - want).abs() / want)[seen].max()) <= 2.0 ** -8
    assert float(got.max()) <= 1.0 and float((got.sum(-1) - 1).abs().max()) <= 2.0 ** -8


def test_subnormal_probabilities(dev):
    """Exponents around -87.3 to -104, whose float32 exponentials are subnormal: the posterior
    keeps what bf16 has of them (steps of 2^-133), the update what float32 has (2^-149)."""
    vocab = 4099
    x = torch.linspace(-104.0, -80.0, vocab).repeat(2, 1)
    x[:, 7] = 0.0
    got = ops.state_embed_rows(_rows(x, dev), 1.0).cpu()[:2].double()
    want = torch.softmax(x.double(), dim=-1)
    assert int(((want < 2.0 ** -126) & (want > 2.0 ** -133)).sum()) > 1000
    # float32's own rounding of the quotient, then half of bf16's step or of its value's ulp
    assert ((got - want).abs() <= 2.0 ** -149 + 2.0 ** -134 + 2.0 ** -8 * want).all()
    logits = x.bfloat16()
    d64 = torch.softmax(logits.double(), dim=-1)
    state = _rows(torch.zeros(2, vocab), dev)
    out = ops.state_update(state, _rows(logits, dev), 0.0, 0.5).cpu().double()
    # two roundings at 2^-149, and 1e-6 of the value as in test_state_update
    assert ((out - 0.5 * d64).abs() <= 2.0 ** -148 + 1e-6 * d64).all()


@pytest.mark.parametrize("vocab", [1003, 16385, 32770, 49157, 151936])
def test_rows_do_not_depend_on_the_others(dev, vocab):
    """A row's values bit for bit, whether the call has 1, 16, 64, 100 or 300 rows (eight to
    one workgroups a row)."""
    print(f"state rows alone and together vocab={vocab}", flush=True)
    g = torch.Generator(device=dev).manual_seed(vocab)
    state = _rows(torch.randn(300, vocab, generator=g, device=dev), dev)
    logits = _rows(2 * torch.randn(300, vocab, generator=g, device=dev, dtype=torch.bfloat16), dev)
    whole = ops.state_embed_rows(state, 3.0)
    moved = ops.state_update(_rows(state, dev), logits, 0.2, 0.7)
    for rows in (1, 16, 64, 100):
        part = ops.state_embed_rows(state[:rows], 3.0)
        assert torch.equal(part[:rows], whole[:rows]), (rows, "posterior")
        assert torch.equal(part[rows:], whole[300:300 + rows]), (rows, "state")
        assert torch.equal(ops.state_update(_rows(state[:rows], dev), logits[:rows], 0.2, 0.7), moved[:rows]), rows


def test_state_kernels_strided_rows(dev):
    """Rows inside a wider buffer (the draft step's padded state), and the state update
    against torch's float32 expression on the same device."""
    g = gen(99)
    base = torch.zeros(8, 1008, device=dev)
    state = base[:, :1001]
    state.copy_(torch.softmax(_state(8, 1001, g), -1).to(dev))
    logits = torch.randn(8, 1001, generator=g).bfloat16().to(dev)
    want = ((1.0 - 0.8) * state + (0.8 - 0.3) * logits.float().softmax(-1)) / (1.0 - 0.3)
    ops.state_update(state, logits, 0.3, 0.8)
    assert torch.allclose(state, want, rtol=1e-6, atol=0)
    assert torch.count_nonzero(base[:, 1001:]) == 0, "the padding is left alone"
    both = ops.state_embed_rows(state, 1.0)
    assert both.shape == (16, 1001) and torch.equal(both[8:], state.bfloat16())


def test_state_wrapper_checks(dev):
    with pytest.raises(ValueError, match="float32"):
        ops.state_embed_rows(torch.zeros(2, 8, dtype=torch.bfloat16, device=dev), 1.0)
    with pytest.raises(ValueError, match="row stride"):
        ops.state_embed_rows(torch.zeros(2, 9, device=dev)[:, :5], 1.0)
    with pytest.raises(ValueError, match="jump times"):
        ops.state_update(torch.zeros(2, 8, device=dev), torch.zeros(2, 8, dtype=torch.bfloat16, device=dev), 1.0, 1.0)
    with pytest.raises(ValueError, match="logits must be bf16"):
        ops.state_update(torch.zeros(2, 8, device=dev), torch.zeros(2, 8, device=dev), 0.0, 0.5)


# rows: 1 and 3 take eight workgroups a row, 64 four, 100 and 128 two, 200 and 300 one; vocab:
# less than a chunk per thread, both sides of the lines between 256, 512 and 1024 threads, around
# what a workgroup keeps in registers (32 values a thread) and the chunks of a step, remainders
# of 1 to 3; (64, 151936) and (100, 131075) read parts of split rows again; the last ones are past
# the size whose accesses are non-temporal, at 1024, 512 and 256 threads.
_EDGES = [(r, v) for r in (1, 3, 128, 200, 300)
          for v in (1, 5, 4099, 8193, 12288, 12291, 32767, 32770, 40960, 40961, 49156)]
_EDGES += [(64, 151936), (100, 131075), (520, 131075), (2100, 32001), (16500, 4099)]


@pytest.mark.parametrize("rows,vocab", _EDGES)
def test_state_kernels_edges(dev, rows, vocab):
    """Masked values (-inf, the lowest finite value), +inf and NaN as torch's softmax takes
    them, and the sizes where a row's workgroups and passes change."""
    print(f"state edges rows={rows} vocab={vocab}", flush=True)
    g = torch.Generator(device=dev).manual_seed(rows * 100003 + vocab)
    state = _rows(torch.randn(rows, vocab, generator=g, device=dev), dev)
    logits = _rows(2 * torch.randn(rows, vocab, generator=g, device=dev, dtype=torch.bfloat16), dev)
    lowest = torch.finfo(torch.bfloat16).min
    for t in (state, logits):
        t[0, ::2] = -torch.inf if vocab > 1 else 0.0
        if rows > 1:
            t[1] = lowest
        if rows > 2:
            t[2] = -torch.inf
        if rows > 4:
            t[3, vocab // 2], t[4, vocab - 1] = torch.inf, torch.nan
    before = state.double()
    post = torch.softmax((1.5 * state).double(), -1)
    both = ops.state_embed_rows(state, 1.5)
    # float32 exponentials and sums to about 1e-6, then bf16: an ulp is 2^-8 of the value, and
    # 2^-133 below its normal range
    assert torch.allclose(both[:rows].double(), post, rtol=2.0 ** -8, atol=2.0 ** -133, equal_nan=True)
    assert torch.equal(both[rows:].view(torch.int16), state.bfloat16().view(torch.int16))
    alone = ops.state_embed_rows(state, 1.5, posterior=False)
    assert torch.equal(alone.view(torch.int16), state.bfloat16().view(torch.int16))
    want = (0.4 * before + 0.3 * torch.softmax(logits.double(), -1)) / 0.7
    out = ops.state_update(state, logits, 0.3, 0.6).double()
    big = want.abs() > 1e38  # beyond float32 on the way to the quotient
    assert torch.allclose(torch.where(big, 0.0, out), torch.where(big, 0.0, want), rtol=2e-5, atol=2e-6,
                          equal_nan=True)
    assert torch.equal(out[big].sign(), want[big].sign())


def test_more_rows_than_a_grid_counts_threads_for(dev):
    """Short rows by the million: 2^22 + 5 workgroups of 1024 threads were past the 2^32 threads
    that a launch counts, and the last rows stayed unwritten, with no error."""
    rows, vocab = (1 << 22) + 5, 3
    g = torch.Generator(device=dev).manual_seed(5)
    state = _rows(torch.randn(rows, vocab, generator=g, device=dev), dev)
    logits = _rows(torch.randn(rows, vocab, generator=g, device=dev, dtype=torch.bfloat16), dev)
    both = ops.state_embed_rows(state, 1.5)
    post = torch.softmax(1.5 * state.double(), -1)
    assert torch.allclose(both[:rows].double(), post, rtol=2.0 ** -8, atol=0)
    assert torch.equal(both[rows:], state.bfloat16())
    assert torch.equal(ops.state_embed_rows(state, 1.5, posterior=False), state.bfloat16())
    want = (0.4 * state.double() + 0.3 * torch.softmax(logits.double(), -1)) / 0.7
    out = ops.state_update(state, logits, 0.3, 0.6).double()
    assert torch.allclose(out, want, rtol=2e-6, atol=1e-6)
