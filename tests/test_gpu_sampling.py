"""GPU parity of the draft step's token selection and noise (csrc/sampling.hip) through
the C ABI, against the CPU oracle (oracle/sampling.py):

- argmax per row: exact (int64 indices) for bf16 / fp16 / fp32 logits, ties to the first
  index, all -inf rows, NaN rows, strided rows, vocabularies that end mid-chunk or on a
  whole number of tiles, a 151936-entry vocabulary;
- the fused sampler: greedy rows exact; sampled rows equal the oracle's tokens wherever
  the oracle's winning key beats the runner-up by more than 1e-4 (the random words are
  exact, the logs may differ in the last ulp); int32 offset wraparound past 2^31;
- seeded normals: within 2e-5 (relative, at least 1 absolute unit) of the oracle, for
  int32 and int64 rows / positions, unseeded rows, seeds with high words.
"""

import numpy as np
import pytest
import torch

from _inputs import gen
from flashmap_amd import ops
from oracle import sampling as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,vocab,stride", [(1, 1, 1), (3, 100, 100), (17, 8193, 8200), (5, 24581, 24581),
                                               (3, 32768, 32768), (64, 151936, 151936)])
def test_argmax_rows(dev, dtype, rows, vocab, stride):
    g = gen(rows + vocab)
    x = torch.randn(rows, stride, generator=g).to(dtype)[:, :vocab]
    if vocab > 10:  # planted ties: the row max at three places, the first must win
        m = x.float().max(dim=1).values + 1
        for r in range(rows):
            cols = torch.randperm(vocab, generator=g)[:3]
            x[r, cols] = m[r].to(dtype)
    got = ops.argmax_rows(x.to(dev))
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), torch.from_numpy(S.argmax_first(x.float().numpy())))
    assert torch.equal(got.cpu(), x.float().argmax(dim=1))


def test_argmax_special_rows(dev):
    x = torch.randn(4, 20000).bfloat16()
    x[0] = -float("inf")
    x[1, 777] = float("nan")
    x[1, 19999] = float("nan")
    x[2] = 0
    x[3, 12345] = float("inf")
    got = ops.argmax_rows(x.to(dev)).cpu()
    assert got.tolist() == [0, 777, 0, 12345]


def test_sample_rows(dev):
    g = gen(5)
    rows, vocab = 40, 50000
    x = (torch.randn(rows, vocab, generator=g) * 3).bfloat16()
    temps = torch.rand(rows, generator=g) + 0.3
    greedy = torch.zeros(rows, dtype=torch.bool)
    greedy[::3] = True
    seed = torch.tensor(0x1234_5678_9ABC, dtype=torch.int64)
    got = ops.sample_rows(x.to(dev), temps.to(dev), greedy.to(dev), seed.to(dev)).cpu().numpy()
    keys = S.sample_keys(x.float().numpy(), temps.numpy(), greedy.numpy(), int(seed))
    want = S.argmax_first(keys)
    gr = greedy.numpy()
    assert (got[gr] == want[gr]).all()
    top2 = np.sort(keys[~gr], axis=1)[:, -2:]
    clear = (top2[:, 1] - top2[:, 0]) > 1e-4
    assert clear.sum() >= (~gr).sum() - 2
    assert (got[~gr][clear] == want[~gr][clear]).all()
    # the sampled rows are not the argmax (noise applied) for most rows
    assert (got[~gr] != x.float().argmax(1).numpy()[~gr]).mean() > 0.5


def _all_keys(x, temps, seed, row0=0):
    """Every logit's key, none skipped."""
    return S.sample_keys(x.float().numpy(), temps.numpy(), np.zeros(len(x), dtype=bool), seed, row0=row0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,vocab,stride", [(1, 1, 1), (2, 7, 8), (3, 100, 100), (5, 8191, 8192), (4, 8193, 8200),
                                               (3, 24581, 24581), (150, 49153, 49160)])
def test_sample_rows_skips_only_losers(dev, dtype, rows, vocab, stride):
    """Rows whose logits are flat (every one can win), peaked, far from zero, mostly -inf or
    steps of about the bound (17 T), at temperatures on both sides of its range: each
    sampled token is the one that the noise of every logit selects."""
    g = gen(rows + vocab)
    x = torch.randn(rows, stride, generator=g)
    temps = 0.3 + torch.rand(rows, generator=g)
    kinds = torch.arange(rows) % 6
    x[kinds == 0] *= 0.1
    x[kinds == 1, :1] += 30.0
    x[kinds == 2] = x[kinds == 2] * 3 - 1000.0
    x[kinds == 3] = torch.where(x[kinds == 3] > 1.0, x[kinds == 3], -float("inf"))
    steps = torch.randint(0, 3, (int((kinds == 4).sum()), stride), generator=g)
    x[kinds == 4] = 17.0 * temps[kinds == 4, None] * steps
    temps[kinds == 5] = 50.0
    x = x.to(dtype)[:, :vocab]
    seed = 0x9_8765_4321
    got = ops.sample_rows(x.to(dev), temps.to(dev), torch.zeros(rows, dtype=torch.bool, device=dev),
                          torch.tensor(seed, device=dev)).cpu().numpy()
    keys = _all_keys(x, temps, seed)
    # A key rounds to float32 twice and its logs are within about two ulps each: the
    # winner's key lies that close to the largest of all.
    won = keys[np.arange(rows), got]
    best = keys.max(axis=1)
    slack = 1e-5 + 4 * 2.0 ** -23 * np.where(np.isfinite(best), np.abs(best), 0)
    assert ((won >= best - slack) | (won == best)).all()


def test_sample_rows_special_rows(dev):
    vocab = 30000
    x = torch.randn(6, vocab).bfloat16()
    x[0] = -float("inf")  # every key -inf: the first index
    x[1, 20000] = float("nan")
    x[1, 29999] = float("nan")
    x[2, 12345] = float("inf")
    temps = torch.tensor([1.0, 1.0, 1.0, 1e-35, 1e35, 1.0])  # rows 3, 4: outside the bound's range
    x[3, 777] = 20.0  # over 1e-35: +inf is the largest key and the first of them wins
    x[3, :777] = -1.0
    x[3, 778:] = -1.0
    greedy = torch.zeros(6, dtype=torch.bool)
    greedy[5] = True
    seed = torch.tensor(5, dtype=torch.int64)
    got = ops.sample_rows(x.to(dev), temps.to(dev), greedy.to(dev), seed.to(dev)).cpu()
    assert got[:4].tolist() == [0, 20000, 12345, 777]
    keys = _all_keys(x[4:5], temps[4:5], 5, row0=4)  # logit / T of about 0: the noise alone
    assert int(got[4]) == int(keys[0].argmax())
    assert int(got[5]) == int(x[5].float().argmax())


def test_sample_rows_offsets_wrap_past_int32(dev):
    """row * V + col passes 2^31 for the last rows: int32 arithmetic, as the reference's."""
    rows, vocab = 300, 7_300_000
    g = torch.Generator(device=dev).manual_seed(6)
    x = torch.randn(rows, vocab, generator=g, device=dev, dtype=torch.bfloat16)
    temps = torch.ones(rows)
    greedy = torch.zeros(rows, dtype=torch.bool)
    seed = torch.tensor(77, dtype=torch.int64)
    got = ops.sample_rows(x, temps.to(dev), greedy.to(dev), seed.to(dev)).cpu().numpy()
    row0 = rows - 3
    assert row0 * vocab > 2 ** 31
    tail = x[row0:].float().cpu().numpy()
    del x
    keys = S.sample_keys(tail, temps[row0:].numpy(), greedy[row0:].numpy(), 77, row0=row0)
    top2 = np.sort(keys, axis=1)[:, -2:]
    clear = (top2[:, 1] - top2[:, 0]) > 1e-4
    assert (got[row0:][clear] == S.argmax_first(keys)[clear]).all()


@pytest.mark.parametrize("idx_dtype", [torch.int32, torch.int64])
def test_seeded_normal(dev, idx_dtype):
    g = gen(7)
    seeds = torch.tensor([3, (1 << 40) + 7, -5, 123456789012345], dtype=torch.int64)
    rows = torch.tensor([0, 1, -1, 2, 3, 3, -2, 1], dtype=idx_dtype)
    pos = torch.randint(0, 10000, (8,), generator=g).to(idx_dtype)
    n_cols = 3000
    got = ops.seeded_normal(seeds.to(dev), rows.to(dev), pos.to(dev), n_cols, 0.7).cpu().numpy()
    want = S.seeded_normal(seeds.numpy(), rows.numpy(), pos.numpy(), n_cols, 0.7)
    err = np.abs(got - want) / np.maximum(1.0, np.abs(want))
    assert err.max() < 2e-5


def test_plugin_entry_points(dev):
    from flashmap_amd import sglang as fs
    from flashmap_amd import vllm as fv

    x = torch.randn(6, 1000).float().to(dev)
    assert torch.equal(fv.split_argmax(x), x.argmax(dim=1))
    seed = torch.tensor(9, dtype=torch.int64, device=dev)
    t = torch.ones(6, device=dev)
    greedy = torch.ones(6, dtype=torch.bool, device=dev)
    assert torch.equal(fs.sample_rows(x, t, greedy, seed), x.argmax(dim=1))
    z = fv.seeded_normal(torch.tensor([1, 2], device=dev), torch.tensor([0, 1], device=dev),
                         torch.tensor([5, 6], device=dev), 10, 2.0)
    assert z.shape == (2, 10) and z.dtype == torch.float32
