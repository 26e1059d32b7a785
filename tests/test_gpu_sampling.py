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


# Rows, vocabulary and row stride of every way a call is taken, well inside each: one wavefront
# per row, 256 threads over a short row and over single tiles, 512 threads over two tiles, and
# 1024 over a whole row (for 2-byte logits; float32 takes 256 throughout); the last two pairs
# once with 16-byte-aligned rows and once without.
_PLANS = [(5000, 1003, 1003), (4096, 2041, 2048), (70, 2041, 2041), (60, 8200, 8200), (30, 50001, 50008),
          (800, 66000, 66000), (700, 98309, 98309), (1024, 65544, 65544), (1024, 98309, 98309)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,vocab,stride", _PLANS)
def test_sample_rows_tiles_and_parts(dev, dtype, rows, vocab, stride):
    """Greedy and sampled rows in one call whose winners, ties, NaN, infinities and -inf
    stretches lie in the first, a later and the last tile: greedy rows exactly, sampled rows
    of every kind the token that the noise of every logit selects."""
    print(f"sample rows={rows} vocab={vocab} stride={stride} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(rows + vocab)
    x = torch.randn(rows, stride, generator=g, device=dev).to(dtype)
    temps = 0.6 + 0.6 * torch.rand(rows, generator=g, device=dev)
    late, mid, last = vocab - vocab // 8, vocab // 2 + 3, vocab - 1
    kinds = 10
    for r in [k + part for k in range(kinds) for part in (0, rows // 3 // kinds * kinds, rows // 2 // kinds * kinds)]:
        k = r % kinds
        if k == 1:  # the largest far on, twice: the first wins if greedy
            x[r, late], x[r, last] = 20.0, 20.0
        elif k == 2:
            x[r, 1], x[r, mid] = 20.0, 20.0
        elif k == 3:
            x[r] = 0.5  # all equal
        elif k == 4:
            x[r] = -torch.inf
        elif k == 5:
            x[r, :late] = -torch.inf  # nothing before the last part
        elif k == 6:
            x[r, mid:] = -torch.inf
        elif k == 7:
            x[r, late], x[r, last] = torch.nan, torch.nan
        elif k == 8:
            x[r, mid] = torch.inf
        elif k == 9:
            temps[r] = 40.0
    pick = torch.arange(rows, device=dev)
    greedy = (pick // kinds) % 2 == 1
    x[:, vocab:] = 30000.0  # what lies between the rows is no logit
    seed = 0x7_1234_5678
    x = x[:, :vocab]
    got = ops.sample_rows(x, temps, greedy, torch.tensor(seed, device=dev)).cpu()
    assert int(got.min()) >= 0 and int(got.max()) < vocab
    want = torch.from_numpy(S.argmax_first(x[greedy].float().cpu().numpy()))
    assert torch.equal(got[greedy.cpu()], want)
    for r in [r for r in list(range(kinds)) + list(range(rows - 20, rows)) if not greedy[r]]:
        row = x[r:r + 1].cpu()
        keys = _all_keys(row, temps[r:r + 1].cpu(), seed, row0=r)[0]
        best, won = S.argmax_first(keys[None])[0], int(got[r])
        if np.isnan(keys).any() or not np.isfinite(keys[best]):
            assert won == best, (r, won, best)
        else:  # as in test_sample_rows_skips_only_losers
            assert keys[won] >= keys[best] - 1e-5 - 4 * 2.0 ** -23 * abs(keys[best]), (r, won, best)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_sample_rows_any_alignment(dev, dtype):
    """Rows that begin at every place of a 16-byte granule and end at every place of one,
    between values that would win: sampled rows exactly the oracle's (its clear winners),
    greedy rows its argmax, rows of -inf the first index."""
    g = gen(11)
    for vocab in (1, 2, 7, 8, 9, 63, 2040, 2041, 2047, 2048, 2049, 8191, 8192, 8193, 16385):
        for offset in range(8):
            rows, stride = 4, vocab + 3
            buf = torch.full((rows * stride + 16,), 30000.0).to(dtype)
            view = buf[offset:offset + rows * stride].view(rows, stride)
            logits = torch.randn(rows, vocab, generator=g).to(dtype)
            logits[3] = -torch.inf
            view[:, :vocab] = logits
            d = buf.to(dev)
            x = torch.as_strided(d, (rows, vocab), (stride, 1), offset)
            temps = 0.3 + torch.rand(rows, generator=g)
            greedy = torch.tensor([False, True, False, offset % 2 == 0])
            got = ops.sample_rows(x, temps.to(dev), greedy.to(dev), torch.tensor(99, device=dev)).cpu()
            keys = S.sample_keys(logits.float().numpy(), temps.numpy(), greedy.numpy(), 99)
            want = S.argmax_first(keys)
            for r in range(rows):
                clear = vocab == 1 or r == 3 or np.diff(np.sort(keys[r])[-2:])[0] > 1e-4 or greedy[r]
                assert not clear or int(got[r]) == want[r], (vocab, offset, r)


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
