"""hy_sample (csrc/sample.hip) against the sort-based path of sample_batch, which
32-bit copies of the same logits take, on the same generator state: the same
draws, since the noise and the order of p / q are the same.

Where a top-p cut falls within rounding of a token's mass the two may keep one
token more or less (sums of up to 151,936 fp32 terms in another order: below
1e-5 of the mass), and small vocabularies are sorted by an unstable sort, which
splits equal scores at the cut differently. So a differing row is accepted
if both tokens are kept by a float64 cut with that slack.
"""

import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from hayate_amd import _native
    from hayate_amd.sampler import sample_batch

DEV = "cuda"
SETTINGS = [(0.0, None, None), (1.0, None, None), (0.7, 1, None), (0.7, 20, None),
            (1.3, 50, 0.8), (1.0, None, 0.05), (0.6, None, 0.5), (1.0, None, 0.95),
            (2.0, 10_000_000, 0.999), (0.3, None, 1.0), (1.0, "half", 0.9), (5.0, "all", None)]


def settings(vocab):
    fix = {"half": vocab // 2 + 1, "all": vocab}
    return [(t, fix.get(k, k), p) for t, k, p in SETTINGS]


def kept(row, t, k, p, token, slack=1e-5):
    x = row.double()
    s = x / t
    if k is not None and k < x.numel() and x[token] < torch.topk(x, k).values[-1]:
        return False
    if k is not None and k < x.numel():
        s = s.masked_fill(x < torch.topk(x, k).values[-1], -math.inf)
    mass = torch.softmax(s, 0)
    above = float(mass[x > x[token]].sum())
    return p is None or p >= 1 or above <= p + slack


def check(logits, seed):
    rows = settings(logits.shape[1])
    t, k, p = map(list, zip(*(rows * (logits.shape[0] // len(rows) + 1))[: logits.shape[0]]))
    gens = [torch.Generator(device=DEV).manual_seed(seed) for _ in range(2)]
    a = sample_batch(logits, t, k, p, gens[0])
    b = sample_batch(logits.float(), t, k, p, gens[1])
    assert a.shape == b.shape and a.dtype == b.dtype
    # both consumed the same noise
    assert torch.equal(gens[0].get_state(), gens[1].get_state())
    differ = (a != b).flatten().nonzero().flatten().tolist()
    for r in differ:
        assert t[r] != 0 and p[r] is not None and p[r] < 1
        for token in (int(a[r]), int(b[r])):
            assert kept(logits[r], t[r], k[r], p[r], token), (r, t[r], k[r], p[r], token)
    return len(differ)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("vocab", [1, 2, 9, 1000, 8191, 8193, 32_771, 151_936])
def test_draws_equal_the_sorted_path(vocab, dtype):
    g = torch.Generator(device=DEV).manual_seed(vocab)
    n = 3 * len(SETTINGS)
    wide = (torch.randn(n, vocab + 3, generator=g, device=DEV) * 2.5).to(getattr(torch, dtype))
    logits = wide[:, 1 : vocab + 1]  # rows at any alignment
    differ = sum(check(logits, s) for s in range(3))
    if vocab >= 1000:  # no row of these sits at a rounding decision
        assert differ <= 1


@pytest.mark.parametrize("value", [0.0, -0.0, 3.0, -2.0])
def test_counters_that_overflow(value):
    """More than 65,535 logits of one value: counted again in 32 bits."""
    g = torch.Generator(device=DEV).manual_seed(5)
    x = torch.full((2 * len(SETTINGS), 151_936), value, device=DEV)
    x[:, ::4] = torch.randn(x.shape[0], x.shape[1] // 4, generator=g, device=DEV)
    if value == 0:
        x[:, 1::4] *= -1  # both zeros, one value
    assert check(x.to(torch.bfloat16), 1) <= 1


def test_more_rows_than_a_launch():
    g = torch.Generator(device=DEV).manual_seed(6)
    assert check(torch.randn(150, 4099, generator=g, device=DEV).to(torch.bfloat16), 2) <= 1


def test_masked_and_extreme_rows():
    g = torch.Generator(device=DEV).manual_seed(7)
    x = torch.randn(2 * len(SETTINGS), 5000, generator=g, device=DEV)
    x[:, 2500:] = -math.inf
    check(x.to(torch.bfloat16), 3)
    x = torch.full((len(SETTINGS), 5000), -math.inf, device=DEV)
    x[:, 77] = 1.0
    out = sample_batch(x.to(torch.bfloat16), *map(list, zip(*settings(5000))),
                       torch.Generator(device=DEV).manual_seed(1))
    assert out.flatten().tolist() == [77] * len(SETTINGS)
    # greedy rows: the first of equal values, zeros of either sign, NaN largest
    x = torch.full((3, 300), -1.0, device=DEV)
    x[0, [40, 200]] = 2.0
    x[1, 50], x[1, 60] = -0.0, 0.0
    x[2, 10], x[2, [20, 30]] = 9.0, math.nan
    out = sample_batch(x.to(torch.bfloat16), [0.0] * 3, [None] * 3, [None] * 3)
    assert out.flatten().tolist() == [40, 50, 20]


@pytest.mark.parametrize("p", [5e-324, 1e-50, 7e-46, 1e-38, 1e-30])
def test_smallest_top_p(p):
    """Down to the smallest positive double: the first of the largest logits."""
    g = torch.Generator(device=DEV).manual_seed(9)
    x = torch.randn(4, 3000, generator=g, device=DEV).to(torch.bfloat16)
    x[0, [700, 40, 2999]] = 9.0
    first = (x == x.max(1, keepdim=True).values).int().argmax(1).tolist()
    assert first[0] == 40
    args = [1.0, 0.5, 2.0, 0.0], [None, 50, None, None], [p, p, p, 1e-50]
    out = sample_batch(x, *args, torch.Generator(device=DEV).manual_seed(1))
    assert out.flatten().tolist() == first
    # the sorted path, whose sort may leave equal scores in any order
    out = sample_batch(x.float(), *args, torch.Generator(device=DEV).manual_seed(1))
    assert torch.equal(x.gather(1, out), x.max(1, keepdim=True).values)


@pytest.mark.parametrize("t", [1e-30, 1e-20, 1e-9, 1e-8, 1e-7, 1e-4, 1e4, 1e30])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_small_and_large_temperatures(t, dtype):
    """Scores of up to 4e31: ties at the maximum are cut by index as at any
    temperature. Below 1e-4 the maximum has all the mass (its neighbour is 1/64
    of it away or more, 150 in the exponent), in equal parts."""
    g = torch.Generator(device=DEV).manual_seed(11)
    for top in (4.0, 17.25, 40.0):
        x = (torch.rand(8, 20_000, generator=g, device=DEV) * 3.5).to(getattr(torch, dtype))
        ties = [5, 800, 801, 9000, 19_999]
        x[:, ties] = top
        p = [0.1, 0.3, 0.39, 0.5, 0.7, 0.81, 0.99, 1.0]
        seen = [set() for _ in p]
        for seed in range(60):
            out = sample_batch(x, [t] * 8, [None] * 8, p,
                               torch.Generator(device=DEV).manual_seed(seed))
            for s, i in zip(seen, out.flatten().tolist()):
                s.add(i)
        if t <= 1e-4:
            # logit j of the five stays while the mass before it, j / 5, is within p
            want = [set(ties[: 1 + sum(j / 5 <= q for j in range(1, 5))]) for q in p]
            assert seen == want, (t, top)
        if t < 1e4:  # (beyond, all logits weigh the same, which the rounding of
            check(x, 1)  # 20,000 sums moves the cuts of)


@pytest.mark.parametrize("n,vocab,native", [
    (1, 9, 0), (1, 65_536, 1), (1, 131_072, 1), (1, 131_073, 0), (2, 65_535, 0), (46, 65_536, 1),
    (47, 65_536, 0), (108, 151_936, 1), (109, 151_936, 0), (300, 1000, 0)])
def test_greedy_batches(n, vocab, native, monkeypatch):
    """All rows greedy, on both sides of the line between hy_sample and argmax; one
    row with a temperature and the whole batch is hy_sample's."""
    from hayate_amd import sampler

    used = []
    real = sampler._sample_native
    monkeypatch.setattr(sampler, "_sample_native", lambda *a: (used.append(1), real(*a))[1])
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(n, vocab, generator=g, device=DEV).to(torch.bfloat16)
    x[:, vocab // 2], x[0, 3] = 9.0, math.nan
    want = [3] + [vocab // 2] * (n - 1)
    out = sample_batch(x, [0.0] * n, [None] * n, [0.5] * n)
    assert out.flatten().tolist() == want and len(used) == native
    x[0, 3] = 0.0
    out = sample_batch(x, [1.0] + [0.0] * (n - 1), [1] + [None] * (n - 1), [None] * n,
                       torch.Generator(device=DEV).manual_seed(1))
    assert out.flatten().tolist() == [vocab // 2] * n and len(used) == native + 1


def test_parameter_types():
    """Settings held in tensors and arrays as in Python numbers; a fractional
    top_k is refused for 16-bit logits as for 32-bit ones."""
    g = torch.Generator(device=DEV).manual_seed(10)
    x = torch.randn(3, 3000, generator=g, device=DEV).to(torch.bfloat16)

    def draw(t, k, p):
        return sample_batch(x, t, k, p, torch.Generator(device=DEV).manual_seed(2)).tolist()

    want = draw([0.5, 0.0, 2.0], [20, None, 7], [0.75, None, 0.5])
    temp, p = torch.tensor([0.5, 0.0, 2.0]), torch.tensor([0.75, 1.0, 0.5])
    for dev in ("cpu", DEV):
        assert draw(temp.to(dev), [20, None, 7], p.to(dev)) == want
        assert draw(list(temp.to(dev)), [20, None, torch.tensor(7, device=dev)], list(p)) == want
    assert draw(temp.numpy(), np.array([20, 3000, 7]), p.numpy()) == want
    for logits in (x, x.float()):
        with pytest.raises((RuntimeError, TypeError)):
            sample_batch(logits, [0.5, 0.0, 2.0], [20.5, None, 7], [None] * 3)


def test_rows_without_a_distribution_are_reported():
    """*valid through the C ABI: a NaN, only -inf, +inf; sample_batch turns it
    into an error as torch.multinomial does."""
    lib = _native.lib()

    def valid(fill):
        x = torch.randn(2, 600, device=DEV).to(torch.bfloat16)
        fill(x)
        t, k, p = (torch.tensor(v) for v in ([0.0, 1.0], [600, 600], [1.0, 0.5]))
        k = k.int()
        noise = torch.rand(1, 600, device=DEV) + 0.1
        out = torch.empty(2, dtype=torch.long, device=DEV)
        ok = torch.empty((), dtype=torch.bool, device=DEV)
        work = torch.empty(lib.hy_sample_workspace_bytes(2, 600), dtype=torch.uint8, device=DEV)
        _native.check(lib.hy_sample(x.data_ptr(), 600, 0, 2, 600, t.data_ptr(), k.data_ptr(),
                                    p.data_ptr(), noise.data_ptr(), out.data_ptr(), ok.data_ptr(),
                                    work.data_ptr(), work.numel(),
                                    torch.cuda.current_stream().cuda_stream), "hy_sample")
        return bool(ok)

    assert valid(lambda x: None)
    assert valid(lambda x: x[0].fill_(math.nan))  # the greedy row
    assert valid(lambda x: x[1, 3:].fill_(-math.inf))
    assert not valid(lambda x: x[1, 5].fill_(math.nan))
    assert not valid(lambda x: x[1].fill_(-math.inf))
    assert not valid(lambda x: x[1, 9].fill_(math.inf))
