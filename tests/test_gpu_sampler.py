"""HIP sampler (sid_sample_rows) vs the exact-rule oracle (oracle/sampler.py
sample_exact_ref), on the reference's test_07 cases and on full-vocabulary rows with
bf16-rounded logits (many exact ties at the top-k / top-p cut), plus its invariants:
batch shape, decode vs verify path, greedy rows, and the empirical distribution."""

from __future__ import annotations

import math

import pytest
import torch

from oracle.sampler import kept_mask_exact, sample_exact_ref, seeded_gumbel_ref

pytestmark = pytest.mark.gpu


def _sample(logits, temps, ks, ps, seeds, pos):
    from sid.engine.sampler import sample
    c = lambda t, dt: torch.as_tensor(t, dtype=dt).cuda()
    return sample(logits.cuda(), c(temps, torch.float32), c(ks, torch.int64), c(ps, torch.float32),
                  c(seeds, torch.int64), c(pos, torch.int64)).cpu()


def _score(logits_row, t, k, p, seed, pos, tok):
    probs = torch.softmax(logits_row.float() / t, dim=-1)
    keep = kept_mask_exact(probs.numpy(), k, p)
    if not keep[tok]:
        return -math.inf
    g = seeded_gumbel_ref(torch.tensor([seed]), torch.tensor([pos]), logits_row.numel())[0]
    return float(torch.log(probs[tok] + 1e-10) + g[tok])


def _check(logits, temps, ks, ps, seeds, pos):
    got = _sample(logits, temps, ks, ps, seeds, pos)
    want = sample_exact_ref(logits, temps, ks, ps, seeds, pos)
    for r in range(logits.shape[0]):
        if got[r] == want[r]:
            continue
        # Only a float near-tie of the final scores may differ (exp/log ulps differ
        # between torch's CPU kernels and the device's): both kept, gap < 1e-4.
        t, k, p, s, q = float(temps[r]), int(ks[r]), float(ps[r]), int(seeds[r]), int(pos[r])
        assert t > 0, (r, got[r], want[r])
        a = _score(logits[r], t, k, p, s, q, int(got[r]))
        b = _score(logits[r], t, k, p, s, q, int(want[r]))
        assert math.isfinite(a) and abs(a - b) < 1e-4, (r, int(got[r]), int(want[r]), a, b)
    return got


def test_greedy_rows_first_index_and_nan():
    logits = torch.zeros(3, 100)
    logits[0, 7] = 5.0
    logits[1, 3] = 2.0
    logits[1, 42] = 2.0
    logits[2, 50] = float("nan")
    logits[2, 60] = float("nan")
    got = _sample(logits, [0.0] * 3, [-1] * 3, [1.0] * 3, [1, 2, 3], [0, 0, 0])
    assert got.tolist() == [7, 3, 50]


def test_reference_known_answer_cases():
    logits = torch.tensor([[10.0, 9.0, 8.0, -20.0, -20.0]])
    for pos in range(64):
        assert _sample(logits, [2.0], [3], [1.0], [5], [pos]).item() in (0, 1, 2)
    peaked = torch.tensor([[10.0, 0.0, 0.0, 0.0, 0.0]])
    for pos in range(32):
        assert _sample(peaked, [1.0], [-1], [0.5], [5], [pos]).item() == 0


@pytest.mark.parametrize("vocab", [151936, 4000, 33])
def test_full_rows_vs_exact_oracle(vocab):
    """bf16-rounded logits (exact duplicates everywhere), every truncation mode."""
    g = torch.Generator().manual_seed(vocab)
    rows = 16
    logits = (torch.randn(rows, vocab, generator=g) * 2.5).to(torch.bfloat16).float()
    temps = [0.0, 0.7, 1.0, 1.5, 0.3, 0.7, 2.0, 0.9] * 2
    ks = [-1, -1, 50, 1, 5, 1000, 40, -1, -1, 3, 200, -1, 10, -1, 2, 64]
    ps = [1.0, 0.9, 1.0, 1.0, 0.8, 0.95, 0.5, 0.0, 0.3, 1.0, 0.99, 0.7, 0.9, 0.6, 1.0, 0.999]
    seeds = [11 * i + 3 for i in range(rows)]
    pos = [100 + 7 * i for i in range(rows)]
    print(f"vocab={vocab}", flush=True)
    _check(logits, temps, ks, ps, seeds, pos)


def test_top_k_boundary_ties_keep_lowest_indices():
    """20 columns share the 3rd-highest value; top_k = 5 keeps the lowest 3 of them."""
    logits = torch.full((1, 300), -30.0)
    logits[0, 10] = 4.0
    logits[0, 20] = 3.0
    tie_cols = list(range(100, 300, 10))
    logits[0, tie_cols] = 2.0
    seen = set()
    for pos in range(400):
        seen.add(_sample(logits, [3.0], [5], [1.0], [9], [pos]).item())
    assert seen <= {10, 20, 100, 110, 120} and {100, 110, 120} <= seen


def test_batch_shape_and_path_invariance():
    torch.manual_seed(0)
    W, seed, base = 32, 777, 250
    logits = torch.randn(W, 151936)
    verify = _sample(logits, [0.7] * W, [50] * W, [0.9] * W, [seed] * W, list(range(base, base + W)))
    for j in (0, 1, W // 2, W - 1):
        dec = _sample(logits[j:j + 1], [0.7], [50], [0.9], [seed], [base + j])
        assert dec.item() == verify[j].item()
    mixed = torch.cat([torch.randn(5, 151936), logits[3:4]])
    out = _sample(mixed, [0.0, 1.0, 0.5, 0.7, 1.2, 0.7], [-1, 3, 9, 50, -1, 50],
                  [1.0, 0.5, 0.9, 0.9, 1.0, 0.9], [1, 2, 3, 4, 5, seed], [9, 8, 7, 6, 5, base + 3])
    assert out[-1].item() == verify[3].item()


def test_positions_draws_equal_oracle_and_respect_top_p():
    """Draws over 2000 positions equal the oracle's token for token. (The reference's hash
    XORs one per-position value with a per-column constant, so the noise of different
    columns is correlated and frequencies over positions need not follow p: equality with
    the oracle, not a frequency test, is what pins the draw.)"""
    probs = torch.tensor([0.5, 0.25, 0.15, 0.10])
    n = 2000
    logits = torch.log(probs).unsqueeze(0).repeat(n, 1)
    args = ([1.0] * n, [-1] * n, [1.0] * n, [42] * n, list(range(n)))
    got = _sample(logits, *args)
    assert torch.equal(got, sample_exact_ref(logits, *args))
    assert len(set(got.tolist())) > 1
    # top_p = 0.6 keeps ranks whose preceding mass <= 0.6: tokens 0 and 1 only
    args = ([1.0] * n, [-1] * n, [0.6] * n, [42] * n, list(range(n)))
    got = _sample(logits, *args)
    assert torch.equal(got, sample_exact_ref(logits, *args))
    assert set(got.tolist()) <= {0, 1}


@pytest.mark.parametrize("vocab", [151936, 20001, 1023, 7, 1])
def test_list_and_full_paths_vs_exact_oracle(vocab):
    """Rows whose cut lies in the listed columns (near the maximum), beyond them (flat rows,
    nuclei wider than the list), with long runs of equal keys at the cut, and with masked
    (-inf) columns; an odd vocabulary puts rows off 16-byte alignment, tiny ones leave most
    parts of a row empty."""
    g = torch.Generator().manual_seed(vocab + 1)
    n = lambda *s: torch.randn(*s, generator=g)
    rows, cfg = [], []

    def add(row, t, k, p):
        rows.append(row.to(torch.bfloat16).float())
        cfg.append((t, k, p))

    peaked = n(vocab) * 2.0
    peaked[torch.randint(0, vocab, (min(40, vocab),), generator=g)] += 11.0
    for t, k, p in ((0.6, 20, 0.95), (1.0, -1, 0.9), (0.7, 50, 1.0), (0.0, 5, 0.5), (1.0, -1, 1.0)):
        add(peaked, t, k, p)
    flat = n(vocab) * 0.3
    for t, k, p in ((1.0, -1, 0.9), (1.0, 40, 1.0), (2.0, 3, 0.2), (1.0, -1, 0.0)):
        add(flat, t, k, p)
    for near in (8191, 8192, 8193):  # that many equal columns, the rest far below
        row = torch.full((vocab,), -40.0)
        row[torch.randperm(vocab, generator=g)[:near]] = 0.0
        row[vocab // 2] = 1.0
        add(row, 1.0, 500, 1.0)
        add(row, 1.0, -1, 0.5)
        add(row, 1.0, 9000, 1.0)  # reaches past the equal columns
    edge = torch.full((vocab,), -9.703125)  # every other column equal
    edge[0] = 0.0
    add(edge, 1.0, 10, 1.0)
    add(edge - 0.0625 * torch.arange(vocab).clamp(max=3), 1.0, 3, 1.0)
    masked = n(vocab) * 3.0
    masked[torch.randperm(vocab, generator=g)[:vocab * 9 // 10]] = -math.inf
    masked[vocab // 3] = 4.0
    add(masked, 0.8, 30, 0.9)
    add(masked, 0.8, vocab - 1, 1.0)
    m = len(rows)
    print(f"vocab={vocab} rows={m}", flush=True)
    t, k, p = (list(x) for x in zip(*cfg))
    _check(torch.stack(rows), t, k, p, [17 * i + 5 for i in range(m)], [31 * i for i in range(m)])


@pytest.mark.parametrize("temp", [1.0425, 1.0495, 1.1])
def test_forced_token_of_the_largest_float(temp):
    """A row whose only likely column holds the largest float, as a forced token does: drawn
    under any limit, also where maximum / T * T rounds to infinity (the first two)."""
    v = 5000
    row = torch.full((3, v), -math.inf)
    row[0, 4321] = row[1, 17] = row[2, 4999] = torch.finfo(torch.float32).max
    row[1] = row[1].clamp(min=torch.finfo(torch.float32).min)
    cfg = ([temp] * 3, [20, 50, -1], [1.0, 0.9, 0.5], [1, 2, 3], [7, 8, 9])
    got = _sample(row, *cfg)
    assert got.tolist() == sample_exact_ref(row, *cfg).tolist() == [4321, 17, 4999]


def test_more_rows_than_one_launch_takes():
    """A million rows and more: 16 workgroups of 256 threads a row would pass a launch's 2^32
    work-items, as one of 1024 would for four million."""
    from sid.kernels.ops import argmax_rows, sample_rows
    n, v = (1 << 20) + 3, 4
    print(f"sampler rows={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    logits = torch.randn(n, v, generator=g, device="cuda")
    temps = (torch.arange(n, device="cuda") % 3 != 0).float()  # every third row greedy
    ids = torch.arange(n, device="cuda")
    got = sample_rows(logits, temps, torch.ones(n, dtype=torch.int64, device="cuda"),
                          torch.ones(n, device="cuda"), ids, ids)
    assert torch.equal(got, logits.argmax(1))  # top-k 1: the argmax for every row
    logits = torch.randn((1 << 22) + 3, 2, generator=g, device="cuda")
    assert torch.equal(argmax_rows(logits), logits.argmax(1))


@pytest.mark.parametrize("vocab", [151936, 65537, 20002])
def test_few_rows_draw_as_among_many(vocab):
    """A few long rows take four launches, many rows one (a workgroup per row): the same tokens
    for greedy, unlimited and limited rows, peaked, flat (past the list), tied and non-finite
    ones, on and off 16-byte alignment."""
    g = torch.Generator().manual_seed(vocab)
    n = lambda *s: torch.randn(*s, generator=g)
    peaked = n(vocab) * 2.0
    peaked[torch.randint(0, vocab, (40,), generator=g)] += 11.0
    tied = torch.full((vocab,), -3.0)
    tied[::7] = 2.0
    bad = n(vocab)
    bad[vocab // 2] = math.nan
    inf = n(vocab)
    inf[vocab // 3] = math.inf
    masked = n(vocab) * 3.0
    masked[torch.randperm(vocab, generator=g)[:vocab * 9 // 10]] = -math.inf
    limits = [(0.0, 5, 0.5), (0.7, -1, 1.0), (0.7, 20, 0.95), (1.3, -1, 0.9), (1.0, 50, 1.0),
              (1.0, 12000, 1.0)]
    rows = [(r, t, k, p) for r in (peaked, n(vocab) * 0.3, tied, masked) for t, k, p in limits]
    rows += [(r, t, k, p) for r in (bad, inf) for t, k, p in limits[:2]]
    few = len(rows)
    assert (144 - few) * vocab > 144 * 16000  # four launches
    logits = torch.stack([r[0] for r in rows]).to(torch.bfloat16).float()
    t, k, p = (torch.tensor([r[i] for r in rows]) for i in (1, 2, 3))
    ids = torch.arange(few)
    want = _sample(logits, t, k, p, 17 * ids + 5, 31 * ids)
    at = torch.arange(160) % few  # one launch
    got = _sample(logits.cuda()[at.cuda()], t[at], k[at], p[at], (17 * ids + 5)[at],
                  (31 * ids)[at])
    assert torch.equal(got, want[at])


@pytest.mark.parametrize("offset", [0, 1])
def test_row_of_the_largest_width(offset):
    """2^31 - 1 columns, where a step past the row's end passes 2^31: greedy, top-k and unlimited
    draws and the argmax of a row that is, and one that is not, 16-byte aligned."""
    from sid.kernels.ops import argmax_rows, sample_rows
    v = (1 << 31) - 1
    print(f"sampler columns={v} offset={offset}", flush=True)
    buf = torch.full((v + 8,), -30.0, device="cuda")
    row = buf[offset:offset + v].view(1, v)
    buf[:offset] = buf[offset + v:] = 9.0  # (outside the row)
    at = [0, 65, v // 2, v - 1000, v - 2, v - 1]
    for c, x in zip(at, (1.0, 2.0, 1.5, 2.5, 2.0, 3.0)):
        buf[offset + c] = x
    assert argmax_rows(row).tolist() == [v - 1]
    one = lambda x, dt=torch.int64: torch.tensor([x], dtype=dt, device="cuda")
    draw = lambda t, k, p, s: sample_rows(row, one(t, torch.float32), one(k), one(p, torch.float32),
                                          one(s), one(3)).item()
    assert draw(0.0, -1, 1.0, 1) == v - 1
    assert draw(0.5, 1, 1.0, 1) == v - 1
    assert draw(0.5, -1, 0.1, 1) == v - 1
    got = {draw(5.0, 6, 1.0, s) for s in range(4)}
    assert got <= set(at) and len(got) > 1
    assert draw(0.25, -1, 1.0, 5) in at  # (elsewhere at most log 1e-10 + 16.7)


def _check_both_forms(rows, cfg):
    """Few rows (four launches where they are long), and the same rows among 160 (one launch)."""
    m = len(rows)
    logits = torch.stack(rows)
    t, k, p = (list(x) for x in zip(*cfg))
    seeds, pos = [17 * i + 5 for i in range(m)], [31 * i for i in range(m)]
    got = _check(logits, t, k, p, seeds, pos)
    at = torch.arange(160) % m
    many = _sample(logits.cuda()[at.cuda()], *(torch.tensor(x)[at] for x in (t, k, p, seeds, pos)))
    assert torch.equal(many, got[at])


LIST_CAP, CUTS = 16384, (6, 9, 12, 15, 18, 21)  # kListCap and -log2 of kCutMin of sample.hip


@pytest.mark.parametrize("vocab", [151936, 40001])
def test_list_capacity_vs_exact_oracle(vocab):
    """Exactly the list's capacity of columns above a threshold, one less and one more, with
    limits at, before and past the last of them."""
    print(f"list capacity vocab={vocab}", flush=True)
    g = torch.Generator().manual_seed(vocab)
    rows, cfg = [], []
    for near in (LIST_CAP - 1, LIST_CAP, LIST_CAP + 1):
        row = torch.full((vocab,), -60.0)
        at = torch.randperm(vocab, generator=g)[:near]
        row[at] = -2.0 * torch.rand(near, generator=g)  # exp of at least 2^-3
        row[at[0]] = 1.0
        for k, p in ((near, 1.0), (near - 1, 1.0), (near + 1, 1.0), (-1, 0.5), (-1, 0.9999)):
            rows.append(row)
            cfg.append((1.0, k, p))
    _check_both_forms(rows, cfg)


@pytest.mark.parametrize("vocab", [151936, 40001])
def test_list_thresholds_vs_exact_oracle(vocab):
    """For each threshold 60 columns just above it and 60 just below (apart by more than the
    roundings of x / T and of the exponential, about 4 ulp), the limit at the last one above,
    at the first below and between; with temperatures and maxima that stretch the logits'
    bound by which the list's candidates are picked."""
    print(f"list thresholds vocab={vocab}", flush=True)
    g = torch.Generator().manual_seed(vocab + 1)
    rows, cfg = [], []
    for i, cut in enumerate(CUTS):
        for t, top in ((1.0, 0.0), (0.3, 300.0), (7.0, -2000.0), (1.7, 40.0))[i % 2::2]:
            gap = 4e-6 + 8 * 2.0 ** -24 * abs(top) / t
            row = torch.full((vocab,), top - 60.0 * t)
            at = torch.randperm(vocab, generator=g)[:121]
            row[at[0]] = top
            row[at[1:61]] = top + t * (-cut * math.log(2) + gap)
            row[at[61:]] = top + t * (-cut * math.log(2) - gap)
            mass = 60 * 2.0 ** -cut  # of each group, the maximum's being 1
            for k, p in ((61, 1.0), (62, 1.0), (31, 1.0), (-1, (1 + 0.5 * mass) / (1 + 2 * mass)),
                         (-1, (1 + 1.5 * mass) / (1 + 2 * mass))):
                rows.append(row)
                cfg.append((t, k, p))
    _check_both_forms(rows, cfg)
