"""Extend (prefill / verify) attention (HIP, MFMA) vs the fp32 oracle, and the two bitwise
properties DVR rests on: window-offset invariance and batch-slot invariance.
Cases follow the reference's tests/test_03_extend_attention.py:56-152."""

from __future__ import annotations

import pytest
import torch

from conftest import HKV, HQ, D, SCALE, assert_close_bf16
from oracle.attention import extend_attention_ref

pytestmark = pytest.mark.gpu


def _fwd(*a):
    from sid.kernels.extend_attention import extend_attention_fwd
    return extend_attention_fwd(*a)


def _make(specs, seed=0):
    g = torch.Generator().manual_seed(seed)
    total_kv = sum(p + e for p, e in specs)
    total_q = sum(e for _, e in specs)
    slots = total_kv + 16
    q = torch.randn(total_q, HQ, D, generator=g).to(torch.bfloat16)
    kb = torch.randn(slots, HKV, D, generator=g).to(torch.bfloat16)
    vb = torch.randn(slots, HKV, D, generator=g).to(torch.bfloat16)
    idx = (torch.randperm(slots - 1, generator=g)[:total_kv] + 1).to(torch.int32)
    qo = torch.zeros(len(specs) + 1, dtype=torch.int32)
    qo[1:] = torch.cumsum(torch.tensor([e for _, e in specs]), 0)
    kvp = torch.zeros(len(specs) + 1, dtype=torch.int32)
    kvp[1:] = torch.cumsum(torch.tensor([p + e for p, e in specs]), 0)
    return [t.cuda() for t in (q, kb, vb, qo, kvp, idx)]


@pytest.mark.parametrize("specs", [
    [(0, 1)], [(0, 32)], [(0, 64)], [(0, 100)], [(0, 500)],
    [(1, 1)], [(100, 32)], [(1000, 64)],
    [(100, 32), (0, 17), (999, 1), (5, 64)],
    [(31, 32), (32, 32), (33, 32), (256, 32)],
    [(7, 1), (100, 1), (5000, 1)],
    [(2048, 32), (2049, 32), (2070, 32), (0, 32)],
], ids=str)
def test_extend_vs_oracle(specs):
    q, kb, vb, qo, kvp, idx = _make(specs)
    out = _fwd(q, kb, vb, qo, kvp, idx, max(e for _, e in specs), SCALE)
    ref = extend_attention_ref(q, kb, vb, qo, kvp, idx, SCALE)
    assert_close_bf16(out, ref)


def test_window_offset_invariance():
    torch.manual_seed(11)
    L = 300
    q_all = torch.randn(L, HQ, D, device="cuda", dtype=torch.bfloat16)
    kb = torch.randn(L + 32, HKV, D, device="cuda", dtype=torch.bfloat16)
    vb = torch.randn(L + 32, HKV, D, device="cuda", dtype=torch.bfloat16)
    idx = (torch.randperm(L + 31, device="cuda")[:L] + 1).to(torch.int32)

    def run(prefix):
        e = L - prefix
        qo = torch.tensor([0, e], dtype=torch.int32, device="cuda")
        kvp = torch.tensor([0, L], dtype=torch.int32, device="cuda")
        return _fwd(q_all[prefix:].contiguous(), kb, vb, qo, kvp, idx, e, SCALE)

    base = run(268)
    for prefix in (233, 245, 267, 269, 236, 0, 100):
        other = run(prefix)
        common = max(268, prefix)
        n = L - common
        assert torch.equal(base[common - 268:common - 268 + n], other[common - prefix:common - prefix + n]), prefix


def test_position_invariance_within_batch():
    torch.manual_seed(7)
    p, e = 100, 32
    q0 = torch.randn(e, HQ, D, device="cuda", dtype=torch.bfloat16)
    kb = torch.randn(4096, HKV, D, device="cuda", dtype=torch.bfloat16)
    vb = torch.randn(4096, HKV, D, device="cuda", dtype=torch.bfloat16)
    idx0 = (torch.randperm(4095, device="cuda")[:p + e] + 1).to(torch.int32)

    def run(slot, others):
        specs, qs, idxs = [], [], []
        g = torch.Generator(device="cuda").manual_seed(1234)
        for i in range(others + 1):
            if i == slot:
                specs.append((p, e)); qs.append(q0); idxs.append(idx0)
            else:
                pe, ee = 40 + 13 * i, 8 + i
                specs.append((pe, ee))
                qs.append(torch.randn(ee, HQ, D, device="cuda", generator=g).to(torch.bfloat16))
                idxs.append(torch.randint(1, 4096, (pe + ee,), device="cuda", generator=g,
                                          dtype=torch.int32))
        qo = torch.zeros(len(specs) + 1, dtype=torch.int32)
        qo[1:] = torch.cumsum(torch.tensor([s[1] for s in specs]), 0)
        kvp = torch.zeros(len(specs) + 1, dtype=torch.int32)
        kvp[1:] = torch.cumsum(torch.tensor([s[0] + s[1] for s in specs]), 0)
        out = _fwd(torch.cat(qs), kb, vb, qo.cuda(), kvp.cuda(), torch.cat(idxs),
                   max(s[1] for s in specs), SCALE)
        return out[qo[slot]:qo[slot] + e]

    base = run(0, 0)
    for slot, others in [(0, 3), (2, 3), (3, 3), (1, 7)]:
        assert torch.equal(base, run(slot, others)), (slot, others)


def test_decode_shape_matches_decode_kernel_numerically():
    """Extend with one query per request == decode attention (tolerance; different kernels)."""
    from oracle.attention import decode_attention_ref
    specs = [(63, 1), (500, 1), (0, 1)]
    q, kb, vb, qo, kvp, idx = _make(specs, seed=5)
    out = _fwd(q, kb, vb, qo, kvp, idx, 1, SCALE)
    assert_close_bf16(out, decode_attention_ref(q, kb, vb, kvp, idx, SCALE))


@pytest.mark.parametrize("specs", [
    [(2048, 32), (2049, 32), (2070, 32), (0, 32)],   # the verify shape with 2k prefixes
    [(100, 32), (0, 17), (999, 1), (5, 64)],
    [(0, 300)],
], ids=str)
def test_split_fanout_bitwise_equals_sequential_fold(specs):
    """With a workspace the kernel gives every 256-key split its own workgroup and folds the
    split states afterwards; without one a workgroup folds them itself: same bits."""
    from sid.kernels.jit import load_ext
    ext = load_ext()
    q, kb, vb, qo, kvp, idx = _make(specs, seed=9)
    max_e = max(e for _, e in specs)
    max_kv = max(p + e for p, e in specs)
    need = ext.extend_attention_workspace_bytes(len(specs), q.shape[0], HQ, HKV, max_e, max_kv)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    a = torch.empty_like(q)
    b = torch.empty_like(q)
    ext.extend_attention_fwd(q, kb, vb, qo, kvp, idx, max_e, SCALE, a, max_kv, ws)
    ext.extend_attention_fwd(q, kb, vb, qo, kvp, idx, max_e, SCALE, b, max_kv, None)
    assert torch.equal(a, b)
    # a looser bound (more, empty splits in the grid) changes nothing either
    ws2 = torch.empty(ext.extend_attention_workspace_bytes(len(specs), q.shape[0], HQ, HKV, max_e,
                                                           4 * max_kv), dtype=torch.uint8, device="cuda")
    c = torch.empty_like(q)
    ext.extend_attention_fwd(q, kb, vb, qo, kvp, idx, max_e, SCALE, c, 4 * max_kv, ws2)
    assert torch.equal(a, c)


@pytest.mark.parametrize("prefix,rows,at", [(48, 32, 70), (16, 64, 64), (1000, 40, 1030)])
def test_hidden_values_do_not_reach_earlier_waves(prefix, rows, at):
    """An infinite and a NaN V row in a tile that only later waves of the query tile see: fan-out
    and sequential walk give the same rows, and the waves before it stay finite."""
    from sid.kernels.jit import load_ext
    ext = load_ext()
    print(f"hidden values prefix={prefix} rows={rows} at={at}", flush=True)
    q, kb, vb, qo, kvp, idx = _make([(prefix, rows)], seed=at)
    vb[idx[at].long(), :, 5] = float("inf")
    vb[idx[at].long(), :, 9] = float("nan")
    kv = prefix + rows
    ws = torch.empty(ext.extend_attention_workspace_bytes(1, rows, HQ, HKV, rows, kv),
                     dtype=torch.uint8, device="cuda")
    a, b = torch.empty_like(q), torch.empty_like(q)
    ext.extend_attention_fwd(q, kb, vb, qo, kvp, idx, rows, SCALE, a, kv, ws)
    ext.extend_attention_fwd(q, kb, vb, qo, kvp, idx, rows, SCALE, b, kv, None)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    before = (at // 64 * 64 - prefix) // 16 * 16  # rows of waves that end before the tile
    assert before > 0 and torch.isfinite(a[:before]).all()


@pytest.mark.parametrize("specs,slots", [
    # 32-row workgroups: one-row requests, tails of 32 rows and 64-key tiles, empty requests
    ([(i % 5, 1 + (37 * i) % 70) for i in range(80)] + [(300, 0)], None),
    # 64-row workgroups: ragged around tile edges
    ([(0, 1024), (3, 1023), (0, 961), (17, 960), (0, 512), (255, 65), (0, 64), (1, 1)] +
     [(0, 577 + i) for i in range(4)], None),
    # a pool of more than 4 GiB a side (64-bit row offsets)
    ([(0, 700), (40, 900)] + [(0, 33)] * 20, 2_200_000),
], ids=["narrow", "wide", "big-pool"])
def test_prefill_kernel_edges_bitwise(specs, slots):
    """The one-workgroup-per-query-tile kernel against the split fan-out: every request's rows,
    recomputed alone through the fan-out (grids below 512 workgroups take it), have the
    same bits, also with out-of-range slots (they read slot 0) and an infinite V row."""
    print(f"prefill edges {len(specs)} requests", flush=True)
    q, kb, vb, qo, kvp, idx = _make(specs, seed=len(specs))
    if slots is not None:  # spread the rows over a large pool, the last slot included
        n = kb.shape[0]
        at = torch.linspace(0, slots - 1, n, device="cuda", dtype=torch.float64).long()
        big_k = torch.zeros(slots, HKV, D, device="cuda", dtype=torch.bfloat16)
        big_v = torch.zeros_like(big_k)
        big_k[at], big_v[at] = kb, vb
        kb, vb, idx = big_k, big_v, at[idx.long()].int()
    first = int(kvp[0])
    hidden = int(kvp[1]) - 1  # the first request's last position
    vb[idx[hidden].long(), :, 3] = float("inf")
    idx[int(kvp[1])] = kb.shape[0]  # out of range: slot 0
    idx[int(kvp[1]) + 1] = -1
    assert first == 0
    longest = max(e for _, e in specs)
    tiles = -(-longest // 32)
    assert len(specs) * HKV * tiles >= 512  # the full batch does not fan out
    from sid.kernels.jit import load_ext
    rows = load_ext().lib.sid_extend_attention_query_rows(len(specs), q.shape[0], HKV, longest)
    assert rows == (64 if longest == 1024 else 32)
    full = _fwd(q, kb, vb, qo, kvp, idx, longest, SCALE)
    assert torch.isinf(full[int(qo[1]) - 1, :, 3]).all()  # (infinite, not NaN: inf / l)
    for b in range(len(specs)):
        lo, hi = int(qo[b]), int(qo[b + 1])
        if hi == lo or (b > 12 and b % 9):
            continue
        one = _fwd(q[lo:hi].contiguous(), kb, vb, torch.tensor([0, hi - lo], dtype=torch.int32, device="cuda"),
                   kvp[b:b + 2] - kvp[b], idx[int(kvp[b]):int(kvp[b + 1])].contiguous(), hi - lo, SCALE)
        assert torch.equal(torch.nan_to_num(one), torch.nan_to_num(full[lo:hi])), (b, specs[b])
        assert torch.equal(torch.isnan(one), torch.isnan(full[lo:hi])), b
