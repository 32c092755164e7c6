"""Decode-step GEMMs (HIP MFMA) vs fp32, and the M-invariance of every row (bitwise).
Shapes: the reference's tests/test_10_batch_invariant.py:18-38 plus the Qwen3-0.6B decode
(M=64) and verify (M=128) projections."""

from __future__ import annotations

import pytest
import torch

from oracle.gemm import linear_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 1024, 1024), (7, 3072, 1024), (128, 151936, 1024), (500, 1024, 3072),
    (64, 4096, 1024), (64, 1024, 2048), (64, 6144, 1024), (64, 1024, 3072), (64, 151936, 1024),
    (128, 6144, 1024), (33, 64, 256), (200, 128, 512), (64, 2048, 1024),
])
def test_linear_vs_fp32(m, n, k):
    from sid.kernels.matmul_persistent import linear
    torch.manual_seed(0)
    x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(n, k, device="cuda") * 0.05).to(torch.bfloat16)
    out = linear(x, w)
    ref = linear_ref(x.cpu(), w.cpu())
    torch.testing.assert_close(out.float().cpu(), ref, atol=3e-2, rtol=2e-2)


def test_bias_and_fp32_output():
    from sid.kernels.matmul_persistent import bi_linear, linear, matmul_persistent
    torch.manual_seed(1)
    x = torch.randn(9, 512, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(128, 512, device="cuda", dtype=torch.bfloat16)
    b = torch.randn(128, device="cuda", dtype=torch.bfloat16)
    y = bi_linear(x, w, b)
    torch.testing.assert_close(y.float().cpu(), linear_ref(x.cpu(), w.cpu(), b.cpu()), atol=2e-1, rtol=2e-2)
    y32 = linear(x, w, b, out_fp32=True)
    assert y32.dtype == torch.float32 and torch.equal(y32.to(torch.bfloat16), y)
    assert torch.equal(matmul_persistent(x, w.t(), b), y)


def test_row_invariance():
    from sid.kernels.matmul_persistent import bi_linear
    torch.manual_seed(2)
    x0 = torch.randn(1, 1024, device="cuda", dtype=torch.bfloat16)
    for n in (3072, 151936):
        w = (torch.randn(n, 1024, device="cuda") * 0.05).to(torch.bfloat16)
        alone = bi_linear(x0, w)
        for m in (2, 64, 65, 333):
            x = torch.cat([torch.randn(m - 1, 1024, device="cuda", dtype=torch.bfloat16), x0])
            assert torch.equal(alone[0], bi_linear(x, w)[-1]), (n, m)


def test_strided_input_rows():
    from sid.kernels.matmul_persistent import linear
    torch.manual_seed(3)
    big = torch.randn(16, 2048, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(64, 1024, device="cuda", dtype=torch.bfloat16)
    assert torch.equal(linear(big[:, :1024], w), linear(big[:, :1024].contiguous(), w))


@pytest.mark.parametrize("m,n,k", [(64, 4096, 1024), (64, 1024, 2048), (64, 6144, 1024),
                                   (64, 1024, 3072), (5, 1024, 3072), (1, 4096, 1024),
                                   (100, 1024, 2048), (512, 1024, 2048), (1024, 1024, 3072),
                                   (300, 4096, 1024)])
def test_partials_fold_equals_linear(m, n, k):
    """Chunk partials folded in increasing chunk order and rounded to bf16 equal sid_linear
    bit for bit (the contract the *_partials consumers rely on)."""
    from sid.kernels.matmul_persistent import linear, linear_partials
    torch.manual_seed(4)
    x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(n, k, device="cuda") * 0.05).to(torch.bfloat16)
    p = linear_partials(x, w)
    assert p.shape == (k // 256, m, n)
    fold = p[0].clone()
    for c in range(1, p.shape[0]):
        fold += p[c]
    assert torch.equal(fold.to(torch.bfloat16), linear(x, w))


@pytest.mark.parametrize("m", [1, 16, 33, 64, 100, 128, 256])
def test_stream_lm_head_path_bitwise_matches_tiled(m):
    """lm_head-shaped GEMMs (K=1024, N >= 32768, M<=256 in 64-row groups) take the persistent
    streaming kernel;
    its bits equal the tiled kernel's (checked on the first and last 4096 columns, which
    the tiled kernel computes separately), for fp32 and bf16 outputs."""
    from sid.kernels.matmul_persistent import linear
    torch.manual_seed(6)
    print(f"m={m}", flush=True)
    x = torch.randn(m, 1024, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(151936, 1024, device="cuda") * 0.05).to(torch.bfloat16)
    full = linear(x, w, out_fp32=True)              # streaming kernel
    head = linear(x, w[:4096].contiguous(), out_fp32=True)  # tiled kernel (small N)
    tail = linear(x, w[-4096:].contiguous(), out_fp32=True)
    assert torch.equal(full[:, :4096], head)
    assert torch.equal(full[:, -4096:], tail)
    assert torch.equal(linear(x, w), full.to(torch.bfloat16))
    ref = x.float().cpu() @ w[:2048].float().cpu().t()
    torch.testing.assert_close(full[:, :2048].cpu(), ref, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("m,n,k", [(1, 151936, 1024), (7, 151936, 1024), (33, 65536, 1024),
                                   (64, 151936, 1024), (64, 4096, 1024), (65, 151936, 1024),
                                   (128, 151936, 1024), (200, 65536, 1024), (300, 151936, 1024),
                                   (512, 151936, 1024), (100, 1088, 512), (3, 4096, 2048)])
def test_linear_argmax_matches_linear_then_argmax(m, n, k):
    """Fused lm_head + greedy argmax == argmax_rows(linear(..., out_fp32=True)), and the
    optional logits output equals linear's: the streaming path (up to 64 rows, K = 1024)
    and the tiled GEMM's argmax epilogue (more rows, other K, a ragged last column tile)."""
    from sid.kernels.matmul_persistent import linear, linear_argmax
    from sid.kernels.ops import argmax_rows
    torch.manual_seed(7 + m)
    print(f"m={m} n={n} k={k}", flush=True)
    x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(n, k, device="cuda") * 0.05).to(torch.bfloat16)
    logits = linear(x, w, out_fp32=True)
    want = argmax_rows(logits)
    assert torch.equal(linear_argmax(x, w), want)
    lg = torch.empty(m, n, device="cuda")
    assert torch.equal(linear_argmax(x, w, logits=lg), want)
    assert torch.equal(lg, logits)


@pytest.mark.parametrize("m", [4, 130])
def test_linear_argmax_ties_and_nan(m):
    """Equal maxima -> first column; a NaN logit wins over every number, first NaN first
    (torch.argmax semantics), also when the tied columns land in different waves (streaming
    path) or column tiles (tiled path)."""
    from sid.kernels.matmul_persistent import linear_argmax
    torch.manual_seed(8)
    n = 151936
    x = torch.randn(m, 1024, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(n, 1024, device="cuda") * 0.01).to(torch.bfloat16)
    hot = (x[0].float() / x[0].float().norm()).to(torch.bfloat16)
    for c in (150000, 70001, 70000, 123):   # identical rows: identical logits for every x
        w[c] = hot
    got = linear_argmax(x, w).cpu()
    assert got[0].item() == 123
    want = torch.argmax(x.float().cpu() @ w.float().cpu().t(), dim=-1)
    assert got[0].item() == want[0].item()
    w[90000, 5] = float("nan")
    w[80000, 7] = float("nan")
    got = linear_argmax(x, w).cpu()
    assert (got == 80000).all()



def _folded(x, w):
    """x w^T in fp32 by the split-K kernel, its chunks folded in order."""
    from sid.kernels.jit import load_ext
    part = torch.empty(x.shape[1] // 256, x.shape[0], w.shape[0], device="cuda",
                       dtype=torch.float32)
    load_ext().linear_partials(x, w, part)
    fold = part[0].clone()
    for c in part[1:]:
        fold += c
    return fold


@pytest.mark.parametrize("m,n,k", [(256, 1024, 1024), (300, 1024, 2048), (1000, 6144, 1024),
                                   (2048, 4096, 1024), (777, 192, 512), (4100, 1024, 3072)])
def test_tiled_large_m_bitwise_matches_folded_chunks(m, n, k):
    """The tile kernel's bits equal the split-K chunks folded in order (rows in groups of 64
    there), and its own on slices of fewer and more than 64 rows, which take other tiles,
    with bias, both output dtypes, ragged M and N tails."""
    from sid.kernels.matmul_persistent import linear
    torch.manual_seed(m + n)
    print(f"m={m} n={n} k={k}", flush=True)
    x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(n, k, device="cuda") * 0.05).to(torch.bfloat16)
    b = torch.randn(n, device="cuda", dtype=torch.bfloat16)
    fold = _folded(x, w)
    for bias in (None, b):
        full = linear(x, w, bias)
        assert torch.equal(full, (fold if bias is None else fold + b.float()).to(torch.bfloat16))
        for lo, hi in ((0, 63), (m - 33, m), (m // 2, m // 2 + 129)):
            assert torch.equal(full[lo:hi], linear(x[lo:hi].contiguous(), w, bias)), (lo, hi)
    f32 = linear(x, w, out_fp32=True)
    assert torch.equal(f32.to(torch.bfloat16), linear(x, w))
    ref = x[:64].float().cpu() @ w.float().cpu().t()
    torch.testing.assert_close(f32[:64].cpu(), ref, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("m,n,k,tile", [
    (1, 64, 256, (64, 64)),          # one row
    (33, 128, 1024, (64, 64)),       # one tile of rows, the first SwiGLU rows on tiles
    (63, 1024, 3072, (64, 64)),      # a row short of a tile
    (64, 64, 256, (64, 64)),         # one tile, one chunk (the shortest K pipeline)
    (300, 1024, 2048, (64, 64)),     # ragged rows
    (1030, 1088, 768, (128, 64)),    # ragged rows
    (1025, 3200, 256, (128, 128)),   # one row in the last tiles, one chunk
    (4353, 8128, 256, (128, 128)),   # several rounds of the grid, one chunk
    (1500, 4032, 512, (256, 128)),   # half a tile of columns left
    (8190, 6144, 256, (256, 128)),   # several rounds of the grid, ragged rows, one chunk
    (8190, 6144, 1024, (256, 128)),  # the same, four chunks
    (4999, 6080, 768, (256, 128)),   # several rounds, ragged rows and columns
])
def test_tile_kernel_edges_bitwise(m, n, k, tile):
    """The pipelined tile GEMM in each tile shape, at the edges of tiles, of the K pipeline and
    of the grid's rounds (a tile's first loads run while the tile before it is stored): bits of
    the split-K kernel's chunks folded in order, for bf16 and fp32 outputs with and without
    bias, from rows inside a wider matrix, into an output that is only 2- (4-) byte aligned,
    with the rows after the output untouched; and the SwiGLU form against sid_silu_mul of the
    folded chunks."""
    from sid.kernels.jit import load_ext
    from sid.kernels.matmul_persistent import linear_silu_mul
    from sid.kernels.ops import silu_mul
    ext = load_ext()
    torch.manual_seed(m + n + k)
    print(f"tile edges m={m} n={n} k={k}", flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        got = ext.lib.sid_linear_tile(m, n)
        assert (got >> 16, got & 0xffff) == tile
    big = torch.randn(m, k + 64, device="cuda", dtype=torch.bfloat16)
    x = big[:, :k]
    w = (torch.randn(n, k, device="cuda") * 0.05).to(torch.bfloat16)
    b = torch.randn(n, device="cuda", dtype=torch.bfloat16)
    fold = _folded(x, w)
    for bias in (None, b):
        ref = (fold if bias is None else fold + b.float()).to(torch.bfloat16)
        for fp32 in (False, True):
            dt = torch.float32 if fp32 else torch.bfloat16
            buf = torch.full((m * n + 9,), 7.0, device="cuda", dtype=dt)
            for off in (0, 1):
                y = buf[off:off + m * n].view(m, n)
                ext.linear(x, w, bias, y, fp32)
                assert torch.equal(y, ref.to(dt)), (bias is not None, fp32, off)
                assert (buf[off + m * n:] == 7.0).all()
    if (n // 2) % 64 == 0:  # the SwiGLU entry takes K = 1024
        x = torch.randn(m, 1024, device="cuda", dtype=torch.bfloat16)
        w = (torch.randn(n, 1024, device="cuda") * 0.05).to(torch.bfloat16)
        assert torch.equal(linear_silu_mul(x, w), silu_mul(_folded(x, w).to(torch.bfloat16)))


@pytest.mark.parametrize("m,ldx", [(2, 1 << 23), (65, 1 << 25)])
def test_wide_row_strides(m, ldx):
    """Rows further apart than 32-bit tile offsets reach (the last token of each of m long
    sequences): the bits of the same rows packed, from sid_linear and the lm_head's argmax."""
    from sid.kernels.jit import load_ext
    from sid.kernels.matmul_persistent import linear
    ext = load_ext()
    print(f"wide row stride m={m} ldx={ldx}", flush=True)
    n, k = 320, 512
    packed = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    big = torch.empty(m, ldx, device="cuda", dtype=torch.bfloat16)
    x = big[:, :k]
    x.copy_(packed)
    w = (torch.randn(n, k, device="cuda") * 0.05).to(torch.bfloat16)
    ref = linear(packed, w, None, True)
    y = torch.empty(m, n, device="cuda", dtype=torch.float32)
    ext.linear(x, w, None, y, True)
    assert torch.equal(y, ref)
    logits = torch.empty_like(y)
    out = torch.empty(m, device="cuda", dtype=torch.int64)
    ws = torch.empty(ext.linear_argmax_workspace_bytes(m), device="cuda", dtype=torch.uint8)
    ext.linear_argmax(x, w, None, logits, ws, out)
    assert torch.equal(logits, ref) and torch.equal(out, ref.argmax(1))


@pytest.mark.parametrize("m,n", [(1, 64), (3, 128)])
def test_weight_rows_past_32_bit_offsets(m, n):
    """K of 2^23, where a tile's weight rows reach past 32-bit offsets: sid_linear's bits against
    the split-K chunks folded in order, and the greedy head's logits and tokens against them."""
    from sid.kernels.jit import load_ext
    ext = load_ext()
    k = 1 << 23
    print(f"long weight rows m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(m, k, device="cuda", generator=g).to(torch.bfloat16)
    w = torch.empty(n, k, device="cuda", dtype=torch.bfloat16)
    for row in w:  # (a row at a time: no second copy of the weights in float)
        row.copy_(torch.randn(k, device="cuda", generator=g) * 0.05)
    b = torch.randn(n, device="cuda", generator=g).to(torch.bfloat16)
    part = torch.empty(k // 256, m, n, device="cuda", dtype=torch.float32)
    ext.linear_partials(x, w, part)
    fold = part[0].clone()
    for c in part[1:]:
        fold += c
    ref = (fold + b.float()).to(torch.bfloat16).float()
    y = torch.empty(m, n, device="cuda", dtype=torch.float32)
    ext.linear(x, w, b, y, True)
    assert torch.equal(y, ref)
    ws = torch.empty(ext.linear_argmax_workspace_bytes(m), device="cuda", dtype=torch.uint8)
    for logits in (torch.empty_like(y), None):
        out = torch.full((m,), -1, device="cuda", dtype=torch.int64)
        ext.linear_argmax(x, w, b, logits, ws, out)
        assert torch.equal(out, ref.argmax(1))
        assert logits is None or torch.equal(logits, ref)
