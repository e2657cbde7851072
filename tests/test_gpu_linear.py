"""The decode step's linear kernels against fp64 products of the same bf16 operands."""

import pytest
import torch

from aspire_amd.decode_step import add_rms_norm, add_rms_norm_partials
from aspire_amd.linear import MAX_ROWS, linear, linear_partials, linear_splits, supported
from aspire_amd.attention.rope import RopeConfig, qk_norm_rope_update_kv, qk_norm_rope_update_kv_partials
from aspire_amd.workloads import PAGE, build_step
from helpers import say

pytestmark = pytest.mark.gpu

# both sides of every row class (16, 32, 64, 128, 224 rows), rows that end inside a 16-row tile
ROWS = [1, 16, 17, 32, 33, 64, 65, 100, 128, 129, 208, 224]


# slabs up to 16, 128 and 224 rows, where a case is there for them
SPLITS = {(1056, 2432): (8, 8, 8), (6144, 4096): (3, 5, 4), (4096, 12288): (4, 8, 5)}


def close_sum(got, x, w, ref, ulps=0.0):
    """Products of bf16 are exact in fp32; a sum of K of them in fp32, in any order, is within
    K * 2^-24 of sum |x w| (gamma_K of the standard bound), plus ``ulps`` roundings to bf16 (8 significant bits: 2^-8 of the value each)."""
    bound = x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    off = (got.double() - ref).abs()
    assert not (off > bound + ulps * 2.0 ** -8 * (ref.abs() + bound)).any(), float(off.max())


def operands(rows, n, k, gpu, pad=0):
    g = torch.Generator(device=gpu).manual_seed(rows * 131 + n + k)
    x = torch.randn(rows, k + pad, device=gpu, generator=g).to(torch.bfloat16)[:, :k]
    w = (torch.randn(n, k + pad, device=gpu, generator=g) * k ** -0.5).to(torch.bfloat16)[:, :k]
    return x, w


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("n,k,pad", [
    (32, 128, 0), (96, 256, 8), (4128, 384, 0), (25600, 128, 16), (12320, 640, 0),
    (1056, 2432, 0),    # 8 splits of 38 steps: unequal ones, rings that wrap a few times
    (6144, 4096, 0),    # 64-row tiles in 3 splits, 128-row in 5, 96-row (past 128 rows) in 4
    (4096, 12288, 8),   # 4, 8 and 5 splits, long walks over k
    (16480, 640, 8),    # 96-row tiles past 64 rows for both outputs, the last one past the weight's end
    (24640, 1152, 0),   # 128-row tiles from 33 rows on
])
def test_linear_and_partials(gpu, rows, n, k, pad):
    """One k step and many, tiles that end past the last weight row, every tile width the chooser takes (few and
    many tiles), row strides longer than k; both outputs, nothing written beside them."""
    say("linear", rows, n, k, pad)
    x, w = operands(rows, n, k, gpu, pad)
    ref = x.double() @ w.double().t()
    out = torch.full((rows + 1, n + 8), 7.0, dtype=torch.bfloat16, device=gpu)
    linear(x, w, out[:rows, :n])
    close_sum(out[:rows, :n], x, w, ref, ulps=1)
    assert (out[rows:] == 7).all() and (out[:, n:] == 7).all()
    s = linear_splits(rows, n, k)
    if (n, k) in SPLITS:
        assert s == SPLITS[n, k][0 if rows <= 16 else 1 if rows <= 128 else 2]
    ws = torch.full((s * rows * n + 64,), 7.0, device=gpu)
    parts = linear_partials(x, w, ws)
    assert parts.shape == (s, rows, n) and (ws[s * rows * n :] == 7).all()
    close_sum(parts.double().sum(0), x, w, ref)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("n,k", [
    (16, 128), (1040, 512), (12304, 256),
    (1040, 2432),       # 64-row tiles, rings that wrap at every row class
    (8224, 2176),       # 96-row tiles past 64 rows, the last one past the weight's end
    (13648, 2304),      # 128-row tiles from 17 to 128 rows
    (12288, 4096),
])
def test_linear_swiglu(gpu, rows, n, k):
    say("linear swiglu", rows, n, k)
    x, w = operands(rows, 2 * n, k, gpu)
    w = w * 4  # gates on both sides of silu's bend
    gu = x.double() @ w.double().t()
    out = torch.full((rows, n + 8), 7.0, dtype=torch.bfloat16, device=gpu)
    linear(x, w, out[:, :n], swiglu=True)
    g, u = gu.chunk(2, dim=-1)
    ref = torch.nn.functional.silu(g) * u
    # g, u, silu(g) and the product are rounded to bf16, 2^-8 each of their size, and fp32 sums moved
    # them by K 2^-24 of sum |x w|; |silu'| <= 1.1, so g's error reaches silu(g) at most 1.1-fold
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    bg, bu = bound.chunk(2, dim=-1)
    dg, du = 2.0 ** -8 * g.abs() + bg, 2.0 ** -8 * u.abs() + bu
    ds = 1.1 * dg + 2.0 ** -8 * torch.nn.functional.silu(g).abs()
    off = (out[:, :n].double() - ref).abs()
    limit = (ds * u.abs() + du * torch.nn.functional.silu(g).abs() + ds * du) * 1.01 + 2.0 ** -8 * ref.abs() + 1e-30
    assert not (off > limit * 1.01).any()
    assert (out[:, n:] == 7).all()


def test_supported_shapes(gpu):
    x, w = operands(4, 64, 256, gpu)
    assert supported(x, w)
    assert not supported(x[:, :192], w[:, :192]) and not supported(x, w[:40])  # K % 128, N % 32
    assert not supported(x.float(), w) and not supported(x.t(), w) and not supported(x[:0], w)
    assert not supported(torch.zeros(MAX_ROWS + 1, 256, dtype=torch.bfloat16, device=gpu), w)
    assert not supported(torch.zeros(4 * 256 + 1, dtype=torch.bfloat16, device=gpu)[1:].view(4, 256), w)
    with pytest.raises(ValueError):
        linear(x, w, torch.empty(4, 32, dtype=torch.bfloat16, device=gpu))
    with pytest.raises(ValueError):
        linear_partials(x, w, torch.empty(8, device=gpu))


@pytest.mark.parametrize("rows,dim,splits", [(1, 8, 1), (37, 4096, 4), (5, 512, 3), (3, 8192, 8), (2, 1024, 9), (3, 520, 17)])
def test_add_rms_norm_partials(gpu, rows, dim, splits):
    """Equal, bit for bit, to add_rms_norm with the slabs' sum rounded to bf16."""
    say("add_rms_norm partials", rows, dim, splits)
    g = torch.Generator(device=gpu).manual_seed(dim + splits)
    x = torch.randn(rows, dim, device=gpu, generator=g).to(torch.bfloat16)
    parts = torch.randn(splits, rows, dim, device=gpu, generator=g)
    w = (torch.rand(dim, device=gpu, generator=g) + 0.5).to(torch.bfloat16)
    total = parts[0].clone()
    for s in range(1, splits):
        total += parts[s]
    x1, x2 = x.clone(), x.clone()
    o1, o2 = torch.empty_like(x), torch.empty_like(x)
    add_rms_norm(x1, w, o1, 1e-6, delta=total.to(torch.bfloat16))
    add_rms_norm_partials(x2, w, o2, 1e-6, parts)
    assert torch.equal(x1, x2) and torch.equal(o1, o2)


@pytest.mark.parametrize("hq,hkv,lens,splits,norm", [(32, 8, [1, 4, 0, 3], 4, True), (7, 3, [40], 1, True),
                                                     (16, 2, [200, 70], 3, False)])
def test_qkv_from_partials(gpu, hq, hkv, lens, splits, norm):
    """Equal, bit for bit, to the q/k preparation of the slabs' sum rounded to bf16."""
    say("qkv from partials", hq, hkv, lens, splits, norm)
    ctx = [n + 33 if n else 0 for n in lens]
    step = build_step(hq=hq, hkv=hkv, ctx_len=ctx, q_len=lens, is_draft=[0] * len(lens), draft_budget=0, seed=3, device=gpu)
    g = torch.Generator(device=gpu).manual_seed(hq + splits)
    T, width = step.total_tokens, (hq + 2 * hkv) * 128
    parts = torch.randn(splits, T, width, device=gpu, generator=g)
    total = parts[0].clone()
    for s in range(1, splits):
        total += parts[s]
    qkv = total.to(torch.bfloat16)
    w = [(torch.rand(128, device=gpu, generator=g) + 0.5).to(torch.bfloat16) if norm else None for _ in range(2)]
    offsets = torch.tensor([c - n for c, n in zip(ctx, lens)] + [0], dtype=torch.int32, device=gpu)
    rest = (*w, 1e-6, step.qo_indptr, offsets)
    pages = (step.kv_indices, step.kv_indptr, step.last_page_len, PAGE)
    c1, c2 = step.cache.clone(), step.cache.clone()
    q1 = qkv[:, : hq * 128].view(T, hq, 128)
    k, v = (qkv[:, (hq + i * hkv) * 128 : (hq + (i + 1) * hkv) * 128].view(T, hkv, 128) for i in range(2))
    qk_norm_rope_update_kv(q1, k, v, *rest, c1, *pages, config=RopeConfig(1e6))
    q2 = torch.empty(T, hq, 128, dtype=torch.bfloat16, device=gpu)
    qk_norm_rope_update_kv_partials(parts, q2, hkv, *rest, c2, *pages, config=RopeConfig(1e6))
    assert torch.equal(q1, q2) and torch.equal(c1, c2)
