"""RoPE, q/k RMSNorm and the fused append on the GPU against the oracle."""

import numpy as np
import pytest
import torch

from aspire_amd.attention.rope import RopeConfig, apply_rope_inplace, qk_norm_rope_update_kv
from aspire_amd.workloads import PAGE, build_step
from helpers import bits, say
from oracle.append import paged_kv_append
from oracle.rope import qk_norm_rope, rope_frequencies, rope_interleaved, token_positions

pytestmark = pytest.mark.gpu


def bf16_close(got: torch.Tensor, ref: torch.Tensor):
    """Within one bf16 rounding step of the reference (relative 2^-8, plus the fp32 work before it)."""
    g, r = got.float().cpu(), ref.float().cpu()
    tol = r.abs() * 2.0 ** -7 + 1e-6
    bad = (g - r).abs() > tol
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} values off; worst {float((g - r).abs().max())}"


@pytest.mark.parametrize("llama31", [False, True])
def test_rope_matches_oracle_up_to_long_positions(gpu, llama31):
    say("rope", llama31)
    g = torch.Generator().manual_seed(3)
    T, HQ, HKV = 40, 32, 8
    q = torch.randn(T, HQ, 128, generator=g).to(torch.bfloat16)
    k = torch.randn(T, HKV, 128, generator=g).to(torch.bfloat16)
    indptr = torch.tensor([0, 1, 5, 5, 30, 36], dtype=torch.int32)  # tokens 36..39 belong to no row
    offsets = torch.tensor([0, 131068, 9, 70000, 32767], dtype=torch.int32)
    cfg = RopeConfig(500000.0, 8.0, 1.0, 4.0, 8192) if llama31 else RopeConfig(1e6)
    ll = dict(low_freq_factor=1.0, high_freq_factor=4.0, old_context_len=8192.0) if llama31 else None
    qd, kd = q.to(gpu), k.to(gpu)
    apply_rope_inplace(qd, kd, indptr.to(gpu), offsets.to(gpu), cfg)
    torch.cuda.synchronize()
    f = rope_frequencies(128, cfg.rope_theta, cfg.rope_scale, ll)
    pos = token_positions(indptr.numpy(), offsets.numpy(), T)
    bf16_close(qd, rope_interleaved(q, pos, f))
    bf16_close(kd, rope_interleaved(k, pos, f))
    assert torch.equal(qd[36:].cpu(), q[36:]) and torch.equal(kd[36:].cpu(), k[36:])  # untouched


def test_fused_norm_rope_append_config1_shape(gpu):
    """Qwen3-8B layer: 32 q / 8 kv heads, q/k RMSNorm, permute, rope theta 1e6, append of the 80 new
    tokens into the random-permutation page pool; q rewritten in place, k and v in the cache."""
    say("fused norm+rope+append")
    step = build_step(hq=32, hkv=8, ctx_len=[2000, 40000, 16, 777], q_len=[1, 4, 4, 1], is_draft=[1, 0, 0, 1],
                      draft_budget=64, seed=8, device=gpu, bucket_tokens=12)
    g = torch.Generator().manual_seed(9)
    T = step.total_tokens
    q = torch.randn(12, 32, 128, generator=g).to(torch.bfloat16) * 3   # bucket of 12: 2 padding tokens
    k = torch.randn(12, 8, 128, generator=g).to(torch.bfloat16) * 3
    v = torch.randn(12, 8, 128, generator=g).to(torch.bfloat16)
    wq = (torch.rand(128, generator=g) + 0.5).to(torch.bfloat16)
    wk = (torch.rand(128, generator=g) + 0.5).to(torch.bfloat16)
    # positions of each row's first new token: its cache length before the append
    offsets = torch.from_numpy(np.append(step.ctx_len - step.q_len, 0).astype(np.int32))
    cache = step.cache.clone()
    before = cache.cpu()
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    qk_norm_rope_update_kv(qd, kd, vd, wq.to(gpu), wk.to(gpu), 1e-6, step.qo_indptr, offsets.to(gpu), cache,
                           step.kv_indices, step.kv_indptr, step.last_page_len, PAGE, config=RopeConfig(1e6))
    torch.cuda.synchronize()
    ref_q, ref_k = qk_norm_rope(q, k, step.qo_indptr_host.numpy(), offsets.numpy(), theta=1e6, q_weight=wq,
                                k_weight=wk, eps=1e-6)
    bf16_close(qd[:T], ref_q[:T])
    # the cache equals the plain append of the oracle's rotated k and of v (padding tokens skipped)
    ref_bits = paged_kv_append(bits(ref_k), bits(v), step.qo_indptr_host.numpy(), bits(before),
                               step.kv_indices.cpu().numpy(), step.kv_indptr_host.numpy(),
                               step.last_page_len.cpu().numpy(), PAGE)
    ref_cache = torch.from_numpy(ref_bits.view(np.int16)).view(torch.bfloat16)
    got = cache.cpu()
    changed = (ref_cache != before).any(dim=-1)
    assert torch.equal(got[~changed], before[~changed])  # untouched rows unchanged (bitwise)
    assert torch.equal(got[:, 1], ref_cache[:, 1])       # V: exact copy
    bf16_close(got[:, 0][changed[:, 0]], ref_cache[:, 0][changed[:, 0]])
    assert torch.equal(kd.cpu(), k)                       # k itself is not rewritten by the fused op


def pairs_close(got: torch.Tensor, ref: torch.Tensor):
    """Rotated pairs against the oracle. The fp32 sums of the norm may be taken in another order, which
    now and then moves one of a pair's two inputs by one bf16 step, at most 2^-7 of it, at each of its
    two roundings; the rotation passes that on in full, so an output may be off by 2 * 2^-7 of the pair's
    length (the rotation keeps it) besides its own step. All but a few are within their own step."""
    g, r = got.double().cpu(), ref.double().cpu()
    step = r.abs() * 2.0 ** -7 + 1e-6
    length = torch.sqrt((r * r).unflatten(-1, (-1, 2)).sum(dim=-1, keepdim=True)).expand(*r.shape[:-1], -1, 2).flatten(-2)
    off = (g - r).abs()
    assert not (off > step + 2 * 2.0 ** -7 * length).any()
    assert (off > step).double().mean().item() < 1e-4


@pytest.mark.parametrize("hq,hkv,lens,width", [
    (32, 8, [1], 128),                       # the smallest call
    (7, 3, [5, 0, 26], 128),                 # heads that fill no quad; 31 tokens, an empty row
    (16, 2, [33], 136),                      # 8 waves a token, more than quads; strided heads
    (6, 6, [100, 156], 130),                 # head rows 4-byte but not 8-byte aligned: the narrow loads
    (32, 8, [257], 128),                     # a last workgroup with waves past the tokens
    (5, 1, [300, 1, 900], 128),
    (64, 8, [3, 28], 128),                   # 20 quads: 32 waves a token, some without heads
    (40, 16, [86], 132),                     # 88 tokens with the padding: the most that 32 waves each are launched for
    (40, 16, [87], 128),                     # and one more: 16 waves, two passes
])
@pytest.mark.parametrize("norm", [True, False])
def test_fused_edges_match_oracle(gpu, hq, hkv, lens, width, norm):
    """Head counts and token counts at the edges of the kernel's quads, waves and workgroups, wide and
    narrow loads, with the norm and permute and without, two padding tokens past the last row."""
    say("fused edges", hq, hkv, lens, width, norm)
    ctx = [n + 21 * (i + 1) if n else 0 for i, n in enumerate(lens)]
    step = build_step(hq=hq, hkv=hkv, ctx_len=ctx, q_len=lens, is_draft=[0] * len(lens), draft_budget=0, seed=17,
                      device=gpu, bucket_tokens=sum(lens) + 2)
    g = torch.Generator().manual_seed(23)
    T = step.total_tokens
    pad = lambda h: torch.randn(T + 2, h, width, generator=g).to(torch.bfloat16)
    qf, kf, v = pad(hq), pad(hkv), torch.randn(T + 2, hkv, 128, generator=g).to(torch.bfloat16)
    q, k = qf[:, :, :128], kf[:, :, :128]
    w = (torch.rand(2, 128, generator=g) + 0.5).to(torch.bfloat16) if norm else (None, None)
    offsets = torch.from_numpy(np.append(step.ctx_len - step.q_len, 0).astype(np.int32))
    before = step.cache.cpu()
    cache = step.cache.clone()
    qd, kd = qf.to(gpu), kf.to(gpu)
    args = [t.to(gpu) if t is not None else None for t in w]
    qk_norm_rope_update_kv(qd[:, :, :128], kd[:, :, :128], v.to(gpu), *args, 1e-6, step.qo_indptr, offsets.to(gpu),
                           cache, step.kv_indices, step.kv_indptr, step.last_page_len, PAGE, config=RopeConfig(1e6))
    torch.cuda.synchronize()
    ref_q, ref_k = qk_norm_rope(q, k, step.qo_indptr_host.numpy()[:-1], offsets.numpy()[:-1], theta=1e6,
                                q_weight=w[0], k_weight=w[1], eps=1e-6)
    pairs_close(qd[:T, :, :128], ref_q[:T])
    assert torch.equal(qd[:, :, 128:].cpu(), qf[:, :, 128:]) and torch.equal(kd.cpu(), kf)
    ref = paged_kv_append(bits(ref_k), bits(v), step.qo_indptr_host.numpy()[:-1], bits(before),
                          step.kv_indices.cpu().numpy(), step.kv_indptr_host.numpy()[:-1],
                          step.last_page_len.cpu().numpy()[:-1], PAGE)
    ref = torch.from_numpy(ref.view(np.int16)).view(torch.bfloat16)
    got = cache.cpu()
    assert torch.equal(got[:, 1], ref[:, 1])              # V: exact copies, nothing else touched
    changed = (ref[:, 0] != before[:, 0]).any(dim=-1)
    assert torch.equal(got[:, 0][~changed], before[:, 0][~changed])
    pairs_close(got[:, 0][changed], ref[:, 0][changed])
