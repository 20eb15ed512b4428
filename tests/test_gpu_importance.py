"""GPU parity of the importance kernel (tm_last_query_importance) and its
Python mirrors against the oracle's last_query_importance, and its use as the
attention input of the expert keep mask."""

import numpy as np
import pytest
import torch

from oracle import tm_oracle as O
from parity_util import ODT, np64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,hkv,d,s,dtype", [(1, 32, 4, 128, 4096, torch.bfloat16),   # Qwen3-VL-30B-A3B heads
                                               (2, 16, 16, 64, 777, torch.float16),
                                               (1, 8, 2, 256, 513, torch.bfloat16),
                                               (3, 4, 1, 192, 100, torch.bfloat16)])
def test_qwen_importance_vs_oracle(hip_device, b, h, hkv, d, s, dtype):
    """Model-dtype scores (the Qwen hook): query_states [B, H, S, D] and
    key_states [B, Hkv, S, D]; the stored weights are the head mean of the
    last query's probabilities."""
    from table_moe.utils import ModalityContext, compute_and_cache_importance

    g = torch.Generator().manual_seed(s + h)
    qs = torch.randn(b, h, 5, d, generator=g).to(dtype)
    ks = torch.randn(b, hkv, s, d, generator=g).to(dtype)
    scale = d ** -0.5
    dev = hip_device
    got = compute_and_cache_importance(qs.to(dev), ks.to(dev), scale)
    torch.cuda.synchronize()
    assert ModalityContext.get_attn_weights() is not None
    assert torch.equal(ModalityContext.get_attn_weights(), got.view(-1))
    want = O.last_query_importance(np64(qs[:, :, -1]), np64(ks.transpose(1, 2)), hkv, scale, ODT[dtype])
    # fp32 accumulation order of the dot products may move a score by one
    # model-dtype ulp; the probabilities then differ by about that ratio
    np.testing.assert_allclose(np64(got), want, rtol=0.02, atol=1e-7)
    assert np.mean(np.abs(np64(got) - want) <= 1e-6 * np.abs(want) + 1e-9) > 0.9
    np.testing.assert_allclose(np64(got).sum(axis=1), 1.0, rtol=1e-5)


def test_deepseek_importance_masked_tail(hip_device):
    """fp32 scores with a key padding mask and only the last query_length keys
    (the DeepSeek hook): query_states [B, q, H, D], key_states [B, kv, H, D]."""
    from table_moe.utils import cache_last_token_attention

    g = torch.Generator().manual_seed(3)
    b, h, d, kv, qlen = 2, 16, 128, 1500, 600
    qs = torch.randn(b, qlen, h, d, generator=g).to(torch.bfloat16)
    ks = torch.randn(b, kv, h, d, generator=g).to(torch.bfloat16)
    mask = torch.rand(b, kv, generator=g) < 0.9
    dev = hip_device
    got = cache_last_token_attention(qs.to(dev), ks.to(dev), 0.088, mask.to(dev), qlen)
    torch.cuda.synchronize()
    want = O.last_query_importance(np64(qs[:, -1]), np64(ks), h, 0.088, O.F32, key_mask=mask.numpy(), out_len=qlen)
    np.testing.assert_allclose(np64(got), want, rtol=1e-4, atol=1e-9)
    assert np.all(np64(got)[~mask.numpy()[:, -qlen:]] == 0.0)


def test_importance_feeds_expert_keep_mask(hip_device):
    """End to end: importance -> tm_expert_keep_mask equals the oracle's
    build_prefill_keep_mask on the device's importance (random scores leave
    no near-tie at the keep boundary here)."""
    from table_moe.skip.pruning import build_prefill_keep_mask
    from table_moe.utils import compute_and_cache_importance

    g = torch.Generator().manual_seed(9)
    n, h, hkv, d, e, k = 1024, 32, 4, 128, 128, 8
    qs = torch.randn(1, h, n, d, generator=g).to(torch.bfloat16)
    ks = torch.randn(1, hkv, n, d, generator=g).to(torch.bfloat16)
    dev = hip_device
    attn = compute_and_cache_importance(qs.to(dev), ks.to(dev), d ** -0.5).view(-1)
    sel = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)])
    w = torch.softmax(torch.randn(n, e, generator=g), dim=1).gather(1, sel)
    mask = build_prefill_keep_mask(sel.to(dev), w.to(dev), attn, e, 0.6)
    torch.cuda.synchronize()
    want, _ = O.build_prefill_keep_mask(sel.numpy(), np64(w), np64(attn), e, 0.6)
    np.testing.assert_array_equal(mask.cpu().numpy(), want)


@pytest.mark.parametrize("b,h,hkv,d,s,out_len", [(1, 8, 1, 128, 1, 1), (1, 3, 3, 64, 63, 63), (2, 16, 2, 128, 65, 40),
                                                 (1, 12, 3, 192, 129, 129), (1, 40, 20, 256, 600, 577),
                                                 (1, 16, 1, 64, 16384, 16384), (1, 8, 4, 128, 16449, 16449),
                                                 (1, 64, 64, 64, 700, 1)])
def test_importance_key_chunks_and_head_sets(hip_device, b, h, hkv, d, s, out_len):
    """Chunk edges of 64 and of 512 keys (from 16385 on), 1 to 16 heads per KV
    head, masked keys (a whole chunk of them too) and a shorter output."""
    from table_moe.utils.importance import last_query_importance

    g = torch.Generator().manual_seed(s + 7 * h)
    q = torch.randn(b, h, d, generator=g).to(torch.bfloat16)
    ks = torch.randn(b, s, hkv, d, generator=g).to(torch.bfloat16)
    mask = torch.rand(b, s, generator=g) < 0.9
    mask[:, -1] = True
    if s > 200:
        mask[:, 64:192] = False
    dev = hip_device
    got = last_query_importance(q.to(dev), ks.to(dev), hkv, d ** -0.5, True, mask.to(dev), out_len)
    torch.cuda.synchronize()
    want = O.last_query_importance(np64(q), np64(ks), hkv, d ** -0.5, O.F32, key_mask=mask.numpy(), out_len=out_len)
    np.testing.assert_allclose(np64(got), want, rtol=1e-4, atol=1e-9)


@pytest.mark.parametrize("s,lo,hi", [(300, 64, 192), (4099, 128, 2700), (16500, 16384, 16500)])
def test_importance_scores_of_minus_infinity(hip_device, s, lo, hi):
    """Keys that score -inf, whole chunks of them, take no weight and leave the
    others' as if they were masked."""
    from table_moe.utils.importance import last_query_importance

    g = torch.Generator().manual_seed(s)
    h, hkv, d = 8, 2, 128
    q = torch.randn(1, h, d, generator=g).to(torch.bfloat16)
    q[:, :, 0] = 1.0
    ks = torch.randn(1, s, hkv, d, generator=g).to(torch.bfloat16)
    mask = torch.ones(1, s, dtype=torch.bool)
    mask[:, lo:hi] = False
    want = O.last_query_importance(np64(q), np64(ks), hkv, d ** -0.5, O.F32, key_mask=mask.numpy(), out_len=s)
    ks[:, lo:hi, :, 0] = -float("inf")
    dev = hip_device
    got = last_query_importance(q.to(dev), ks.to(dev), hkv, d ** -0.5, True, None, s)
    torch.cuda.synchronize()
    np.testing.assert_allclose(np64(got), want, rtol=1e-4, atol=1e-9)


@pytest.mark.parametrize("s", [65, 4099, 16384])
def test_importance_in_the_least_workspace(hip_device, s):
    """The scores and a statistic per 512 keys are enough (one byte less is
    refused): the same importance up to the order of the sums, and nothing past
    the workspace is written."""
    from table_moe import _native as N
    from table_moe.utils.importance import last_query_importance

    g = torch.Generator().manual_seed(s)
    h, hkv, d = 8, 2, 128
    dev = hip_device
    q = torch.randn(1, h, d, generator=g).to(torch.bfloat16).to(dev)
    ks = torch.randn(1, s, hkv, d, generator=g).to(torch.bfloat16).to(dev)
    want = last_query_importance(q, ks, hkv, d ** -0.5, True)
    need = (4 * h * s + 255) // 256 * 256 + 8 * h * ((s + 511) // 512)
    assert need < N.lib().tm_importance_workspace_size(1, h, s)
    ws = torch.full((need + 4096,), 77, dtype=torch.uint8, device=dev)
    out = torch.empty(1, s, device=dev)

    def call(nbytes):
        N.call("tm_last_query_importance", N.dtype_tag(q.dtype), q.data_ptr(), q.stride(0), q.stride(1), ks.data_ptr(),
               ks.stride(0), ks.stride(1), ks.stride(2), 1, h, hkv, d, s, d ** -0.5, N.TM_SCORE_F32, None, 0, s,
               out.data_ptr(), s, ws.data_ptr(), nbytes, N.stream(dev))

    with pytest.raises(ValueError):
        call(need - 1)
    call(need)
    torch.cuda.synchronize()
    np.testing.assert_allclose(np64(out), np64(want), rtol=1e-5, atol=0)
    assert bool((ws[need:] == 77).all())
