"""The wide KIVI decode over few KV heads, split over the GPU, and (in one
pass) at per-sequence lengths: window-old group counts around the kernel's and
the plan's limits and uneven splits, steady state and ramp-up (fewer groups than
the workspace was planned for), every workspace size, against the fp64 oracle."""

import numpy as np
import pytest
import torch

from helpers import ATTN_TOL, SCALE, assert_nearly_rounded, dev, host, max_abs, randn, say
from oracle import kvdec_oracle as O

pytestmark = pytest.mark.gpu


def _problem(B, H, KVH, S, W, seed, device):
    from quant_kernel import build_quantized_kv_cache
    kc = randn((B, KVH, S + W, 128), seed).astype(np.float16)
    kc[..., 3] *= 10
    vc = randn((B, KVH, S + W, 128), seed + 1).astype(np.float16)
    q = randn((B, H, 128), seed + 2).astype(np.float16)
    c = build_quantized_kv_cache(dev(kc, device), dev(vc, device), sink=S)
    return q, {k: host(v) for k, v in c.items()}, c


def _attend(q, c, L, W, S, device):
    from quant_kernel import sparse_decode_attention_quantized
    return host(sparse_decode_attention_quantized(dev(q, device), *[c[k] for k in O.CACHE_KEYS], seq_len=L,
                                                  window=W, sink=S))


@pytest.mark.parametrize("B,H,KVH", [(1, 64, 8), (3, 8, 8), (1, 12, 2), (40, 16, 2)])
@pytest.mark.parametrize("groups,S,splits", [(12, 4, 1), (16, 1, 1), (17, 16, 1), (29, 4, 3), (33, 16, 4), (77, 4, 9)])
def test_split_over_few_heads(B, H, KVH, groups, S, splits, device):
    import _kvdec as K
    W = 128 + 32 * groups
    if B > 4 and groups > 40:
        pytest.skip("covered by the smaller batches")
    # (a workgroup per CU: at most 3 splits of 80 KV heads)
    assert K.lib.kvdec_num_splits(K.KIND_KIVI_SPLIT, B, KVH, W - 128) == min(splits, 256 // (B * KVH))
    q, hc, c = _problem(B, H, KVH, S, W, 40 + groups, device)
    for L in (163840, S + W - 7, S + W // 2, 100, 1):
        say(f"kivi split B={B} H={H} KVH={KVH} groups={groups} S={S} L={L}")
        o = _attend(q, c, L, W, S, device)
        ref = O.quantized_attention_masked(q, hc, L, W, SCALE, sink=S)
        assert max_abs(o, ref) < ATTN_TOL, L
        assert_nearly_rounded(o, ref)
    rng = np.random.default_rng(groups)
    lens = np.where(rng.random(B) < 0.6, rng.integers(1, S + W, B), 100000).astype(np.int32)
    o = _attend(q, c, dev(lens, device), W, S, device)
    ref = O.quantized_attention_varlen(q, hc, lens, W, SCALE, sink=S)
    assert_nearly_rounded(o, ref)


@pytest.mark.parametrize("held", [0, 1, 2, 3, 5, 1000])
def test_any_workspace(held, device):
    """Fewer splits in a smaller workspace, one pass in none; nothing past
    the workspace's end is written."""
    import _kvdec as K
    B, H, KVH, S, W, R = 1, 64, 8, 4, 128 + 32 * 45, 128
    q, hc, c = _problem(B, H, KVH, S, W, 7, device)
    qd = dev(q, device)
    o = torch.empty_like(qd)
    nbytes = held * B * H * 130 * 4
    ws = torch.full((nbytes // 4 + 1024,), 7.0, device=device)
    arr = (K._vp * 12)(*[K.ptr(c[k]) for k in O.CACHE_KEYS[2:]])
    say(f"kivi split workspace of {held} splits")
    rc = K.lib.kvdec_sparse_decode_kivi(K.ptr(qd), K.ptr(c["k_residual"]), K.ptr(c["v_residual"]), arr, K.ptr(o),
                                        B, H, KVH, 163840, W, S, R, 32, 2, SCALE, K.ptr(ws) if held else None,
                                        nbytes, K.stream_of(qd))
    assert rc == 0
    assert_nearly_rounded(host(o), O.quantized_attention_masked(q, hc, 163840, W, SCALE, sink=S))
    assert bool((ws[nbytes // 4:] == 7.0).all())


@pytest.mark.parametrize("token", [0, 700, 1279])
def test_infinite_partials(token, device):
    """An infinite V row in the first, a middle and the last window-old split
    of a 4-bit call reaches its channels as that infinity, and no others."""
    import _kvdec as K
    from quant_kernel import sparse_decode_attention_quantized
    B, H, KVH, S, R, bits = 1, 8, 1, 4, 128, 4
    W = R + 32 * 40
    assert K.lib.kvdec_num_splits(K.KIND_KIVI_SPLIT, B, KVH, W - R) == 5
    kc, vc, q = randn((B, KVH, S + W, 128), 81), randn((B, KVH, S + W, 128), 82), randn((B, H, 128), 83)
    hc = O.build_quantized_kv_cache(kc, vc, residual_size=R, sink=S, bits=bits)
    hc = {k: v.astype(np.float16) if k.endswith("residual") else v for k, v in hc.items()}
    hc["v_win_zero"][:, :, token, 1] = np.inf
    q = q.astype(np.float16)
    say(f"kivi 4-bit split, infinite V of token {token}")
    o = host(sparse_decode_attention_quantized(dev(q, device), *[dev(hc[k], device) for k in O.CACHE_KEYS],
                                               seq_len=163840, window=W, sink=S, bits=bits))
    ref = O.quantized_attention_masked(q, hc, 163840, W, SCALE, sink=S, bits=bits)
    assert (ref[..., 32:64] == -np.inf).all() and (o[..., 32:64] == -np.inf).all()
    rest = np.r_[0:32, 64:128]
    assert_nearly_rounded(o[..., rest], ref[..., rest])
