"""The generic decode kernel's 16-token tiles at their edges: row counts around a
tile, a round of the waves and a split, every query group size, tensors off a
16-byte boundary, slots that were never written (NaN behind the mask), logits
far outside the usual range; and KIVI caches whose groups hold fewer than four
channels, one code per byte to eight, sinks and residuals of no whole tile."""

import numpy as np
import pytest
import torch

from helpers import SCALE, assert_nearly_rounded, dev, randn
from oracle import kvdec_oracle as O

pytestmark = pytest.mark.gpu

DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _ref(q, k, v):
    """[B, H, 128] fp64 attention of q over k, v [B, KVH, n, 128]."""
    B, H, _ = q.shape
    KVH = k.shape[1]
    s = torch.matmul(q.double().view(B, KVH, H // KVH, 128), k.double().transpose(2, 3).contiguous()) * SCALE
    return torch.matmul(torch.softmax(s, -1), v.double()).view(B, H, 128)


def _rows(shape, dt, seed, offset=0):
    """Random rows, `offset` elements past an aligned address."""
    n = int(np.prod(shape))
    flat = torch.empty(n + offset, dtype=DT[dt], device="cuda")
    x = flat[offset:].view(shape)
    x.copy_(torch.from_numpy(randn(shape, seed)).to(DT[dt]))
    return x


def _check(o, ref, dt):
    # fp32: the repository's 2e-6 for N(0, 1) rows; bf16: half an ulp more
    half_ulp = 2.0 ** (torch.floor(torch.log2(ref.abs().clamp(min=2.0**-126))) - 8) if dt == "bf16" else 0.0
    assert ((o.double() - ref).abs() - half_ulp).max().item() <= 2e-6


@pytest.mark.parametrize("L", [1, 15, 16, 17, 127, 128, 129, 255, 257, 2047, 4113])
@pytest.mark.parametrize("dt,offset", [("fp32", 0), ("fp32", 1), ("bf16", 1)])
def test_rows_edges(L, dt, offset, device):
    from dense_kernel import dense_decode_attention
    for B, H, KVH in ((1, 16, 1), (2, 6, 2), (3, 5, 5)):
        q = _rows((B, H, 128), dt, L)
        k, v = _rows((B, KVH, L, 128), dt, L + 1, offset), _rows((B, KVH, L, 128), dt, L + 2, offset)
        _check(dense_decode_attention(q, k, v, L), _ref(q, k, v), dt)


@pytest.mark.parametrize("W,sink", [(12, 4), (61, 3), (300, 5), (8000, 4)])
def test_masked_slots_hold_anything(W, sink, device):
    from sparse_kernel import sparse_decode_attention
    q = _rows((3, 16, 128), "fp32", 1)
    k, v = _rows((3, 2, sink + W, 128), "fp32", 2), _rows((3, 2, sink + W, 128), "fp32", 3)
    lens = torch.tensor([1, sink + W // 2, 10 * W], dtype=torch.int32, device=device)
    slots = torch.arange(sink + W, device=device)
    refs = []
    for b, n in enumerate(lens.tolist()):
        ok = torch.where(slots < sink, slots < n, n - W + slots - sink >= sink)
        refs.append(_ref(q[b:b + 1], k[b:b + 1, :, ok], v[b:b + 1, :, ok])[0])
        k[b, :, ~ok], v[b, :, ~ok] = float("nan"), float("inf")
    _check(sparse_decode_attention(q, k, v, lens, W, sink=sink), torch.stack(refs), "fp32")
    _check(sparse_decode_attention(q[1:2], k[1:2], v[1:2], int(lens[1]), W, sink=sink), refs[1][None], "fp32")


@pytest.mark.parametrize("size", [1e-30, 1e12])
def test_logits_of_any_size(size, device):
    """Uniform weights, or one row's value: no starting maximum stands in the way."""
    from dense_kernel import dense_decode_attention
    q, k, v = _rows((1, 8, 128), "fp32", 1) * size, _rows((1, 1, 900, 128), "fp32", 2), _rows((1, 1, 900, 128), "fp32", 3)
    k -= 40 * torch.sign(q.sum(1, keepdim=True))[:, None]     # most logits far below zero
    k = k.contiguous()
    _check(dense_decode_attention(q, k * size, v, 900), _ref(q, k * size, v), "fp32")


@pytest.mark.parametrize("L,at", [(17, 16), (900, 0), (5000, 4999)])
def test_nan_reaches_the_output(L, at, device):
    """An attended token's NaN, also where its tile holds no other logit."""
    from dense_kernel import dense_decode_attention
    q, k, v = _rows((1, 8, 128), "fp32", 1), _rows((1, 1, L, 128), "fp32", 2), _rows((1, 1, L, 128), "fp32", 3)
    k[:, :, at, 5] = float("nan")
    assert dense_decode_attention(q, k, v, L).isnan().all()


@pytest.mark.parametrize("L", [4007, 4039, 4331])
def test_split_sums_are_divided_once(L, device):
    """Equal logits over rows of ones, split: n / n is 1, n * (1 / n) is not."""
    from dense_kernel import dense_decode_attention
    assert np.float32(L) * (np.float32(1) / np.float32(L)) != 1
    q, v = torch.zeros((1, 16, 128), device=device), torch.ones((1, 2, L, 128), device=device)
    print(f"fp32 dense of ones L={L}", flush=True)
    assert (dense_decode_attention(q, v, v, seq_len=L) == 1).all()


@pytest.mark.parametrize("bits,group", [(8, 1), (8, 2), (5, 4), (8, 32), (4, 2), (3, 4), (4, 64), (2, 4), (1, 8),
                                        (1, 128)])
@pytest.mark.parametrize("q_dt,res_dt", [("fp16", "fp16"), ("fp32", "bf16")])
def test_kivi_forms(bits, group, q_dt, res_dt, device):
    from quant_kernel import sparse_decode_attention_quantized
    B, H, KVH, S, R = 2, 12, 2, min(group, 3), 37
    W = R + group * (-(-150 // group))
    # neighbours of opposite sign: every group of two or more spans 1 at least,
    # so that no zero point leaves fp16's range
    sign = torch.tensor([1.0, -1.0]).repeat(64)[None] * torch.tensor([1.0, -1.0]).repeat(S + W)[:S + W, None]
    kc, vc = (((torch.from_numpy(randn((B, KVH, S + W, 128), s)).abs() + 0.5) * sign).to(DT[res_dt]) for s in (5, 6))
    kc[..., 3] *= 10
    hc = O.build_quantized_kv_cache(kc.float().numpy(), vc.float().numpy(), residual_size=R, sink=S, group_size=group,
                                    bits=bits)
    hc["k_residual"], hc["v_residual"] = (x[:, :, -R:].float().numpy() for x in (kc, vc))
    c = {n: dev(x, device).to(DT[res_dt]) if n.endswith("residual") else dev(x, device) for n, x in hc.items()}
    q = torch.from_numpy(randn((B, H, 128), 7)).to(DT[q_dt])
    for L in (100000, S + W - 9, S + 20):
        o = sparse_decode_attention_quantized(q.to(device), *[c[n] for n in O.CACHE_KEYS], seq_len=L, window=W, sink=S,
                                              residual_size=R, group_size=group, bits=bits)
        ref = O.quantized_attention_masked(q.float().numpy(), hc, L, W, SCALE, sink=S, residual_size=R,
                                           group_size=group, bits=bits)
        if q_dt == "fp32":
            # logits up to ~20 (the x10 channel): their fp32 products' error, 2e-6, in the weights
            assert np.abs(o.cpu().numpy() - ref).max() <= 1e-5
        else:
            assert_nearly_rounded(o.cpu().numpy(), ref)
