"""bf16 dense and sparse decode on the matrix cores, at the sizes where tiles,
splits and kernels change (32-row tiles, the 16-tile and 16-tile-plus-tail
limits of the single-pass kernel, split contexts), with a workspace, with none
and from tensors that start off a 16-byte boundary, against the fp64 oracle."""

import numpy as np
import pytest
import torch

from helpers import SCALE, dev, randn, say
from oracle import kvdec_oracle as O

pytestmark = pytest.mark.gpu


def _bf16(shape, seed):
    return torch.from_numpy(randn(shape, seed)).to(torch.bfloat16)


def _check(o, ref):
    """One rounding to bf16 of a result within 2e-6 of the oracle's: fp32 sums
    of logits and outputs of order 1 (a few units of 2^-23 each)."""
    ref = np.asarray(ref, dtype=np.float64)
    e = np.floor(np.log2(np.maximum(np.abs(ref), 2.0**-126)))
    assert (np.abs(o.float().cpu().numpy() - ref) - 2.0 ** (e - 8)).max() <= 2e-6


@pytest.mark.parametrize("H,KVH", [(64, 8), (32, 2), (8, 8)])
@pytest.mark.parametrize("L", [1, 31, 33, 511, 512, 516, 517, 545, 4100])
def test_dense(H, KVH, L, device):
    from dense_kernel import dense_decode_attention
    q, k, v = _bf16((2, H, 128), 1), _bf16((2, KVH, L, 128), 2), _bf16((2, KVH, L, 128), 3)
    say(f"dense bf16 H={H} KVH={KVH} L={L}")
    o = dense_decode_attention(q.to(device), k.to(device), v.to(device), seq_len=L)
    _check(o, O.dense_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), SCALE))


@pytest.mark.parametrize("W", [29, 508, 512, 1500])
@pytest.mark.parametrize("layout", ["linear", "ring"])
def test_sparse_lengths_and_garbage_rows(W, layout, device):
    """Rows past the valid slots hold NaN: they must not reach the output."""
    from sparse_kernel import sparse_decode_attention
    B, H, KVH, S = 3, 64, 8, 4
    q, k, v = _bf16((B, H, 128), 4), _bf16((B, KVH, S + W, 128), 5), _bf16((B, KVH, S + W, 128), 6)
    f = [x.float().numpy() for x in (q, k, v)]
    lay = 0 if layout == "linear" else 1
    for L in (1, S + W // 2, S + W, 100000):
        valid = O.slot_validity(L, W, S, lay)
        kd, vd = k.clone(), v.clone()
        kd[:, :, ~torch.from_numpy(valid)] = float("nan")
        vd[:, :, ~torch.from_numpy(valid)] = float("nan")
        say(f"sparse bf16 {layout} W={W} L={L}")
        o = sparse_decode_attention(q.to(device), kd.to(device), vd.to(device), seq_len=L, window=W, sink=S,
                                    layout=layout)
        _check(o, O.masked_attention(*f, valid, SCALE))
    lens = np.array([1, S + W // 3, S + W + 9], dtype=np.int32)
    o = sparse_decode_attention(q.to(device), k.to(device), v.to(device), seq_len=dev(lens, device), window=W,
                                sink=S, layout=layout)
    _check(o, O.sparse_attention_varlen(*f, lens, W, S, SCALE, layout=lay))


@pytest.mark.parametrize("L,splits_held", [(517, 0), (9000, 0), (9000, 3), (9000, 1000)])
def test_any_workspace(L, splits_held, device):
    """bf16 calls run with whatever workspace they are given."""
    import _kvdec as K
    B, H, KVH = 1, 64, 8
    q, k, v = (x.to(device) for x in (_bf16((B, H, 128), 7), _bf16((B, KVH, L, 128), 8), _bf16((B, KVH, L, 128), 9)))
    o = torch.empty_like(q)
    nbytes = splits_held * KVH * (H // KVH) * 130 * 4
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=device)
    say(f"dense bf16 L={L} workspace {nbytes}")
    rc = K.lib.kvdec_dense_decode(K.ptr(q), K.ptr(k), K.ptr(v), K.ptr(o), K.BF16, B, H, KVH, L, 128, SCALE,
                                  K.ptr(ws) if nbytes else None, nbytes, K.stream_of(q))
    assert rc == 0
    _check(o, O.dense_attention(*(x.float().cpu().numpy() for x in (q, k, v)), SCALE))


def test_off_16_byte_boundary(device):
    from dense_kernel import dense_decode_attention
    B, H, KVH, L = 2, 64, 8, 700
    k, v, q = _bf16((B, KVH, L, 128), 10), _bf16((B, KVH, L, 128), 11), _bf16((B, H, 128), 12)
    buf = torch.zeros(k.numel() + 1, dtype=torch.bfloat16, device=device)
    buf[1:] = k.flatten().to(device)
    say("dense bf16, k one element off alignment")
    o = dense_decode_attention(q.to(device), buf[1:].view(k.shape), v.to(device), seq_len=L)
    _check(o, O.dense_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), SCALE))


def test_dominant_token(device):
    """A token that carries nearly all of a head's weight: the probabilities'
    three bf16 parts leave one output rounding."""
    from dense_kernel import dense_decode_attention
    B, H, KVH, L = 1, 16, 2, 600
    q, k, v = _bf16((B, H, 128), 13), _bf16((B, KVH, L, 128), 14), _bf16((B, KVH, L, 128), 15)
    k[:, :, 77] = (q.view(B, KVH, 8, 128).mean(2) * 2).to(torch.bfloat16)
    v *= 3
    say("dense bf16 dominant token")
    o = dense_decode_attention(q.to(device), k.to(device), v.to(device), seq_len=L)
    _check(o, O.dense_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), SCALE))


@pytest.mark.parametrize("L", [20, 600, 9000])
def test_logits_far_below_zero(L, device):
    """Every logit near -1e33: still weights that sum to 1."""
    from dense_kernel import dense_decode_attention
    q = torch.full((1, 16, 128), 1e16, dtype=torch.bfloat16)
    k = torch.full((1, 2, L, 128), -1e15, dtype=torch.bfloat16)
    v = _bf16((1, 2, L, 128), 16)
    say(f"dense bf16 low logits L={L}")
    o = dense_decode_attention(q.to(device), k.to(device), v.to(device), seq_len=L)
    # equal logits: the mean of V
    want = v.double().mean(2, keepdim=True).expand(1, 2, 8, 128).reshape(1, 16, 128).numpy()
    _check(o, want)


def _check_infinite(o, ref):
    got, fin = o.double().cpu().numpy(), np.isfinite(ref)
    assert np.array_equal(got[~fin], ref[~fin]) and (~fin).any()
    _check(torch.where(torch.from_numpy(fin).to(o.device), o, torch.zeros_like(o)), np.where(fin, ref, 0.0))


@pytest.mark.parametrize("H,KVH", [(32, 2), (3, 1)])
@pytest.mark.parametrize("L,at", [(20, 3), (500, 499), (515, 512), (9000, 0), (9000, 4700), (9000, 8999)])
def test_infinite_value_rows(H, KVH, L, at, device):
    """An attended infinity in V is that infinity in its channel's output."""
    from dense_kernel import dense_decode_attention
    q, k, v = _bf16((2, H, 128), 17), _bf16((2, KVH, L, 128), 18), _bf16((2, KVH, L, 128), 19)
    v[:, :, at, 5], v[:, 0, at, 77] = float("inf"), float("-inf")
    say(f"dense bf16 H={H} L={L} infinite V at {at}")
    o = dense_decode_attention(q.to(device), k.to(device), v.to(device), seq_len=L)
    _check_infinite(o, O.dense_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), SCALE))


@pytest.mark.parametrize("W", [29, 512, 1500])
@pytest.mark.parametrize("layout", ["linear", "ring"])
def test_infinite_sparse_rows(W, layout, device):
    """The same under the sink and window rule, NaN in the slots it masks."""
    from sparse_kernel import sparse_decode_attention
    B, H, KVH, S = 3, 24, 8, 4
    q, k, v = _bf16((B, H, 128), 20), _bf16((B, KVH, S + W, 128), 21), _bf16((B, KVH, S + W, 128), 22)
    v[:, :, 1, 9] = float("inf")
    f = [x.float().numpy() for x in (q, k, v)]
    lay = 0 if layout == "linear" else 1
    for L in (2, S + W // 2, 100000):
        valid = O.slot_validity(L, W, S, lay)
        kd, vd = k.clone(), v.clone()
        kd[:, :, ~torch.from_numpy(valid)] = float("nan")
        vd[:, :, ~torch.from_numpy(valid)] = float("nan")
        say(f"sparse bf16 {layout} W={W} L={L} infinite V")
        o = sparse_decode_attention(q.to(device), kd.to(device), vd.to(device), seq_len=L, window=W, sink=S,
                                    layout=layout)
        _check_infinite(o, O.masked_attention(*f, valid, SCALE))
    lens = np.array([2, S + W // 3, S + W + 9], dtype=np.int32)
    o = sparse_decode_attention(q.to(device), k.to(device), v.to(device), seq_len=dev(lens, device), window=W,
                                sink=S, layout=layout)
    _check_infinite(o, O.sparse_attention_varlen(*f, lens, W, S, SCALE, layout=lay))
