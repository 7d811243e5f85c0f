"""The KIVI decode on the matrix cores at 4-bit codes and under bf16 queries,
against the fp64 oracle: window-old group counts from none to several per wave,
partial residuals, sinks up to the form's limit and past it, ramp-up with
never-written slots, per-sequence lengths, scales far from 1, and the calls
that stay with the generic kernel (other widths, types, groups, alignments)."""

import numpy as np
import pytest
import torch

from helpers import SCALE, assert_nearly_rounded, dev, randn, say
from oracle import kvdec_oracle as O

pytestmark = pytest.mark.gpu

DT = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _check(o, ref, dt):
    """fp16: half an ulp plus the repository's 5e-5; bf16: half an ulp plus
    1e-5, a few fp32 ulps of logits up to ~20 (the x10 channel) and of the
    two-part products."""
    ref = np.asarray(ref, dtype=np.float64)
    if dt == "fp16":
        return assert_nearly_rounded(o.cpu().numpy(), ref)
    e = np.floor(np.log2(np.maximum(np.abs(ref), 2.0**-126)))
    assert (np.abs(o.float().cpu().numpy() - ref) - 2.0 ** (e - 8)).max() <= 1e-5


def _cache(B, KVH, S, W, R, bits, dt, seed, k_mul=1.0, v_mul=1.0):
    kc = randn((B, KVH, S + W, 128), seed) * k_mul
    kc[..., 3] *= 10
    vc = randn((B, KVH, S + W, 128), seed + 1) * v_mul
    kc, vc = (torch.from_numpy(x).to(DT[dt]) for x in (kc, vc))
    hc = O.build_quantized_kv_cache(kc.float().numpy(), vc.float().numpy(), residual_size=R, sink=S, bits=bits)
    res = min(R, W)
    hc["k_residual"], hc["v_residual"] = (x[:, :, -res:].float().numpy() for x in (kc, vc))
    return hc


def _upload(hc, dt, device):
    return {k: dev(v, device).to(DT[dt]) if k.endswith("residual") else dev(v, device) for k, v in hc.items()}


def _attend(q, c, L, W, S, R, bits):
    from quant_kernel import sparse_decode_attention_quantized
    return sparse_decode_attention_quantized(q, *[c[k] for k in O.CACHE_KEYS], seq_len=L, window=W, sink=S,
                                             residual_size=R, bits=bits)


@pytest.mark.parametrize("bits,dt", [(4, "fp16"), (4, "bf16"), (2, "bf16")])
@pytest.mark.parametrize("W,S,R", [(40, 4, 128), (128, 16, 128), (160, 4, 128), (128 + 32 * 9, 1, 128),
                                   (100 + 32 * 3, 4, 100), (128 + 32 * 61, 3, 128), (256, 17, 128), (352, 4, 160)])
def test_forms(bits, dt, W, S, R, device):
    B, H, KVH = 2, 64, 8
    hc = _cache(B, KVH, S, W, R, bits, dt, 10 * bits + W)
    c = _upload(hc, dt, device)
    q = torch.from_numpy(randn((B, H, 128), 3)).to(DT[dt])
    qh = q.float().numpy()
    for L in (163840, S + W - 5, S + W // 3, 2):
        say(f"kivi bits={bits} {dt} W={W} S={S} R={R} L={L}")
        o = _attend(q.to(device), c, L, W, S, R, bits)
        _check(o, O.quantized_attention_masked(qh, hc, L, W, SCALE, sink=S, residual_size=R, bits=bits), dt)
    lens = np.array([S + W // 2, 90000], dtype=np.int32)
    o = _attend(q.to(device), c, dev(lens, device), W, S, R, bits)
    _check(o, O.quantized_attention_varlen(qh, hc, lens, W, SCALE, sink=S, residual_size=R, bits=bits), dt)


@pytest.mark.parametrize("bits,dt", [(4, "fp16"), (4, "bf16"), (2, "bf16")])
@pytest.mark.parametrize("q_mul,k_mul,v_mul", [(1e-3, 1e3, 1.0), (300.0, 1e-3, 1.0), (1.0, 1.0, 300.0),
                                               (1.0, 1.0, 1e-3)])
def test_scales_far_from_one(bits, dt, q_mul, k_mul, v_mul, device):
    """Logits of the usual size from large and small factors, and outputs of
    any size: relative to the largest output the bounds above hold."""
    B, H, KVH, S, W, R = 1, 16, 2, 4, 448, 128
    hc = _cache(B, KVH, S, W, R, bits, dt, 77, k_mul, v_mul)
    q = (torch.from_numpy(randn((B, H, 128), 5)) * q_mul).to(DT[dt])
    say(f"kivi bits={bits} {dt} q x {q_mul} k x {k_mul} v x {v_mul}")
    o = _attend(q.to(device), _upload(hc, dt, device), 163840, W, S, R, bits)
    ref = O.quantized_attention_masked(q.float().numpy(), hc, 163840, W, SCALE, sink=S, residual_size=R, bits=bits)
    got, top = o.double().cpu().numpy(), np.abs(ref).max()
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ref), 1e-30))) - (11 if dt == "fp16" else 8))
    # below fp16's normal range the output's own spacing is 2^-24
    assert (np.abs(got - ref) - ulp).max() <= 1e-5 * top + (2.0**-25 if dt == "fp16" else 0.0)


@pytest.mark.parametrize("bits,dt", [(4, "fp16"), (4, "bf16"), (2, "bf16")])
@pytest.mark.parametrize("odd", ["x2^14", "x2^-14", "nan", "inf", "-inf"])
def test_heads_stand_alone(bits, dt, odd, device):
    """One query head far from the size of the others of its KV head, or with
    one element that is not finite: the others' results do not change by it."""
    B, H, KVH, S, W, R = 1, 16, 2, 4, 448, 128
    hc = _cache(B, KVH, S, W, R, bits, dt, 55)
    q = torch.from_numpy(randn((B, H, 128), 9))
    q[:, 2] *= {"x2^14": 2.0**14, "x2^-14": 2.0**-14}.get(odd, 1.0)
    q = q.to(DT[dt])
    ref = O.quantized_attention_masked(q.float().numpy(), hc, 163840, W, SCALE, sink=S, residual_size=R, bits=bits)
    if odd[0] != "x":
        q[:, 2, 40] = float(odd)
    say(f"kivi bits={bits} {dt} head 2 {odd}")
    o = _attend(q.to(device), _upload(hc, dt, device), 163840, W, S, R, bits)
    rest = [h for h in range(H) if h != 2]
    _check(o[:, rest], ref[:, rest], dt)
    if odd == "nan":
        assert o[:, 2].isnan().all()


def _same(o, ref, dt):
    """_check where the oracle is finite, the same infinities where not."""
    got, fin = o.double().cpu().numpy(), np.isfinite(ref)
    assert np.array_equal(got[~fin], ref[~fin])
    _check(torch.where(torch.from_numpy(fin).to(o.device), o, torch.zeros_like(o)), np.where(fin, ref, 0.0), dt)


@pytest.mark.parametrize("bits,dt", [(4, "fp16"), (4, "bf16"), (2, "bf16")])
@pytest.mark.parametrize("what", ["k_zero", "k_scale", "v_zero", "v_scale", "v_residual"])
def test_infinities_in_the_cache(bits, dt, what, device):
    """A nearly constant channel far from 0 has an infinite zero point once
    quantized: its 32 keys are -inf, weight 0 under a positive query.  Infinite
    scales, V zero points and V rows likewise give scale * (code - zero)."""
    B, H, KVH, S, W, R = 2, 16, 2, 4, 448, 128
    kc, vc = randn((B, KVH, S + W, 128), 71), randn((B, KVH, S + W, 128), 72)
    if what == "k_zero":
        kc[:, :, S + 32:S + 64, 40] = -20000 + 0.05 * randn((B, KVH, 32), 73)
    hc = O.build_quantized_kv_cache(kc, vc, residual_size=R, sink=S, bits=bits)
    hc["k_residual"], hc["v_residual"] = (
        torch.from_numpy(x[:, :, -R:]).to(DT[dt]).float().numpy() for x in (kc, vc))
    if what == "k_zero":
        assert (hc["k_win_zero"][:, :, 1, 40] == np.inf).all()
    elif what == "k_scale":
        hc["k_win_scale"][:, :, 1, 40], hc["k_win_zero"][:, :, 1, 40] = np.inf, 20
    elif what == "v_zero":
        hc["v_win_zero"][:, :, 37, 2] = np.inf
    elif what == "v_scale":
        hc["v_win_scale"][:, :, 37, 2], hc["v_win_zero"][:, :, 37, 2] = np.inf, -1
    else:
        hc["v_residual"][:, :, 3, 7] = np.inf
    q = torch.from_numpy(randn((B, H, 128), 74))
    q[..., 40] = q[..., 40].abs() + 0.1
    q = q.to(DT[dt])
    c = _upload(hc, dt, device)
    say(f"kivi bits={bits} {dt} infinite {what}")
    for L in (163840, S + W - 20):
        ref = O.quantized_attention_masked(q.float().numpy(), hc, L, W, SCALE, sink=S, residual_size=R, bits=bits)
        assert not np.isnan(ref).any() and np.isinf(ref).any() == (what[0] == "v")
        _same(_attend(q.to(device), c, L, W, S, R, bits), ref, dt)
    lens = np.array([S + W - 20, 90000], dtype=np.int32)
    ref = O.quantized_attention_varlen(q.float().numpy(), hc, lens, W, SCALE, sink=S, residual_size=R, bits=bits)
    _same(_attend(q.to(device), c, dev(lens, device), W, S, R, bits), ref, dt)


@pytest.mark.parametrize("bits", [2, 4])
def test_channels_far_apart(bits, device):
    """Query channels 2^-20 the size of the head's largest, against keys 2^10
    times the others': the small ones keep all their bits."""
    B, H, KVH, S, W, R = 1, 16, 2, 4, 448, 128
    small = torch.arange(128) % 2 == 0
    kc, vc = (torch.from_numpy(randn((B, KVH, S + W, 128), n)) for n in (61, 62))
    kc = torch.where(small, kc * 2.0**10, kc).to(torch.bfloat16)
    vc = vc.to(torch.bfloat16)
    q = torch.from_numpy(randn((B, H, 128), 63)) * 8
    q = torch.where(small, q * 2.0**-20, q).to(torch.bfloat16)
    hc = O.build_quantized_kv_cache(kc.float().numpy(), vc.float().numpy(), residual_size=R, sink=S, bits=bits)
    hc["k_residual"], hc["v_residual"] = (x[:, :, -R:].float().numpy() for x in (kc, vc))
    ref = O.quantized_attention_masked(q.float().numpy(), hc, 163840, W, SCALE, sink=S, residual_size=R, bits=bits)
    say(f"kivi bits={bits} channels far apart")
    o = _attend(q.to(device), _upload(hc, "bf16", device), 163840, W, S, R, bits)
    _check(o, ref, "bf16")


def _relative(o, ref, dt):
    """Half an ulp plus 1e-5 of the head's largest output (2^-25: fp16's own
    spacing below its normal range)."""
    got, top = o.double().cpu().numpy(), np.abs(ref).max(-1, keepdims=True)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ref), 1e-30))) - (11 if dt == "fp16" else 8))
    assert (np.abs(got - ref) - ulp - 1e-5 * top).max() <= (2.0**-25 if dt == "fp16" else 0.0)


@pytest.mark.parametrize("bits,dt", [(4, "fp16"), (4, "bf16"), (2, "bf16")])
@pytest.mark.parametrize("span,at", [(8, 4), (16, 8), (17, 8), (18, 9), (24, 12), (17, 15), (20, 17)])
def test_key_scales_far_apart(bits, dt, span, at, device):
    """Every other channel's keys 2^span the others' (2^-at), its query as much
    smaller; at the low ends the small scales are subnormal fp16."""
    if dt == "fp16" and at > 12:
        pytest.skip("no fp16 query makes so small a key count")
    B, H, KVH, S, W, R = 1, 16, 2, 4, 448, 128
    big = torch.arange(128) % 2 == 0
    lo, hi = 2.0**-at, 2.0 ** (span - at)
    kc, vc, q = (torch.from_numpy(randn(n, i)) for n, i in
                 (((B, KVH, S + W, 128), 91), ((B, KVH, S + W, 128), 92), ((B, H, 128), 93)))
    kc = torch.where(big, kc * hi, kc * lo).to(DT[dt])
    q = (torch.where(big, q / hi, q / lo) * 2).to(DT[dt])
    vc = vc.to(DT[dt])
    hc = O.build_quantized_kv_cache(kc.float().numpy(), vc.float().numpy(), residual_size=R, sink=S, bits=bits)
    hc["k_residual"], hc["v_residual"] = (x[:, :, -R:].float().numpy() for x in (kc, vc))
    ref = O.quantized_attention_masked(q.float().numpy(), hc, 163840, W, SCALE, sink=S, residual_size=R, bits=bits)
    say(f"kivi bits={bits} {dt} key scales 2^{span} apart")
    _relative(_attend(q.to(device), _upload(hc, dt, device), 163840, W, S, R, bits), ref, dt)


@pytest.mark.parametrize("bits,dt", [(4, "fp16"), (4, "bf16"), (2, "bf16")])
@pytest.mark.parametrize("span,at", [(8, 10), (10, 10), (12, 10), (20, 10), (24, 10), (14, 18)])
def test_value_scales_far_apart(bits, dt, span, at, device):
    """Two tokens of weight 0 whose values are 2^span the others' (2^-at), and
    two whose values are 0."""
    B, H, KVH, S, W, R = 1, 16, 2, 4, 448, 128
    kc, vc, q = (torch.from_numpy(randn(n, i)) for n, i in
                 (((B, KVH, S + W, 128), 94), ((B, KVH, S + W, 128), 95), ((B, H, 128), 96)))
    q[..., 40] = 4
    out = [S + 5, S + 200]
    kc[:, :, out, 40] = -300
    vc *= 2.0**-at
    vc[:, :, out] *= 2.0**span
    vc[:, :, [S + 9, S + 100]] = 0
    kc, vc, q = (x.to(DT[dt]) for x in (kc, vc, q))
    hc = O.build_quantized_kv_cache(kc.float().numpy(), vc.float().numpy(), residual_size=R, sink=S, bits=bits)
    hc["k_residual"], hc["v_residual"] = (x[:, :, -R:].float().numpy() for x in (kc, vc))
    ref = O.quantized_attention_masked(q.float().numpy(), hc, 163840, W, SCALE, sink=S, residual_size=R, bits=bits)
    say(f"kivi bits={bits} {dt} value scales 2^{span} apart")
    _relative(_attend(q.to(device), _upload(hc, dt, device), 163840, W, S, R, bits), ref, dt)


@pytest.mark.parametrize("bits,dt", [(4, "fp16"), (2, "bf16")])
def test_slots_never_written(bits, dt, device):
    """NaN patterns in every quantized byte and residual row of slots past the
    sequence's length must not reach the output."""
    B, H, KVH, S, W, R, L = 1, 64, 8, 4, 512, 128, 300
    hc = _cache(B, KVH, S, W, R, bits, dt, 21)
    c = _upload(hc, dt, device)
    valid = O.slot_validity(L, W, S, 0)
    dead = (~valid[S:S + W - R]).reshape(-1, 32)
    whole = torch.from_numpy(dead.all(1))
    tok = torch.from_numpy(~valid[S:S + W - R])
    for n in ("k_win_scale", "k_win_zero"):
        c[n][:, :, whole] = float("nan")
    for n in ("v_win_scale", "v_win_zero"):
        c[n][:, :, tok] = float("nan")
    q = torch.from_numpy(randn((B, H, 128), 6)).to(DT[dt])
    say(f"kivi bits={bits} {dt} with never-written slots")
    o = _attend(q.to(device), c, L, W, S, R, bits)
    _check(o, O.quantized_attention_masked(q.float().numpy(), hc, L, W, SCALE, sink=S, residual_size=R, bits=bits), dt)


def test_stays_generic(device):
    """Groups of more than 8 query heads and tensors off a 16-byte boundary."""
    B, H, KVH, S, W, R, bits = 1, 32, 2, 4, 320, 128, 4
    hc = _cache(B, KVH, S, W, R, bits, "bf16", 31)
    c = _upload(hc, "bf16", device)
    q = torch.from_numpy(randn((B, H, 128), 8)).to(torch.bfloat16)
    ref = O.quantized_attention_masked(q.float().numpy(), hc, 9999, W, SCALE, sink=S, residual_size=R, bits=bits)
    say("kivi 4-bit, 16 heads per KV head")
    _check(_attend(q.to(device), c, 9999, W, S, R, bits), ref, "bf16")
    q = q[:, :16].contiguous()
    ref = O.quantized_attention_masked(q.float().numpy(), hc, 9999, W, SCALE, sink=S, residual_size=R, bits=bits)
    x = c["v_win_packed"]
    buf = torch.zeros(x.numel() + 1, dtype=torch.uint8, device=device)
    buf[1:] = x.flatten()
    c["v_win_packed"] = buf[1:].view(x.shape)
    say("kivi 4-bit, codes off a 16-byte boundary")
    _check(_attend(q.to(device), c, 9999, W, S, R, bits), ref, "bf16")
