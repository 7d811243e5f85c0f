"""The one-launch cache builder bit for bit against the oracle's over the
remainders of its work split (channel counts that are no multiple of a wave's
128, window-old groups that are no multiple of a workgroup's four, residual
rows that are no multiple of its steps), sinks of 1 to 32 tokens, every type of
input and residual, and caches off a 16-byte boundary."""

import numpy as np
import pytest
import torch

from helpers import randn, say
from oracle import kvdec_oracle as O

pytestmark = pytest.mark.gpu

DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _check(kc, vc, S, R, res_dt):
    from quant_kernel import build_quantized_kv_cache
    got = build_quantized_kv_cache(kc, vc, residual_size=R, sink=S, residual_dtype=res_dt)
    kh, vh = kc.float().cpu().numpy(), vc.float().cpu().numpy()
    want = O.build_quantized_kv_cache(kh, vh, residual_size=R, sink=S)
    for key in O.CACHE_KEYS:
        g, w = got[key], np.asarray(want[key])
        if key.endswith("residual"):
            w = torch.from_numpy((kh if key[0] == "k" else vh)[:, :, -w.shape[2]:].copy()).to(got[key].dtype).float().numpy()
            g = g.float()
        assert tuple(g.shape) == w.shape, key
        np.testing.assert_array_equal(g.cpu().numpy(), w, err_msg=key)


@pytest.mark.parametrize("dt,res", [("fp16", None), ("bf16", None), ("bf16", torch.float16), ("fp32", None),
                                    ("fp32", torch.float16)])
@pytest.mark.parametrize("D,S,W,R", [(32, 1, 20, 128), (128, 4, 128, 128), (128, 4, 288, 128), (96, 32, 192, 96),
                                     (288, 17, 128 + 96, 100), (128, 3, 33 + 32 * 5, 33)])
def test_bit_exact(dt, res, D, S, W, R, device):
    if (W - min(W, R)) % 32:
        W = min(W, R) + 32 * ((W - min(W, R)) // 32)
    say(f"build {dt} -> {res} D={D} S={S} W={W} R={R}")
    x = [torch.from_numpy(randn((2, 3, S + W, D), 50 + i)).to(DT[dt]).to(device) for i in (0, 1)]
    _check(*x, S, R, res)


@pytest.mark.parametrize("dt", ["fp16", "fp32"])
def test_off_16_byte_boundary(dt, device):
    shape = (1, 2, 4 + 192, 128)
    views = []
    for i in (0, 1):
        buf = torch.zeros(int(np.prod(shape)) + 1, dtype=DT[dt], device=device)
        buf[1:] = torch.from_numpy(randn(shape, 60 + i)).flatten().to(DT[dt]).to(device)
        views.append(buf[1:].view(shape))
    say(f"build {dt} one element off alignment")
    _check(*views, 4, 128, None)
