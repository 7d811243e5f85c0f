"""The streaming quantizers at 1, 4 and 8 bits in groups of 32 (2 bits has its
own tests): bit-exact codes, scales and zeros against the oracle over lane and
wave remainders (token groups and channel counts that are no multiple of a
wave's), every input type, groups that take the exact slow path, and tensors
that do not allow the wide accesses."""

import numpy as np
import pytest
import torch

from helpers import host, randn, say
from oracle import kvdec_oracle as O

pytestmark = pytest.mark.gpu

DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _compare(x, bits, what):
    from quant_kernel import quantize_k_cache, quantize_v_cache
    say(what)
    with np.errstate(over="ignore", invalid="ignore"):
        for fn, ofn in ((quantize_k_cache, O.quantize_k), (quantize_v_cache, O.quantize_v)):
            got = [host(t) for t in fn(x, bits=bits)]
            for name, g, w in zip(("packed", "scale", "zero"), got, ofn(x.float().cpu().numpy(), 32, bits)):
                np.testing.assert_array_equal(g, w, err_msg=f"{fn.__name__} {name}")


@pytest.mark.parametrize("bits", [1, 4, 8])
@pytest.mark.parametrize("dt", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("shape", [(1, 1, 32, 32), (1, 3, 96, 128), (2, 2, 64, 96), (1, 1, 160, 288)])
def test_bit_exact(bits, dt, shape, device):
    x = torch.from_numpy(randn(shape, bits + shape[2])).to(DT[dt])
    x[..., 5] *= 30
    x[:, :, ::7] += 4
    x[:, :, :32, 1] = 1.5   # a constant group
    _compare(x.to(device), bits, f"quantize bits={bits} {dt} {shape}")


@pytest.mark.parametrize("bits", [1, 4, 8])
@pytest.mark.parametrize("mul", [1e-20, 1e30])
def test_slow_path_scales(bits, mul, device):
    x = torch.from_numpy(randn((1, 2, 64, 128), 9)) * mul
    _compare(x.to(device), bits, f"quantize bits={bits} x {mul}")


@pytest.mark.parametrize("dt", ["fp32", "bf16"])
def test_off_16_byte_boundary(dt, device):
    x = torch.from_numpy(randn((1, 2, 64, 128), 11)).to(DT[dt])
    buf = torch.zeros(x.numel() + 1, dtype=DT[dt], device=device)
    buf[1:] = x.flatten().to(device)
    _compare(buf[1:].view(x.shape), 4, f"quantize 4 bits {dt}, one element off alignment")


@pytest.mark.parametrize("dt", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_two_bits_off_16_byte_boundary(dt, off, device):
    """2-bit input `off` elements off alignment, codes as many bytes and scales
    and zeros as many halves off, bit for bit; nothing around them is written."""
    import _kvdec as K
    B, KVH, N, D = 1, 2, 64, 128
    x = torch.from_numpy(randn((B, KVH, N, D), 12 + off)).to(DT[dt])
    buf = torch.zeros(x.numel() + off, dtype=DT[dt], device=device)
    buf[off:] = x.flatten().to(device)
    xd = buf[off:].view(x.shape)
    _compare(xd, 2, f"quantize 2 bits {dt}, {off} elements off alignment")
    for fn, ofn in ((K.lib.kvdec_quantize_k, O.quantize_k), (K.lib.kvdec_quantize_v, O.quantize_v)):
        want = ofn(x.float().numpy(), 32, 2)
        out = [torch.full((w.size + off + 16,), 77, dtype=torch.uint8 if w.dtype == np.uint8 else torch.float16,
                          device=device) for w in want]
        say(f"quantize 2 bits {dt}, outputs {off} off alignment")
        rc = fn(K.ptr(xd), {"fp32": K.F32, "fp16": K.F16, "bf16": K.BF16}[dt], *[K.ptr(o[off:]) for o in out],
                B, KVH, N, D, 32, 2, K.stream_of(xd))
        assert rc == 0
        for o, w in zip(out, want):
            np.testing.assert_array_equal(host(o[off:off + w.size]).reshape(w.shape), w)
            assert (host(o[:off]) == 77).all() and (host(o[off + w.size:]) == 77).all()
