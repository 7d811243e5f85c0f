"""Evictions of the one-launch step of a decode-time KIVI cache (the K half and
the V half of a block quantized by two waves): every ring block into every
window-old slot, against the quantizers on the block's tokens, blocks with
infinities, zero spans and NaN (whose groups take the double quotient) among
ordinary ones; and the attention of each evicting step against the two-launch
form."""

import pytest
import torch

from kivi_stream import KiviStreamBatch
from quant_kernel import quantize_k_cache, quantize_v_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [1, 2, 3, 4])
def test_every_block_and_slot(groups, device):
    B, H, KVH, W = 3, 16, 2, 128 + 32 * groups
    n = 32 * 10
    torch.manual_seed(groups)

    def r(*shape):
        return torch.randn(*shape, device=device, dtype=torch.float16)
    k, v = r(B, KVH, W + 4, 128), r(B, KVH, W + 4, 128)
    kt, vt, q = r(B, KVH, n, 128), r(B, KVH, n, 128), r(B, H, 128)
    # sequence 1 evicts groups with no finite scale, sequence 2 groups of one value
    for x in (kt, vt):
        x[1, 0, 40, 7] = float("inf")
        x[1, 1, 75, 96] = float("-inf")
        x[1, 1, 100, 31] = float("nan")
        x[2, 0, 64:96] = 0.25
    caches = [KiviStreamBatch.from_prefill(k, v, window=W) for _ in range(2)]
    hist = {"k": torch.cat([k[:, :, -128:], kt], 2), "v": torch.cat([v[:, :, -128:], vt], 2)}
    off = torch.tensor([0, 11, 20], device=device)   # evictions on different steps
    for i in range(n):
        active = (i >= off).to(torch.int32)
        at = (i - off).clamp(min=0)[:, None, None, None].expand(-1, KVH, 1, 128)
        kn, vn = kt.gather(2, at)[:, :, 0].contiguous(), vt.gather(2, at)[:, :, 0].contiguous()
        one = caches[0].step_attend(q, kn, vn, active=active)
        caches[1].append(kn, vn, active=active)
        two = caches[1].attend(q)
        done = [i + 1 - o for o in off.tolist()]
        if not any(d > 0 and d % 32 == 0 for d in done):
            continue
        finite = torch.isfinite(two)
        assert torch.equal(torch.isfinite(one), finite)
        assert torch.allclose(one[finite].float(), two[finite].float(), rtol=2**-10, atol=5e-5)
        for b, d in enumerate(done):
            if d <= 0 or d % 32:
                continue
            e = d // 32 - 1                         # this sequence's eviction number
            tok = slice(32 * e, 32 * e + 32)
            slot = e % groups
            for side, quantize in (("k", quantize_k_cache), ("v", quantize_v_cache)):
                codes, scale, zero = quantize(hist[side][b:b + 1, :, tok].contiguous())
                t = caches[0].t
                at_c = slice(8 * slot, 8 * slot + 8) if side == "k" else slice(32 * slot, 32 * slot + 32)
                at_s = slice(slot, slot + 1) if side == "k" else at_c
                assert torch.equal(t[f"{side}_win_packed"][b:b + 1, :, at_c], codes), (i, b, side)
                for name, x in (("scale", scale), ("zero", zero)):
                    got = t[f"{side}_win_{name}"][b:b + 1, :, at_s]
                    assert torch.equal(got.nan_to_num(9.0), x.nan_to_num(9.0)), (i, b, side, name)
