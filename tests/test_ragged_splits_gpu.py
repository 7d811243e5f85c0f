"""Splits shared out by the sequences' own lengths: lengths of nothing, of one
token, of tiles' edges and of the whole context together; few and the most
sequences that share, one more; lengths past the context (clamped).  Each case
says whether its plan shares (2 to 64 sequences, splits of at least 64 tiles)."""

import pytest
import torch

from helpers import SCALE

pytestmark = pytest.mark.gpu


def _ref(q, k, v):
    s = torch.matmul(q.double().view(k.shape[0], -1, 128), k.double().transpose(1, 2).contiguous()) * SCALE
    return torch.matmul(torch.softmax(s, -1), v.double()).view(-1, 128)


def _check(o, q, k, v, lens):
    for b, n in enumerate(min(n, k.shape[2]) for n in lens):
        if n <= 0:
            assert (o[b] == 0).all()
            continue
        ref = _ref(q[b], k[b, :, :n], v[b, :, :n])
        # one fp16 rounding of a result within 2e-6
        half_ulp = 2.0 ** (torch.floor(torch.log2(ref.abs().clamp(min=2.0**-14))) - 11)
        assert ((o[b].double() - ref).abs() - half_ulp).max().item() <= 2e-6, (b, n)


@pytest.mark.parametrize("B,KVH,L,lens,shares", [
    (1, 2, 9000, [7001], False),
    (2, 8, 33000, [0, 33000], True),
    (3, 30, 5000, [1, 5000, 33], False),
    (3, 30, 6300, [1, 6300, 33], True),
    (4, 16, 9000, [9000, 9000, 9000, 9000], True),
    (5, 8, 15000, [0, 0, 0, 0, 0], True),
    (5, 8, 15000, [3000, 6000, 9000, 12000, 15000], True),
    (7, 16, 5000, [5000, 31, 32, 33, -5, 2049, 99999], False),
    (7, 16, 6300, [6300, 31, 32, 33, -5, 2049, 99999], True),
    (7, 16, 6300, [-2147483648, 2147483647, 1, 0, 6299, 6301, 64], True),
    (30, 8, 4500, None, True),
    (64, 2, 4500, None, True),
    (65, 2, 4500, None, False),
])
def test_dense_lengths(B, KVH, L, lens, shares, device):
    import _kvdec as K
    from dense_kernel import dense_decode_attention
    splits, tiles = K.lib.kvdec_num_splits(K.KIND_DENSE, B, KVH, L), (L + 31) // 32
    assert shares == (2 <= B <= 64 and splits > 1 and -(-tiles // splits) >= 64)
    g = torch.Generator(device=device).manual_seed(B)
    q = torch.randn((B, 4 * KVH, 128), generator=g, device=device, dtype=torch.float16)
    k, v = (torch.randn((B, KVH, L, 128), generator=g, device=device, dtype=torch.float16) for _ in range(2))
    lens = lens or [L if b == B // 2 else 13 * b * b % 1500 for b in range(B)]
    print(f"ragged dense B={B} KVH={KVH} L={L}", flush=True)
    _check(dense_decode_attention(q, k, v, torch.tensor(lens, dtype=torch.int32, device=device)), q, k, v, lens)


def test_pages_and_changed_lengths_under_replay(device):
    """A captured call reads the lengths of each replay."""
    from paged_kernel import paged_decode_attention
    B, KVH, L, page = 6, 16, 8192, 16
    g = torch.Generator(device=device).manual_seed(1)
    q = torch.randn((B, 2 * KVH, 128), generator=g, device=device, dtype=torch.float16)
    k, v = (torch.randn((B, KVH, L, 128), generator=g, device=device, dtype=torch.float16) for _ in range(2))
    table = torch.randperm(B * L // page, generator=g, device=device).to(torch.int32)
    pools = []
    for x in (k, v):
        pool = torch.empty((B * L // page, page, KVH, 128), device=device, dtype=torch.float16)
        pool[table.long()] = x.transpose(1, 2).reshape(-1, page, KVH, 128)
        pools.append(pool)
    table = table.view(B, -1)
    lens = torch.full((B,), L, dtype=torch.int32, device=device)
    call = lambda: paged_decode_attention(q, *pools, table, lens, max_seq_len=L)  # noqa: E731
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = call()
    for now in ([L] * B, [1, L, 0, 4000, 17, 300], [L, 1, 1, 1, 1, 1], [64, 64, 64, 64, 64, 65]):
        lens.copy_(torch.tensor(now, dtype=torch.int32))
        print(f"ragged pages {now}", flush=True)
        graph.replay()
        torch.cuda.synchronize()
        _check(o, q, k, v, now)
        # eager too (not bit for bit: a workgroup's waves claim tiles as they come free)
        _check(call(), q, k, v, now)
