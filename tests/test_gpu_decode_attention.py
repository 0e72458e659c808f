"""Block-table decode attention whose kernels read lengths and tables themselves, against the same attention over prefix sums
and a slot map (which the oracle tests cover): the same kernel and the same bits.  Units of one head in one, two and four
workgroups, of two and of four heads, requests past the table entries that a wave holds at once (4096 keys), block sizes that the direct form takes and does not take, key counts at the edges of chunks and of cache blocks, requests without
keys, absent blocks, tables that are too short, lengths that sum to more than the caller said, more than 64 requests."""
import pytest
import torch

from acache_amd import ops
from tests.test_attention_form import ANY_HEAD_DIM, GROUP, PAIRS, SHORT, form

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,D,B,kind", [(32, 32, 128, 1, (SHORT, 4)), (28, 4, 128, 2, (SHORT, 4)), (28, 4, 128, 3, (SHORT, 2)),
                                            (32, 32, 128, 5, (SHORT, 1)), (16, 4, 64, 6, (SHORT, 1)), (28, 4, 128, 12, (GROUP, 2)),
                                            (32, 8, 128, 16, (GROUP, 2)), (28, 4, 128, 30, (GROUP, 4)), (14, 2, 128, 64, (GROUP, 4)),
                                            (8, 2, 128, 65, (PAIRS, 2)), (4, 2, 128, 70, (GROUP, 2)), (4, 4, 80, 3, (ANY_HEAD_DIM, 1))])
@pytest.mark.parametrize("bs", [16, 32, 48, 256])
@pytest.mark.parametrize("how", ["whole", "holes", "short", "cut"])
def test_equals_attention_over_the_slot_map(device, H, Hkv, D, B, kind, bs, how):
    g = torch.Generator().manual_seed(B + bs)
    dtype = torch.float16 if B % 2 else torch.bfloat16
    edges = [1, 0, 31, 32, 33, 255, 256, 257, 2 * bs, bs + 1]
    lens = [edges[i % len(edges)] for i in range(B)]
    lens[B // 2] = 4500 if kind[0] == SHORT and D == 128 else 512 * B  # a few hundred keys on average at least
    blocks = [-(-n // bs) for n in lens]
    pool, at = torch.randperm(sum(blocks) + 3, generator=g).to(torch.int32), 0
    tables = torch.full((B, max(blocks) + 1), -1, dtype=torch.int32)
    for b, n in enumerate(blocks):
        tables[b, :n] = pool[at:at + n]
        at += n
    if how == "holes":
        tables[:, 1::3] = -1
    if how == "short":
        tables = tables[:, :max(max(blocks) // 2, 1)].contiguous()
    total = sum(lens) - (300 if how == "cut" else 0)
    q_len = 32 if B % 3 else 7
    assert form(B, B * q_len, total, H, Hkv, D, 0)[:2] == kind
    rand = lambda *shape: torch.randn(*shape, generator=g).to(dtype).to(device)
    q, k, v = rand(B, q_len, H, D), rand(len(pool), bs, Hkv, D), rand(len(pool), bs, Hkv, D)
    tables = tables.to(device)
    got = ops.baseline_decode_attention(q, k, v, torch.tensor(lens, device=device), tables, total_k=total)
    whole = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    slots = ops.block_table_slots(tables, whole.to(device), bs, sum(lens))[:total]
    cu_q = torch.arange(0, B * q_len + 1, q_len, dtype=torch.int32, device=device)
    want = ops.acache_attention(q.flatten(0, 1), k, v, cu_q, whole.clamp(max=total).to(device), slots)
    assert torch.equal(got.flatten(0, 1), want)
    assert torch.isfinite(got).all() and got.any()
