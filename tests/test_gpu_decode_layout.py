"""acache_decode_layout against the prefix sums of torch and the slot map of block_table_slots, exactly."""
import pytest
import torch

from acache_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _layout(seqlens, tables, q_len, bs, total_k, device):
    B = seqlens.numel()
    cu_q = torch.full((B + 1,), -7, dtype=torch.int32, device=device)
    cu_k = cu_q.clone()
    out = torch.full((sum(seqlens.tolist()) + 5,), -9, dtype=torch.int32, device=device)
    s, t = seqlens.to(device), tables.to(device)
    rc = _lib.load().acache_decode_layout(cu_q.data_ptr(), cu_k.data_ptr(), out.data_ptr(), s.data_ptr(), t.data_ptr(), B,
                                          q_len, t.shape[1], bs, total_k, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "decode_layout")
    return cu_q, cu_k, out


@pytest.mark.parametrize("B,longest,bs", [(1, 1, 8), (2, 70, 16), (16, 1512, 256), (255, 40, 8), (256, 3, 4), (257, 33, 8),
                                          (700, 20, 16)])
def test_equals_scan_and_slot_map(device, B, longest, bs):
    g = torch.Generator().manual_seed(B)
    seqlens = torch.randint(0, longest + 1, (B,), generator=g, dtype=torch.int32)
    seqlens[-1] = longest
    tables = torch.randint(-1, 900, (B, -(-longest // bs)), generator=g, dtype=torch.int32)
    total = int(seqlens.sum())
    cu_q, cu_k, out = _layout(seqlens, tables, 32, bs, total, device)
    want = torch.tensor([0] + seqlens.cumsum(0).tolist(), dtype=torch.int32)
    assert torch.equal(cu_k.cpu(), want) and cu_q.tolist() == [32 * i for i in range(B + 1)]
    assert torch.equal(out[:total], ops.block_table_slots(tables.to(device), want.to(device), bs, total))
    assert out[total:].tolist() == [-9] * 5
    # a short table maps to -1 and nothing is written past total_k
    if total > 1:
        cut = _layout(seqlens, tables[:, :1].contiguous(), 1, bs, total - 1, device)[2]
        assert torch.equal(cut[:total - 1],
                           ops.block_table_slots(tables[:, :1].contiguous().to(device), want.to(device), bs, total)[:-1])
        assert cut[total - 1:].tolist() == [-9] * 6


def test_lengths_beyond_the_slot_map_are_cut(device):
    """No reader of cu_k gets past the slots that exist, whatever the lengths on the device say."""
    lens = torch.tensor([5, 9, 3, 4], dtype=torch.int32)
    tables = torch.arange(8, dtype=torch.int32).view(4, 2)
    for total, want in ((21, [0, 5, 14, 17, 21]), (14, [0, 5, 14, 14, 14]), (8, [0, 5, 8, 8, 8]), (0, [0, 0, 0, 0, 0])):
        assert _layout(lens, tables, 2, 8, total, device)[1].tolist() == want


@pytest.mark.parametrize("known", [True, False])
def test_batched_decode_attention_equals_the_ragged_call(device, known):
    g = torch.Generator(device=device).manual_seed(3)
    seqlens = [257, 1, 700]
    q = torch.randn(3, 32, 28, 128, generator=g, device=device).to(torch.bfloat16)
    k, v = (torch.randn(8, 256, 4, 128, generator=g, device=device).to(torch.bfloat16) for _ in range(2))
    tables = torch.tensor([[5, 2, -1], [0, -1, -1], [7, 1, 3]], dtype=torch.int32, device=device)
    got = ops.baseline_decode_attention(q, k, v, torch.tensor(seqlens, device=device), tables,
                                        total_k=sum(seqlens) if known else None)
    cu = lambda lens: torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=device)
    want = ops.baseline_ragged_attention(q.flatten(0, 1), k, v, cu([32] * 3), cu(seqlens), tables)
    assert torch.equal(got.flatten(0, 1), want)


def test_calls_that_the_layout_launch_does_not_cover(device):
    """A table without rows for trailing requests that have no keys, or with more rows than requests; one length for a batch
    (a prefix sum that broadcasts: the first request has the keys); no requests; no query rows."""
    g = torch.Generator(device=device).manual_seed(4)
    q = torch.randn(3, 4, 4, 128, generator=g, device=device).to(torch.bfloat16)
    k, v = (torch.randn(8, 16, 4, 128, generator=g, device=device).to(torch.bfloat16) for _ in range(2))
    tables = torch.tensor([[5, 2], [0, -1], [7, 1], [3, 4]], dtype=torch.int32, device=device)
    lens = lambda *n: torch.tensor(n, device=device)
    full = ops.baseline_decode_attention(q, k, v, lens(20, 9, 0), tables[:3])
    assert torch.equal(ops.baseline_decode_attention(q, k, v, lens(20, 9, 0), tables[:2]), full)
    assert torch.equal(ops.baseline_decode_attention(q, k, v, lens(20, 9, 0), tables), full)
    assert torch.equal(full[0], ops.baseline_decode_attention(q[:1], k, v, lens(20), tables[:1])[0])
    assert not full[2].any()
    one = ops.baseline_decode_attention(q, k, v, lens(20), tables[:3])
    assert torch.equal(one[0], full[0]) and not one[1:].any()
    assert ops.baseline_decode_attention(q[:0], k, v, lens()[:0], tables[:0]).shape == (0, 4, 4, 128)
    with pytest.raises(RuntimeError):
        ops.baseline_decode_attention(q[:, :0], k, v, lens(20, 9, 0), tables[:3])
