"""Attention of short query blocks (at most 32 rows per request on average), every relocation mode against the CPU oracle:
batches that fit one (request, head) per CU and have a thousand keys per request on average (wave-private key chunks) at
the edges of the 32-key chunks, of a wave's register-held slots (4096 keys) and of the 32-row query tiles; the same batches
without the long request that raises the average (per-head units); and grouped-query batches of two heads per unit.  Bound:
2e-2, that of the other attention tests (rounding of probabilities and outputs to 16 bits)."""
import pytest
import torch

from acache_amd import ops
from oracle import acache_oracle as O
from tests.test_attention_form import SHORT, form

pytestmark = pytest.mark.gpu
A, START = 40, 9      # shared rows (slots 0 .. A-1) and, in the relocation modes, private keys in front of them


def _case(q_lens, tails, H, Hkv, D, dtype, mode, seed, holes=False, keys_per_request=0):
    """`keys_per_request`: one more request, of three rows and of as many keys as that average takes."""
    g = torch.Generator().manual_seed(seed)
    if keys_per_request:
        q_lens, tails = q_lens + [3], tails + [keys_per_request * (len(q_lens) + 1)]
    reads, nxt = [], A
    for i, tail in enumerate(tails):
        if tail < 0:
            reads.append([])                                     # no keys at all
            continue
        a0 = START + i if mode != "plain" else 0
        mine = list(range(nxt, nxt + a0 + tail))
        nxt += a0 + tail
        shared = list(range(A)) if mode != "plain" else []
        reads.append(mine[:a0] + shared + mine[a0:] if mode == "key" else shared + mine)
    S = 16 * (nxt // 16 + 2)
    slots = torch.tensor(sum(reads, []), dtype=torch.int32)
    if holes:
        slots[5::11] = -1                                        # absent rows
        slots[7::13] = S + 3
    cu = lambda lens: torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    t = [(torch.randn(sum(q_lens), H, D, generator=g) / D ** 0.25).to(dtype),
         (torch.randn(S, Hkv, D, generator=g) / D ** 0.25).to(dtype), torch.randn(S, Hkv, D, generator=g).to(dtype),
         cu(q_lens), cu([len(r) for r in reads]), slots]
    kw = {}
    if mode != "plain":
        cos, sin = O.rope_table(4400, D, 5e5)
        kw = dict(shared_prefix_len=A, rope_cos=cos, rope_sin=sin,
                  affix_shifts=torch.tensor([START + i for i in range(len(tails))], dtype=torch.int32))
        if mode == "query":
            kw["shared_kv_lens"] = torch.tensor([A if n >= 0 else 0 for n in tails], dtype=torch.int32)
    return t, kw


def _device_call(t, kw, device, plan=None):
    q, kc, vc, cu_q, cu_k, slots = (x.to(device) for x in t)
    shape = (kc.shape[0] // 16, 16, *kc.shape[1:])
    kw = {k: v.to(device) if torch.is_tensor(v) else v for k, v in kw.items()}
    return ops.acache_attention(q, kc.view(shape), vc.view(shape), cu_q, cu_k, slots, plan=plan, **kw).cpu()


def _check(t, kw, device):
    got = _device_call(t, kw, device)
    want = O.acache_attention(*t, **kw)
    assert torch.isfinite(got.float()).all()
    assert (got.float() - want.float()).abs().max().item() <= 2e-2
    return got


@pytest.mark.parametrize("keys_per_request", [0, 1024])
@pytest.mark.parametrize("mode", ["plain", "key", "query"])
@pytest.mark.parametrize("H,Hkv,D,dtype", [(4, 4, 128, torch.bfloat16), (7, 1, 128, torch.float16),
                                           (6, 3, 64, torch.bfloat16), (8, 8, 64, torch.float16)])
def test_edges_against_the_oracle(device, mode, H, Hkv, D, dtype, keys_per_request):
    case = lambda q_lens, tails, seed: _check(*_case(q_lens, tails, H, Hkv, D, dtype, mode, seed,
                                                     keys_per_request=keys_per_request), device)
    case([1, 16, 17, 32, 31], [1, 31, 33, 257, 223], 1)
    case([40, 33, 20], [300, 90, 64], 2)                                                 # five tiles, three requests
    case([8, 0, 32, 4], [70, 20, -1, 0 if mode != "plain" else 1], 3)


@pytest.mark.parametrize("mode", ["plain", "query"])
@pytest.mark.parametrize("H,Hkv,q_lens", [(32, 4, [33, 31, 64, 0, 33, 25]), (16, 8, [161, 1, 1, 1, 20, 1, 1, 1, 1, 1, 1, 2])])
def test_more_tiles_than_units(device, mode, H, Hkv, q_lens):
    """A grid of one unit per request and head, so that tiles of long requests run in further turns."""
    t, kw = _case(q_lens, [30 * i + 1 for i in range(len(q_lens))], H, Hkv, 128, torch.bfloat16, mode, 8, keys_per_request=1024)
    B, total = len(q_lens) + 1, sum(q_lens) + 3
    assert total % B == 0 and H * ((total + 31 * B) // 32) > 256 and H * B <= 256
    _check(t, kw, device)


@pytest.mark.parametrize("H,Hkv,parts", [(2, 1, 4), (96, 8, 2), (160, 8, 1)])
@pytest.mark.parametrize("mode", ["plain", "key", "query"])
def test_slots_are_refilled_and_absent_rows_are_zero(device, mode, H, Hkv, parts):
    # the keys behind the first 4096 have values around 40: they carry 145 / 4241 of the weight, so the result moves by more
    # than 1 without them and by 0.3 for every chunk of 32 that is read from other slots
    t, kw = _case([32], [4241], H, Hkv, 128, torch.bfloat16, mode, 4)
    assert form(1, 32, t[5].numel(), H, Hkv, 128, 0)[:2] == (SHORT, parts)
    t[2][t[5][4096:].long()] += 40
    assert _check(t, kw, device).float().mean() > 1
    if mode == "plain" and H == 2:
        t, kw = _case([20, 32], [150, 77], 2, 2, 128, torch.bfloat16, mode, 5, holes=True, keys_per_request=1024)
        present = (t[5] >= 0) & (t[5] < t[1].shape[0])
        zero = t[1].shape[0] - 1                                 # what an absent row reads as
        t2 = [t[0], t[1].clone(), t[2].clone(), t[3], t[4], torch.where(present, t[5], zero).to(torch.int32)]
        t2[1][zero], t2[2][zero] = 0, 0
        assert (_device_call(t, kw, device).float() - O.acache_attention(*t2).float()).abs().max().item() <= 2e-2


@pytest.mark.parametrize("keys_per_request", [0, 1024])
@pytest.mark.parametrize("mode", ["plain", "query"])
def test_more_requests_than_one_ballot_holds(device, mode, keys_per_request):
    n = 70
    _check(*_case([(5 * i) % 33 for i in range(n)], [(37 * i) % 130 + 1 for i in range(n)], 1, 1, 64, torch.bfloat16, mode,
                  6, keys_per_request=keys_per_request), device)


@pytest.mark.parametrize("mode", ["plain", "key", "query"])
@pytest.mark.parametrize("B,H,Hkv,dtype", [(19, 28, 4, torch.bfloat16), (18, 32, 8, torch.float16),
                                           (44, 12, 3, torch.float16), (70, 10, 2, torch.bfloat16)])
def test_two_heads_of_a_group_per_unit(device, mode, B, H, Hkv, dtype):
    """Grouped-query batches beyond two units per CU: odd and even groups, all three ways KV heads meet XCDs, requests
    without queries, without keys and with more than one query tile; the bits of the per-head units (which a few of the
    requests by themselves are) up to 64 rows, beyond which those do not split the keys."""
    q_lens = [(7 * i) % 33 for i in range(B)]
    q_lens[3], q_lens[4], q_lens[5] = 0, 70, 33
    q_lens[7] += -sum(q_lens) % B
    tails = [(29 * i) % 140 + 1 for i in range(B)]
    tails[6] = -1
    t, kw = _case(q_lens, tails, H, Hkv, 128, dtype, mode, B)
    assert sum(q_lens) <= 32 * B and sum(q_lens) % B == 0 and B * H > 512
    got = _check(t, kw, device)
    cu_q, cu_k = t[3].tolist(), t[4].tolist()
    for first in (0, 4, 8, B - 2):
        last = first + 2
        some = {k: v[first:last] if k in ("affix_shifts", "shared_kv_lens") else v for k, v in kw.items()}
        part = _device_call([t[0][cu_q[first]:cu_q[last]], t[1], t[2], t[3][first:last + 1] - cu_q[first],
                             t[4][first:last + 1] - cu_k[first], t[5][cu_k[first]:cu_k[last]]], some, device)
        for r in range(first, last):
            if q_lens[r] <= 64:
                assert torch.equal(part[cu_q[r] - cu_q[first]:cu_q[r + 1] - cu_q[first]], got[cu_q[r]:cu_q[r + 1]]), r


def test_plan_and_slot_pitch_do_not_change_the_bits(device):
    t, kw = _case([32, 7], [190, 61], 8, 8, 128, torch.bfloat16, "plain", 7)
    got = _check(t, kw, device)
    plan = ops.attention_plan(t[3], t[4], 8, 8, device, slots_per_xcd=2)
    assert torch.equal(_device_call(t, kw, device, plan), got)   # (per-head units: few keys)
    # slots 16 MiB apart: 64-bit copy addresses, in per-head units and in wave-private chunks
    q, kc, vc = t[0].to(device), t[1][:24].to(device), t[2][:24].to(device)
    wide = [torch.zeros(24 << 23, dtype=torch.bfloat16, device=device).as_strided((24, 8, 128), (1 << 23, 128, 1))
            for _ in range(2)]
    wide[0].copy_(kc)
    wide[1].copy_(vc)
    for turns in (1, 43):
        few = torch.arange(24, dtype=torch.int32).repeat(2 * turns)
        args = (t[3].to(device), torch.tensor([0, 24 * turns, 48 * turns], dtype=torch.int32, device=device), few.to(device))
        assert torch.equal(ops.acache_attention(q, *wide, *args), ops.acache_attention(q, kc, vc, *args))


@pytest.mark.parametrize("D,keys", [(128, 300), (128, 399), (128, 400), (128, 700), (128, 900), (128, 1100), (64, 400), (64, 511),
                                    (64, 512), (64, 600)])
@pytest.mark.parametrize("H,Hkv,B", [(4, 4, 3), (28, 4, 7), (16, 16, 8), (16, 16, 9)])
def test_key_side_equals_a_materialised_copy(device, D, keys, H, Hkv, B):
    """On both sides of every line of the dispatch, plain attention over a relocated copy takes the form that key-side
    relocation takes: the same bits.  All requests have their shared rows at the same position."""
    g, S = torch.Generator(device=device).manual_seed(keys), A + 16 * (keys // 16 + 1)
    q = torch.randn(32 * B, H, D, generator=g, device=device).to(torch.bfloat16)
    kc, vc = (torch.randn(1, S + A + 8, Hkv, D, generator=g, device=device).to(torch.bfloat16) for _ in range(2))
    own = torch.randperm(S - A)[:keys - A] + A
    at = torch.cat([own[:START], torch.arange(A), own[START:]])
    cu = lambda n: torch.arange(0, n * B + 1, n, dtype=torch.int32, device=device)
    call = lambda slots, **kw: ops.acache_attention(q, kc[0], vc[0], cu(32), cu(keys),
                                                    slots.to(torch.int32).repeat(B).to(device), **kw)
    cos, sin = (t.to(device) for t in O.rope_table(64, D, 5e5))
    key_side = call(at, shared_prefix_len=A, rope_cos=cos, rope_sin=sin,
                    affix_shifts=torch.full((B,), START, dtype=torch.int32, device=device))
    ops.materialize_relocated_affix(kc, vc, cos, sin, S, A, START)
    at[START:START + A] = torch.arange(S, S + A)
    assert torch.equal(call(at), key_side)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("logit", [-20.0, -100.0])
@pytest.mark.parametrize("shared", [1, 31, 32, 33])
@pytest.mark.parametrize("H,Hkv,q_lens", [(4, 2, [40, 64]), (4, 2, [16, 64]), (28, 4, [32] * 19), (4, 2, [32, 32])])
def test_few_shared_keys_and_scores_far_below_zero(device, H, Hkv, q_lens, shared, logit, dtype):
    """Query-side relocation whose shared range ends inside the first half of its tile: the waves that take the second half
    of a tile's keys have none there, and later keys that all score near `logit`.  Tiles of up to 32 and of up to 64 rows in
    per-head units, and two heads per unit.  A softmax does not know such an offset: 2e-2 as above."""
    D, g = 128, torch.Generator().manual_seed(shared)
    level = (-logit / D ** 0.5) ** 0.5
    kv = [shared + 70 + i for i in range(len(q_lens))]
    S = shared + sum(kv)
    q = (level + 0.3 * torch.randn(sum(q_lens), H, D, generator=g)).to(dtype)
    kc = (-level + 0.3 * torch.randn(S + 16 - S % 16, Hkv, D, generator=g)).to(dtype)
    vc = torch.randn(kc.shape, generator=g).to(dtype)
    own = iter(range(shared, S))
    slots = torch.tensor([s for n in kv for s in list(range(shared)) + [next(own) for _ in range(n - shared)]], dtype=torch.int32)
    cu = lambda lens: torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    cos, sin = O.rope_table(64, D, 5e5)
    B = len(q_lens)
    _check([q, kc, vc, cu(q_lens), cu(kv), slots],
           dict(shared_prefix_len=shared, rope_cos=cos, rope_sin=sin, affix_shifts=torch.zeros(B, dtype=torch.int32),
                shared_kv_lens=torch.full((B,), shared, dtype=torch.int32)), device)
