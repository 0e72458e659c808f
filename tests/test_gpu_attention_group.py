"""Grouped-query batches of short query blocks that run two or four heads per unit of eight waves, every relocation mode
against the CPU oracle: ragged batches with requests without queries, without keys and with several query tiles, key counts
at the edges of the 32-key chunks and of the rounds, odd and even groups, all three ways KV heads meet XCDs, more requests
than one ballot holds.  Bound: 2e-2, that of the other attention tests (rounding of probabilities and outputs to 16 bits)."""
import pytest
import torch

from acache_amd import ops
from oracle import acache_oracle as O
from tests.test_attention_form import GROUP, SHORT, form, grid
from tests.test_gpu_attention_short import A, START, _case, _check

pytestmark = pytest.mark.gpu
EDGES = [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 95, 97]


def _units(B, H, Hkv, heads):
    per_kv = -(-(H // Hkv) // heads)
    tiles = -(-B // (8 // Hkv)) * (8 // Hkv) if Hkv < 8 and 8 % Hkv == 0 else B
    return -(-tiles * Hkv * per_kv // 8) * 8


@pytest.mark.parametrize("mode", ["plain", "key", "query"])
@pytest.mark.parametrize("heads,B,H,Hkv,dtype", [(2, 10, 28, 4, torch.bfloat16), (2, 16, 32, 8, torch.float16),
                                                 (2, 23, 12, 3, torch.float16), (2, 28, 10, 2, torch.bfloat16),
                                                 (4, 30, 24, 8, torch.bfloat16), (4, 29, 28, 4, torch.bfloat16), (4, 52, 10, 2, torch.float16),
                                                 (4, 118, 14, 2, torch.bfloat16), (4, 32, 48, 8, torch.float16)])
def test_ragged_batches_against_the_oracle(device, mode, heads, B, H, Hkv, dtype):
    n = B - 1                                                    # the last request raises the average to 256 keys
    q_lens = [(7 * i) % 33 for i in range(n)]
    q_lens[2], q_lens[4], q_lens[5] = 0, 70, 33                  # three and two query tiles
    q_lens[7] += -(sum(q_lens) + 3) % B
    tails = [EDGES[i % len(EDGES)] - (A if mode == "plain" and i % 2 else 0) for i in range(n)]
    tails = [max(t, 1) for t in tails]
    tails[6] = -1
    assert sum(q_lens) + 3 <= 32 * B and (sum(q_lens) + 3) % B == 0
    assert _units(B, H, Hkv, 1) > 256
    if heads == 2:
        assert _units(B, H, Hkv, 2) <= 256
    else:
        assert _units(B, H, Hkv, 2) > 256 and (512 - _units(B, H, Hkv, 4)) % 256 < 64
    _check(*_case(q_lens, tails, H, Hkv, 128, dtype, mode, B, keys_per_request=256), device)


def test_absent_rows_are_zero_and_64_bit_addresses_change_nothing(device):
    B, keys = 12, 288
    t, kw = _case([32] * B, [keys] * B, 28, 4, 128, torch.bfloat16, "plain", 5, holes=True)
    present = (t[5] >= 0) & (t[5] < t[1].shape[0])
    zero = t[1].shape[0] - 1                                     # what an absent row reads as
    t2 = [t[0], t[1].clone(), t[2].clone(), t[3], t[4], torch.where(present, t[5], zero).to(torch.int32)]
    t2[1][zero], t2[2][zero] = 0, 0
    q, kc, vc, cu_q, cu_k, slots = (x.to(device) for x in t)
    shape = (kc.shape[0] // 16, 16, 4, 128)
    got = ops.acache_attention(q, kc.view(shape), vc.view(shape), cu_q, cu_k, slots).cpu()
    assert (got.float() - O.acache_attention(*t2).float()).abs().max().item() <= 2e-2
    # slots 16 MiB apart
    wide = [torch.zeros(24 << 23, dtype=torch.bfloat16, device=device).as_strided((24, 4, 128), (1 << 23, 128, 1))
            for _ in range(2)]
    wide[0].copy_(kc[:24])
    wide[1].copy_(vc[:24])
    few = torch.arange(24, dtype=torch.int32, device=device).repeat(keys // 24 * B)
    assert torch.equal(ops.acache_attention(q, *wide, cu_q, cu_k, few), ops.acache_attention(q, kc[:24], vc[:24], cu_q, cu_k, few))


@pytest.mark.parametrize("keys", [200, 255, 256, 300, 1536, 1537])
@pytest.mark.parametrize("H,Hkv,B", [(28, 4, 10), (32, 8, 16), (28, 4, 30)])
def test_key_side_equals_a_materialised_copy(device, keys, H, Hkv, B):
    """On both sides of the lines of the dispatch, plain attention over a relocated copy takes the form that key-side
    relocation takes: the same bits."""
    g, S, D = torch.Generator(device=device).manual_seed(keys), A + 16 * (keys // 16 + 1), 128
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


@pytest.mark.parametrize("shared", [1, 31, 33, 97])
@pytest.mark.parametrize("B", [12, 30])
def test_scores_far_below_zero(device, B, shared):
    """Query-side relocation with streams that hold few or no shared keys, and all scores near -100: a softmax does not
    know such an offset."""
    D, g = 128, torch.Generator().manual_seed(shared)
    level = (100.0 / D ** 0.5) ** 0.5
    kv = [shared + 40 + i for i in range(B)]
    S = shared + sum(kv)
    q = (level + 0.3 * torch.randn(32 * B, 28, D, generator=g)).to(torch.bfloat16)
    kc = (-level + 0.3 * torch.randn(S + 16 - S % 16, 4, D, generator=g)).to(torch.bfloat16)
    vc = torch.randn(kc.shape, generator=g).to(torch.bfloat16)
    own = iter(range(shared, S))
    slots = torch.tensor([s for n in kv for s in list(range(shared)) + [next(own) for _ in range(n - shared)]], dtype=torch.int32)
    cu = lambda lens: torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    cos, sin = O.rope_table(64, D, 5e5)
    _check([q, kc, vc, cu([32] * B), cu(kv), slots],
           dict(shared_prefix_len=shared, rope_cos=cos, rope_sin=sin, affix_shifts=torch.zeros(B, dtype=torch.int32),
                shared_kv_lens=torch.full((B,), shared, dtype=torch.int32)), device)


@pytest.mark.parametrize("mode", ["plain", "key", "query"])
@pytest.mark.parametrize("H,Hkv,D,dtype", [(32, 32, 128, torch.bfloat16), (28, 4, 128, torch.float16), (16, 4, 64, torch.bfloat16)])
@pytest.mark.parametrize("keys", [256, 400, 512])
def test_one_head_per_unit_from_a_few_hundred_keys(device, mode, H, Hkv, D, dtype, keys):
    """Batches of up to 256 units of one head take the wave-private form from 256, 400 or 512 keys on average."""
    _check(*_case([32, 1, 17, 0, 33], [31, 97, -1, 64, 255], H, Hkv, D, dtype, mode, keys, keys_per_request=keys), device)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mode", ["plain", "key", "query"])
@pytest.mark.parametrize("H,Hkv,batches", [(32, 32, (2, 4, 6)), (28, 4, (2, 4, 7)), (12, 3, (5, 10, 15))])
def test_few_units_in_parts_have_the_same_bits(device, mode, H, Hkv, batches, dtype):
    """One request alone (up to 64 units: its features over four workgroups) and repeated in batches of up to 64, 128 and more
    units (four, two, one workgroup each): the same bits, in the bound against the oracle."""
    assert [1 + (B * H > 64) + (B * H > 128) for B in batches] == [1, 2, 3]
    q_len, keys = 32 if Hkv == 32 else 13, 515
    t, kw = _case([q_len], [keys], H, Hkv, 128, dtype, mode, H)
    alone = _check(t, kw, device)
    for B in batches:
        rep = lambda cu: torch.arange(B + 1, dtype=torch.int32) * cu[1]
        tb = [t[0].repeat(B, 1, 1), t[1], t[2], rep(t[3]), rep(t[4]), t[5].repeat(B)]
        kwb = {k: v.repeat(B) if k in ("affix_shifts", "shared_kv_lens") else v for k, v in kw.items()}
        q, kc, vc, cu_q, cu_k, slots = (x.to(device) for x in tb)
        shape = (kc.shape[0] // 16, 16, *kc.shape[1:])
        kwb = {k: v.to(device) if torch.is_tensor(v) else v for k, v in kwb.items()}
        got = ops.acache_attention(q, kc.view(shape), vc.view(shape), cu_q, cu_k, slots, **kwb).cpu()
        for b in range(B):
            assert torch.equal(got[b * q_len:(b + 1) * q_len], alone), (B, b)


MODES = ["plain", "key", "query"]


def _alternating(B):
    q_lens = [33 - 2 * (b % 2) for b in range(B)]
    q_lens[-1] += 32 * B - sum(q_lens)
    return q_lens, sum(-(-q // 32) for q in q_lens)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("H,Hkv,B,parts", [(32, 32, 2, 4), (28, 4, 4, 2), (12, 3, 5, 4), (12, 3, 8, 2), (7, 1, 16, 2)])
def test_more_tiles_than_requests_run_in_fewer_parts(device, mode, H, Hkv, B, parts, dtype):
    """Blocks of 33 and 31 rows look like blocks of 32: their grid holds a tile per request (and what CUs are left), the
    kernel deals all tiles in half as many parts.  The bits of whole units, which three times as many requests are."""
    q_lens, tiles = _alternating(B)
    t, kw = _case(q_lens, [470 + 13 * b for b in range(B)], H, Hkv, 128, dtype, mode, H + B)
    total_k = t[5].numel()
    kind, share, room, _ = form(B, 32 * B, total_k, H, Hkv, 128, MODES.index(mode))
    assert (kind, share) == (SHORT, parts) and room < tiles
    got = _check(t, kw, device)
    n = 1
    while form(n * B, 32 * n * B, n * total_k, H, Hkv, 128, MODES.index(mode))[:2] != (SHORT, 1):
        n += 1
    cu = lambda c: torch.cat([c[:1]] + [c[1:] + i * c[-1] for i in range(n)])
    tb = [t[0].repeat(n, 1, 1), t[1], t[2], cu(t[3]), cu(t[4]), t[5].repeat(n)]
    kwb = {k: v.repeat(n) if k in ("affix_shifts", "shared_kv_lens") else v for k, v in kw.items()}
    assert torch.equal(_check(tb, kwb, device)[-32 * B:], got)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("H,Hkv,B,fits", [(28, 4, 16, True), (24, 8, 16, True), (12, 3, 40, True), (32, 8, 12, True), (32, 16, 16, False)])
def test_more_tiles_than_requests_run_four_heads_per_unit(device, mode, H, Hkv, B, fits, dtype):
    """The same for two heads per unit: units of four where the grid holds them, otherwise in a second turn."""
    q_lens, tiles = _alternating(B)
    t, kw = _case(q_lens, [250 + 5 * b for b in range(B)], H, Hkv, 128, dtype, mode, H + B)
    kind, share, room, blocks = form(B, 32 * B, t[5].numel(), H, Hkv, 128, MODES.index(mode))
    assert (kind, share) == (GROUP, 2) and room < tiles
    assert (grid(tiles, H, Hkv, -(-(H // Hkv) // 4)) <= blocks) == fits
    _check(t, kw, device)


@pytest.mark.parametrize("mode", ["key", "query"])
@pytest.mark.parametrize("H,Hkv,D,B,kind", [(32, 32, 128, 1, SHORT), (16, 16, 64, 3, SHORT), (28, 4, 128, 12, GROUP), (28, 4, 128, 30, GROUP)])
def test_rope_tables_of_any_alignment(device, mode, H, Hkv, D, B, kind):
    """Tables are contiguous floats, not 16-byte aligned ones: the same bits from a view one float into an allocation."""
    t, kw = _case([32] * B, [560] * B, H, Hkv, D, torch.bfloat16, mode, B)
    assert form(B, 32 * B, t[5].numel(), H, Hkv, D, MODES.index(mode))[0] == kind
    got = _check(t, kw, device)
    q, kc, vc, cu_q, cu_k, slots = (x.to(device) for x in t)
    kw = {k: v.to(device) if torch.is_tensor(v) else v for k, v in kw.items()}
    for name, by in (("rope_cos", 1), ("rope_sin", 3)):
        moved = torch.empty(kw[name].numel() + by, device=device)[by:].view(kw[name].shape)
        kw[name] = moved.copy_(kw[name])
        assert moved.data_ptr() % 16 == 4 * by and moved.is_contiguous()
    shape = (kc.shape[0] // 16, 16, *kc.shape[1:])
    assert torch.equal(ops.acache_attention(q, kc.view(shape), vc.view(shape), cu_q, cu_k, slots, **kw).cpu(), got)
