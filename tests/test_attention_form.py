"""The rule that picks the attention kernel of a call, over sizes alone (host side, no GPU work)."""
import ctypes

import pytest

from acache_amd import _lib

UNITS, SHORT, GROUP, PAIRS, ANY_HEAD_DIM = range(5)
PLAIN, KEY_SIDE, QUERY_SIDE = range(3)
HEADS = [(32, 32), (28, 4), (32, 8), (32, 16), (24, 8), (40, 8), (48, 8), (14, 2), (8, 2), (6, 2), (12, 3), (12, 4), (8, 1), (5, 5), (1, 1)]


def form(B, total_q, total_k, H, Hkv, D, mode):
    out = (ctypes.c_int64 * 4)()
    _lib.check(_lib.load().acache_varlen_attn_form(out, B, total_q, total_k, H, Hkv, D, mode), "form")
    return tuple(out)


def sizes():
    for H, Hkv in HEADS:
        for B in [1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 28, 30, 32, 48, 64, 65, 96, 128]:
            for q in (1, 8, 13, 31, 32, 33, 200):
                for keys in (0, 60, 255, 256, 399, 400, 512, 1024, 1536, 1537, 4000):
                    for D in (128, 64):
                        yield B, q * B, keys * B, H, Hkv, D


def test_plain_and_key_side_take_the_same_form():
    """A key-side call has the bits of a plain one over a materialised copy, so no line may come between them."""
    kinds = set()
    for B, total_q, total_k, H, Hkv, D in sizes():
        for q in (total_q, total_q + 1):
            plain = form(B, q, total_k, H, Hkv, D, PLAIN)
            assert plain == form(B, q, total_k, H, Hkv, D, KEY_SIDE), (B, q, total_k, H, Hkv, D)
            kinds.add(plain[:2])
    assert kinds == {(UNITS, 1), (SHORT, 1), (SHORT, 2), (SHORT, 4), (GROUP, 2), (GROUP, 4), (PAIRS, 2)}


def test_other_head_dims_and_bad_sizes():
    assert form(3, 40, 900, 8, 2, 80, PLAIN)[0] == ANY_HEAD_DIM
    for bad in [(0, 1, 1, 1, 1, 128, 0), (1, 0, 1, 1, 1, 128, 0), (1, 1, -1, 1, 1, 128, 0), (1, 1, 1, 3, 2, 128, 0),
                (1, 1, 1, 1, 1, 100, 0), (1, 1, 1, 1, 1, 128, 3)]:
        with pytest.raises(ValueError):
            form(*bad)


def most_tiles(B, total_q):
    return (total_q + 31 * B) // 32                              # of 32 rows, whatever the lengths


def grid(tiles, H, Hkv, slices):
    """Workgroups for `slices` units per tile and KV head: the fullest of the eight XCDs, times eight."""
    if Hkv < 8 and 8 % Hkv == 0:
        return 8 * slices * -(-tiles * Hkv // 8)
    return -(-tiles * slices * Hkv // 8) * 8


def test_wave_private_units_run_at_once():
    """A workgroup of these fills its CU: blocks of one length never wait for a second turn, and where CUs are left, their
    tiles are those of the longest blocks that the total allows."""
    seen = set()
    for B, total_q, total_k, H, Hkv, D in sizes():
        for q in (total_q, total_q + 1):
            for mode in (PLAIN, QUERY_SIDE):
                kind, parts, tiles, blocks = form(B, q, total_k, H, Hkv, D, mode)
                if kind == SHORT:
                    assert blocks <= 256, (B, q, total_k, H, Hkv, D, mode)
                    assert tiles >= (B if q % B == 0 else most_tiles(B, q))
                    assert blocks == grid(tiles, H, Hkv, H // Hkv * parts)
                    assert tiles == most_tiles(B, q) or grid(tiles + 1, H, Hkv, H // Hkv * parts) > 256
                    seen.add((Hkv, parts))
    assert {(3, 2), (3, 4), (4, 4), (32, 4), (8, 1)} <= seen


def test_grouped_units_have_room_for_longer_blocks():
    """Two heads per unit: a turn of the CUs.  Four: up to two.  Where CUs are left, for the tiles of the longest blocks that
    the total allows."""
    seen = set()
    for B, total_q, total_k, H, Hkv, D in sizes():
        for q in (total_q, total_q + 1):
            for mode in (PLAIN, QUERY_SIDE):
                kind, heads, tiles, blocks = form(B, q, total_k, H, Hkv, D, mode)
                if kind == GROUP:
                    slices = -(-(H // Hkv) // heads)
                    turns = 1 if heads == 2 or grid(B, H, Hkv, slices) <= 256 else 2
                    assert blocks == grid(tiles, H, Hkv, slices) <= 256 * turns
                    assert tiles >= (B if q % B == 0 else most_tiles(B, q))
                    assert tiles == most_tiles(B, q) or grid(tiles + 1, H, Hkv, slices) > 256 * turns, (B, q, total_k, H, Hkv, D, mode)
                    seen.add((heads, turns))
    assert seen == {(2, 1), (4, 1), (4, 2)}


def test_four_heads_per_unit_keep_most_waves_busy():
    """Units of four heads have two waves per head: groups of two would leave half of them without one."""
    groups = set()
    for B, total_q, total_k, H, Hkv, D in sizes():
        for mode in (PLAIN, QUERY_SIDE):
            kind, heads, _, _ = form(B, total_q, total_k, H, Hkv, D, mode)
            if kind == GROUP and heads == 4:
                turns = 1 if grid(B, H, Hkv, -(-(H // Hkv) // 4)) <= 256 else 2
                assert 8 * 256 * turns < 2 * 2 * B * H, (B, H, Hkv, mode)
                groups.add(H // Hkv)
    assert groups >= {3, 4, 7} and 2 not in groups
