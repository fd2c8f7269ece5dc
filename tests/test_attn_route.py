"""Which kernel a call's sizes lead to (localrouter_amd/csrc/lr_abi.hip, through lr_attention_route: host arithmetic, no GPU),
on 256 compute units: the lines the rules draw, from both sides."""
from __future__ import annotations

import pytest

from tests._util import KEY_RANGES, KEYSPLIT, PIPE_W4, PIPE_W8, STREAM, route


def test_sizes_no_call_takes():
    for bad in (dict(W=0), dict(H=0), dict(HK=0), dict(nkeys=0), dict(p0=-1)):
        assert route(**{**dict(W=8, H=2, nkeys=8), **bad}) == 0


@pytest.mark.parametrize("W,H,nkeys,want", [
    (1280, 24, 1280, KEYSPLIT),      # 240 blocks of 128 queries: one round
    (2000, 24, 2000, PIPE_W4),       # 384: past one round
    (16384, 4, 2000, PIPE_W8),       # 256 blocks of 256 queries
    (4608, 24, 4608, STREAM),        # from 4,096 keys on, 432 blocks of 256 queries
    (560, 24, 560, PIPE_W4),         # too few key tiles for the key-split kernel's longer start
])
def test_rows(W, H, nkeys, want):
    assert route(W, H, nkeys) == want


@pytest.mark.parametrize("W,H,nkeys,want", [(218, 16, 50220, KEY_RANGES), (4608, 24, 4608, STREAM), (218, 16, 300, PIPE_W4)])
def test_rows_with_a_workspace(W, H, nkeys, want):
    assert route(W, H, nkeys, workspace=True) == want


@pytest.mark.parametrize("W,H", [(32, 40), (64, 33), (513, 12), (600, 16), (2048, 16), (1000, 32)])
def test_split_area_keeps_the_streaming_kernel(W, H):
    """From 4,096 keys and 33 blocks of 256 queries on, a workspace call runs the streaming kernel with its split tail."""
    for nkeys in (4096, 8192, 16384):
        assert route(W, H, nkeys, workspace=True) == STREAM
    assert route(W, H, 4095, workspace=True) != STREAM


@pytest.mark.parametrize("W,H,nkeys,want", [
    (1, 16, 961, KEY_RANGES), (128, 16, 961, KEY_RANGES), (128, 32, 961, KEY_RANGES),   # one wave a SIMD
    (218, 8, 961, KEY_RANGES), (218, 16, 1024, KEYSPLIT), (218, 16, 1025, KEY_RANGES),  # 1,744 rows; 3,488: 16 tiles
    (400, 16, 1280, KEYSPLIT), (400, 16, 1281, KEY_RANGES),                             # 6,400: 20
    (218, 16, 960, KEYSPLIT)])                                                          # below 16 tiles nothing is split
def test_split_over_workgroups_or_key_split(W, H, nkeys, want):
    assert route(W, H, nkeys, workspace=True) == want


@pytest.mark.parametrize("W,nkeys,causal,want", [
    (1, 1500, 0, PIPE_W4), (1, 3000, 1, PIPE_W4), (64, 3000, 0, PIPE_W4), (65, 3000, 0, KEYSPLIT), (65, 3000, 1, KEYSPLIT),
    (128, 576, 0, PIPE_W4), (128, 577, 0, KEYSPLIT), (128, 449, 1, KEYSPLIT), (128, 448, 1, PIPE_W4)])
def test_few_rows_and_short_calls_keep_the_pipelined_kernel(W, nkeys, causal, want):
    assert route(W, 16, nkeys, causal=causal, p0=(nkeys - W) * causal) == want


@pytest.mark.parametrize("W,p0,want", [
    (1280, 100000, KEYSPLIT),                               # 240 blocks: one round
    (1500, 1500, KEYSPLIT), (1500, 1501, PIPE_W4),          # 288, 1.1 rounds: as many keys before the chunk as in it
    (2688, 30000, PIPE_W4), (2816, 30000, KEYSPLIT)])       # 504 and 528: two rounds
def test_causal_chunks_behind_many_keys(W, p0, want):
    """Blocks of about the same length fill whole rounds or lose one, as a non-causal call's."""
    assert route(W, 24, p0 + W, HK=1, causal=1, p0=p0) == want


@pytest.mark.parametrize("W,H,HK,causal", [(300, 16, 16, 0), (500, 32, 32, 1), (1500, 24, 24, 1),
                                             (1000, 64, 8, 1)])
def test_keys_beyond_the_cache_keep_the_pipelined_kernel(W, H, HK, causal):
    """512 bytes a key and key head: 256 MB are 2^19 of them."""
    last = (1 << 19) // HK
    assert route(W, H, last + 64, HK, causal, p0=last + 64 - W) == PIPE_W4
    assert route(W, H, last, HK, causal, p0=last - W) == (KEYSPLIT if (W + 127) // 128 * H <= 256 else PIPE_W4)


def test_keys_beyond_the_cache_without_scratch():
    """Past half a round of 256-query blocks the other kernel is the streaming one's whole blocks: the key-split kernel."""
    assert route(1000, 32, 50000) == KEYSPLIT and route(1000, 24, 50000) == PIPE_W4


@pytest.mark.parametrize("W,p0,want", [(100, 0, PIPE_W4), (448, 0, PIPE_W4), (128, 320, PIPE_W4), (449, 0, KEYSPLIT),
                                       (128, 321, KEYSPLIT)])
def test_causal_calls_count_the_keys_they_see(W, p0, want):
    """A causal chunk sees p0 + W keys, however long the buffer behind them is."""
    for nkeys in (p0 + W, 512, 3000, 100000):
        if nkeys >= p0 + W:
            assert route(W, 16, nkeys, causal=1, p0=p0) == want, nkeys


@pytest.mark.parametrize("Sq,H,Sk,want", [(320, 4, 320, KEYSPLIT), (1280, 24, 1280, KEYSPLIT), (4608, 24, 4608, STREAM)])
def test_images(Sq, H, Sk, want):
    assert route(Sq, H, Sk, images=True) == want
    assert route(Sq, H, Sk, images=True, causal=1) == STREAM


@pytest.mark.parametrize("Sq,Sk,want", [(3300, 3300, KEYSPLIT), (3300, 3500, STREAM), (4200, 4200, STREAM), (100, 2000, KEYSPLIT),
                                        (100, 5000, STREAM)])
def test_images_beside_the_split_tail(Sq, Sk, want):
    assert route(Sq, 4, Sk, images=True) == want
