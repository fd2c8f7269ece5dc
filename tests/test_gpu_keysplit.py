"""GPU parity of the key-split kernel (localrouter_amd/csrc/attn_keysplit.hip): 128-query blocks whose waves are two groups
over alternating 64-key tiles, merged through LDS. The sizes are those where its cut can go wrong: one query row, the
edges of a 128-query block, an odd number of key tiles (the second group's last tile is masked whole), a partial last
tile in either group, one step in all, causal blocks whose second group sees no key, GQA. The calls take it by their
sizes (LR_ATTN_CFG_AUTO), which every test asserts first; each is checked against the oracle at the bar of tests/_util.py, and over every stride form
against the pipelined kernel (an explicit configuration) to within two bf16 roundings."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests._util import KEYSPLIT, assert_close, bf16_f32, from_dev, route, to_dev
from tests.test_gpu_attention import _qkv, _ref, _sign_ramp, _sign_ramp_expected

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from localrouter_amd import _lib, ops  # noqa: E402


def _takes_keysplit(W, nk, H, HK, causal=0, p0=0, images=False):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert route(W, H, nk, HK, causal=causal, p0=p0, images=images, cus=cus) == KEYSPLIT


@pytest.mark.parametrize("W,nk,H,HK,causal,p0", [
    (65, 577, 3, 3, 0, 0),       # a wave with one row, one with none; 10 tiles, the last with one key (second group)
    (127, 640, 2, 1, 0, 0), (128, 641, 2, 2, 0, 0), (129, 704, 4, 2, 0, 0),
    (300, 1000, 5, 5, 0, 0),     # 16 tiles, a partial one last
    (130, 500, 2, 2, 1, 370),    # causal: the diagonal in the last tiles
    (513, 513, 8, 2, 1, 0),      # causal from position 0: first blocks with an empty second group, H a multiple of 8
    (600, 449, 3, 1, 1, 0),      # queries past the keys see all of them
    (570, 1200, 7, 7, 1, 77)])   # keys past the queries are seen by none
def test_keysplit_rows(W, nk, H, HK, causal, p0):
    print(f"\n[keysplit rows] W={W} nk={nk} H={H} HK={HK} causal={causal} p0={p0}", flush=True)
    _takes_keysplit(W, nk, H, HK, causal, p0)
    q, k, v = _qkv(71, W, nk, H, HK)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    got = from_dev(ops.attention(dq, dk, dv, causal=bool(causal), p0=p0))
    assert_close(got, _ref(q, k, v, causal=bool(causal), p0=p0), what="keysplit")
    # in place: each block reads its queries before it writes over them
    ops.attention(dq, dk, dv, dq, causal=bool(causal), p0=p0)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(dq), got)


@pytest.mark.parametrize("layout", ["packed", "head-major", "wide"])
def test_keysplit_strides_against_the_pipelined_kernel(layout):
    W, nk, H, HK = 261, 613, 4, 2
    print(f"\n[keysplit strides] {layout}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    rand = lambda n: torch.randn(n, generator=g, device="cuda").to(torch.bfloat16)
    if layout == "packed":       # q, k, v views of one [rows, (H + 2 HK) * 128] buffer
        rs = (H + 2 * HK) * 128
        buf = rand(nk * rs)
        q, k, v = buf, buf[H * 128:], buf[(H + HK) * 128:]
        args = (rs, rs, rs, 128, 128)
    elif layout == "head-major":
        q, k, v = rand(W * H * 128), rand(nk * HK * 128), rand(nk * HK * 128)
        args = (H * 128, 128, 128, nk * 128, nk * 128)
    else:                        # different strides for every tensor
        q, k, v = rand(W * 1032), rand(nk * 520), rand(nk * 776)
        args = (1032, 520, 776, 136, 256)
    q_rs, k_rs, v_rs, k_hs, v_hs = args
    outs = []
    for cfg in (ops.CFG_AUTO, ops.CFG_PIPE_W4):
        for causal, p0 in ((0, 0), (1, 352)):
            _takes_keysplit(W, nk, H, HK, causal, p0)
            out = torch.zeros(W, H, 136, dtype=torch.bfloat16, device="cuda")   # rows 544 elements apart, 8 of them unused
            _lib.call("lr_attention_bf16_ex", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), p0, W, H, HK, nk,
                      causal, ops.SCALE_128, q_rs, k_rs, v_rs, H * 136, k_hs, v_hs, cfg,
                      torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            flat = out.view(W, H * 136)
            assert not flat[:, H * 128:].any(), "past the row's heads nothing is written"
            outs.append(from_dev(flat[:, :H * 128].contiguous()))
    for a, b in ((0, 2), (1, 3)):   # twice the relative-L2 bar: two outputs, each rounded once from its own fp32 result
        assert_close(outs[a], bf16_f32(outs[b]).astype(np.float64), rel=6e-3, what=layout)


@pytest.mark.parametrize("rows", [True, False])
def test_keysplit_overflow_reaches_exact_recomputation(rows):
    """Scores rising by ~400 (exp2 domain) along the keys: both groups of the rising rows overflow their fixed reference,
    those of the falling rows do not; queries and outputs in the same rows."""
    Sq, Sk, H = 260, 700, 2
    print(f"\n[keysplit overflow] rows={rows}", flush=True)
    _takes_keysplit(Sq, Sk, H, H, images=not rows)
    q, k = _sign_ramp(Sq, Sk, H)
    v = oracle.synth_bf16(72, 3, (Sk, H, 128))
    exp = _sign_ramp_expected(q, k, v, 5.0, ops.SCALE_128)
    if rows:
        dq = to_dev(oracle.f32_to_bf16(bf16_f32(q) * 5.0))
        ops.attention(dq, to_dev(oracle.f32_to_bf16(bf16_f32(k) * 5.0)), to_dev(v), dq)
        got = from_dev(dq)
    else:
        w5 = torch.full((128,), 5.0, dtype=torch.float32, device="cuda")
        got = from_dev(ops.joint_attention(to_dev(q), to_dev(k), to_dev(v), q_norm=w5, k_norm=w5, table_kind=0, eps=0.0))
    torch.cuda.synchronize()
    assert_close(got, exp, what="keysplit overflow")


def test_keysplit_one_group_far_above_the_other():
    """Every second key tile scores ~100 (exp2 domain) above the others: one group's result must vanish beside the
    other's, whichever holds the larger scores."""
    W, nk, H = 96, 640, 2
    _takes_keysplit(W, nk, H, H)
    q, k, v = _qkv(73, W, nk, H, H)
    kf = bf16_f32(k)
    for odd in (0, 1):
        kk = kf.copy()
        tile = (np.arange(nk) // 64) % 2 == odd
        # +-: the query's own direction, so that the boosted tiles' scores rise for every row
        qf = np.ones((W, H, 128), np.float32)
        kk[tile] = kk[tile] * 0.25 + 6.0
        qb, kb = oracle.f32_to_bf16(qf), oracle.f32_to_bf16(kk)
        got = from_dev(ops.attention(to_dev(qb), to_dev(kb), to_dev(v)))
        torch.cuda.synchronize()
        assert_close(got, _ref(qb, kb, v), what=f"odd={odd}")


@pytest.mark.parametrize("Sq,Sk,H,HK", [(64, 1, 1, 1), (1, 65, 2, 2), (200, 64, 2, 2), (129, 130, 6, 2), (1280, 1280, 24, 24),
                                        (1000, 3000, 4, 4)])
def test_keysplit_images_against_the_streaming_kernel(Sq, Sk, H, HK):
    """The fused call at sizes that take the key-split kernel over tile images, against the explicit streaming
    configuration."""
    print(f"\n[keysplit images] Sq={Sq} Sk={Sk} H={H} HK={HK}", flush=True)
    _takes_keysplit(Sq, Sk, H, HK, images=True)
    q, _, _ = _qkv(74, Sq, 1, H, HK)
    _, k, v = _qkv(75, 1, Sk, H, HK)
    rng = np.random.default_rng(3)
    ang = rng.uniform(-np.pi, np.pi, size=(max(Sq, Sk), 64)).astype(np.float32)
    tab = (torch.from_numpy(np.cos(ang)).cuda(), torch.from_numpy(np.sin(ang)).cuda())
    got, ref = (from_dev(ops.joint_attention(to_dev(q), to_dev(k), to_dev(v), q_table=tab, config=c))
                for c in (ops.CFG_AUTO, ops.CFG_STREAM_W8))
    torch.cuda.synchronize()
    assert_close(got, bf16_f32(ref).astype(np.float64), rel=6e-3, what="images")


def test_keysplit_row_of_one_key_is_its_value():
    """A row that sees one key returns that key's value to the bit: the probabilities are normalised by the sum of their
    rounded values, so the one factor left is p * (1 / p) in fp32, far below a bf16 rounding. Over rows the first row of a
    causal call (its second group of waves sees no key), over images a call of one key."""
    W, H = 600, 3
    _takes_keysplit(W, W, H, H, causal=1)
    _takes_keysplit(W, 1, H, H, images=True)
    q, k, v = _qkv(76, W, W, H, H)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    got = from_dev(ops.attention(dq, dk, dv, causal=True))
    assert np.array_equal(got[0], from_dev(dv)[0])
    got = from_dev(ops.joint_attention(dq, dk[:1].contiguous(), dv[:1].contiguous(), table_kind=0))
    torch.cuda.synchronize()
    assert np.array_equal(got, np.broadcast_to(from_dev(dv)[:1], got.shape))


@pytest.mark.parametrize("W,nk,H,HK", [(300, 2500, 17, 17), (513, 2497, 12, 6), (65, 650, 33, 33), (129, 704, 4, 1)])
def test_keysplit_rows_equal_images(W, nk, H, HK):
    """Over key rows the key-split kernel gathers each key tile into the layout of a tile image: the same bits as over images
    of the same keys (lr_joint_kv_prepare with every key a prefix key: copied unchanged)."""
    print(f"\n[keysplit rows = images] W={W} nk={nk} H={H} HK={HK}", flush=True)
    _takes_keysplit(W, nk, H, HK)
    _takes_keysplit(W, nk, H, HK, images=True)
    q, k, v = _qkv(77, W, nk, H, HK)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    ws = torch.empty(ops.workspace_bytes(nk, HK), dtype=torch.uint8, device="cuda")
    ops.joint_kv_prepare(dk, dv, ws, table_kind=ops.TABLE_NONE, n_pre=nk)
    img, rows = ops.joint_attention_images(dq, ws, nk, HK), ops.attention(dq, dk, dv)
    torch.cuda.synchronize()
    assert torch.equal(rows, img)
