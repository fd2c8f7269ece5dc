"""GPU test of the key compaction (localrouter_amd/csrc/keys.hip) behind lr_attention_kmask_bf16: the masked call must be,
bit for bit, the plain call over the kept keys' rows, wherever the compaction's blocks end: masks off a 16-byte boundary,
key counts around its 16-key passes and past 8,192 (several passes a block), rows narrower and wider than its 1 KB column
slabs, mask bytes other than 1, strided key rows, and a mask keeping more keys than declared (the first n_valid count)."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from localrouter_amd import ops  # noqa: E402


@pytest.mark.parametrize("nkeys,HK,offset,extra", [(1, 1, 0, 0), (15, 3, 1, 0), (16, 4, 0, 0), (17, 5, 3, 0), (700, 8, 0, 0),
                                                   (1000, 1, 5, 64), (8192, 2, 0, 0), (8209, 2, 7, 8), (20000, 1, 0, 0)])
def test_compaction_equals_gathered_rows(nkeys, HK, offset, extra):
    print(f"\n[compaction] nkeys={nkeys} HK={HK} offset={offset} extra={extra}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(nkeys + HK)
    rs = HK * 128 + extra
    q = torch.randn(40, HK, 128, generator=g, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn(nkeys, rs, generator=g, device="cuda").to(torch.bfloat16)[:, :HK * 128].view(nkeys, HK, 128)
            if not extra else torch.randn(nkeys, rs, generator=g, device="cuda").to(torch.bfloat16)
            .as_strided((nkeys, HK, 128), (rs, 128, 1)) for _ in range(2))
    buf = torch.zeros(nkeys + 16, dtype=torch.uint8, device="cuda")
    mask = buf[offset:offset + nkeys]
    mask.copy_(torch.randint(0, 256, (nkeys,), generator=g, device="cuda") * (torch.rand(nkeys, generator=g, device="cuda") < 0.6))
    mask[nkeys // 2] = 0x80
    keep = mask.nonzero()[:, 0]
    for n_valid in {len(keep), max(1, len(keep) // 2)}:   # (fewer than the mask keeps: the first ones)
        got = ops.attention_kmask(q, k, v, mask, n_valid=n_valid)
        idx = keep[:n_valid]
        want = ops.attention(q, k[idx].contiguous(), v[idx].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(got, want), (nkeys, n_valid)
