"""fp32 pooling: the block means against the float64 mean (edges of the row
groups and of the last block, both head dims, strided keys, block 64 / 128 /
256), from the one-launch plan + pooling and from the separate launches."""

import pytest
import torch

from flashprefill_amd.runtime import FlashPrefillCall

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("lens", [[1], [7, 8, 9], [63, 64, 65, 15, 17], [127, 0, 129, 300, 1000],
                                  [33] * 17])
def test_block_means(lens, d, block):
    g = torch.Generator().manual_seed(len(lens) + d)
    T, hkv = sum(lens), 3
    k = torch.randn(T, hkv + 2, d, generator=g) * 10.0 ** torch.randn(T, 1, 1, generator=g)
    k = k.to(DEV)[:, 1:1 + hkv]
    q = torch.randn(T, hkv, d, generator=g).to(DEV)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    calls = []
    for whole in (True, False):
        o = torch.empty_like(q)
        c = FlashPrefillCall(q, k, k, o, cu, max(lens), alpha=0.5, block_size=block)
        if whole:
            c.run()
        else:
            c.plan()
            c.pool()
        torch.cuda.synchronize()
        calls.append(c.pooled_k().cpu())
    assert torch.equal(*calls)
    want = []
    for b, n in enumerate(lens):
        for s in range(0, n, block):
            want.append(k[int(cu[b]) + s:int(cu[b]) + min(s + block, n)].double().mean(0).cpu())
    want = torch.stack(want)
    # rounded once from a float64 sum: half a spacing, 2^-24 of the value, plus
    # the float64 sum's own error (terms of up to ~1e4 against small means)
    bound = want.abs() * 2.0 ** -24 * 1.0001 + 1e-11
    assert ((calls[0].double() - want).abs() <= bound).all()
