"""Few-row calls (at most one attention workgroup per CU): every count of blocks
per row from 1 on, rows without their diagonal block or with no block at all,
partial last blocks, split dense rows, both block sizes, head dims and types,
against float32 attention over the call's own lists; and the bits of a sequence
do not depend on what else is in the call."""

import math

import pytest
import torch

from flashprefill_amd.runtime import FlashPrefillCall

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,hq,hkv,rules", [([1], 1, 1, (2, 4, 2)), ([300, 5, 1000], 8, 2, (2, 4, 2)),
                                               ([1100], 7, 7, (1, 2, 1)), ([3000], 2, 1, (0, 1, 2)),
                                               ([1500], 4, 2, (3, 0, 0)), ([2000], 4, 1, (2, 4, 30))])
def test_few_rows(lens, hq, hkv, rules, d, block, dtype):
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + d)
    T = sum(lens)
    q, k, v = [torch.randn(T, h, d, generator=g, device=DEV).to(dtype) for h in (hq, hkv, hkv)]
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    o = torch.full_like(q, float("nan"))
    call = FlashPrefillCall(q, k, v, o, torch.tensor(cu, dtype=torch.int32, device=DEV), max(lens),
                            alpha=0.6, attention_sink=rules[0], window_size=rules[1],
                            last_n_block=rules[2], block_size=block)
    call.run()
    for b, n in enumerate(lens):
        sl = slice(cu[b], cu[b + 1])
        mask = call.selection_masks()[b].to(DEV)  # (Hq, NB, NB)
        keep = mask.repeat_interleave(block, 1).repeat_interleave(block, 2)[:, :n, :n]
        keep = keep & torch.ones(n, n, dtype=torch.bool, device=DEV).tril()
        qf, kf, vf = [t[sl].float().permute(1, 0, 2) for t in (q, k, v)]
        kf, vf = kf.repeat_interleave(hq // hkv, 0), vf.repeat_interleave(hq // hkv, 0)
        s = torch.matmul(qf, kf.transpose(1, 2).contiguous()) / math.sqrt(d)
        p = torch.softmax(s.masked_fill(~keep, -math.inf), -1)
        want = torch.matmul(p.nan_to_num(0.0), vf).permute(1, 0, 2)  # no key: 0 (l starts at 1)
        err = (o[sl].float() - want).abs()
        # P rounded to the input type against fp32 weights that sum to 1, and
        # one rounding of the result: 2^-9 (2^-12) of |v| <= ~5 each, as a bound
        # on every element and a tenth of it on the mean
        bar = 2.0 ** -8 * 5 if dtype == torch.bfloat16 else 2.0 ** -11 * 5
        assert err.max().item() <= bar and err.mean().item() <= bar / 10, (b, n, err.max())


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bits_of_a_sequence_do_not_depend_on_the_batch(d, block, dtype):
    """One short sequence alone (fewer rows than CUs) against the same sequence as
    the first of twelve: eight blocks a row, so that no row is split either way."""
    n, hq, hkv = 8 * block - 24, 32, 8
    g = torch.Generator(device=DEV).manual_seed(d + block)
    q, k, v = [torch.randn(12 * n, h, d, generator=g, device=DEV).to(dtype) for h in (hq, hkv, hkv)]
    outs = []
    for b in (1, 12):
        o = torch.empty_like(q[:b * n])
        cu = torch.arange(0, b * n + 1, n, dtype=torch.int32, device=DEV)
        FlashPrefillCall(q[:b * n], k[:b * n], v[:b * n], o, cu, n, alpha=0.18, attention_sink=2,
                         window_size=4, last_n_block=2, block_size=block).run()
        outs.append(o[:n])
    assert torch.equal(*outs)
