"""Calls whose rules alone keep every block (sequences of at most sink + window
+ last_n blocks): the selection that k_plan_pool writes against the staged
search's on the same inputs (counts, lists, row records) and the outputs, at the
last length that takes it and the first that does not, ragged batches, GQA
ratios, block sizes, fp32, and more sequences than the one launch plans."""

import pytest
import torch

from flashprefill_amd.runtime import FlashPrefillCall

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _call(t, cu, lens, rules, block, native):
    q, k, v = t
    o = torch.full_like(q, float("nan"))
    sink, window, last_n = rules
    return FlashPrefillCall(q, k, v, o, cu, max(lens), alpha=0.9, attention_sink=sink,
                            window_size=window, last_n_block=last_n, block_size=block,
                            native_normalize=native, min_budget=3 if native else 0), o


@pytest.mark.parametrize("block,dtype,d", [(128, torch.bfloat16, 128), (64, torch.float16, 64),
                                           (128, torch.float32, 64), (128, torch.bfloat16, 256),
                                           (256, torch.bfloat16, 128)])
@pytest.mark.parametrize("lens", [[1], [1000, 1024, 0, 127], [1025, 3], [512, 300, 128, 129],
                                  [60] * 17])
@pytest.mark.parametrize("rules", [(2, 4, 2), (0, 1, 7), (8, 0, 0), (-1, 20, -3)])
@pytest.mark.parametrize("hq,hkv,native", [(8, 2, False), (7, 1, True)])
def test_same_selection_and_output_as_the_staged_path(lens, rules, block, dtype, d, hq, hkv, native):
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    T = sum(lens)
    t = [torch.randn(T, h, d, generator=g, device=DEV).to(dtype) for h in (hq, hkv, hkv)]
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    whole, o1 = _call(t, cu, lens, rules, block, native)
    staged, o2 = _call(t, cu, lens, rules, block, native)
    whole.run()
    for stage in (staged.plan, staged.pool, staged.search, staged.attn):
        stage()
    torch.cuda.synchronize()
    assert whole.ordered_lists_ok() and staged.ordered_lists_ok()
    tile = whole.seq_tables()[0]
    assert torch.equal(whole.counts()[:, :tile[-1]], staged.counts()[:, :tile[-1]])
    for x, y in zip(whole.selection_masks(), staged.selection_masks()):
        assert torch.equal(x, y)
    assert torch.equal(o1, o2)
