"""head_dim 256 attention at the edges of its tile ring: rows of one, two, three
and more blocks, partial last blocks around every 32-key tile boundary, both
block sizes and types, one workgroup per row and the persistent grid, against
float32 causal attention over every block (alpha 0)."""

import math

import pytest
import torch

from flashprefill_amd import flash_prefill_varlen_func
from tests._parity import persistent_grid_slots

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(lens, hq, hkv, block, dtype):
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + block)
    T, d = sum(lens), 256
    q = torch.randn(T, hq, d, generator=g, device=DEV).to(dtype)
    k = torch.randn(T, hkv, d, generator=g, device=DEV).to(dtype)
    v = torch.randn(T, hkv, d, generator=g, device=DEV).to(dtype)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    o = torch.full_like(q, float("nan"))
    flash_prefill_varlen_func(q, k, v, o, torch.tensor(cu, dtype=torch.int32, device=DEV),
                              max(lens), 0.0, block)
    for b, n in enumerate(lens):
        if n == 0:
            continue
        sl = slice(cu[b], cu[b + 1])
        qf, kf, vf = [t[sl].float().permute(1, 0, 2) for t in (q, k, v)]
        kf, vf = kf.repeat_interleave(hq // hkv, 0), vf.repeat_interleave(hq // hkv, 0)
        s = torch.matmul(qf, kf.transpose(1, 2).contiguous()) / math.sqrt(d)
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1), -math.inf)
        want = torch.matmul(torch.softmax(s, -1), vf).permute(1, 0, 2)
        err = (o[sl].float() - want).abs()
        # P rounded to the input type against fp32 weights that sum to 1, and
        # one rounding of the result: 2^-9 (2^-12) of |v| <= ~5 each, as a bound
        # on every element and a tenth of it on the mean
        bar = 2.0 ** -8 * 5 if dtype == torch.bfloat16 else 2.0 ** -11 * 5
        assert err.max().item() <= bar and err.mean().item() <= bar / 10, (b, n, err.max())


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens", [[1, 31, 32, 33], [63, 64, 65, 95, 96, 97], [127, 128, 129],
                                  [160, 191, 193, 224, 225, 255, 256, 257], [383, 385, 400, 0, 513],
                                  [900, 1100]])
def test_rows_of_few_blocks(lens, block, dtype):
    _check(lens, 4, 2, block, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block,lens", [(128, [2100, 1900]), (64, [2300, 2500])])
def test_persistent_grid_and_split_rows(block, lens, dtype):
    slots, least = persistent_grid_slots(32, lens, block, 256)
    assert slots >= least
    _check(lens, 32, 8, block, dtype)
