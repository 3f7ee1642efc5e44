"""head_dim 64 attention in 64-key passes (block 128) and at three waves per SIMD
(blocks 64 and 128): lengths around every 32- and 64-key boundary of the first
blocks, and enough rows for the persistent grid, against float32 causal
attention over every block (alpha 0)."""

import math

import pytest
import torch

from flashprefill_amd import flash_prefill_varlen_func
from tests._parity import persistent_grid_slots

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,hq,hkv", [([1, 31, 32, 33, 63, 64, 65], 4, 2),
                                         ([96, 127, 128, 129, 191, 192, 193], 4, 1),
                                         ([255, 256, 257, 320, 0, 385], 6, 3),
                                         ([6300, 6200], 32, 8)])
def test_dense_rows(lens, hq, hkv, block, dtype):
    if hq == 32:
        slots, least = persistent_grid_slots(hq, lens, block, 64)
        assert slots >= least
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + block)
    T, d = sum(lens), 64
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
        err = (o[sl].float() - torch.matmul(torch.softmax(s, -1), vf).permute(1, 0, 2)).abs()
        # P rounded to the input type against fp32 weights that sum to 1, and
        # one rounding of the result: 2^-9 (2^-12) of |v| <= ~5 each, as a bound
        # on every element and a tenth of it on the mean
        bar = 2.0 ** -8 * 5 if dtype == torch.bfloat16 else 2.0 ** -11 * 5
        assert err.max().item() <= bar and err.mean().item() <= bar / 10, (b, n, err.max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,hq", [(700, 4), (13000, 32)])
def test_runs_of_keys_of_score_minus_infinity(n, hq, dtype):
    """A row's first 64-key pass without a finite score drops out, also in a
    diagonal block; rows that see nothing else in their first block are NaN, as the
    softmax of that tile is."""
    d, block, run = 64, 128, 100
    slots, least = persistent_grid_slots(hq, [n], block, d)
    assert (slots >= least) == (hq == 32)
    g = torch.Generator(device=DEV).manual_seed(n)
    q = (torch.rand(n, hq, d, generator=g, device=DEV) + 0.5).to(dtype)
    k = torch.randn(n, 1, d, generator=g, device=DEV).to(dtype)
    v = torch.randn(n, 1, d, generator=g, device=DEV).to(dtype)
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    outs = []
    for low in (-math.inf, -200.0):  # far below: P = 0 there too
        kk = k.clone()
        kk[:run] = low
        o = torch.empty_like(q)
        flash_prefill_varlen_func(q, kk, v, o, cu, n, 0.0, block)
        outs.append(o)
    assert outs[0][:run].isnan().all()
    assert not outs[0][run:].isnan().any()
    # the same scores but for the run's, so P and the sums differ by the maximum
    # that the first pass leaves: a rounding of P and one of the result
    err = (outs[0][run:].float() - outs[1][run:].float()).abs()
    bar = 2.0 ** -8 * 5 if dtype == torch.bfloat16 else 2.0 ** -11 * 5
    assert err.max().item() <= bar and err.mean().item() <= bar / 10


@pytest.mark.parametrize("sharp,one_tile", [(1.0, 2.0787e-3), (2.0, 2.0462e-3), (4.0, 1.8369e-3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_error_against_float64_no_larger_than_as_one_tile(dtype, sharp, one_tile):
    """2-norm error of four dense 4,000-token inputs, against what the kernel that
    took a block as one 128-key tile gave on the same inputs (bf16; fp16 keeps three
    more bits: 2.6037e-4, 2.5575e-4 and 2.2984e-4)."""
    if dtype == torch.float16:
        one_tile = {1.0: 2.6037e-4, 2.0: 2.5575e-4, 4.0: 2.2984e-4}[sharp]
    n, hq, d = 4000, 8, 64
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    errs = []
    for seed in range(4):
        g = torch.Generator(device=DEV).manual_seed(seed)
        q = (sharp * torch.randn(n, hq, d, generator=g, device=DEV)).to(dtype)
        k = torch.randn(n, 1, d, generator=g, device=DEV).to(dtype)
        v = torch.randn(n, 1, d, generator=g, device=DEV).to(dtype)
        o = torch.empty_like(q)
        flash_prefill_varlen_func(q, k, v, o, cu, n, 0.0, 128)
        qd, kd, vd = [t.double().permute(1, 0, 2) for t in (q, k, v)]
        s = torch.matmul(qd, kd.transpose(1, 2).contiguous().expand(hq, -1, -1)) / math.sqrt(d)
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1), -math.inf)
        want = torch.matmul(torch.softmax(s, -1), vd.expand(hq, -1, -1)).permute(1, 0, 2)
        errs.append(((o.double() - want).norm() / want.norm()).item())
    assert sum(errs) / 4 <= one_tile, errs
