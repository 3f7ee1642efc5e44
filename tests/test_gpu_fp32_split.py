"""fp32 attention on three-part bf16 products: error against float64 over
magnitudes, rows in one and in several chunk slots, and the values that do not
go through the split (2^56 and above, infinities, NaN)."""

import math

import pytest
import torch

from flashprefill_amd import flash_prefill, flash_prefill_varlen_func

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dense(q, k, v):
    """causal attention in float64, q (S, Hq, d)"""
    S, hq, d = q.shape
    g = hq // k.shape[1]
    q, k, v = [t.double().permute(1, 0, 2) for t in (q, k, v)]
    k, v = k.repeat_interleave(g, 0), v.repeat_interleave(g, 0)
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(d)
    s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    return torch.matmul(torch.softmax(s, -1), v).permute(1, 0, 2)


def _run(q, k, v, block=128, last_n=2):
    o = torch.empty_like(q)
    cu = torch.tensor([0, q.shape[0]], dtype=torch.int32, device=DEV)
    # alpha 0: every block (of finite pooled keys; with last_n rows dense, any)
    flash_prefill_varlen_func(q, k, v, o, cu, q.shape[0], 0.0, block, last_n_block=last_n)
    return o


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("S,hq,hkv", [(1, 2, 1), (129, 2, 1), (700, 4, 2), (2100, 2, 2),
                                      (1023, 24, 8)])
@pytest.mark.parametrize("kscale,vscale", [(1.0, 1.0), (1e-3, 1e6), (30.0, 1e-12)])
def test_error_against_float64(block, d, S, hq, hkv, kscale, vscale):
    # 2 heads: several chunk slots per row; (1023, 24): one or two
    g = torch.Generator(device=DEV).manual_seed(S + d)
    q = torch.randn(S, hq, d, generator=g, device=DEV)
    k = torch.randn(S, hkv, d, generator=g, device=DEV) * kscale
    v = torch.randn(S, hkv, d, generator=g, device=DEV) * vscale
    got, want = _run(q, k, v, block).double(), _dense(q, k, v)
    # a score s = sum_d q_d k_d / sqrt(d) in fp32 has an error of about
    # sqrt(d) 2^-24 |q_d k_d| ~ 2^-24 |s|_rms, which shifts log P; the sums of P
    # and P.V add a few 2^-24: 16 x 2^-24 (1 + rms of the scores)
    rel = ((got - want).norm() / want.norm()).item()
    assert rel <= 16 * 2.0 ** -24 * (1 + kscale), rel


@pytest.mark.parametrize("value", [2.0 ** 31, 2.0 ** 32, 2.0 ** 56, 1e30, 3.4028234e38, math.inf, -math.inf])
def test_a_key_of_score_minus_infinity_or_far_below_drops_out(value):
    # keys whose score is hugely negative (or -inf) get P = 0: the rows equal
    # those computed without them, with no NaN from the parts
    S, d = 300, 64
    g = torch.Generator(device=DEV).manual_seed(1)
    q = torch.rand(S, 2, d, generator=g, device=DEV) + 0.5
    k = torch.randn(S, 1, d, generator=g, device=DEV)
    v = torch.randn(S, 1, d, generator=g, device=DEV)
    at = torch.tensor([7, 150, 290], device=DEV)
    k[at] = -abs(value)
    got = _run(q, k, v)
    kk = k.clone()
    kk[at] = -1e3
    want = _run(q, kk, v)
    assert not got.isnan().any()
    # the scalar products add in another order (see the bound above; 4: the rms
    # of these scores)
    assert ((got - want).norm() / want.norm()).item() <= 32 * 2.0 ** -24 * 4


def test_large_and_infinite_values():
    S, d = 300, 64
    g = torch.Generator(device=DEV).manual_seed(2)
    q = torch.randn(S, 1, d, generator=g, device=DEV)
    k = torch.randn(S, 1, d, generator=g, device=DEV)
    v = torch.randn(S, 1, d, generator=g, device=DEV)
    v[3, 0, 5] = 1e35  # finite: the result is finite
    got, want = _run(q, k, v).double(), _dense(q, k, v)
    assert ((got - want)[:, 0, 5].norm() / want[:, 0, 5].norm()).item() <= 64 * 2.0 ** -24
    # every row from 3 on holds inf in that dim (rows 0 .. 2 multiply it by the
    # P = 0 of a masked key, which is NaN, as the reference's masked tile does);
    # the other dims stay finite
    v[3, 0, 5] = math.inf
    got = _run(q, k, v)
    assert got[3:, 0, 5].isinf().all()
    assert got[:, 0, :5].isfinite().all() and got[:, 0, 6:].isfinite().all()
    v[3, 0, 5] = math.nan
    got = _run(q, k, v)
    assert got[3:, 0, 5].isnan().all() and got[:, 0, 6:].isfinite().all()


def test_sparse_lists_in_chunks_match_one_slot_per_row():
    # 4000 tokens of 2 heads (several chunk slots) against the same rows in a
    # batch of enough heads for one slot per row
    from flashprefill_amd import synth
    spec = synth.SynthSpec(seq_lens=(4000,), num_q_heads=2, num_kv_heads=1, head_dim=64,
                           dtype=torch.float32, seed=5)
    q, k, v, _ = synth.make_inputs(spec, "cpu")
    one = [t.to(DEV).unsqueeze(0) for t in (q, k, v)]
    many = [t.repeat(16, 1, 1, 1) for t in one]
    o1, o16 = torch.empty_like(one[0]), torch.empty_like(many[0])
    flash_prefill(*one, o1, 128, 2, 4, 0.3, 2, 0)
    flash_prefill(*many, o16, 128, 2, 4, 0.3, 2, 0)
    # the same products; the chunks' merge adds a rounding per chunk
    assert ((o1 - o16[:1]).norm() / o1.norm()).item() <= 8 * 2.0 ** -24
    assert torch.equal(o16[0], o16[15])


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("scale", [1e-32, 1e-34, 1e-35, 1e-36])
def test_tiny_values_keep_their_bits(d, scale):
    # V, and K against a Q that makes up for it, near the end of fp32's normal
    # range (1.2e-38), where the third of three bf16 parts would be a subnormal
    S = 700
    g = torch.Generator(device=DEV).manual_seed(d)
    q = torch.randn(S, 2, d, generator=g, device=DEV)
    k = torch.randn(S, 1, d, generator=g, device=DEV)
    if scale == 1e-32:  # and near the split's upper end, 2^56 = 7.2e16
        v = torch.randn(S, 1, d, generator=g, device=DEV).clamp(-7, 7) * 1e16
        got, want = _run(q * 1e-16, k * 1e16, v).double(), _dense(q * 1e-16, k * 1e16, v)
        assert ((got - want).norm() / want.norm()).item() <= 32 * 2.0 ** -24
    # magnitudes above 1 / 16, so that no element is a subnormal of its own
    v = torch.randn(S, 1, d, generator=g, device=DEV)
    v = (v + 0.0625 * v.sign()) * scale
    got, want = _run(q, k, v).double(), _dense(q, k, v)
    assert ((got - want).norm() / want.norm()).item() <= 32 * 2.0 ** -24
    up = 2.0 ** 20  # (below the bound of the split)
    down = scale * 64
    got, want = _run(q * up, k * down, v / scale).double(), _dense(q * up, k * down, v / scale)
    assert ((got - want).norm() / want.norm()).item() <= 32 * 2.0 ** -24


def test_tiny_probabilities_keep_their_bits():
    # a V of one non-zero entry at a key of P = 2^-t: the output is P V however
    # small P is (exp2 of an exponent t held in fp32: 2^-24 t)
    S, d, H = 128, 64, 64
    ts = torch.linspace(100, 124, H)
    q = torch.zeros(S, H, d, device=DEV)
    k, v = torch.zeros(S, H, d, device=DEV), torch.zeros(S, H, d, device=DEV)
    q[:, :, 0] = 8 * math.log(2.0)
    k[1, :, 0] = -ts.to(DEV)
    k[2:, :, 0] = -1e4  # P = 0
    v[1, :, 4] = 2.0 ** 20
    got, want = _run(q, k, v).double()[1:, :, 4], _dense(q, k, v)[1:, :, 4]
    assert ((got - want) / want).abs().max().item() <= 124 * 4 * 2.0 ** -24


def _small_products(q, k, truncate):
    """relative weight of the part products that are left out (second by third,
    third by third), the first parts truncated or rounded to nearest"""
    def parts(x):
        x1 = (x.view(torch.int32) & -65536).view(torch.float32) if truncate else x.bfloat16().float()
        x2 = (x - x1).bfloat16().float()
        return x2.double(), (x - x1).double() - x2.double()
    (q2, q3), (k2, k3) = parts(q), parts(k)
    return ((q2 * k3 + q3 * k2 + q3 * k3) / (q.double() * k.double())).abs()


def test_a_score_of_one_product():
    """Scores that are one product q k each (the other dims are 0), for the pairs
    whose small part products weigh most: no further off than a rounded product."""
    g = torch.Generator().manual_seed(11)
    q = 8 * (1 + torch.rand(1000000, generator=g) / 8)
    k = -32 * (1 + torch.rand(1000000, generator=g) / 8)
    top = torch.cat([_small_products(q, k, t).topk(128).indices for t in (False, True)])
    q, k = q[top], k[top]
    assert _small_products(q, k, False).max() <= 2.0 ** -24
    H, d = 256, 64
    Q = torch.zeros(2, H, d)
    K, V = torch.zeros(2, H, d), torch.zeros(2, H, d)
    Q[:, :, 9] = q
    K[0, :, 9] = k
    V[0] = 1.0
    got = _run(Q.to(DEV), K.to(DEV), V.to(DEV)).double().cpu()[1, :, 0]
    s = (q.double() * k.double()) / 8
    want = 1 / (1 + torch.exp(-s))
    # |s| times what its relative error may be: 2^-24 for the product, 2^-24 for its
    # rounding, 2^-24 for that of the scaled exponent, 2^-26 for the scale's; and
    # 2^-22 for exp2, the sum and the quotient
    bound = s.abs() * (3 * 2.0 ** -24 + 2.0 ** -26) + 2.0 ** -22
    rel = ((got - want) / want).abs()
    assert (rel <= bound).all(), (rel / bound).max()


@pytest.mark.parametrize("d,block", [(64, 128), (128, 128), (128, 64), (64, 64)])
@pytest.mark.parametrize("hq", [2, 32])
def test_runs_of_keys_of_score_minus_infinity(d, block, hq):
    # whole tiles of such keys at the start of a row, of a diagonal block and of a
    # chunk drop out (2 heads: several chunk slots per row); a row whose first
    # selected block holds nothing else is NaN, as softmax over that tile is
    S = 1500
    g = torch.Generator(device=DEV).manual_seed(d + block)
    q = torch.rand(S, hq, d, generator=g, device=DEV) + 0.5
    k = torch.randn(S, 1, d, generator=g, device=DEV)
    v = torch.randn(S, 1, d, generator=g, device=DEV)
    gone = torch.zeros(S, dtype=torch.bool, device=DEV)
    gone[:block - 16] = True
    gone[2 * block:2 * block + 64] = True
    gone[4 * block:7 * block] = True
    kk = k.clone()
    kk[gone] = -math.inf
    got = _run(q, kk, v, block, 100).double()
    want = _dense(q, torch.where(gone[:, None, None], torch.full_like(k, -1e4), k), v)
    first = block - 16
    assert got[:first].isnan().all()
    assert ((got - want)[first:].norm() / want[first:].norm()).item() <= 32 * 2.0 ** -24 * 4
    kk[:block] = -math.inf
    assert _run(q, kk, v, block, 100).isnan().all()


@pytest.mark.parametrize("hq", [2, 32])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("large,top", [((10, 11), 100), ((1000, 1001), 5)])
def test_values_whose_sum_overflows_only_without_the_row_maximum(hq, d, large, top):
    # two values of 3e38 at keys e^-8 below the row's largest, which lies in another
    # tile of their block or in another chunk: the result is finite
    S = 1500
    q = torch.zeros(S, hq, d, device=DEV)
    k, v = torch.zeros(S, 1, d, device=DEV), torch.zeros(S, 1, d, device=DEV)
    q[..., 0] = math.sqrt(d)
    k[:, 0, 0] = -1000.0
    k[list(large), 0, 0] = 0.0
    k[top, 0, 0] = 8.0
    v[list(large), 0, 5] = 3e38
    got = _run(q, k, v, 128, 100)[1002:, :, 5].double()
    want = 6e38 * math.exp(-8) / (1 + 2 * math.exp(-8))
    assert ((got - want) / want).abs().max().item() <= 9 * 8 * 2.0 ** -24
