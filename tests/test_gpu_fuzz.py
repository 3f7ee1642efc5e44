"""Seeded random configurations through every stage, against the oracle.

Each case draws sequence lengths (including 1-token and partial-block
sequences), head counts with a GQA ratio, head dim, dtype, selection
parameters and the native / varlen mode, and runs the staged parity check:
pooled K, block scores, exact selection in both directions from identical
fp32 scores, and the attention output within the bf16 (fp32) tolerance. Seeds
from 12 on also vary the block size (64 / 128) and include fp32 inputs. The sequences are short (at most ~10 blocks),
so sink / window / last-n rules keep most blocks: these cases stress the
edges (1-token and partial blocks, GQA ratios, d = 64, fp16, native mode,
min_budget); sparse selection at length is covered by the structured 4K and
128K tests. A third set draws block sizes up to 256 and head dims up to 256. Four larger seeded cases (ragged batches of 19K-55K tokens from
the structured synthetic distribution, sampled attention rows) are sized so
that the attention stage runs as the persistent grid."""

import random

import pytest
import torch

from flashprefill_amd import synth
from tests._parity import (OUT_MAX_ABS, OUT_MAX_ABS_F32, OUT_MEAN_ABS, OUT_MEAN_ABS_F32,
                           assert_pool, persistent_grid_slots, run_stages)

pytestmark = pytest.mark.gpu


def _case(seed):
    rnd = random.Random(seed)
    nseq = rnd.randint(1, 4)
    lens = [rnd.choice([1, rnd.randint(2, 127), rnd.randint(128, 1500), 128 * rnd.randint(1, 10)])
            for _ in range(nseq)]
    hkv = rnd.choice([1, 2, 4])
    hq = hkv * rnd.choice([1, 2, 4, 7])
    d = rnd.choice([64, 128])
    dtype = rnd.choice([torch.bfloat16, torch.float16])
    params = dict(alpha=rnd.choice([0.0, 0.05, 0.12, 0.18, 0.5, 0.9]),
                  sink=rnd.randint(0, 4), window=rnd.randint(0, 6), last_n=rnd.randint(0, 3),
                  native=rnd.random() < 0.3)
    if params["native"] and rnd.random() < 0.5:
        params["min_budget"] = rnd.randint(1, 12)
    # score spread: unit-scale inputs give flat block scores (every block
    # kept); larger Q/K scales, sink rows and a shared direction in a few key
    # blocks give peaked, sparse selections
    shape = dict(scale=rnd.uniform(1.0, 4.0), sink=rnd.random() < 0.7, stripes=rnd.randint(0, 4))
    # seeds from 1012 on also draw the block size and fp32 inputs (the draws
    # above are unchanged for every seed)
    block = 128
    if seed >= 1012:
        block = rnd.choice([64, 128])
        if rnd.random() < 0.4:
            dtype = torch.float32
    return lens, hq, hkv, d, dtype, params, shape, block


# seeds 50 and 130 (and 53, 56, 91, 105 of the wide set) reach outputs of
# magnitude >= 4, where a bf16 ulp (2^-5) exceeds the max-abs bar and the
# parity helper holds elements to one ulp (output_errors)
@pytest.mark.parametrize("seed", list(range(24)) + [50, 130])
def test_random_configuration(seed):
    lens, hq, hkv, d, dtype, params, shape, block = _case(1000 + seed)
    g = torch.Generator().manual_seed(seed)
    T = sum(lens)
    q = torch.randn(T, hq, d, generator=g) * shape["scale"]
    k = torch.randn(T, hkv, d, generator=g) * shape["scale"]
    v = torch.randn(T, hkv, d, generator=g)
    cu = [0]
    for s in lens:
        cu.append(cu[-1] + s)
    u = torch.randn(d, generator=g)
    u = u / u.norm()
    for b in range(len(lens)):
        a0, a1 = cu[b], cu[b + 1]
        if shape["sink"]:
            k[a0:min(a0 + 4, a1)] *= 4.0
        for _ in range(shape["stripes"]):  # a key block aligned with the queries' shared direction
            if a1 - a0 >= block:
                j0 = a0 + block * int(torch.randint(0, (a1 - a0) // block, (1,), generator=g))
                k[j0:j0 + block] += 3.0 * shape["scale"] * u
    q += 0.5 * shape["scale"] * u
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    print(f"\n  seed={seed} lens={lens} hq={hq} hkv={hkv} d={d} {dtype} block={block} {params} "
          f"{shape}", flush=True)
    rep = run_stages(q, k, v, cu, max(lens), block=block, **params)
    print(f"  flips={rep.e2e_flips}/{rep.cells} density={rep.density:.3f} "
          f"out_max={rep.out_max_abs:.2e} out_mean={rep.out_mean_abs:.2e} "
          f"coarse={rep.out_coarse} ({rep.out_coarse_ulp} ulp)", flush=True)
    assert_pool(rep)
    assert rep.m_max_rel < 1e-4
    assert rep.p_max_rel < 1e-3
    assert rep.sel_from_gpu_scores_mismatch == 0
    assert rep.sel_from_oracle_scores_mismatch == 0
    assert rep.e2e_flips <= max(2, 2e-3 * rep.cells)
    f32 = dtype == torch.float32
    assert rep.out_max_abs <= (OUT_MAX_ABS_F32 if f32 else OUT_MAX_ABS)
    assert rep.out_mean_abs <= (OUT_MEAN_ABS_F32 if f32 else OUT_MEAN_ABS)


def _wide_case(seed):
    """Block sizes 64 / 128 / 256 and head dims 64 / 128 / 256 over the same
    random edges (the supported combinations: head_dim 256 for 16-bit inputs at
    blocks of 64 and 128)."""
    lens, hq, hkv, _, _, params, shape, _ = _case(seed)
    rnd = random.Random(seed * 7 + 3)
    # (block, head_dim) in turn over the seeds
    block, d = [(256, 128), (64, 256), (256, 64), (128, 256)][seed % 4]
    dtype = rnd.choice([torch.bfloat16, torch.float16, torch.bfloat16, torch.float16, torch.float32])
    if d == 256 and dtype == torch.float32:
        dtype = torch.bfloat16
    return lens, hq, hkv, d, dtype, params, shape, block


@pytest.mark.parametrize("seed", list(range(16)) + [53, 56, 91, 105])
def test_random_configuration_wide_blocks_and_head_dims(seed):
    lens, hq, hkv, d, dtype, params, shape, block = _wide_case(3000 + seed)
    g = torch.Generator().manual_seed(300 + seed)
    T = sum(lens)
    q = torch.randn(T, hq, d, generator=g) * shape["scale"]
    k = torch.randn(T, hkv, d, generator=g) * shape["scale"]
    v = torch.randn(T, hkv, d, generator=g)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    if shape["sink"]:
        for b in range(len(lens)):
            k[cu[b]:min(cu[b] + 4, cu[b + 1])] *= 4.0
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    print(f"\n  seed={seed} lens={lens} hq={hq} hkv={hkv} d={d} {dtype} block={block} {params}",
          flush=True)
    rep = run_stages(q, k, v, cu, max(lens), block=block, **params)
    print(f"  flips={rep.e2e_flips}/{rep.cells} density={rep.density:.3f} "
          f"out_max={rep.out_max_abs:.2e} out_mean={rep.out_mean_abs:.2e} "
          f"coarse={rep.out_coarse} ({rep.out_coarse_ulp} ulp)", flush=True)
    assert_pool(rep)
    assert rep.m_max_rel < 1e-4
    assert rep.p_max_rel < 1e-3
    assert rep.sel_from_gpu_scores_mismatch == 0
    assert rep.sel_from_oracle_scores_mismatch == 0
    assert rep.e2e_flips <= max(2, 2e-3 * rep.cells)
    f32 = dtype == torch.float32
    assert rep.out_max_abs <= (OUT_MAX_ABS_F32 if f32 else OUT_MAX_ABS)
    assert rep.out_mean_abs <= (OUT_MEAN_ABS_F32 if f32 else OUT_MEAN_ABS)


def _large_case(seed):
    """Ragged batches; the test grows them until the attention stage runs as the
    persistent grid."""
    rnd = random.Random(seed)
    block = rnd.choice([64, 128])
    hkv = rnd.choice([2, 4, 8])
    hq = hkv * rnd.choice([4, 7, 8]) if hkv < 8 else 32
    d = rnd.choice([64, 128])
    dtype = rnd.choice([torch.bfloat16, torch.float16])
    nseq = rnd.randint(2, 4)
    lens = [rnd.choice([rnd.randint(1, 300), rnd.randint(2000, 9000), rnd.randint(9000, 24000)])
            for _ in range(nseq)]
    params = dict(alpha=rnd.choice([0.05, 0.12, 0.18]), sink=rnd.randint(0, 3),
                  window=rnd.randint(1, 6), last_n=rnd.randint(0, 3))
    return lens, hq, hkv, d, dtype, params, block


@pytest.mark.parametrize("seed", range(4))
def test_random_large_configuration_persistent_attention(seed):
    lens, hq, hkv, d, dtype, params, block = _large_case(2000 + seed)
    # grow the longest sequence until the slots reach twice the host's threshold
    # for the persistent grid, so that every workgroup claims several
    while True:
        slots, least = persistent_grid_slots(hq, lens, block, d)
        if slots >= 2 * least:
            break
        lens[lens.index(max(lens))] += 4096
    # the structured synthetic distribution of the benchmark (sinks, stripes,
    # a rotary local band, hot blocks): sparse selections with ragged lists
    spec = synth.SynthSpec(seq_lens=tuple(lens), num_q_heads=hq, num_kv_heads=hkv, head_dim=d,
                           dtype=dtype, seed=seed, block=block)
    q, k, v, cu_t = synth.make_inputs(spec, device="cpu")
    cu = [int(x) for x in cu_t]
    rows = {}
    for b, n in enumerate(lens):
        nb = (n + block - 1) // block
        rows[b] = sorted({(h, i) for h in (0, hq // 2, hq - 1) for i in (0, nb // 2, nb - 1)})
    print(f"\n  seed={seed} lens={lens} hq={hq} hkv={hkv} d={d} {dtype} block={block} {params}",
          flush=True)
    rep = run_stages(q, k, v, cu, max(lens), block=block, attn_rows=rows, **params)
    print(f"  flips={rep.e2e_flips}/{rep.cells} density={rep.density:.3f} "
          f"out_max={rep.out_max_abs:.2e} out_mean={rep.out_mean_abs:.2e} "
          f"coarse={rep.out_coarse} ({rep.out_coarse_ulp} ulp)", flush=True)
    assert_pool(rep)
    assert rep.m_max_rel < 1e-4
    assert rep.p_max_rel < 1e-3
    assert rep.sel_from_gpu_scores_mismatch == 0
    assert rep.sel_from_oracle_scores_mismatch == 0
    assert rep.e2e_flips <= max(2, 2e-3 * rep.cells)
    assert rep.out_max_abs <= OUT_MAX_ABS
    assert rep.out_mean_abs <= OUT_MEAN_ABS
