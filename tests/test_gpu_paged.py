"""Paged attention kernels (fp_paged_attention) against float64 attention over
the gathered pages: decode and several queries per sequence, edges of the
16-key tiles, of the 32- and 128-key rounds and of the chunks, page sizes that
are and are not multiples of 16, head dims, GQA ratios, metadata types."""

import math

import pytest
import torch

from flashprefill_amd import vllm_backend as vb

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(lens, news, hq, hkv, d, page, dtype, seed=0, index=torch.int32, width=None, spare=3):
    g = torch.Generator().manual_seed(seed)
    per = [(n + page - 1) // page for n in lens]
    total = sum(per) + spare
    perm = torch.randperm(total, generator=g)
    table = torch.full((len(lens), max(width or 0, max(per), 1)), -1, dtype=index)
    at = 0
    for b, m in enumerate(per):
        table[b, :m] = perm[at:at + m].to(index)
        at += m
    # slots past a sequence's end hold NaN: they must never reach the output
    kc = torch.full((total, page, hkv, d), float("nan"), dtype=dtype)
    vc = torch.full((total, page, hkv, d), float("nan"), dtype=dtype)
    for b, n in enumerate(lens):
        for j in range(per[b]):
            m = min(page, n - j * page)
            kc[table[b, j], :m] = torch.randn(m, hkv, d, generator=g).to(dtype)
            vc[table[b, j], :m] = torch.randn(m, hkv, d, generator=g).to(dtype)
    q = (1.5 * torch.randn(sum(news), hq, d, generator=g)).to(dtype)
    cu = torch.tensor([0] + list(torch.tensor(news).cumsum(0)), dtype=index)
    used = torch.tensor(lens, dtype=index)
    return q, kc, vc, cu, used, table


def _want(q, kc, vc, cu, used, table, scale):
    out = torch.zeros(q.shape, dtype=torch.float64)
    hq, hkv, page = q.shape[1], kc.shape[2], kc.shape[1]
    for b in range(used.numel()):
        n, q0, q1 = int(used[b]), int(cu[b]), int(cu[b + 1])
        if n == 0:
            continue
        rows = table[b, :(n + page - 1) // page].long()
        k = kc[rows].reshape(-1, hkv, q.shape[2])[:n].double().repeat_interleave(hq // hkv, 1)
        v = vc[rows].reshape(-1, hkv, q.shape[2])[:n].double().repeat_interleave(hq // hkv, 1)
        s = torch.einsum("qhd,khd->hqk", q[q0:q1].double(), k) * scale
        pos = torch.arange(n - (q1 - q0), n).view(1, -1, 1)
        s = s.masked_fill(torch.arange(n).view(1, 1, -1) > pos, float("-inf"))
        out[q0:q1] = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), v)
    return out


def _run(args, scale):
    dev = [t.to(DEV) for t in args]
    out = torch.full(args[0].shape, 7.0, dtype=args[0].dtype, device=DEV)
    assert vb._paged_kernel_takes(dev[0], dev[1], dev[2], out, *dev[3:])
    vb.paged_decode_attention(dev[0], dev[1], dev[2], out, *dev[3:], scale)
    return out.cpu()


def _check(args, scale):
    got, want = _run(args, scale).double(), _want(*args, scale)
    # the output is rounded once to the input type: half a spacing, i.e. 2^-8
    # (bf16, 8-bit significand) or 2^-11 (fp16, 11-bit) of the value at most;
    # the fp32 scores, sums and exp2 before it add a few 2^-24 of |v| ~ 4
    eps = 2.0 ** -8 if args[0].dtype == torch.bfloat16 else 2.0 ** -11
    bound = want.abs() * eps * 1.01 + 2e-6
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    assert ((got - want).abs()[~nan] <= bound[~nan]).all(), (got - want)[~nan].abs().max()


@pytest.mark.parametrize("lens", [[1, 15, 16, 17], [31, 32, 33, 127], [128, 129, 255, 256],
                                  [257, 384, 511, 640], [3000, 1, 40, 700]])
@pytest.mark.parametrize("hq,hkv,d,dtype", [(32, 8, 128, torch.bfloat16), (28, 4, 128, torch.float16),
                                            (8, 8, 64, torch.float16), (40, 2, 64, torch.bfloat16),
                                            (8, 2, 256, torch.bfloat16), (6, 3, 256, torch.float16)])
def test_decode(lens, hq, hkv, d, dtype):
    _check(_case(lens, [1] * len(lens), hq, hkv, d, 16, dtype), 1 / math.sqrt(d))


@pytest.mark.parametrize("page", [1, 5, 16, 24, 32, 48, 256])
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
def test_page_sizes_and_index_types(page, index):
    _check(_case([700, 33, 260], [1, 2, 1], 8, 2, 128, page, torch.bfloat16, index=index),
           1 / math.sqrt(128))


@pytest.mark.parametrize("lens,news", [([40, 300, 2100], [1, 7, 33]), ([5, 600, 64], [5, 0, 64]),
                                       ([900, 0, 1300], [200, 3, 130]), ([3, 50], [6, 1]),
                                       ([1500], [700])])
@pytest.mark.parametrize("hq,hkv,d,dtype", [(28, 4, 128, torch.bfloat16), (8, 8, 64, torch.float16),
                                            (8, 2, 256, torch.bfloat16), (32, 8, 128, torch.float16),
                                            (4, 1, 64, torch.bfloat16), (4, 2, 256, torch.float16)])
def test_several_queries(lens, news, hq, hkv, d, dtype):
    # [3, 50] / [6, 1]: rows before the first cached token see nothing (NaN, as
    # softmax over no key); a sequence of no cached tokens gives 0
    _check(_case(lens, news, hq, hkv, d, 16, dtype), 1 / math.sqrt(d))


@pytest.mark.parametrize("page", [1, 16, 24, 64])
@pytest.mark.parametrize("d,dtype", [(128, torch.bfloat16), (64, torch.float16), (128, torch.float16),
                                     (64, torch.bfloat16)])
def test_many_rows_at_tile_edges(page, d, dtype):
    # 128-row tiles (31, 32, 33, 64 queries x 4 heads), 64-key tiles (sequence
    # ends one before, at and after a boundary, inside a page), one chunk and
    # several; queries that see no key (nk < nq)
    for lens, news in (([127, 128, 129, 64], [31, 32, 33, 64]), ([1000, 65, 320], [65, 65, 1]),
                       ([2049, 30], [97, 40])):
        _check(_case(lens, news, 8, 2, d, page, dtype, seed=page), 1 / math.sqrt(d))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("news", [1, 40])
@pytest.mark.parametrize("scale", [0.5, -0.3, 1e-3])
def test_peaked_and_flat_rows(dtype, news, scale):
    # sharp softmax rows (most P far below the largest), a negative scale and
    # nearly uniform rows; V of one sign, so that small P add up
    q, kc, vc, cu, used, table = _case([3000, 700], [news, news], 8, 2, 128, 16, dtype, seed=9)
    vc = vc.abs()
    _check((q, kc, vc, cu, used, table), scale)


def test_wide_table_and_many_sequences():
    # a table far wider than the sequences (a server's limit), and more
    # sequences than one round of the tile search covers
    _check(_case([100, 2000], [1, 1], 8, 2, 128, 16, torch.bfloat16, width=4096), 0.08)
    lens = [(37 * i) % 300 + 1 for i in range(150)]
    _check(_case(lens, [1 + (i % 3 == 0) for i in range(150)], 4, 2, 64, 16, torch.bfloat16), 0.125)


def test_one_long_sequence_uses_every_chunk_slot():
    _check(_case([40000], [1], 4, 1, 128, 16, torch.bfloat16), 0.09)


def test_strided_inputs_and_untouched_rows():
    q, kc, vc, cu, used, table = _case([300, 70], [1, 1], 8, 2, 128, 16, torch.bfloat16)
    T = 5
    qkv = torch.zeros(T, 12, 128, dtype=torch.bfloat16)
    qkv[:2, 2:10] = q
    qd = qkv.to(DEV)[:, 2:10]
    out = torch.full((T, 8, 128), 7.0, dtype=torch.bfloat16, device=DEV)
    vb.paged_decode_attention(qd, kc.to(DEV), vc.to(DEV), out, cu.to(DEV), used.to(DEV),
                              table.to(DEV), 0.1)
    want = _run((q, kc, vc, cu, used, table), 0.1)
    assert torch.equal(out[:2].cpu(), want)
    assert (out[2:] == 7.0).all()


def test_what_only_the_device_sees():
    # a length beyond the table and a page outside the cache: NaN rows, the
    # other sequences as they are; no access outside the cache
    q, kc, vc, cu, used, table = _case([300, 70, 40], [1, 1, 1], 8, 2, 128, 16, torch.bfloat16)
    want = _run((q, kc, vc, cu, used, table), 0.1)
    u2 = used.clone()
    u2[0] = table.shape[1] * 16 + 1
    t2 = table.clone()
    t2[2, 1] = kc.shape[0]
    got = _run((q, kc, vc, cu, u2, t2), 0.1)
    assert got[0].isnan().all() and got[2].isnan().all()
    assert torch.equal(got[1], want[1])


@pytest.mark.parametrize("page", [16, 24, 64])
@pytest.mark.parametrize("d,dtype", [(128, torch.bfloat16), (64, torch.float16)])
def test_a_page_outside_the_cache_at_many_rows(page, d, dtype):
    """40 queries per sequence share the loaded tiles: a bad page at any of the
    tile's four 16-key positions makes every row of its sequence NaN, in several
    chunks (1000 tokens) and in one (200); the other sequence keeps its bits."""
    args = _case([1000, 200], [40, 40], 8, 2, d, page, dtype, seed=page)
    want = _run(args, 0.1)
    for b, first in ((0, 384), (1, 64)):
        for pos in range(4):
            t2 = args[5].clone()
            t2[b, (first + 16 * pos) // page] = (args[1].shape[0], -args[1].shape[0] - 1)[pos % 2]
            got = _run((*args[:5], t2), 0.1)
            rows, rest = slice(40 * b, 40 * b + 40), slice(40 - 40 * b, 80 - 40 * b)
            assert got[rows].isnan().all(), (b, pos, got[rows].isnan().float().mean())
            assert torch.equal(got[rest], want[rest]), (b, pos)


def test_capture_and_replay():
    q, kc, vc, cu, used, table = [t.to(DEV) for t in
                                  _case([900, 70], [1, 1], 8, 2, 128, 16, torch.bfloat16)]
    out = torch.zeros_like(q)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        vb.paged_decode_attention(q, kc, vc, out, cu, used, table, 0.1)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        vb.paged_decode_attention(q, kc, vc, out, cu, used, table, 0.1)
    for n in (900, 300, 897):
        used[0] = n
        want = torch.zeros_like(q)
        vb.paged_decode_attention(q, kc, vc, want, cu, used, table, 0.1)
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_threads_on_one_stream():
    """Two threads on the default stream, chunked calls: neither's partial sums
    reach the other's merge."""
    import threading

    cases = [_case([3000 + 500 * i, 700], [1, 1], 8, 2, 128, 16, torch.bfloat16, seed=60 + i)
             for i in range(2)]
    dev = [[t.to(DEV) for t in c] for c in cases]
    scale = 1 / math.sqrt(128)
    want, got = [], [[], []]
    for c in dev:
        out = torch.empty_like(c[0])
        vb.paged_decode_attention(c[0], c[1], c[2], out, *c[3:], scale)
        want.append(out.clone())

    def work(i):
        c = dev[i]
        for _ in range(200):
            out = torch.empty_like(c[0])
            vb.paged_decode_attention(c[0], c[1], c[2], out, *c[3:], scale)
            got[i].append(out)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 200 and all(torch.equal(o, want[i]) for o in got[i])


def test_forward_mode_keeps_its_tangent():
    """Dual numbers take the torch composition, which carries the tangent: the
    derivative of the output in the values is the attention of the tangent."""
    from torch.autograd import forward_ad

    q, kc, vc, cu, used, table = [t.to(DEV) for t in
                                  _case([48, 32], [1, 1], 8, 2, 64, 16, torch.bfloat16, spare=0)]
    tv = torch.randn(vc.shape, device=DEV).to(vc.dtype)
    want, out = torch.empty_like(q), torch.zeros_like(q)
    vb.paged_attention_reference(q, kc, tv, want, cu, used, table, 0.125)
    with forward_ad.dual_level():
        vb.paged_decode_attention(q, kc, forward_ad.make_dual(vc, tv), out, cu, used, table, 0.125)
        tangent = forward_ad.unpack_dual(out).tangent
        assert tangent is not None
        assert torch.equal(tangent, want)


@pytest.mark.parametrize("hq,hkv", [(1, 1), (5, 5), (6, 3), (7, 1), (9, 3)])
@pytest.mark.parametrize("d", [64, 128])
def test_merge_of_many_rows_at_head_counts(hq, hkv, d):
    """Head counts that are no multiple of the merge's four heads per wave, with
    sequences of one, two and several chunks and one of no query."""
    _check(_case([1300, 70, 700, 40], [41, 33, 35, 0], hq, hkv, d, 16, torch.bfloat16),
           1 / math.sqrt(d))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("news", [1, 40])
@pytest.mark.parametrize("d,page", [(128, 16), (64, 24)])
def test_infinite_values(dtype, news, d, page):
    """+inf and -inf in V at keys that every row sees: those dims are infinite, the
    others what they are without; in several chunks and in one."""
    lens = [1000, 200]
    args = _case(lens, [news] * 2, 8, 2, d, page, dtype, seed=3)
    scale = 1 / math.sqrt(d)
    for b, key in ((0, 500), (1, 77)):
        at = int(args[5][b, key // page]), key % page
        args[2][at[0], at[1], 0, 5] = math.inf
        args[2][at[0], at[1], 1, d - 1] = -math.inf
    got, want = _run(args, scale).double(), _want(*args, scale)
    assert not want.isnan().any() and want.isinf().sum() == 2 * news * 8
    inf = want.isinf()
    assert torch.equal(got[inf], want[inf])
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11  # as in _check
    assert ((got - want).abs()[~inf] <= (want.abs() * eps * 1.01 + 2e-6)[~inf]).all()


@pytest.mark.parametrize("value", [math.inf, math.nan])
@pytest.mark.parametrize("news,d", [(40, 128), (3, 128), (3, 64), (3, 256)])
def test_a_value_that_a_row_does_not_see(value, news, d):
    """An infinity or NaN in V at the last new token reaches the last query only,
    the rows before it stay finite."""
    args = _case([500], [news], 8, 2, d, 16, torch.bfloat16, seed=4)
    want = _want(*args, 0.1)
    args[2][args[5][0, 499 // 16], 499 % 16, :, 7] = value
    got = _run(args, 0.1).double()
    last = news - 1
    assert torch.equal(got[last, :, 7].isnan(), torch.full((8,), math.isnan(value)))
    assert not got[last, :, 7].isfinite().any()
    bound = want.abs()[:last] * 2.0 ** -8 * 1.01 + 2e-6
    assert ((got - want).abs()[:last] <= bound).all()


@pytest.mark.parametrize("news", [1, 40])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("page", [16, 24])
def test_values_near_the_largest(news, d, page):
    """V of 3.3e38 at every key of a dim: the weighted mean is that value, whatever
    the sum of the weights before the division, in one chunk and in several."""
    args = _case([3000, 200], [news] * 2, 8, 2, d, page, torch.bfloat16, seed=5)
    args[2][:, :, 0, 3] = 3.3e38
    args[2][:, :, 1, d - 2] = -3.3e38
    got, want = _run(args, 0.05).double(), _want(*args, 0.05)
    assert want.isfinite().all()
    assert ((got - want).abs() <= want.abs() * 2.0 ** -8 * 1.01 + 2e-6).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("news", [1, 40])
def test_small_probabilities_of_fp16_calls(d, news):
    """A value of 60000 at a key of probability 2^-t, 0 at the key that holds the
    rest: the output is 60000 x 2^-t to half a step of fp16 (2^-25 below its
    normal range) however far t lies below the row's largest probability."""
    ts = [12 + i / 8 for i in range(200)]
    args = _case([64] * len(ts), [news] * len(ts), 4, 1, d, 16, torch.float16, seed=6)
    q, kc, vc, cu, used, table = args
    q.zero_()
    q[..., 0] = 1.0
    for b, t in enumerate(ts):
        kc[table[b]] = 0.0
        kc[table[b], :, :, 0] = -1000.0  # P = 0
        vc[table[b]] = 0.0
        kc[table[b, 0], 0, 0, 0] = 0.0
        kc[table[b, 0], 1, 0, 0] = -t
        vc[table[b, 0], 1, 0, 3] = 60000.0
    got, want = _run(args, math.log(2.0)).double(), _want(*args, math.log(2.0))
    # half a step of the rounded output, and about 2^-20 of the value for the
    # exponent t <= 37 held in fp32 (2^-19 of a step of one, scale included)
    step = torch.clamp(2.0 ** (want.abs().clamp_min(1e-30).log2().floor() - 10), min=2.0 ** -24)
    assert ((got - want).abs() <= 0.5 * step + 2.0 ** -18 * want.abs()).all(), \
        ((got - want).abs() / step).max()


@pytest.mark.parametrize("news", [1, 40])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (8, 4, 256)])
def test_offsets_that_do_not_fit(news, hq, hkv, d):
    """Query offsets past the tokens, below zero or descending, seen only on the
    device: every row of the call is NaN. On the host, these and lengths beyond
    the table are refused."""
    args = _case([1000, 200, 300], [news] * 3, hq, hkv, d, 16, torch.bfloat16)
    n = news
    for cu in ([0, n, 2 * n, 3 * n + 1], [-1, n, 2 * n, 3 * n], [0, 2 * n + 1, 2 * n, 3 * n],
               [0, n, 2 * n, 2 ** 30]):
        bad = torch.tensor(cu, dtype=torch.int32)
        got = _run((*args[:3], bad, *args[4:]), 0.1)
        assert got.isnan().all(), cu
        if max(cu) == 2 ** 30:  # (refused only after masks of that size)
            continue
        dev = [t.to(DEV) for t in args]
        with pytest.raises((RuntimeError, IndexError)):
            vb.paged_decode_attention(*dev[:3], torch.empty_like(dev[0]), bad, *dev[4:], 0.1)
    dev = [t.to(DEV) for t in args]
    with pytest.raises(RuntimeError):
        vb.paged_decode_attention(*dev[:3], torch.empty_like(dev[0]), dev[3],
                                  args[4] + 16 * args[5].shape[1], dev[5], 0.1)
    # fewer rows than tokens: the others stay as they were
    short = torch.tensor([0, n, 2 * n, 3 * n - 1], dtype=torch.int32)
    got = _run((*args[:3], short, *args[4:]), 0.1)
    assert (got[3 * n - 1:] == 7.0).all() and not got[:3 * n - 1].isnan().any()


def test_transforms_take_the_torch_composition():
    """vmap, a trace and a dispatch mode see torch operations: a vmapped call is
    the calls of its slices, and a trace, which cannot follow the lengths, fails
    instead of recording nothing."""
    from torch.utils._python_dispatch import TorchDispatchMode

    args = [t.to(DEV) for t in _case([48, 32], [1, 1], 8, 2, 64, 16, torch.bfloat16, spare=0)]

    def call(q):
        out = torch.zeros_like(q)
        vb.paged_attention_reference(q, *args[1:3], out, *args[3:], 0.125)
        return out

    qs = torch.stack([args[0], 2 * args[0], -args[0]])
    want = torch.stack([call(q) for q in qs])

    def entry(q):
        out = torch.zeros_like(q)
        vb.paged_decode_attention(q, *args[1:3], out, *args[3:], 0.125)
        return out

    # a batched product adds in another order: one rounding to bf16 apart
    assert torch.allclose(torch.vmap(entry)(qs).float(), want.float(), rtol=2.0 ** -7, atol=1e-5)
    with pytest.raises(RuntimeError):
        torch.jit.trace(entry, (qs[0],), check_trace=False)

    class Ops(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, a=(), kw=None):
            seen.append(func.overloadpacket.__name__)
            return func(*a, **(kw or {}))

    seen = []
    with Ops():
        got = entry(qs[2])
    assert "copy_" in seen and torch.equal(got, want[2])


def test_an_output_that_must_not_be_written_is_refused():
    q, kc, vc, cu, used, table = [t.to(DEV) for t in
                                  _case([48, 32], [2, 2], 8, 2, 64, 16, torch.bfloat16)]
    for out in (torch.zeros(1, 8, 64, dtype=q.dtype, device=DEV).expand(4, 8, 64),
                torch.zeros(4, 1, 64, dtype=q.dtype, device=DEV).expand(4, 8, 64)):
        with pytest.raises(RuntimeError):
            vb.paged_decode_attention(q, kc, vc, out, cu, used, table, 0.125)
    with torch.inference_mode():
        out = torch.zeros_like(q)
    with pytest.raises(RuntimeError, match="inference"):
        vb.paged_decode_attention(q, kc, vc, out, cu, used, table, 0.125)


def test_the_write_counts_as_an_in_place_change():
    q, kc, vc, cu, used, table = [t.to(DEV) for t in
                                  _case([48, 32], [1, 1], 8, 2, 64, 16, torch.bfloat16)]
    out = torch.ones_like(q)
    w = torch.ones_like(q, requires_grad=True)
    y = (w * out).sum()  # saves out
    with torch.no_grad():
        vb.paged_decode_attention(q, kc, vc, out, cu, used, table, 0.125)
    with pytest.raises(RuntimeError, match="inplace"):
        y.backward()
