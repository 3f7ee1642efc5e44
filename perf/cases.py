"""The framework's performance cases: what a user's program has it do.

``listed()`` names the fixed cases, ``draw(rng)`` gives further ones of the
same ranges. A case is a dict of plain values; ``prepare(case, seed)`` makes
what a program holds before the call (tensors on the GPU, weights, the paged
cache), ``run(state)`` is one pass through the public entry points,
``work(case)`` the bytes and operations such a pass cannot do without,
``tolerance(case)`` how far two correct implementations at the same precision
may lie apart, and ``exact(case, seed)`` the same outputs in 64 bits by plain
torch.

Five kinds of case:

* ``varlen``: ``flash_prefill_varlen_func`` on packed sequences (the entry
  point that a serving engine calls);
* ``native``: ``flash_prefill`` on a (batch, seq, heads, dim) batch with
  ``min_budget`` (the entry point that the model files call);
* ``hook``: the serving hook's forward on a prefill step, i.e. the paged
  KV-cache write and the sparse prefill;
* ``paged``: ``paged_decode_attention`` over a paged cache, decode steps
  (one query per sequence) and prefix-cache prefill (many);
* ``layer``: the decoder layer's attention block (QKV projection, q/k norm and
  RoPE, sparse prefill, output projection).
"""

import math
from types import SimpleNamespace

import torch

from flashprefill_amd import synth
from flashprefill_amd.attention_layer import PrefillAttention
from flashprefill_amd.flashprefill_native_forward import flash_prefill
from flashprefill_amd.flashprefill_varlen_func import flash_prefill_varlen_func
from flashprefill_amd.vllm_backend import make_forward, paged_decode_attention

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# selection settings that every caller of the operator passes
SINK, WINDOW, LAST_N = 2, 4, 2
PAGE = 16  # tokens per page of the paged KV cache


def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def _attn(kind, name, lens, hq, hkv, d, dtype="bf16", alpha=0.18, block=128, **more):
    case = {"kind": kind, "lens": ",".join(str(int(x)) for x in lens), "hq": hq, "hkv": hkv,
            "d": d, "dtype": dtype, "alpha": alpha, "block": block}
    case.update(more)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # a short prompt: launches, host work and one wave of rows
        _attn("varlen", "prompt_1k", [1000], 32, 8, 128),
        # an ordinary chat prompt with the Llama head shapes
        _attn("varlen", "prompt_4k", [4096], 32, 8, 128),
        # a document
        _attn("varlen", "prompt_32k", [32768], 32, 8, 128),
        # the headline: one long-context prompt
        _attn("varlen", "prompt_128k", [131072], 32, 8, 128),
        # a serving step of ragged prompts with the Qwen2.5 head shapes, through
        # the serving hook (KV-cache write included)
        _attn("hook", "serving_step_ragged", [40001, 17408, 3072, 1023, 129, 1], 28, 4, 128,
              alpha=0.08),
        # a batch through the model files' entry point: fp16, head_dim 64, a budget
        _attn("native", "batch_fp16_d64", [8192] * 4, 32, 8, 64, dtype="fp16", alpha=0.12,
              budget=16),
        # full-precision inputs (the CPU-sized configuration's shape)
        _attn("native", "full_precision_4k", [4096], 8, 2, 64, dtype="fp32", alpha=0.12, budget=0),
        # wide heads
        _attn("varlen", "wide_heads_16k", [16384], 32, 8, 256),
        # a decode step of 32 running requests of mixed context lengths
        _attn("paged", "decode_32", [(211 + 977 * i * i) % 15000 + 300 for i in range(32)],
              32, 8, 128, new=1),
        # decode of one long request: too few sequences to fill the card by themselves
        _attn("paged", "decode_one_long", [65000], 32, 8, 128, new=1),
        # prompts whose prefix is cached: the new tokens attend over the pages
        _attn("paged", "prefix_prefill", [6144, 2500, 1111], 28, 4, 128, new=500),
        # the attention block of a decoder layer (Qwen3-MoE head shapes)
        _attn("layer", "decoder_layer_16k", [12000, 4384], 32, 4, 128, alpha=0.12, hidden=4096),
    ]


def _split(rng, total, n):
    """total tokens as n ragged lengths, odd ones among them"""
    w = [rng.random() ** 2 + 0.01 for _ in range(n)]
    s = sum(w)
    return [max(1, int(total * x / s)) for x in w]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["varlen", "varlen", "varlen", "native", "hook", "paged", "paged", "layer"])
    alpha = rng.choice([0.08, 0.12, 0.18])
    if kind == "paged":
        hq, hkv = rng.choice([(32, 8), (28, 4), (32, 4), (8, 2)])
        d = rng.choice([64, 128, 128])
        dtype = rng.choice(["bf16", "bf16", "fp16"])
        n = _log_uniform(rng, 1, 32)
        if rng.random() < 0.7:  # decode
            return _attn(kind, None, [_log_uniform(rng, 40, 15000) for _ in range(n)], hq, hkv, d,
                         dtype, new=1)
        n = min(n, 3)
        new = _log_uniform(rng, 2, 500)
        return _attn(kind, None, [new + _log_uniform(rng, 1, 5500) for _ in range(n)], hq, hkv, d,
                     dtype, new=new)
    if kind == "layer":
        total = _log_uniform(rng, 200, 16000)
        return _attn(kind, None, _split(rng, total, rng.randint(1, 4)), 32, 4, 128,
                     alpha=alpha, hidden=rng.choice([2048, 4096]))
    hq, hkv = rng.choice([(32, 8), (32, 8), (28, 4), (32, 4), (8, 2), (4, 1)])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    d = rng.choice([128, 128, 128, 64, 256])
    if dtype == "fp32":
        d = min(d, 128)
    block = rng.choice([128, 128, 128, 64] if d == 256 else [128, 128, 128, 64, 256])
    if kind == "hook":
        dtype, block = ("bf16" if dtype == "fp32" else dtype), 128
    top = 4096 if dtype == "fp32" else 16384 if d == 256 else 65536
    total = _log_uniform(rng, 150, top)
    if kind == "native":
        b = rng.randint(1, 4)
        return _attn(kind, None, [max(1, total // b)] * b, hq, hkv, d, dtype, alpha, block,
                     budget=rng.choice([0, 0, 8, 40]))
    return _attn(kind, None, _split(rng, total, rng.randint(1, 6)), hq, hkv, d, dtype, alpha, block)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1234577 * (seed + 1))
    return g


def _qkv(case, seed):
    """Structured prefill inputs: sinks, stripes, a local band, topics and hot
    blocks, so that the selection is sparse as it is on real prompts."""
    spec = synth.SynthSpec(seq_lens=tuple(_lens(case)), num_q_heads=case["hq"],
                           num_kv_heads=case["hkv"], head_dim=case["d"],
                           dtype=DTYPES[case["dtype"]], seed=seed)
    return synth.make_inputs(spec, "cuda")


def _paged_cache(case, lens, g):
    """A cache of shuffled pages, the block table and the lengths."""
    hkv, d, dtype = case["hkv"], case["d"], DTYPES[case["dtype"]]
    pages = [(n + PAGE - 1) // PAGE for n in lens]
    total = sum(pages)
    perm = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32, device="cuda")
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        at += n
    return total, table


def prepare(case, seed):
    kind, lens = case["kind"], _lens(case)
    hq, hkv, d, dtype = case["hq"], case["hkv"], case["d"], DTYPES[case["dtype"]]
    st = SimpleNamespace(case=case, kind=kind)
    if kind == "paged":
        g = _generator(seed)
        total, st.table = _paged_cache(case, lens, g)
        shape = (total, PAGE, hkv, d)
        st.key_cache = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
        st.value_cache = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
        n = len(lens) * case["new"]
        # queries a little sharper than unit variance, as trained heads are
        st.query = 1.5 * torch.randn(n, hq, d, generator=g, device="cuda", dtype=dtype)
        st.out = torch.empty_like(st.query)
        st.cu = torch.arange(0, n + 1, case["new"], dtype=torch.int32, device="cuda")
        st.used = torch.tensor(lens, dtype=torch.int32, device="cuda")
        return st
    if kind == "layer":
        g = _generator(seed)
        st.module = PrefillAttention(case["hidden"], hq, hkv, d, qk_norm=True,
                                     alpha=case["alpha"], dtype=dtype, device="cuda", seed=seed)
        st.x = torch.randn(sum(lens), case["hidden"], generator=g, device="cuda", dtype=dtype)
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        st.cu = torch.tensor(cu, dtype=torch.int32, device="cuda")
        st.max_len = max(lens)
        return st
    st.q, st.k, st.v, st.cu = _qkv(case, seed)
    st.o = torch.empty_like(st.q)
    st.max_len = max(lens)
    if kind == "native":
        b, s = len(lens), lens[0]
        st.q, st.o = st.q.view(b, s, hq, d), st.o.view(b, s, hq, d)
        st.k, st.v = st.k.view(b, s, hkv, d), st.v.view(b, s, hkv, d)
    if kind == "hook":
        total, table = _paged_cache(case, lens, _generator(seed))
        st.kv_cache = torch.zeros(2, total, PAGE, hkv, d, dtype=dtype, device="cuda")
        slots = []
        for b, n in enumerate(lens):
            pos = torch.arange(n, device="cuda")
            slots.append(table[b, pos // PAGE].long() * PAGE + pos % PAGE)
        st.meta = SimpleNamespace(num_actual_tokens=sum(lens), slot_mapping=torch.cat(slots),
                                  query_start_loc=st.cu, max_query_len=max(lens),
                                  seq_lens=None, block_table=table, use_cascade=False)
        st.impl = SimpleNamespace(scale=1.0 / math.sqrt(d), attn_type="decoder",
                                  kv_cache_dtype="auto")
        st.forward = make_forward({"block_size": case["block"], "attention_sink": SINK,
                                   "window_size": WINDOW, "alpha": case["alpha"],
                                   "last_n_full_block": LAST_N})
    return st


def run(st):
    case = st.case
    if st.kind == "varlen":
        flash_prefill_varlen_func(st.q, st.k, st.v, st.o, st.cu, st.max_len, case["alpha"],
                                  case["block"], SINK, WINDOW, LAST_N)
        return st.o
    if st.kind == "native":
        flash_prefill(st.q, st.k, st.v, st.o, case["block"], SINK, WINDOW, case["alpha"], LAST_N,
                      case["budget"])
        return st.o
    if st.kind == "hook":
        out = st.forward(st.impl, None, st.q, st.k, st.v, st.kv_cache, st.meta, st.o)
        return [out, st.kv_cache]
    if st.kind == "paged":
        paged_decode_attention(st.query, st.key_cache, st.value_cache, st.out, st.cu, st.used,
                               st.table, 1.0 / math.sqrt(case["d"]))
        return st.out
    return st.module(st.x, st.cu, st.max_len)


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------

def _selected_blocks(case, n):
    """About how many 128-token key blocks the selection keeps for a sequence
    of n tokens and one query head: every causal block of the last rows, and
    about 3.3 log2(nb) - 8 of the others on these inputs at alpha 0.18 (8.4,
    13.5, 18 and 24 measured at 4K, 16K, 32K and 128K), more at smaller alpha
    (about 1.3 x at 0.12, 1.7 x at 0.08); never more than are causal. Random
    weights (the layer) keep every block."""
    nb = (n + 127) // 128
    if case["kind"] == "layer":
        return nb * (nb + 1) / 2
    per = max(6.0, 3.3 * math.log2(max(nb, 2)) - 8.0) * min(2.0, (0.18 / case["alpha"]) ** 0.65)
    per = max(per, case.get("budget", 0) * case["block"] / 128)
    return sum(i + 1 if i >= nb - LAST_N else min(i + 1, per) for i in range(nb))


def work(case):
    lens, hq, hkv, d = _lens(case), case["hq"], case["hkv"], case["d"]
    eb = 4 if case["dtype"] == "fp32" else 2
    total = sum(lens)
    if case["kind"] == "paged":
        new = case["new"]
        pairs = sum(new * (n - new) + new * (new + 1) / 2 for n in lens)
        return {"bytes": 2 * total * hkv * d * eb + 2 * len(lens) * new * hq * d * eb,
                "flops": 4 * d * hq * pairs}
    byts = 2 * total * (hq + hkv) * d * eb
    flops = 0.0
    for n in lens:
        nb = (n + case["block"] - 1) // case["block"]
        flops += 2 * d * hq * n * (nb + 1) / 2  # every query against the pooled keys
        # a diagonal block is half a block
        nb = (n + 127) // 128
        flops += hq * 4 * 128 * 128 * d * (_selected_blocks(case, n) - nb / 2)
    if case["kind"] == "hook":
        byts += 2 * total * hkv * d * eb  # the cache pages written
    if case["kind"] == "layer":
        hid = case["hidden"]
        flops += 2 * total * hid * d * (2 * hq + 2 * hkv)
        byts = eb * (2 * total * hid + hid * d * (2 * hq + 2 * hkv))
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """fp32: sums in another order. 16 bits: the outputs and the probabilities
    are rounded to the input type (bf16 keeps 8 bits, fp16 11), and a block
    near the selection's threshold may fall on the other side of it."""
    return {"rel": {"fp32": 1e-5, "bf16": 1e-2, "fp16": 2e-3}[case["dtype"]]}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _exact_sequence(q, k, v, case, native):
    """Sparse prefill of one sequence, q (S, Hq, d), k / v (S, Hkv, d) float64
    tensors of the (16- or 32-bit) inputs: pooled keys rounded to the input
    type, everything else in float64."""
    S, hq, d = q.shape
    blk, g = case["block"], hq // k.shape[1]
    nb = (S + blk - 1) // blk
    pad = nb * blk - S
    c = math.log2(math.e) / math.sqrt(d)
    counts = torch.full((nb,), blk, dtype=torch.float64, device=q.device)
    counts[-1] = blk - pad
    at = torch.arange(nb, device=q.device)
    causal = at[None, :] <= at[:, None]
    forced = (at[None, :] < SINK) | (at[:, None] - at[None, :] < WINDOW) | \
        (at[:, None] >= nb - LAST_N)
    out = torch.zeros_like(q)
    pos = torch.arange(nb * blk, device=q.device).view(nb, blk)
    for h in range(hq):
        kp = torch.nn.functional.pad(k[:, h // g], (0, 0, 0, pad)).view(nb, blk, d)
        vp = torch.nn.functional.pad(v[:, h // g], (0, 0, 0, pad)).view(nb, blk, d)
        qp = torch.nn.functional.pad(q[:, h], (0, 0, 0, pad)).view(nb, blk, d)
        mk = (kp.sum(1) / counts[:, None]).to(DTYPES[case["dtype"]]).double()
        s = torch.matmul(qp.reshape(nb * blk, d), mk.t().contiguous()).view(nb, blk, nb) * c
        m = s.amax(1)
        p = torch.exp2(s - m[:, None]).sum(1)
        # the diagonal block counts the block's last row only
        m.diagonal().copy_(s[:, blk - 1].diagonal())
        p.diagonal().fill_(1.0)
        del s
        m.masked_fill_(~causal, -math.inf)
        sc = torch.where(causal, p * torch.exp2(m - m.amax(1, keepdim=True)), 0.0)
        if native:
            sc = sc / (sc.sum(1, keepdim=True) + 1e-9)
        keep = (sc >= case["alpha"] * sc.amax(1, keepdim=True)) | forced
        budget = case.get("budget", 0)
        if budget > 0:  # the largest scores of the row, lower blocks first among equals
            order = torch.where(causal, sc, -1.0).sort(dim=1, descending=True, stable=True).indices
            top = torch.zeros_like(keep)
            top.scatter_(1, order[:, :min(budget, nb)], True)
            keep = keep | top
        keep = keep & causal
        n_keep = keep.sum(1).tolist()
        cols = keep.nonzero()[:, 1]
        first = 0
        for i in range(nb):
            js = cols[first:first + n_keep[i]]
            first += n_keep[i]
            kk, vv = kp[js].reshape(-1, d), vp[js].reshape(-1, d)
            a = torch.matmul(qp[i], kk.t().contiguous()) * c
            a[:, -blk:].masked_fill_(pos[i][None, :] > pos[i][:, None], -math.inf)
            a = torch.exp2(a - a.amax(1, keepdim=True))
            r = torch.matmul(a / a.sum(1, keepdim=True), vv)
            rows = min(blk, S - i * blk)
            out[i * blk:i * blk + rows, h] = r[:rows]
    return out


def _exact_paged(st, case, lens):
    outs = []
    hq, hkv, d, new = case["hq"], case["hkv"], case["d"], case["new"]
    for b, n in enumerate(lens):
        pages = st.table[b, :(n + PAGE - 1) // PAGE].long()
        k = st.key_cache[pages].reshape(-1, hkv, d)[:n].double()
        v = st.value_cache[pages].reshape(-1, hkv, d)[:n].double()
        q = st.query[b * new:(b + 1) * new].double()
        hidden = torch.arange(n, device=q.device)[None] > \
            torch.arange(n - new, n, device=q.device)[:, None]
        o = torch.empty_like(q)
        for h in range(hq):
            s = torch.matmul(q[:, h], k[:, h // (hq // hkv)].t().contiguous()) / math.sqrt(d)
            s.masked_fill_(hidden, -math.inf)
            o[:, h] = torch.matmul(torch.softmax(s, -1), v[:, h // (hq // hkv)])
        outs.append(o)
    return torch.cat(outs)


def _exact_layer(st, case, lens):
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    mod, half = st.module, case["d"] // 2
    qkv = torch.matmul(st.x.double(), mod.w_qkv.double().t().contiguous())
    qkv = qkv.view(-1, hq + 2 * hkv, d)

    def norm(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + mod.rms_eps) * w.double()

    def rope(x):
        inv = mod.rope_theta ** (-torch.arange(0, d, 2, device=x.device, dtype=torch.float64) / d)
        ang = torch.arange(x.shape[0], device=x.device, dtype=torch.float64)[:, None] * inv
        cos, sin = ang.cos()[:, None], ang.sin()[:, None]
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    outs, at = [], 0
    for n in lens:
        x = qkv[at:at + n]
        at += n
        q = rope(norm(x[:, :hq], mod.q_norm))
        k = rope(norm(x[:, hq:hq + hkv], mod.k_norm))
        outs.append(_exact_sequence(q, k, x[:, hq + hkv:], case, False))
    o = torch.cat(outs).view(-1, hq * d)
    return torch.matmul(o, mod.w_o.double().t().contiguous())


def exact(case, seed):
    st, lens = prepare(case, seed), _lens(case)
    if case["kind"] == "paged":
        return _exact_paged(st, case, lens)
    if case["kind"] == "layer":
        return _exact_layer(st, case, lens)
    native = case["kind"] == "native"
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    q, k, v = st.q.reshape(-1, hq, d), st.k.reshape(-1, hkv, d), st.v.reshape(-1, hkv, d)
    outs, at = [], 0
    for n in lens:
        outs.append(_exact_sequence(q[at:at + n].double(), k[at:at + n].double(),
                                    v[at:at + n].double(), case, native))
        at += n
    out = torch.cat(outs)
    if native:
        return out.view(st.q.shape)
    if case["kind"] == "hook":
        cache = torch.zeros(st.kv_cache.shape, dtype=torch.float64, device=q.device)
        flat = cache.view(2, -1, hkv, d)
        flat[0, st.meta.slot_mapping] = k.double()
        flat[1, st.meta.slot_mapping] = v.double()
        return [out, cache]
    return out
