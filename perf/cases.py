"""The decode calls that the performance of this package is judged by.

A case is one decode step's call (or, for an engine that plans once per step,
the plan and its layers' calls) as a serving program makes it: a batch of
sequences whose K/V pages are scattered over one paged cache, one query per
sequence and query head.  The listed cases stand for the uses named beside
them; ``draw`` gives others from the same ranges.

Fields of a case:

* ``batch``, ``hq``, ``hkv``, ``d``, ``ps``: sequences, query heads, kv heads,
  head dimension, tokens per page;
* ``lo``, ``hi``: lengths are uniform in [lo, hi], drawn from ``lens``, with
  the two ends among them (their order over the batch comes from the seed);
* ``room``: tokens that a row of the dense block table has columns for;
* ``q``, ``kv``: element types of q (and the output) and of the caches;
* ``index``: how the pages are given: ``dense`` (block_table, seq_lens),
  ``csr`` (indptr, indices, last_page_len), or a ``BatchDecodeWrapper`` planned
  in the pass over either (``planned``, ``planned_csr``) and run for every layer;
* ``layers``: caches (and queries) that one pass decodes from.
"""

import math
import random

import torch

import paged_attention_decode_amd as pad

_TYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
_FP8_MAX = {"e4m3": 448.0, "e5m2": 57344.0}
# One key row in this many is scaled by 8: the outliers that move a running
# softmax maximum in the middle of a sequence.
_OUTLIERS = 4096


def _case(name, batch, hq, hkv, d, ps, lo, hi, room=None, q="fp16", kv=None, index="dense", layers=1, lens=1):
    c = {"name": name} if name else {}
    c.update(batch=batch, hq=hq, hkv=hkv, d=d, ps=ps, lo=lo, hi=hi, room=room or hi, q=q, kv=kv or q, index=index,
             layers=layers, lens=lens)
    return c


def listed():
    return [
        # One user, a short context: the smallest call, where latency counts.
        _case("b1_1k", 1, 12, 2, 128, 16, 1024, 1024),
        # A few users of one server, whose block table has a column for every
        # page of the model's context.
        _case("b4_chat_wide_table", 4, 12, 2, 128, 16, 200, 3000, room=32768),
        # The two ordinary uniform batches of the latency / bandwidth sweep.
        _case("b16_4k", 16, 12, 2, 128, 16, 4096, 4096),
        _case("b64_4k", 64, 12, 2, 128, 16, 4096, 4096),
        # A ragged batch of everything from one token to 8192.
        _case("b32_ragged_page32", 32, 12, 2, 128, 32, 1, 8192),
        # One long document.
        _case("b1_128k", 1, 32, 8, 128, 16, 131072, 131072),
        # A full server: 17 GB of K/V for one call, the largest.
        _case("b256_ragged_32k", 256, 64, 8, 128, 16, 512, 32768),
        # Quantised caches under a bfloat16 model.
        _case("b64_fp8_ragged", 64, 32, 8, 128, 16, 1, 8192, q="bf16", kv="e4m3"),
        # An engine that keeps a token-granular page pool (page size 1) as a
        # CSR index, plans once per step and runs its layers from the plan.
        _case("b48_planned_csr_page1", 48, 32, 8, 128, 1, 1, 4096, q="bf16", index="planned_csr", layers=4),
        # Small head dimension, odd batch.
        _case("b24_d64_ragged", 24, 32, 8, 64, 16, 1, 4096),
        # Large head dimension, all query heads over one kv head.
        _case("b8_d256_mqa_8k", 8, 16, 1, 256, 16, 8192, 8192, q="bf16"),
        # Many short conversations on one GPU of a tensor-parallel group.
        _case("b512_short_one_kv_head", 512, 8, 1, 128, 16, 1, 2048),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 1e-9))))


# (query heads, kv heads, head_dim) of the configurations, the shape survey
# and the tests.
_HEADS = [(12, 2, 128), (12, 2, 128), (32, 8, 128), (32, 8, 128), (64, 8, 128), (8, 1, 128), (16, 2, 128),
          (32, 32, 128), (32, 8, 64), (16, 16, 64), (24, 8, 96), (16, 4, 32), (16, 4, 256), (16, 1, 256)]
_MOST_BYTES = 2.5e9  # of K and V in a drawn case, all layers


def draw(rng):
    """One more case: batch 1-512, 64-131072 tokens, even and ragged, every page mode, type and index."""
    hq, hkv, d = rng.choice(_HEADS)
    ps = rng.choice([16, 16, 16, 32, 64, 1, 1, 8, rng.choice([2, 3, 4, 12, 24, 48])])
    q = rng.choice(["fp16", "fp16", "bf16"])
    kv = rng.choice(["e4m3", "e4m3", "e5m2"]) if d in (64, 128, 256) and rng.random() < 0.3 else q
    index = rng.choice(["dense", "dense", "csr", "planned", "planned_csr"])
    layers = rng.choice([2, 3, 4]) if index.startswith("planned") else 1
    batch = _log_int(rng, 1, 512)
    token_bytes = 2 * hkv * d * (1 if kv in _FP8_MAX else 2) * layers
    most = int(min(131072, max(64, _MOST_BYTES / (token_bytes * batch))))
    hi = _log_int(rng, 64, most)
    lo = hi if rng.random() < 0.35 else rng.randint(1, max(1, hi // 2))
    room = hi if rng.random() < 0.6 else min(131072, hi * rng.randint(2, 8))
    return _case(None, batch, hq, hkv, d, ps, lo, hi, room, q, kv, index, layers, lens=rng.randrange(1 << 30))


def _lengths(case):
    """The lengths of the case's sequences, in no order that means anything."""
    rng = random.Random(case["lens"])
    lens = [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    lens[-1] = case["hi"]
    if case["batch"] > 1:
        lens[0] = case["lo"]
    return lens


def _pages(n, ps):
    return -(-n // ps)


def _caches(case, gen, num_pages):
    """One layer's K and V: standard normal, a few outlying keys; fp8 codes of them with per-tensor scales."""
    shape = (num_pages, case["ps"], case["hkv"], case["d"])
    dt = _TYPES[case["q"]]
    out, scales = [], []
    for which in ("k", "v"):
        x = torch.randn(shape, generator=gen, device="cuda", dtype=dt)
        if which == "k":
            rows = x.view(-1, case["hkv"], case["d"])
            hot = torch.randint(0, rows.shape[0], (max(1, rows.shape[0] // _OUTLIERS),), generator=gen, device="cuda")
            rows[hot] = rows[hot] * 8
        scale = 1.0
        if case["kv"] in _FP8_MAX:
            scale = float(x.abs().max()) / (0.875 * _FP8_MAX[case["kv"]])
            x = torch.cat([p.float().div_(scale).to(_TYPES[case["kv"]]) for p in x.split(max(1, (1 << 28) // x[0].numel()))])
        out.append(x)
        scales.append(scale)
    return out, scales


def prepare(case, seed):
    """Paged caches with scattered pages, queries, and the page index as the program holds it."""
    rng = random.Random(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lens = _lengths(case)
    rng.shuffle(lens)
    ps = case["ps"]
    pages = [_pages(n, ps) for n in lens]
    total = sum(pages)
    perm = torch.randperm(total, generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    width = max(_pages(case["room"], ps), max(pages))
    table = torch.zeros(case["batch"], width, dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        at += n
    st = {"case": dict(case), "layers": []}
    if case["index"] in ("dense", "planned"):
        st["table"] = table.cuda()
        st["lens"] = torch.tensor(lens, dtype=torch.int32).cuda()
    else:
        used = torch.arange(width).unsqueeze(0) < torch.tensor(pages).unsqueeze(1)
        st["indices"] = table[used].cuda()
        st["indptr"] = torch.tensor([0] + pages, dtype=torch.int32).cumsum(0).to(torch.int32).cuda()
        st["last"] = torch.tensor([n - (p - 1) * ps for n, p in zip(lens, pages)], dtype=torch.int32).cuda()
    for _ in range(case["layers"]):
        (k, v), (ks, vs) = _caches(case, gen, total)
        q = torch.randn(case["batch"], case["hq"], case["d"], generator=gen, device="cuda", dtype=_TYPES[case["q"]])
        st["layers"].append({"q": q, "k": k, "v": v, "ks": ks, "vs": vs})
    if case["index"].startswith("planned"):
        st["wrapper"] = pad.BatchDecodeWrapper()
    st["host"] = (lens, table)
    return st


def run(st):
    c = st["case"]
    fp8 = c["kv"] in _FP8_MAX
    if c["index"].startswith("planned"):
        w = st["wrapper"]
        geometry = dict(kv_data_type=_TYPES[c["kv"]], q_data_type=_TYPES[c["q"]])
        if c["index"] == "planned":
            w.plan_block_table(st["table"], st["lens"], c["hq"], c["hkv"], c["d"], c["ps"], **geometry)
        else:
            w.plan(st["indptr"], st["indices"], st["last"], c["hq"], c["hkv"], c["d"], c["ps"], **geometry)
        scales = (lambda y: {"k_scale": y["ks"], "v_scale": y["vs"]}) if fp8 else (lambda y: {})
        return [w.run(y["q"], (y["k"], y["v"]), **scales(y)) for y in st["layers"]]
    y = st["layers"][0]
    if c["index"] == "csr":
        scales = {"k_scale": y["ks"], "v_scale": y["vs"]} if fp8 else {}
        return pad.paged_attention_decode_csr(y["q"], y["k"], y["v"], st["indptr"], st["indices"], st["last"], **scales)
    if fp8:
        return pad.paged_attention_decode_fp8(y["q"], y["k"], y["v"], st["table"], st["lens"], y["ks"], y["vs"])
    if c["q"] == "bf16":
        return pad.paged_attention_decode_ex(y["q"], y["k"], y["v"], st["table"], st["lens"])
    return pad.paged_attention_decode(y["q"], y["k"], y["v"], st["table"], st["lens"])


def work(case):
    """K and V of every token, q, the output and the index entries in use, once each; 2 products of 2 operations."""
    lens = _lengths(case)
    tokens, b = sum(lens), case["batch"]
    kv = tokens * case["hkv"] * case["d"] * 2 * (1 if case["kv"] in _FP8_MAX else 2)
    qo = 2 * b * case["hq"] * case["d"] * 2
    index = 4 * sum(_pages(n, case["ps"]) for n in lens) + 4 * b
    if case["index"] in ("csr", "planned_csr"):
        index += 4 * (b + 1)
    return {"bytes": case["layers"] * (kv + qo) + index, "flops": case["layers"] * 4 * tokens * case["hq"] * case["d"]}


def tolerance(case):
    # Four times the 2-norm error against 64 bits (measured over the listed
    # and some drawn cases: fp16 1.6e-4 to 2.5e-4, bf16 1.2e-3 to 2.0e-3): the
    # rounding of the output and of the softmax weights to 16 bits.  A single
    # value may be off by a few of its own roundings (2^-11, 2^-8) and by
    # those of a weight that carries it: 24 roundings of a value.
    return {"rel": 1e-3, "max": 1.2e-2} if case["q"] == "fp16" else {"rel": 8e-3, "max": 9e-2}


def exact(case, seed):
    """softmax(q K^T / sqrt(d)) V in 64 bits, sequence by sequence."""
    st = prepare(case, seed)
    lens, table = st["host"]
    hq, hkv, d, ps = case["hq"], case["hkv"], case["d"], case["ps"]
    outs = []
    for y in st["layers"]:
        out = torch.zeros(case["batch"], hq, d, dtype=torch.float64, device="cuda")
        for b, n in enumerate(lens):
            ids = table[b, :_pages(n, ps)].cuda().long()

            def rows(cache, scale):
                x = cache.view(torch.uint8)[ids].view(cache.dtype) if case["kv"] in _FP8_MAX else cache[ids]
                return (x.float().double() * scale).reshape(-1, hkv, d)[:n].transpose(0, 1).contiguous()

            k, v = rows(y["k"], y["ks"]), rows(y["v"], y["vs"])
            q = y["q"][b].double().view(hkv, hq // hkv, d)
            s = (q @ k.transpose(1, 2).contiguous()) / math.sqrt(d)
            out[b] = (torch.softmax(s, dim=-1) @ v).view(hq, d)
        outs.append(out)
    return outs if case["index"].startswith("planned") else outs[0]
