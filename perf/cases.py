"""The indexer's work as its users call it, with sizes, seeded inputs, the work that cannot be
avoided, tolerances and a 64-bit restatement of the computed outputs.

Five kinds of call, each through the public ``hcu_ops`` operators:
  decode    bf16 q -> quant_q_fp8 -> mqa_logits -> top-2048 + page-table transform, one token step of
            a serving loop; captured once in a graph and replayed (as serving loops run it) or eager
  prefill   bf16 q -> quant_q_fp8 -> prefill_indexer: a prompt or a chunk of one over its cached prefix
  logits    mqa_logits_prefill: the query rows of a chunk against its whole cached prefix
  topk      sparse_mask_topk_transform of given scores and nonzero mask
  mla       dequantize_k_cache_paged: 656-B MLA slots to bf16
  kcache    store_k_cache of a chunk's new keys, then the request's keys read back from the cache
            (dequant_k_paged to bf16, or gather_k_paged to contiguous fp8 + scales)

Sizes are the repository's benchmark and test configurations and ragged ones between them.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sglang0.5.18-opt_amd"))

import hcu_ops  # noqa: E402

PAGE = 64
DIM = 128
TOPK = 2048
OTHER = 64  # pages of the cache that belong to other requests
DEV = "cuda:0"


def listed():
    return [
        # one request, one row, a short context, no graph: a single user's latency, launches included
        dict(name="decode_1x4k", kind="decode", req=1, group=1, lo=4096, hi=4096, heads=64, graph=False, blocks=False),
        # a batch of equal contexts, one row a request: steady serving
        dict(name="decode_32x16k", kind="decode", req=32, group=1, lo=16384, hi=16384, heads=64, graph=True, blocks=False),
        # speculative verify with two rows a request over ragged contexts: the quoted decode configuration
        dict(name="decode_mtp64", kind="decode", req=64, group=2, lo=2048, hi=65536, heads=64, graph=True, blocks=False),
        # deep speculative verify: six rows a request, 32 heads, long ragged contexts, block-table transform
        dict(name="decode_mtp6", kind="decode", req=8, group=6, lo=16384, hi=131072, heads=32, graph=True, blocks=True),
        # a whole prompt of an odd length with nothing cached; default page table and budget
        dict(name="prefill_prompt", kind="prefill", rows=5003, prefix=0, heads=64, keys="normal", table=False),
        # a small chunk over a medium cached prefix, as chunked prefill mixes it into decode steps
        dict(name="prefill_chunk", kind="prefill", rows=509, prefix=20480, heads=32, keys="normal", table=False),
        # an 8K chunk over a 64K cached prefix: the quoted prefill configuration
        dict(name="prefill_8k_64k", kind="prefill", rows=8192, prefix=65536, heads=64, keys="normal", table=True),
        # the long-context prefill, heavy-tailed keys
        dict(name="prefill_16k_128k", kind="prefill", rows=16384, prefix=131072, heads=64, keys="student_t4", table=True),
        # logits of a chunk's rows against its cached prefix, for a caller with its own selection
        dict(name="logits_1k_8k", kind="logits", rows=1024, width=8192, heads=64),
        # the top-k alone at the reference's production shape: few long ReLU-sum rows in a wider block
        dict(name="topk_48x128k", kind="topk", rows=48, width=131072, dist="relu_sum"),
        # MLA cache read-back of a long context, random slots
        dict(name="mla_393k", kind="mla", tokens=392832),
        # a chunk's new keys written, then the 72K-key context read back as bf16
        dict(name="kcache_74k", kind="kcache", new=8192, tokens=73728, gather=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 4 + ["logits", "topk", "mla", "kcache"])
    if kind == "decode":
        group = rng.choice([1, 1, 2, 2, 4, 6])
        heads = rng.choice([32, 64])
        hi = _log_int(rng, 3000, 131072)
        lo = rng.randint(max(1, hi // 8), hi)
        # at most the K tokens of decode_mtp64
        req = min(_log_int(rng, 1, 96), max(1, 2200000 // hi))
        return dict(kind=kind, req=req, group=group, lo=lo, hi=hi, heads=heads, graph=rng.random() < 0.75,
                    blocks=rng.random() < 0.3)
    if kind == "prefill":
        prefix = 0 if rng.random() < 0.3 else _log_int(rng, 500, 131072)
        rows = _log_int(rng, 40, 12000)
        return dict(kind=kind, rows=rows, prefix=prefix, heads=rng.choice([32, 64]),
                    keys=rng.choice(["normal", "student_t4"]), table=rng.random() < 0.5)
    if kind == "logits":
        return dict(kind=kind, rows=_log_int(rng, 30, 4096), width=_log_int(rng, 1000, 65536), heads=rng.choice([32, 64]))
    if kind == "topk":
        width = _log_int(rng, 2500, 131072) // 64 * 64
        rows = min(_log_int(rng, 1, 1024), max(1, (256 << 20) // (4 * width)))
        return dict(kind=kind, rows=rows, width=width, dist=rng.choice(["relu_sum", "relu_sum", "pos", "sparse30", "sparse2"]))
    if kind == "mla":
        return dict(kind=kind, tokens=_log_int(rng, 500, 390000))
    tokens = _log_int(rng, 1000, 400000)
    return dict(kind=kind, new=min(tokens, _log_int(rng, 1, 16384)), tokens=tokens, gather=rng.random() < 0.5)


# ------------------------------------------------------------------------------------------------
# inputs

def _keys(g, n, keys):
    x = torch.randn(n, DIM, generator=g, device=DEV)
    if keys == "student_t4":
        chi = torch.zeros_like(x)
        for _ in range(4):
            chi += torch.randn(n, DIM, generator=g, device=DEV).square_()
        x /= (chi / 4.0).sqrt_()
    return x


def _pages(g, n_pages, keys="normal"):
    """Paged K cache uint8 [n_pages, 64, 1, 132]: a page holds 64 x 128 fp8 codes, then 64 f32 scales."""
    kv = torch.empty(n_pages, PAGE * (DIM + 4), dtype=torch.uint8, device=DEV)
    for p in range(0, n_pages, 4096):
        n = min(4096, n_pages - p)
        x = _keys(g, n * PAGE, keys)
        amax = x.abs().amax(-1).clamp_(min=1e-30)
        kv[p:p + n, :PAGE * DIM] = (x * (448.0 / amax)[:, None]).to(torch.float8_e4m3fn).view(torch.uint8).view(n, -1)
        kv[p:p + n, PAGE * DIM:] = (amax / 448.0).view(torch.uint8).view(n, -1)
    return kv.view(n_pages, PAGE, 1, DIM + 4)


def _q(g, rows, heads):
    q = torch.randn(rows, heads, DIM, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(rows, heads, generator=g, device=DEV) * math.sqrt(1.0 / 8.0)
    return q, w


def _slots(bt, width):
    t = torch.arange(width, device=DEV)
    return (bt.long()[..., t // PAGE] * PAGE + t % PAGE).to(torch.int32).contiguous()


def _decode_lens(case, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(case["lo"], case["hi"] + 1, (case["req"],), generator=g)


def _decode(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    req, group = case["req"], case["group"]
    first = _decode_lens(case, seed)  # a request's rows see 0, 1, ... further tokens
    lens = (first[:, None] + torch.arange(group)).reshape(-1).to(torch.int32)
    n_pages = [(int(v) + group - 1 + PAGE - 1) // PAGE for v in first]
    cap = (case["hi"] + group - 1 + PAGE - 1) // PAGE
    perm = torch.randperm(sum(n_pages) + OTHER, generator=g, device=DEV).to(torch.int32)
    bt = torch.zeros(req, cap, dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(n_pages):
        bt[i, :n] = perm[at:at + n]
        at += n
    bt = bt.repeat_interleave(group, 0).contiguous()
    q, w = _q(g, req * group, case["heads"])
    st = dict(case=case, q=q, w=w, kv=_pages(g, sum(n_pages) + OTHER), lens=lens.to(DEV), bt=bt, width=cap * PAGE,
              cu=torch.arange(req * group + 1, dtype=torch.int32, device=DEV))
    if not case["blocks"]:
        st["pt"] = _slots(bt, cap * PAGE)
    st["full"] = case["lo"] == case["hi"] == cap * PAGE and group == 1
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _decode_step(st)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        st["step"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["step"]):
            st["out"] = _decode_step(st)
        st["step"].replay()
    return st


def _decode_step(st):
    c = st["case"]
    q8, w = hcu_ops.quant_q_fp8(st["q"], st["w"])
    logits, mask = hcu_ops.mqa_logits(q8.unsqueeze(1), st["kv"], w, st["lens"], st["bt"], st["width"], c["group"],
                                      hist_lens=st["lens"])
    if c["blocks"]:
        top = hcu_ops.sparse_mask_topk_transform_blocks(logits, mask, st["lens"], st["bt"], st["cu"])
    else:
        top = hcu_ops.sparse_mask_topk_transform(logits, mask, st["lens"], st["pt"], st["cu"])
    out = dict(mask=mask, top=top)
    if st["full"]:  # logits at and past a row's length are not written
        out["logits"] = logits
    return out


def _prefill(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    width = case["prefix"] + case["rows"]
    n_pages = (width + PAGE - 1) // PAGE
    bt = torch.randperm(n_pages + OTHER, generator=g, device=DEV)[:n_pages].to(torch.int32)
    q, w = _q(g, case["rows"], case["heads"])
    lens = (case["prefix"] + 1 + torch.arange(case["rows"], device=DEV)).to(torch.int32)
    return dict(case=case, q=q, w=w, kv=_pages(g, n_pages + OTHER, case["keys"]), bt=bt, lens=lens, width=width,
                pt=_slots(bt, width) if case["table"] else None)


def _logits(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    n_pages = (case["width"] + PAGE - 1) // PAGE
    bt = torch.randperm(n_pages + OTHER, generator=g, device=DEV)[:n_pages].to(torch.int32)
    q, w = _q(g, case["rows"], case["heads"])
    q8, w = _quant(q, w)
    return dict(case=case, q8=q8, w=w, kv=_pages(g, n_pages + OTHER), bt=bt,
                lens=torch.full((case["rows"],), case["width"], dtype=torch.int32, device=DEV))


def _topk(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rows, width, dist = case["rows"], case["width"], case["dist"]
    x = torch.empty(rows, width, device=DEV)
    c = torch.rand(8, generator=g, device=DEV) - 0.3
    for r in range(0, rows, 16):
        n = min(16, rows - r)
        if dist == "relu_sum":
            x[r:r + n] = (torch.relu(torch.randn(n, width, 8, generator=g, device=DEV)) * c).sum(-1)
            continue
        u = torch.rand(n, width, generator=g, device=DEV) * 10
        keep = {"pos": 1.0, "sparse30": 0.3, "sparse2": min(1.0, 1500.0 / width)}[dist]
        x[r:r + n] = torch.where(torch.rand(n, width, generator=g, device=DEV) <= keep, u, torch.zeros_like(u))
    bits = ((x != 0).view(rows, -1, 16).to(torch.int32) << torch.arange(16, device=DEV, dtype=torch.int32)).sum(-1)
    mask = torch.where(bits > 32767, bits - 65536, bits).to(torch.int16).contiguous()
    lens = (width - torch.arange(rows, device=DEV) * 37 % (width // 4) - 3).to(torch.int32)
    pt = torch.stack([torch.randperm(width, generator=g, device=DEV) for _ in range(min(rows, 8))]).to(torch.int32)
    pt = pt[torch.arange(rows, device=DEV) % pt.shape[0]].contiguous()
    return dict(case=case, x=x, mask=mask, lens=lens, pt=pt, cu=torch.arange(rows + 1, dtype=torch.int32, device=DEV))


def _mla(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    pool = 1 << 19
    codes = torch.randint(0, 254, (pool, 512), generator=g, device=DEV, dtype=torch.int32)
    cache = torch.empty(pool, 656, dtype=torch.uint8, device=DEV)
    cache[:, :512] = (codes + (codes >= 0x7F).int()).to(torch.uint8)  # no NaN codes
    scale = torch.rand(pool, 4, generator=g, device=DEV) * 0.01 + 1e-3
    cache[:, 512:528] = scale.view(torch.uint8)
    cache[:, 528:] = torch.randn(pool, 64, generator=g, device=DEV).to(torch.bfloat16).view(torch.uint8)
    slots = torch.randint(0, pool, (case["tokens"],), generator=g, device=DEV, dtype=torch.int32)
    return dict(case=case, cache=cache.view(pool, 1, 656), slots=slots)


def _kcache(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    n_pages = (case["tokens"] + PAGE - 1) // PAGE
    bt = torch.randperm(n_pages + OTHER, generator=g, device=DEV)[:n_pages].to(torch.int32)
    slots = _slots(bt, case["tokens"])
    return dict(case=case, kv=_pages(g, n_pages + OTHER), slots=slots, new_slots=slots[case["tokens"] - case["new"]:].contiguous(),
                k=torch.randn(case["new"], DIM, generator=g, device=DEV).to(torch.bfloat16))


def prepare(case, seed):
    return {"decode": _decode, "prefill": _prefill, "logits": _logits, "topk": _topk, "mla": _mla,
            "kcache": _kcache}[case["kind"]](case, seed)


# ------------------------------------------------------------------------------------------------
# one pass

def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "decode":
        if not c["graph"]:
            return _decode_step(st)
        st["step"].replay()
        return st["out"]
    if kind == "prefill":
        q8, w = hcu_ops.quant_q_fp8(st["q"], st["w"])
        return hcu_ops.prefill_indexer(q8, w, st["kv"], st["bt"], st["lens"], st["width"], st["pt"])
    if kind == "logits":
        return hcu_ops.mqa_logits_prefill(st["q8"], st["w"], st["kv"], st["bt"], st["lens"], c["width"])
    if kind == "topk":
        return hcu_ops.sparse_mask_topk_transform(st["x"], st["mask"], st["lens"], st["pt"], st["cu"])
    if kind == "mla":
        return hcu_ops.dequantize_k_cache_paged(st["cache"], st["slots"])
    hcu_ops.store_k_cache(st["k"], st["new_slots"], st["kv"])
    read = hcu_ops.gather_k_paged if c["gather"] else hcu_ops.dequant_k_paged
    out = read(st["kv"], st["slots"])
    return dict(kv=st["kv"], out=list(out) if c["gather"] else out)


# ------------------------------------------------------------------------------------------------
# work, tolerance, 64-bit results

def work(case):
    kind = case["kind"]
    if kind == "decode":
        # the middle of the drawn lengths; K once a request, logits written and read back, mask likewise
        rows, mean = case["req"] * case["group"], (case["lo"] + case["hi"]) / 2
        keys = rows * mean
        h = case["heads"]
        b = (case["req"] * mean * (DIM + 4 + 4 / PAGE) + rows * h * (DIM * 2 + 4) + 2 * keys * 4 + 2 * keys / 8
             + rows * TOPK * 8)
        return dict(bytes=b, flops=2 * h * DIM * keys)
    if kind == "prefill":
        r, p, h = case["rows"], case["prefix"], case["heads"]
        first = min(r, max(0, TOPK - p))  # rows of at most 2048 keys select all of them
        keys = (r - first) * (p + (first + 1 + r) / 2)
        return dict(bytes=(p + r) * (DIM + 4 + 4) + r * (h * (DIM * 2 + 4) + TOPK * 4 + 4), flops=2 * h * DIM * keys)
    if kind == "logits":
        r, n, h = case["rows"], case["width"], case["heads"]
        return dict(bytes=n * (DIM + 4) + r * h * (DIM + 4) + r * n * 4, flops=2 * h * DIM * r * n)
    if kind == "topk":
        r, n = case["rows"], case["width"]
        keep = {"sparse30": 0.3, "sparse2": min(1.0, 1500.0 / n)}.get(case["dist"], 1.0)
        return dict(bytes=r * (n * 4 * keep + n / 8 + TOPK * 8), flops=0)
    if kind == "mla":
        return dict(bytes=case["tokens"] * (4 + 656 + 576 * 2), flops=0)
    n, m = case["tokens"], case["new"]
    return dict(bytes=m * (4 + DIM * 2 + DIM + 4) + n * (4 + DIM + 4 + (DIM + 4 if case["gather"] else DIM * 2)), flops=0)


def tolerance(case):
    # The fp8 matrix products are not fp32 sums: an instruction's 128 products are off by up to 5e-5 of
    # their summed magnitudes, and another order of the same sum by as much (1.4e-5 measured against
    # the 64-bit logits).  The selections turn such a difference into other tokens near the
    # threshold.  Everything else is exact.
    if case["kind"] in ("decode", "logits"):
        return {"rel": 6e-5, "max": 2e-3, "differ": 0.01}
    if case["kind"] == "prefill":
        return {"rel": 0.0, "differ": 0.01}
    return "exact"


def _quant(q, w):
    """fp8 codes amax / 448 per (row, head) and the scale folded into the weight, in f32 as the format has it."""
    codes, scale = _codes(q)
    return codes, w * scale


def _codes(x):
    x = x.float()
    amax = x.abs().amax(-1)
    top = torch.full_like(amax, 448.0)  # a tensor: with a plain number torch multiplies by a reciprocal
    inv = torch.where(amax == 0, torch.zeros_like(amax), top / amax)
    return (x * inv[..., None]).to(torch.float8_e4m3fn), amax / top


def _k64(kv, bt):
    """The keys of a block table's pages, f64 [tokens, 128] and their scales."""
    p = kv.view(kv.shape[0], -1)[bt.long()]
    k = p[:, :PAGE * DIM].contiguous().view(torch.float8_e4m3fn).double().view(-1, DIM)
    return k, p[:, PAGE * DIM:].contiguous().view(torch.float32).double().view(-1)


def _scores64(q8, w, k, s):
    """f64 logits [rows, tokens]: scale * sum over heads of w * relu(q . k)."""
    rows, heads = w.shape
    out = torch.empty(rows, k.shape[0], dtype=torch.float64, device=DEV)
    kt = k.t().contiguous()
    for r in range(rows):
        dots = torch.relu_(q8[r].double() @ kt)
        out[r] = (w[r].double()[None, :] @ dots)[0] * s
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        st = _decode(dict(case, graph=False), seed)
        if not st["full"]:
            return None
        q8, w = _quant(st["q"], st["w"])
        rows = []
        for i in range(case["req"]):
            k, s = _k64(st["kv"], st["bt"][i])
            rows.append(_scores64(q8[i:i + 1], w[i:i + 1], k, s))
        return dict(mask=None, top=None, logits=torch.cat(rows))
    if kind == "logits":
        if case["rows"] * case["width"] * case["heads"] > 2 << 30:
            return None
        st = _logits(case, seed)
        k, s = _k64(st["kv"], st["bt"])
        return _scores64(st["q8"], st["w"], k[:case["width"]], s[:case["width"]])
    if kind == "mla":
        st = _mla(case, seed)
        c = st["cache"].view(-1, 656)[st["slots"].long()]
        out = torch.empty(case["tokens"], 1, 576, dtype=torch.float64, device=DEV)
        for i in range(0, case["tokens"], 65536):
            x = c[i:i + 65536]
            v = x[:, :512].contiguous().view(torch.float8_e4m3fn).double().view(-1, 4, DIM)
            s = x[:, 512:528].contiguous().view(torch.float32).double()
            out[i:i + 65536, 0, :512] = (v * s[:, :, None]).view(-1, 512)
            out[i:i + 65536, 0, 512:] = x[:, 528:].contiguous().view(torch.bfloat16).double()
        return out
    if kind == "kcache" and not case["gather"]:
        st = _kcache(case, seed)
        codes, scale = _codes(st["k"])
        flat = st["kv"].view(st["kv"].shape[0], -1)
        page, off = (st["new_slots"] // PAGE).long(), (st["new_slots"] % PAGE).long()
        d = torch.arange(DIM, device=DEV)
        flat[page[:, None], off[:, None] * DIM + d] = codes.view(torch.uint8)
        flat[page[:, None], PAGE * DIM + off[:, None] * 4 + d[:4]] = scale.view(torch.uint8).view(-1, 4)
        k, s = _k64(st["kv"], torch.arange(flat.shape[0], device=DEV))
        slots = st["slots"].long()
        return dict(kv=None, out=k[slots] * s[slots][:, None])
    return None
