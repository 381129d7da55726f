"""Decode workloads of seoulkv_amd: what they are, how they are made, and
their 64-bit answers in plain torch.

Three kinds of work, each through a public entry point:

``step``     one sparse decode step of a prefilled layer,
             ``SeoulKV4.run(q)`` with a host query, the call a decoder makes
             once per layer and token; contiguous records, or records in the
             pages of a ``KVPagePool`` (``page_tokens`` > 0).
``dense``    one dense FP8 decode over every key of caller-owned records,
             ``dense_decode_static``: what short contexts, and callers that
             may not allocate, run instead of the sparse step.
``session``  the life of one sequence's layer: instance from K, V and an
             index (uploads, key codec, FP8 records, first checked step),
             then ``tokens`` times append one token, run, read the output
             back; close.

Keys are what a RoPE attention layer holds: per KV head a mixture of
``components`` directions with spread 0.3 (0: i.i.d. directions), rotated to
their positions; queries are noisy retrieval-zone keys rotated to the
decoding position.  Everything is made on the GPU from the seed.  The
instances of a program share one stream, as the layers of a decoder do:
each step follows the one before it.
"""

import functools
import math

import torch

from seoulkv_amd import KVPagePool, SeoulKV4, SeoulKV4Config, SeoulKV4Index
from seoulkv_amd._hip import dense_decode_static

KV_HEADS, HEADS, DIM, TOPK = 4, 4, 256, 100  # heads: query heads per KV head
THETA = 1e6
DEVICE = "cuda:0"


@functools.cache
def _stream():
    return torch.cuda.Stream(DEVICE)


def _step(name, context, components, n_centroids, nprobe, sink=128, local=256, capacity=0,
          page_tokens=0):
    """capacity: pool capacity per KV head (0: sized for the worst case);
    n_centroids 0: the index builder's default, about T / 4."""
    return {"name": name, "kind": "step", "context": context, "components": components,
            "n_centroids": n_centroids, "nprobe": nprobe, "sink": sink, "local": local,
            "capacity": capacity, "page_tokens": page_tokens}


def _dense(name, context, components, spare=0):
    return {"name": name, "kind": "dense", "context": context, "components": components,
            "spare": spare}


def listed():
    return [
        # the shortest context worth an index: launches and latency only
        _step("step_8k", 8192, 256, 512, 64),
        # a chat-length context
        _step("step_32k", 32768, 1024, 2048, 384),
        # no power of two anywhere: ragged tiles, a long local window
        _step("step_50k_ragged", 50020, 1500, 3104, 304, sink=37, local=601),
        # the headline: a long document
        _step("step_128k", 131072, 4096, 8192, 384),
        # the same through a serving engine's page table
        _step("step_128k_paged", 131072, 4096, 8192, 384, page_tokens=256),
        # the index builder's and the configuration's defaults (32672
        # centroids per KV head, small pools)
        _step("step_128k_default_index", 131072, 4096, 0, 256, capacity=13056),
        # a whole repository or book in context
        _step("step_512k", 524288, 16384, 32768, 512),
        # dense: a short prompt
        _dense("dense_1k", 1000, 64),
        # dense: an odd context in a larger record buffer
        _dense("dense_40k_ragged", 40009, 1024, spare=503),
        # dense: the headline context
        _dense("dense_128k", 131072, 4096),
        # dense: the longest context
        _dense("dense_1m", 1048576, 4096),
        # prefill of one layer, then a short reply
        {"name": "session_32k", "kind": "session", "context": 32768, "components": 1024,
         "n_centroids": 2048, "nprobe": 384, "sink": 128, "local": 256, "capacity": 0,
         "page_tokens": 0, "tokens": 16},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _draw_step(rng, lo, hi):
    """A sparse shape: contexts are multiples of 4 (the index takes no other)."""
    context = 4 * int(_log_uniform(rng, lo, hi) / 4)
    sink, local = rng.randrange(0, 257), rng.randrange(16, 1025)
    retrieval = context - sink - local
    while True:
        nc = 32 * max(3, round(context / rng.choice([16, 8, 4]) * rng.uniform(0.8, 1.2) / 32))
        # probes: multiples of 16, enough that every pool passes the 2048-key minimum
        low = math.ceil(4800 / (2 * retrieval / nc) / 16)
        high = min(512, nc) // 16
        if low <= high and nc <= 65536:
            break
    return {"context": context, "components": rng.choice([0, context // 32, context // 32]),
            "n_centroids": nc, "nprobe": 16 * rng.randint(max(low, high // 4), high),
            "sink": sink, "local": local, "capacity": 0,
            "page_tokens": rng.choice([0, 0, 64, 256, 1024])}


def draw(rng):
    kind = rng.choices(["step", "dense", "session"], [6, 3, 1])[0]
    if kind == "dense":
        context = int(_log_uniform(rng, 200, 800000))
        return {"kind": kind, "context": context, "components": max(1, min(4096, context // 32)),
                "spare": rng.choice([0, rng.randrange(1, 600)])}
    if kind == "session":
        return dict(_draw_step(rng, 8192, 30000), kind=kind, tokens=rng.randrange(4, 16))
    return dict(_draw_step(rng, 8192, 300000), kind=kind)


# ------------------------------------------------------------------- inputs
def _generator(seed, stream):
    return torch.Generator(DEVICE).manual_seed(1_000_003 * (seed + 1) + stream)


def _rope(x, positions):
    """Rotate-half RoPE of rows x [N, 256] at positions [N]."""
    half = DIM // 2
    inv = THETA ** (-torch.arange(half, dtype=torch.float64, device=x.device) * 2 / DIM)
    angle = positions.to(torch.float64)[:, None] * inv
    cos, sin = torch.cos(angle).float(), torch.sin(angle).float()
    a, b = x[:, :half], x[:, half:]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEVICE)


def _cache(context, components, sink, local, seed, queries=1):
    """K, V [4, context, 256] and queries [queries, 16, 256], BF16 on the GPU;
    the context's last ``queries - 1`` tokens decode queries 1.. (query i sits
    at position context - (queries - 1) + i)."""
    gen = _generator(seed, 0)
    positions = torch.arange(context, device=DEVICE)
    k = torch.empty(KV_HEADS, context, DIM, dtype=torch.bfloat16, device=DEVICE)
    v = torch.empty_like(k)
    q = torch.empty(queries, KV_HEADS, HEADS, DIM, dtype=torch.bfloat16, device=DEVICE)
    first = context - (queries - 1)
    for g in range(KV_HEADS):
        pre = _randn(gen, context, DIM)
        if components:
            centres = _randn(gen, components, DIM)
            pick = torch.randint(components, (context,), generator=gen, device=DEVICE)
            pre = centres[pick] + 0.3 * pre
        k[g] = _rope(pre, positions)
        v[g] = _randn(gen, context, DIM)
        at = torch.randint(sink, first - local, (queries, HEADS), generator=gen, device=DEVICE)
        noisy = pre[at.reshape(-1)] + 0.5 * _randn(gen, queries * HEADS, DIM)
        where = first + torch.arange(queries, device=DEVICE).repeat_interleave(HEADS)
        q[:, g] = _rope(noisy, where).reshape(queries, HEADS, DIM).bfloat16()
    return k, v, q.reshape(queries, KV_HEADS * HEADS, DIM)


def _records(k, v):
    """FP8 e4m3 [V || K] records, uint8 [.., 512]."""
    return torch.cat((v.to(torch.float8_e4m3fn).view(torch.uint8),
                      k.to(torch.float8_e4m3fn).view(torch.uint8)), dim=-1)


def _index(case, k_cpu):
    return SeoulKV4Index.build(k_cpu, sink=case["sink"], local=case["local"],
                               nprobe=case["nprobe"], build_device=DEVICE,
                               n_centroids=case["n_centroids"] or None)


def _dense_inputs(case, seed):
    context = case["context"]
    k, v, q = _cache(context, case["components"], 0, 0, seed)
    rows = context + case["spare"]
    kv8 = torch.full((KV_HEADS, rows, 2 * DIM), 0x7f, dtype=torch.uint8, device=DEVICE)
    for g in range(KV_HEADS):  # rows past the context hold NaN records
        kv8[g, :context] = _records(k[g], v[g])
    return kv8, q[0].contiguous()


def _instance(case, k, v, index, append=0):
    pool = None
    if case["page_tokens"]:
        tokens = case["page_tokens"]
        pool = KVPagePool(-(-(case["context"] + append) // tokens) + 3, page_tokens=tokens,
                          device=DEVICE)
        # a pool in use: its free pages come in no order
        pages = pool.allocate(pool.n_pages)
        pool.release(pages[1::2] + pages[::2])
    config = SeoulKV4Config(stage15_capacity=case["capacity"] or None, append_capacity=append)
    return SeoulKV4(device=DEVICE, k=k, v=v, index=index, config=config, kv_pool=pool)


def prepare(case, seed):
    if case["kind"] == "dense":
        kv8, q = _dense_inputs(case, seed)
        return {"case": case, "kv8": kv8, "q": q, "out": torch.empty_like(q)}
    tokens = case.get("tokens", 0)
    k, v, q = _cache(case["context"] + tokens, case["components"], case["sink"], case["local"],
                     seed, tokens + 1)
    k, v = k.cpu(), v.cpu()
    queries = [x.reshape(1, 1, KV_HEADS * HEADS, DIM) for x in q.cpu()]
    prompt = [x[:, :case["context"]].contiguous() for x in (k, v)] if tokens else [k, v]
    index = _index(case, prompt[0])
    if case["kind"] == "session":
        new = [tuple(x[:, case["context"] + i:][:, :1].contiguous() for x in (k, v))
               for i in range(tokens)]
        return {"case": case, "k": prompt[0], "v": prompt[1], "index": index, "new": new,
                "queries": queries}
    with torch.cuda.stream(_stream()):  # the instance keeps its caller's stream
        attn = _instance(case, *prompt, index)
        first = attn.run(queries[0])
    attn.synchronize()
    # the output buffer that every step writes
    return {"case": case, "attn": attn, "q": queries[0], "out": first.device_tensors}


# ---------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    if case["kind"] == "dense":
        dense_decode_static(state["kv8"], case["context"], state["q"], state["out"])
        return state["out"]
    if case["kind"] == "step":
        state["attn"].run(state["q"])
        return state["out"]
    with torch.cuda.stream(_stream()), \
            _instance(case, state["k"], state["v"], state["index"], append=case["tokens"]) as attn:
        outs = [attn.run(state["queries"][0]).to_torch()]
        for (k, v), q in zip(state["new"], state["queries"][1:]):
            attn.append(k, v)
            outs.append(attn.run(q).to_torch())
    return outs


# --------------------------------------------------------------------- work
def _step_work(case):
    """Bytes and flops one step cannot do without: every centroid's two 2-bit
    planes and factors, the posting lists and prefix rows of the clusters
    that four heads' probes cover (about 3.5 probes' worth, half of their
    postings shared between two clusters), the 256-byte records of the
    union of four top-1600, and the attended FP8 records."""
    retrieval = case["context"] - case["sink"] - case["local"]
    nc = case["n_centroids"] or 32 * math.ceil(retrieval / 128)
    lists = min(nc, 3.5 * case["nprobe"])
    postings = 2 * retrieval * lists / nc
    pool = min(retrieval, 0.88 * postings)
    union = min(pool, HEADS * 1600 * 0.94)
    attended = case["sink"] + case["local"]
    by = KV_HEADS * (nc * 134 + lists * 8 + postings * 8 + pool * 64 + union * 256
                     + attended * 512 + HEADS * TOPK * 512) + 4 * HEADS * KV_HEADS * DIM
    fl = KV_HEADS * HEADS * 2 * DIM * (2 * nc + pool + 2 * union + 2 * (attended + TOPK))
    return by, fl


def work(case):
    context = case["context"]
    if case["kind"] == "dense":
        return {"bytes": KV_HEADS * context * 512 + 4 * KV_HEADS * HEADS * DIM,
                "flops": 4 * KV_HEADS * HEADS * DIM * context}
    by, fl = _step_work(case)
    if case["kind"] == "session":  # K and V once, key and FP8 records written, the steps
        steps = case["tokens"] + 1
        by = KV_HEADS * context * (4 * DIM + DIM + 2 * DIM) + steps * by
        fl = steps * fl
    return {"bytes": by, "flops": fl}


def tolerance(case):
    # BF16 outputs of exactly selected FP8 records: the outputs are about
    # 1.7e-3 off the 64-bit values by their own rounding, one BF16 step
    # (2^-7 of a value) at most where two correct sums round apart
    return {"rel": 7e-3, "max": 2e-2}


# -------------------------------------------------------- the 64-bit answers
def _fixed(x):
    """BF16 rows x [N, 256] as integers X and scales 2^fx with X 2^fx = x,
    elements more than 14 binades below their row's largest truncated."""
    x = x.double()
    _, e = torch.frexp(x)
    fx = torch.where(x != 0, e, -(1 << 20)).amax(-1, keepdim=True) - 8 - 14
    return torch.trunc(torch.ldexp(x, -fx)), fx


def _centred(x, codes, centre, up):
    """bf16(f32(sum x (2 code - centre) 2^up)), the sum exact: [heads, N]."""
    ints, fx = _fixed(x)
    dot = 2 * (ints @ codes.double().T) - centre * ints.sum(-1, keepdim=True)
    return torch.ldexp(dot, fx + up).float()


def _ordered(x):
    """BF16 values as integers of the same order."""
    b = x.bfloat16().view(torch.int16).long() & 0xffff
    return torch.where(b >= 0x8000, 0xffff - b, b + 0x8000)


def _best(order, ids, k):
    """Per head the members [heads, N] with the k largest (order, -id)."""
    keys = torch.where(order >= 0, (order << 20) + (0xfffff - ids), -1)
    top = keys.topk(min(k, keys.shape[1]), dim=-1)
    member = torch.zeros_like(keys, dtype=torch.bool).scatter_(1, top.indices, True)
    return member & (keys >= 0), top.indices


def _two_bit(packed):
    p = packed.to(DEVICE)[..., None]
    shift = torch.tensor([0, 2, 4, 6], device=DEVICE, dtype=torch.uint8)
    return ((p >> shift) & 3).reshape(*packed.shape[:-1], -1)


def _selected(cell, k, q):
    """Token IDs [4, 100] that one KV head's query heads q [4, 256] attend
    beside the windows, from its index cell and prefill keys k."""
    upper, lower = _two_bit(cell["upper"]), _two_bit(cell["lower"])
    nc = len(upper)
    cid = torch.arange(nc, device=DEVICE)
    # interval scores, the probe budget's threshold, the best fine scores
    value = _centred(q, upper, 3, 0) * (cell["scale"].float().to(DEVICE) / 4)
    ints, fx = _fixed(q)
    norm = torch.ldexp(ints.square().sum(-1, keepdim=True).sqrt(), fx).float()
    norm = norm * torch.tensor(float(cell["lam"]), dtype=torch.float32, device=DEVICE)
    margin = norm * cell["coarse_residual_norm"].to(DEVICE).half().bfloat16().float()
    low, high = _ordered(value - margin), _ordered(value + margin)
    p = int(cell["p"])
    eligible = high >= low.topk(p, dim=-1).values[:, -1:]
    scale = cell["group_fine_scale"].to(DEVICE).half().float().repeat_interleave(32)[:nc]
    fine = _ordered(_centred(q, 4 * upper + lower, 15, 0) * scale)
    member, _ = _best(torch.where(eligible, fine, -1), cid, p)
    lists = member.any(0).nonzero()[:, 0]
    # their postings, each token at its first occurrence
    off = cell["offsets"].to(DEVICE).long()
    size = off[lists + 1] - off[lists]
    at = torch.arange(int(size.sum()), device=DEVICE)
    at = at - (size.cumsum(0) - size).repeat_interleave(size) + off[lists].repeat_interleave(size)
    tokens = cell["values"].to(DEVICE).long()[at]
    place = torch.arange(len(tokens), device=DEVICE)
    first = torch.full((len(k),), len(tokens), device=DEVICE)
    first.scatter_reduce_(0, tokens, place, "amin")
    pool = tokens[first[tokens] == place]
    # 2-, 4- and 8-bit key codes
    s = k.abs().amax(0).float().clamp_min(1e-9)
    code = torch.floor((k[pool].float() + s) / (2 * s / 256)).clamp(0, 255)
    q15, qs = ((q.float() * s / w).bfloat16() for w in (64, 256))
    keep = _best(_ordered(_centred(q15, torch.floor(code / 64), 3, 4)), pool, 1600)[0].any(0)
    pool, code = pool[keep], code[keep]
    keep = _best(_ordered(_centred(qs, torch.floor(code / 16), 15, 4)), pool, 256)[0].any(0)
    pool, code = pool[keep], code[keep]
    return pool[_best(_ordered(_centred(qs, code, 255, 0)), pool, TOPK)[1]]


def _attend(q, k8, v8):
    """softmax(q k / 16) v in 64 bits; q [.., 256], k8, v8 [.., N, 256]."""
    logits = (k8.double() @ q.double()[..., None])[..., 0] / 16
    return (torch.softmax(logits, -1)[..., None, :] @ v8.double())[..., 0, :]


def _dense_exact(case, seed):
    kv8, q = _dense_inputs(case, seed)
    out = []
    for g in range(KV_HEADS):
        x = q[HEADS * g:HEADS * (g + 1)].double()
        m = torch.full((HEADS, 1), -math.inf, dtype=torch.float64, device=DEVICE)
        total, acc = torch.zeros_like(m), torch.zeros_like(x)
        for rows in kv8[g, :case["context"]].split(1 << 17):
            both = rows.view(torch.float8_e4m3fn).double()
            logits = x @ both[:, DIM:].T.contiguous() / 16
            new = torch.maximum(m, logits.amax(-1, keepdim=True))
            p = torch.exp(logits - new)
            total = total * torch.exp(m - new) + p.sum(-1, keepdim=True)
            acc = acc * torch.exp(m - new) + p @ both[:, :DIM].contiguous()
            m = new
        out.append(acc / total)
    return torch.cat(out)


def exact(case, seed):
    """64-bit values of run()'s outputs.  The selection is defined by exact
    integer dots rounded as the scores are, so it is computed, not copied;
    the posting lists and centroid codes are those of the index, which is
    the step's input."""
    if case["kind"] == "dense":
        return _dense_exact(case, seed)
    tokens, context = case.get("tokens", 0), case["context"]
    k, v, q = _cache(context + tokens, case["components"], case["sink"], case["local"], seed,
                     tokens + 1)
    cells = _index(case, k[:, :context].contiguous().cpu()).cells
    k8, v8 = k.to(torch.float8_e4m3fn), v.to(torch.float8_e4m3fn)
    out = torch.empty(tokens + 1, KV_HEADS, HEADS, DIM, dtype=torch.float64, device=DEVICE)
    for i in range(tokens + 1):
        window = torch.cat((torch.arange(case["sink"], device=DEVICE),
                            torch.arange(context - case["local"], context + i, device=DEVICE)))
        for g in range(KV_HEADS):
            x = q[i, HEADS * g:HEADS * (g + 1)]
            ids = _selected(cells[g], k[g, :context], x)
            ids = torch.cat((window.expand(HEADS, -1), ids), -1)
            kk, vv = (t[g].view(torch.uint8)[ids].view(torch.float8_e4m3fn) for t in (k8, v8))
            out[i, g] = _attend(x, kk, vv)
    if case["kind"] == "session":
        return [o.reshape(1, 1, KV_HEADS * HEADS, DIM) for o in out]
    tiles = torch.zeros(KV_HEADS, 1, 32, HEADS, DIM, dtype=torch.float64, device=DEVICE)
    for h in range(HEADS):
        tiles[:, 0, h, h] = out[0, :, h]
    return tuple(tiles)
