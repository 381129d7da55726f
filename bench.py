#!/usr/bin/env python3
"""SeoulKV4 sparse decode step on one MI355X at T = 128K.

One "step" is one ``SeoulKV4.run`` decode step (all 16 query heads of the 4 KV
heads of one layer) with the query already resident on the device.  Prints one
JSON line: µs per layer-step (device time, HIP events), the roofline of the
dominant kernel, the step's algorithmic HBM bytes and GB/s, whether the
top-100 IDs match the CPU oracle bit for bit, the oracle's own CPU time on a
bounded sample of the same workload, and the dense FP8 decode over all T keys
on the same GPU (the sparse step's comparison).

    python bench.py [--steps K] [--warmup W] [--config cfg2] [--no-cpu-baseline]
"""

from __future__ import annotations

import argparse
import json
import os
import random
import statistics
import sys
import time

import numpy as np
import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

from seoulkv_amd import KVPagePool, SeoulKV4, SeoulKV4Config, SeoulKV4Index  # noqa: E402
from seoulkv_amd.index import (  # noqa: E402
    build_cell,
    centroid_count,
    list_agreement,
    posting_cosine,
)
from seoulkv_amd.synthetic import PROFILES, make_profile  # noqa: E402

HBM_PEAK_GBS = 8000.0
G_KV = 4  # KV heads of the layer
APPEND_BULK = 64  # tokens of the bulk host and device appends after the measured steps
APPEND_BULK_REPS = 3  # bulk appends of each kind (median reported)
N_COLD = 10  # independent instances the cold-cache steps rotate over
PAGE_TOKENS = 256  # tokens per page of the paged-records measurement
METRIC = "µs/layer decode step at T=128K (1 GPU); achieved HBM GB/s; top-100 ID match"


def log(msg: str) -> None:
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def kernel_bytes(status: dict, p, nc: int) -> dict:
    """Algorithmic HBM bytes of each kernel for one step (all 4 KV groups),
    from the live stage sizes.  Reads of each input once plus the outputs the
    next stage needs.  Member bitmaps are (n + 63) / 64 words of 8 B per
    (group, head) over a group's n items."""
    G, H = 4, 4
    sel = sum(status["selected"])
    scanned = sum(status["scanned"])
    pool = sum(status["pool"])
    u1 = sum(status["u1"])
    bm_pool = H * sum((n + 63) // 64 * 8 for n in status["pool"])  # top-1600 members
    bm_u1 = H * sum((n + 63) // 64 * 8 for n in status["u1"])      # top-256 members
    return {
        # Q + key scales in (per block, from L2); both centroid planes, scale,
        # residual norm in; lower/upper bounds and fine scores out; three
        # query operand blocks out
        "front": G * nc * (128 + 4 + H * 6) + G * (nc // 32) * 8 + 16 * 256 * 2
        + 3 * G * 8400,
        # lower, upper and fine scores in (per head); selected bitmap out; the
        # extra blocks' sink/local FP8 [V||K] records (once per group) in and
        # their slice partials out
        "select": G * H * nc * 6 + G * nc // 8 + G * (p.sink + p.local) * 512
        + 16 * ((p.sink + p.local + 255) // 256) * 258 * 4,
        # upper bounds in, survivor masks out; CSR bounds of the selected
        # lists, mate and token of each of their postings in; pool tokens
        # out; the 64 B prefix row of each pool key in, its 2-bit scores and
        # the 16-key tile maxima out
        "pool": G * nc * (H * 2 + 1) + sel * 8 + scanned * (4 + 4) + pool * 4
        + pool * (64 + H * 2) + H * pool // 16 * 2,
        # pool scores in; member bitmaps out
        "top1600": pool * H * 2 + bm_pool,
        # member bitmaps + pool tokens in; U1 tokens, their full 256 B key
        # records in; U1 tokens, 4-bit and 8-bit scores out
        "union_score": bm_pool + u1 * (4 + 4 + 256 + H * 4),
        "top256": u1 * (4 + H * 2) + bm_u1,
        # per head: U1 8-bit scores and tokens, the 4 heads' top-256 bitmaps
        # in, top-100 IDs out; the 100 FP8 [V||K] records of each head, the
        # sink/local slice partials in; BF16 output out
        "top100_sdpa": H * u1 * (4 + 2) + H * bm_u1 + 16 * 100 * 4 + 16 * 100 * 512
        + 16 * ((p.sink + p.local + 255) // 256) * 258 * 4 + 16 * 256 * 2,
    }


def kv_gather_bytes(top_ids, p) -> tuple[int, int]:
    """FP8 [V || K] record bytes the sparse SDPA gathers in one step, as
    (sink/local, top-100): each KV group's sink and local records once (read
    for its 4 query heads) and the distinct top-100 tokens of its heads (a
    token chosen by several heads of a group is one record)."""
    rec = 512
    top = 0
    for g in range(4):
        ids = np.unique(np.asarray(top_ids[g]).ravel())
        top += int((ids >= 0).sum()) * rec
    return 4 * (p.sink + p.local) * rec, top


# The gather's latency bound: an 8 KB read of records nobody touched recently
# takes one CU 0.64 us from issue to arrival (MI355X, device clock), so the
# top-100 part (~51 KB per query-head block, 16 blocks) cannot beat ~1 TB/s
# however it is spread: ~16 % of the HBM peak for ~0.8 MB.
GATHER_LATENCY_CAP_FRAC = 0.16


def gather_phases(k, v, index, q, steps: int):
    """Record-gather phases of the sparse SDPA from the trace build of the
    library (same kernels plus per-block device timestamps), or None when it
    was not built.  Per step: the top-100 gather (k_top100 blocks: record
    loads issued -> the last wave's records arrived) and the sink/local
    gather (the attention-slice blocks of k_select, the same two points);
    `window` = first issue to last arrival over the blocks of the part,
    `per_block` = the blocks' mean issue -> arrival; medians over steps."""
    from seoulkv_amd import _hip

    lib = _hip.load_trace_library()
    if lib is None:
        return None
    zones = index.zones
    slices = -(-(zones.sink + zones.local) // 256)
    rt = _hip.Runtime(0, k, v, index, pool_min=0, pool_capacity=None, debug=False, lib=lib)
    try:
        rt.bind_query(q)
        for _ in range(20):
            rt.enqueue()
        rt.synchronize()
        parts = {"top100": [], "sink_local": []}
        for _ in range(steps):
            rt.enqueue()
            rt.synchronize()
            bl = rt.trace_blocks().astype(np.int64)
            for name, rows in (("top100", bl[9][:16]), ("sink_local", bl[5][16:16 + 16 * slices])):
                issue, arrive = rows[:, 1], rows[:, 2]
                parts[name].append(((arrive.max() - issue.min()) * 0.01,
                                    float(np.mean(arrive - issue)) * 0.01))
    finally:
        rt.close()
    return {name: {"window_us": round(statistics.median(w for w, _ in vals), 3),
                   "per_block_us": round(statistics.median(b for _, b in vals), 3),
                   "steps": len(vals)}
            for name, vals in parts.items()}


def cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(index, k, v, q, top_gpu, budget_s: float):
    """Time the oracle (numpy restatement of the step) on this host; also
    check the GPU's top-100 against it.  Prefill work is not timed."""
    from threadpoolctl import threadpool_info

    from oracle import decode as od

    kb = k.view(torch.int16).numpy().view(np.uint16)
    vb = v.view(torch.int16).numpy().view(np.uint16)
    t0 = time.time()
    code8, scales = od.key_codec(kb)
    k8, v8 = od.fp8_records(kb, vb)
    cells = [od.GroupCell.from_cell(c) for c in index.cells]
    log(f"oracle prefill {time.time() - t0:.1f}s (untimed)")
    qb = q.view(torch.int16).numpy().view(np.uint16).reshape(16, 256)
    zones = index.zones
    times, traces, out = [], None, None
    t_end = time.time() + budget_s
    while len(times) < 3 or (time.time() < t_end and len(times) < 50):
        t = time.perf_counter()
        traces, out = od.decode_step(cells, code8, scales, k8, v8, qb,
                                     sink=zones.sink, local=zones.local)
        times.append(time.perf_counter() - t)
    ref_top = np.stack([tr.top100 for tr in traces])  # [4, 4, 100]
    match = float((ref_top == top_gpu).mean())
    # dense fp32 decode over every token (the reference's dense comparison)
    kf = od.arith.bf16_to_f32(kb)
    vf = od.arith.bf16_to_f32(vb)
    qf = od.arith.bf16_to_f32(qb)
    dt = []
    for _ in range(3):
        t = time.perf_counter()
        od.dense_decode(kf, vf, qf)
        dt.append(time.perf_counter() - t)
    # the same dense decode over the FP8-cast records (like-for-like bytes with
    # the GPU's dense FP8 path, whose reference output it also is)
    d8 = []
    dense_fp8 = None
    for _ in range(3):
        t = time.perf_counter()
        dense_fp8 = od.dense_decode(k8, v8, qf)
        d8.append(time.perf_counter() - t)
    threads = max((i.get("num_threads", 1) for i in threadpool_info()), default=1)
    return {
        "value": statistics.median(times) * 1e6,
        "unit": "µs/step",
        "cores": int(threads),
        "kind": "port",
        "sample": (
            f"{len(times)} full sparse decode steps of the same {args_config()} workload "
            "(numpy oracle: query prep, coarse, fine, pool, 2/4/8-bit scoring, top-k, FP8 "
            "SDPA), median; prefill untimed; `cores` = BLAS threads the oracle ran on"
        ),
        "host_cpus": os.cpu_count(),
        "cpu_model": cpu_model(),
        "dense_fp32_us": statistics.median(dt) * 1e6,
        "dense_fp8_cast_us": statistics.median(d8) * 1e6,
    }, match, out, dense_fp8, (code8, scales, k8, v8)


def reference_profile_check(entry, indexes, q, prefill) -> None:
    """Top-100 IDs of the reference-profile runs against the oracle on the
    same index (the checker of that leg; untimed)."""
    from oracle import decode as od

    code8, scales, k8, v8 = prefill
    qb = q.view(torch.int16).numpy().view(np.uint16).reshape(16, 256)
    for nprobe, (ix, ids) in indexes.items():
        cells = [od.GroupCell.from_cell(c) for c in ix.cells]
        traces, _ = od.decode_step(cells, code8, scales, k8, v8, qb, sink=ix.zones.sink,
                                   local=ix.zones.local)
        ref = np.stack([tr.top100 for tr in traces])
        entry["nprobe"][str(nprobe)]["top100_match"] = float((ref == ids).mean())


_CONFIG = {"name": "cfg2"}


def args_config() -> str:
    return _CONFIG["name"]


def workload_name(config: str) -> str:
    if config.startswith("cfg"):
        return f"BASELINE config {config[3:]}"
    return "the reference's default index profile (SeoulKV4Index.build defaults)"


def calibrate_copy(mib: int) -> int:
    """Copy ``mib`` MiB between two device buffers 5 times: a dispatch that
    reads and writes exactly ``mib`` MiB, for scaling the HBM counters."""
    n = mib << 20
    src = torch.ones(n, dtype=torch.uint8, device="cuda:0")
    dst = torch.empty_like(src)
    torch.cuda.synchronize()
    for _ in range(5):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"calibrate_copy_bytes": n, "dispatches": 5}), flush=True)
    return 0


def measured_traffic(kernel: str, config: str):
    """HBM bytes per launch of ``kernel`` on ``config`` from the committed
    counter summary of that config (``profiles/hbm_traffic_<config>.txt``:
    lines ``traffic <kernel> <bytes>``), or None when that kernel was not
    measured on it."""
    path = os.path.join(ROOT, "profiles", f"hbm_traffic_{config}.txt")
    try:
        with open(path) as f:
            for line in f:
                parts = line.split()
                if len(parts) == 3 and parts[0] == "traffic" and parts[1] == kernel:
                    return int(parts[2])
    except OSError:
        pass
    return None


def index_build(args) -> int:
    """Index build time on the host CPU and on the GPU for one config, and how
    far the GPU-built cells agree with the CPU-built ones (the build starts
    both from the same seeds; a difference is a floating-point rounding
    change of an assignment).  Cells are built one at a time exactly as
    ``SeoulKV4Index.build`` builds them (one log line per cell).  One JSON
    line."""
    p, k, v, _ = make_profile(args.config, n_queries=1)
    r0, r1 = p.sink, p.context - p.local
    nc = p.n_centroids or centroid_count(r1 - r0)
    log(f"{args.config}: T={p.context}, nc={nc}")

    def build(device: str):
        cells, t0 = [], time.time()
        for head in range(4):
            cells.append(build_cell(k[head], p=p.nprobe, lam=0.0625, seed=0, r0=r0, r1=r1,
                                    nc=nc, device=torch.device(device)))
            if device != "cpu":
                torch.cuda.synchronize()
            log(f"{device} build: cell {head} done at {time.time() - t0:.1f} s")
        return SeoulKV4Index(cells, {"nprobe_source": "explicit (build)"}), time.time() - t0

    SeoulKV4Index.build(k[:, :8192].contiguous(), v[:, :8192].contiguous(), sink=p.sink,
                        local=p.local, nprobe=64, n_centroids=512, build_device="cuda:0")
    torch.cuda.synchronize()  # warm the GPU build path (kernels, allocator)
    gpu, gpu_s = build("cuda:0")
    cpu, cpu_s = build("cpu")
    log(f"GPU build {gpu_s:.1f} s, CPU build {cpu_s:.1f} s ({torch.get_num_threads()} threads)")
    agree, identical, quality = [], [], {"cpu": [], "gpu": []}
    for h, (c, g) in enumerate(zip(cpu.cells, gpu.cells)):
        agree.append(round(list_agreement(c, g), 6))
        quality["cpu"].append(round(posting_cosine(c, k[h]), 5))
        quality["gpu"].append(round(posting_cosine(g, k[h]), 5))
        identical.append(bool(torch.equal(c["offsets"], g["offsets"])
                              and torch.equal(c["values"], g["values"])))
    print(json.dumps({
        "metric": "index build seconds (4 KV heads, one cell at a time)",
        "config": {"workload": args.config, "context": p.context,
                   "n_centroids": nc, "nprobe": p.nprobe},
        "cpu_s": round(cpu_s, 2), "gpu_s": round(gpu_s, 2),
        "cpu_threads": torch.get_num_threads(), "host_cpus": os.cpu_count(),
        "cpu_model": cpu_model(),
        "list_agreement": agree, "csr_identical": identical,
        "posting_cosine": quality,
    }), flush=True)
    return 0


def kv_gather_entry(sl_bytes: int, top_bytes: int, phases, alone_ms: dict) -> dict:
    """The K/V gather stage: its two parts' bytes over their own gather phase
    (trace build) and, beside them, over the whole kernel that holds each
    part (k_select for sink/local, k_top100 for the top-100 records)."""
    def rate(nbytes, us):
        if not us:
            return None, None
        gbs = nbytes / (us * 1e-6) / 1e9
        return round(gbs, 1), round(gbs / HBM_PEAK_GBS, 4)

    entry = {"bytes": sl_bytes + top_bytes, "latency_cap_frac": GATHER_LATENCY_CAP_FRAC,
             "target_frac": 0.5}
    for name, nbytes, kernel in (("top100", top_bytes, "top100_sdpa"),
                                 ("sink_local", sl_bytes, "select")):
        part = {"bytes": nbytes, "kernel": kernel,
                "kernel_us": round(alone_ms[kernel] * 1e3, 2)}
        part["kernel_GB/s"], part["kernel_frac"] = rate(nbytes, part["kernel_us"])
        if phases is not None:
            ph = phases[name]
            part.update(phase_us=ph["window_us"], per_block_us=ph["per_block_us"])
            part["GB/s"], part["frac"] = rate(nbytes, ph["window_us"])
        entry[name] = part
    if phases is not None:
        both = phases["top100"]["window_us"] + phases["sink_local"]["window_us"]
        entry["phase_us"] = round(both, 3)
        entry["GB/s"], entry["frac"] = rate(sl_bytes + top_bytes, both)
    entry["note"] = (
        "unique FP8 [V||K] records of each KV group: sink/local (gathered by the attention-"
        "slice blocks of the select launch while the centroid selections run) and top-100 "
        "(gathered by k_top100 after its selection); phase = record loads issued -> last "
        "wave's records arrived, first block to last (trace build of the same kernels); "
        "kernel_* = the same bytes over the whole holding kernel alone; latency_cap_frac = "
        "the fraction a 0.64 us issue-to-arrival floor per block allows for the top-100 part")
    return entry


def time_steps(inst, stream, steps: int, warmup: int) -> float:
    """µs per step of ``steps`` back-to-back steps of an initialised instance
    on its bound query (HIP events on ``stream``) after ``warmup``."""
    for _ in range(warmup):
        inst._run_bound()
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    inst._run_bound()  # untimed lead step (see the main timed loop)
    start.record(stream)
    for _ in range(steps):
        inst._run_bound()
    end.record(stream)
    end.synchronize()
    return start.elapsed_time(end) / steps * 1e3


def reference_profile(k, v, q, dev, stream, steps: int, warmup: int) -> dict:
    """The reference's own 128K profile on the same cache: the index that
    ``SeoulKV4Index.build(k, v)`` makes at its defaults (ceil(R / 128) * 32 =
    32672 centroids per KV head, nprobe 256; reference
    ``_index_build.py:16-19``, ``config.py:5``) run with ``SeoulKV4Config()``
    (pool capacity 13056, ``config.py:10-22``), and the same index re-probed
    at nprobe 384 (the README's figure, ``README.md:50``) through
    ``SeoulKV4Index.load(path, nprobe=384)``.  Device time of back-to-back
    steps, timed like ``value``."""
    import tempfile

    t0 = time.time()
    index = SeoulKV4Index.build(k, v)
    build_s = time.time() - t0
    log(f"reference profile: default index (nc={index.n_centroids}) built in {build_s:.1f}s")
    entry = {"n_centroids": index.n_centroids, "stage15_capacity": 13056,
             "index_build_s": round(build_s, 2), "nprobe": {}}
    indexes = {}
    with tempfile.TemporaryDirectory(prefix="skv_ref128k_") as tmp:
        path = os.path.join(tmp, "index.npz")
        index.dump(path)
        indexes[256] = index
        indexes[384] = SeoulKV4Index.load(path, nprobe=384)
    for nprobe, ix in indexes.items():
        with SeoulKV4(device=dev, k=k, v=v, index=ix,
                      config=SeoulKV4Config(debug=True)) as inst:
            inst.run(q)
            inst.synchronize()
            status = inst._state.synchronize()
            ids = inst.debug_snapshot()["selected_ids"].numpy()
            us = time_steps(inst, stream, steps, warmup)
            rt = inst._state
            rt.profile(True)
            for _ in range(steps):
                inst._run_bound()
            kernel_ms, _ = rt.profile_read()
            rt.profile(False)
            inst.synchronize()
        log(f"reference profile nprobe {nprobe}: {us:.1f} µs/step, pools {status['pool']}")
        entry["nprobe"][str(nprobe)] = {
            "us": round(us, 2),
            "vs_published": round(us / 518.0, 4),
            "in_step_us": {n: round(t * 1e3, 2) for n, t in kernel_ms.items()},
            "stage_sizes": {k_: status[k_] for k_ in ("selected", "pool", "u1", "u2")},
            "source": "SeoulKV4Index.build(k, v)" if nprobe == 256
                      else "SeoulKV4Index.load(path, nprobe=384)",
        }
        indexes[nprobe] = (ix, ids)
    entry["note"] = ("same cache, query and timing as `value`; index and pool capacity at the "
                     "reference's defaults (the profile of its published 518 µs/layer on a "
                     "Tenstorrent Blackhole p150a, README.md:7); vs_published = µs / 518")
    return entry, indexes


def dense_layouts(args) -> int:
    """Only the dense FP8 decode over one config's cache in four record
    layouts: contiguous, and 256-token pages of a pool holding exactly the
    pages needed or twice that, handed out in order or scrambled.  Two sets
    of 20 back-to-back calls per layout (skv_time_dense, after a warm-up
    set); one JSON line.  The layouts the bench's "paged" leg compares, for
    counter runs."""
    p, k, v, qs = make_profile(args.config, n_queries=1)
    index = SeoulKV4Index.build(k, v, sink=p.sink, local=p.local, nprobe=p.nprobe,
                                n_centroids=p.n_centroids)
    from seoulkv_amd import _hip

    need = -(-p.context // PAGE_TOKENS)
    out = {}

    def run(label, pages=None):
        rt = _hip.Runtime(0, k, v, index, pool_min=0, pool_capacity=None, debug=False,
                          kv_pages=pages)
        try:
            rt.bind_query(qs[0])
            rt.enqueue()
            rt.synchronize()
            rt.dense_decode()
            rt.read_dense_output()
            rt.time_dense(reps=5)
            sets = [rt.time_dense(reps=20) for _ in range(2)]
        finally:
            rt.close()
        out[label] = [{"partials_us": round(a * 1e3, 2), "call_us": round(c * 1e3, 2)}
                      for a, _, c in sets]
        log(f"{label}: {out[label]}")

    run("contiguous")
    for mult in (1, 2):
        pool = KVPagePool(mult * need, page_tokens=PAGE_TOKENS, device="cuda:0")
        order = list(range(mult * need))
        random.Random(5).shuffle(order)
        run(f"pool_x{mult}_in_order", (pool, list(range(need))))
        run(f"pool_x{mult}_scrambled", (pool, order[:need]))
        del pool
    print(json.dumps({"metric": "dense FP8 decode µs by record layout", "config": args.config,
                      "page_tokens": PAGE_TOKENS, "layouts": out}), flush=True)
    return 0


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--config", default="cfg2", choices=sorted(PROFILES))
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-reference-profile", action="store_true",
                    help="skip the reference's default 128K profile leg (config 2 only)")
    ap.add_argument("--no-append", action="store_true",
                    help="skip the cache-append decode loops")
    ap.add_argument("--no-gather-phases", action="store_true",
                    help="skip the K/V gather phase timing (trace build of the library)")
    ap.add_argument("--cpu-budget", type=float, default=12.0)
    ap.add_argument("--build-device", default="cpu")
    ap.add_argument("--calibrate-copy", type=int, default=0, metavar="MIB",
                    help="only copy MIB MiB device-to-device 5 times (the known-size "
                         "kernel that scales the FETCH_SIZE / WRITE_SIZE counters)")
    ap.add_argument("--index-build", action="store_true",
                    help="only time SeoulKV4Index.build on the CPU and the GPU for --config "
                         "and compare the two indexes")
    ap.add_argument("--dense-layouts", action="store_true",
                    help="only time the dense FP8 decode in contiguous and paged record "
                         "layouts (for counter runs)")
    args = ap.parse_args()
    _CONFIG["name"] = args.config
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(
            "bench.py measures one MI355X: this build runs one GPU per process and the "
            "4 KV groups of a layer on that GPU; multi-GPU (--gpus > 1) is not part of "
            "this build: the 4 KV groups would shard one per GPU with a single 8 KiB "
            "all-gather of the outputs.",
            file=sys.stderr,
        )
        return 2
    if not torch.cuda.is_available():
        print("bench.py needs a ROCm GPU", file=sys.stderr)
        return 1
    if args.calibrate_copy:
        return calibrate_copy(args.calibrate_copy)
    if args.index_build:
        return index_build(args)
    if args.dense_layouts:
        return dense_layouts(args)

    t0 = time.time()
    p, k, v, qs = make_profile(args.config, n_queries=1)
    q = qs[0]
    log(f"generated {args.config} T={p.context} in {time.time() - t0:.1f}s")
    t0 = time.time()
    index = SeoulKV4Index.build(k, v, sink=p.sink, local=p.local, nprobe=p.nprobe,
                                n_centroids=p.n_centroids, build_device=args.build_device)
    nc = index.n_centroids
    log(f"index built in {time.time() - t0:.1f}s (nc={nc}, nprobe={p.nprobe})")

    dev = torch.device("cuda", 0)
    stream = torch.cuda.Stream(dev)
    # token IDs stay below 2^20: at T = 2^20 (config 4) there is no room to append
    # the decode loops append one token per step (host, then device), then
    # two bulk appends; token IDs stay below 2^20, so config 4 has no room
    loop_steps = max(args.steps, 200)
    n_append = min(2 * loop_steps + 2 * APPEND_BULK_REPS * APPEND_BULK, (1 << 20) - p.context)
    config = SeoulKV4Config(stage15_capacity=None, debug=True, append_capacity=n_append)
    with torch.cuda.stream(stream):
        attn = SeoulKV4(device=dev, k=k, v=v, index=index, config=config)
        t0 = time.time()
        attn.run(q)
        attn.synchronize()
        log(f"initialised in {time.time() - t0:.1f}s")
        status = attn._state.synchronize()
        top_gpu = attn.debug_snapshot()["selected_ids"].numpy()
        out_gpu = attn.run(q).to_torch().float().numpy().reshape(16, 256)

        for _ in range(args.warmup):
            attn._run_bound()
        torch.cuda.synchronize()
        start = torch.cuda.Event(enable_timing=True)
        end = torch.cuda.Event(enable_timing=True)
        # one untimed step between the synchronize and the start event (here
        # and in every timed loop below): the timed steps then follow queued
        # work, so the window holds their device time, not the idle GPU's
        # wait for the host's first launches (~28 us over the window, which
        # a 20-step run would spread as +1.4 us per step; the host's own cost
        # is host_inclusive_us)
        attn._run_bound()
        start.record(stream)
        for _ in range(args.steps):
            attn._run_bound()
        end.record(stream)
        end.synchronize()
        torch.cuda.synchronize()
        ms_per_step = start.elapsed_time(end) / args.steps
        log(f"device time {ms_per_step * 1e3:.1f} µs/step over {args.steps} steps")

        # cold cache: steps rotate over N_COLD instances of the same cache, each
        # with its own device copy of the index, key rows and FP8 records, so
        # the ~30-40 MB a step touches was last read N_COLD - 1 steps (over
        # 300 MB) earlier and is no longer in the L2s or the 256 MB MALL, as
        # for a decoder that visits every other layer between two steps of
        # this one
        cold = [attn]
        cold_cfg = SeoulKV4Config(stage15_capacity=None)
        for _ in range(N_COLD - 1):
            inst = SeoulKV4(device=dev, k=k, v=v, index=index, config=cold_cfg)
            inst.run(q)
            cold.append(inst)
        for inst in cold:
            inst._run_bound()
        torch.cuda.synchronize()
        n_cold = max(N_COLD, (args.steps // N_COLD) * N_COLD)
        cold[-1]._run_bound()  # untimed lead step (the last instance, just used)
        start.record(stream)
        for i in range(n_cold):
            cold[i % N_COLD]._run_bound()
        end.record(stream)
        end.synchronize()
        cold_ms = start.elapsed_time(end) / n_cold
        for inst in cold[1:]:
            inst.close()
        del cold
        log(f"cold-cache device time {cold_ms * 1e3:.1f} µs/step over {n_cold} steps "
            f"({N_COLD} instances)")

        # host-inclusive: the product call with a host query, ``run(q)`` (the
        # query rides with the front kernel), and beside it the query's upload
        # and the enqueue as two calls; host clock from the first call to the
        # last step's end, over at least 200 steps (a short run's start-up and
        # final drain would weigh on each step)
        def bind_enqueue():
            attn._bind_query(q)
            attn._run_bound()

        host_us = {}
        for name, call in (("run", lambda: attn.run(q)), ("bind_enqueue", bind_enqueue)):
            for _ in range(args.warmup):
                call()
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(loop_steps):
                call()
            torch.cuda.synchronize()
            host_us[name] = (time.perf_counter() - t) / loop_steps * 1e6

        # per-kernel HIP-event profile of the same steps, each with its host
        # query (includes the gaps between dependent kernels)
        rt = attn._state
        rt.profile(True)
        for _ in range(args.steps):
            attn.run(q)
        kernel_ms, n_prof = rt.profile_read()
        rt.profile(False)
        attn.synchronize()
        # each kernel alone: `reps` back-to-back launches between HIP events on
        # the library's stream (what rocprofv3 reports as the kernel duration)
        names = list(kernel_ms)
        alone_ms = {name: rt.time_kernel(i, reps=max(20, args.steps // 4))
                    for i, name in enumerate(names)}
        attn.synchronize()

        # the dense FP8 decode over all T keys, the sparse step's comparison
        rt.dense_decode()
        dense_gpu = rt.read_dense_output().float().numpy().reshape(16, 256)
        rt.time_dense(reps=5)  # warm-up: the first timed set runs 1-4 µs slower
        dn_kernel_ms, dn_merge_ms, dn_ms = rt.time_dense(reps=max(20, args.steps // 4))
        log(f"dense FP8 decode {dn_ms * 1e3:.1f} µs (partials {dn_kernel_ms * 1e3:.1f} µs)")

        # the same cache with its FP8 records in 256-token pages of a shared
        # pool, handed out in a scrambled order: same results, step and dense
        # decode timed the same way
        pool = KVPagePool(2 * (-(-p.context // PAGE_TOKENS)), page_tokens=PAGE_TOKENS,
                          device=dev)
        scrambled = pool.allocate(pool.n_pages)
        random.Random(5).shuffle(scrambled)
        pool.release(scrambled)
        paged = SeoulKV4(device=dev, k=k, v=v, index=index,
                         config=SeoulKV4Config(stage15_capacity=None, debug=True), kv_pool=pool)
        paged_out = paged.run(q).to_torch().view(torch.int16).clone()
        paged_ids = paged.debug_snapshot()["selected_ids"].numpy()
        attn.run(q)
        same_out = bool(torch.equal(paged_out, attn.run(q).to_torch().view(torch.int16)))
        for _ in range(args.warmup):
            paged._run_bound()
        torch.cuda.synchronize()
        paged._run_bound()  # untimed lead step
        start.record(stream)
        for _ in range(args.steps):
            paged._run_bound()
        end.record(stream)
        end.synchronize()
        paged_us = start.elapsed_time(end) / args.steps * 1e3
        prt = paged._state
        prt.dense_decode()
        paged_dense_same = bool(torch.equal(prt.read_dense_output(), rt.read_dense_output()))
        prt.time_dense(reps=5)  # warm-up, as for the contiguous records
        _, _, paged_dn_ms = prt.time_dense(reps=max(20, args.steps // 4))
        paged.close()
        del pool
        log(f"paged records ({PAGE_TOKENS}-token pages): step {paged_us:.1f} µs, dense "
            f"{paged_dn_ms * 1e3:.1f} µs, results identical: {same_out and paged_dense_same}")
        paged_entry = {
            "page_tokens": PAGE_TOKENS, "step_us": round(paged_us, 2),
            "dense_us": round(paged_dn_ms * 1e3, 2),
            "top100_equal": bool(np.array_equal(paged_ids, top_gpu)),
            "output_equal": same_out, "dense_output_equal": paged_dense_same,
            "note": "FP8 records in pool pages handed out in a scrambled order, read through "
                    "the page table; device time of back-to-back steps",
        }

        ref_entry, ref_indexes = None, None
        if args.config == "cfg2" and not args.no_reference_profile:
            ref_entry, ref_indexes = reference_profile(k, v, q, dev, stream, args.steps,
                                                       args.warmup)

        # cache append (after every measurement above: it grows the local
        # window).  A decoder's loop: each step appends the token it decoded
        # (1 token, from the host or from the device), binds the next query
        # and enqueues the step, with no host synchronisation; device time of
        # `loop_steps` such iterations against the same loop without appends.
        append = None
        if not args.no_append and n_append >= 2 * loop_steps + 2 * APPEND_BULK_REPS * APPEND_BULK:
            rt = attn._state
            kn = k[:, -n_append:].clone()
            vn = v[:, -n_append:].clone()
            kd, vd = kn.to(dev), vn.to(dev)
            torch.cuda.synchronize()

            def loop(append_fn) -> tuple[float, float]:
                """(device µs per iteration, host µs per append call)."""
                host = 0.0
                start.record(stream)
                for i in range(loop_steps):
                    if append_fn is not None:
                        t = time.perf_counter()
                        append_fn(i)
                        host += time.perf_counter() - t
                    rt.bind_query(q)
                    rt.enqueue()
                end.record(stream)
                end.synchronize()
                return start.elapsed_time(end) / loop_steps * 1e3, host / loop_steps * 1e6

            loop(None)  # warm-up of the bind + step loop
            # each append loop is bracketed by the loop without appends, since
            # the step itself grows with the local window
            base_us, _ = loop(None)
            used = 0
            host_slices = [(kn[:, i:i + 1].contiguous(), vn[:, i:i + 1].contiguous())
                           for i in range(loop_steps)]

            def host_one(i):
                rt.append(*host_slices[i])

            host_us_, host_call_us = loop(host_one)
            used += loop_steps
            mid_us, _ = loop(None)
            dev_slices = [(kd[:, used + i:used + i + 1].contiguous(),
                           vd[:, used + i:used + i + 1].contiguous()) for i in range(loop_steps)]
            torch.cuda.synchronize()

            def dev_one(i):
                rt.append(*dev_slices[i])

            dev_us_, dev_call_us = loop(dev_one)
            used += loop_steps
            after_us, _ = loop(None)
            # bulk appends (wall time including the host sync), median of
            # APPEND_BULK_REPS each
            attn.synchronize()

            def bulk(kk, vv) -> tuple[float, list, list]:
                # (median wall time, each append's wall time, each append
                # call's own time before the host sync), µs
                nonlocal used
                times, calls = [], []
                # the K/V of each append made contiguous before the clock
                # starts (as the 1-token loop's slices): the timed call is
                # the append, not the caller's copy into fresh pages
                parts = [(kk[:, u:u + APPEND_BULK].contiguous(), vv[:, u:u + APPEND_BULK].contiguous())
                         for u in range(used, used + APPEND_BULK_REPS * APPEND_BULK, APPEND_BULK)]
                if kk.is_cuda:
                    torch.cuda.synchronize()
                for ks, vs in parts:
                    t = time.perf_counter()
                    attn.append(ks, vs)
                    tc = time.perf_counter()
                    attn.synchronize()
                    times.append((time.perf_counter() - t) * 1e6)
                    calls.append((tc - t) * 1e6)
                    used += APPEND_BULK
                return (float(np.median(times)), [round(x, 1) for x in times],
                        [round(x, 1) for x in calls])

            bulk_host_us, bulk_host_each, bulk_host_calls = bulk(kn, vn)
            bulk_dev_us, bulk_dev_each, bulk_dev_calls = bulk(kd, vd)
            host_ref, dev_ref = (base_us + mid_us) / 2, (mid_us + after_us) / 2
            log(f"decode loop: step {base_us:.1f} / {mid_us:.1f} / {after_us:.1f} µs (local "
                f"window {p.local} / +{loop_steps} / +{2 * loop_steps}); with a 1-token host "
                f"append {host_us_:.1f} µs ({host_call_us:.1f} µs host per append call), device "
                f"append {dev_us_:.1f} µs; bulk {APPEND_BULK} tokens host {bulk_host_us:.0f} µs, "
                f"device {bulk_dev_us:.0f} µs")
            append = {
                "loop_steps": loop_steps,
                "step_us": round(base_us, 2),
                "host_1token_step_us": round(host_us_, 2),
                "device_1token_step_us": round(dev_us_, 2),
                "host_over_step": round(host_us_ / host_ref, 4),
                "device_over_step": round(dev_us_ / dev_ref, 4),
                "host_append_call_us": round(host_call_us, 1),
                "device_append_call_us": round(dev_call_us, 1),
                "step_us_between_loops": round(mid_us, 2),
                "step_us_after_loops": round(after_us, 2),
                "bulk_tokens": APPEND_BULK,
                "bulk_host_us": round(bulk_host_us, 1),
                "bulk_device_us": round(bulk_dev_us, 1),
                "bulk_host_each_us": bulk_host_each,
                "bulk_host_call_us": bulk_host_calls,
                "bulk_device_each_us": bulk_dev_each,
                "bulk_device_call_us": bulk_dev_calls,
                "appended": used,
                "note": "decode loop per iteration: append 1 token, bind the query (8 KiB "
                        "upload; a host token rides along and the step's first kernel packs "
                        "it), enqueue the step; device time between HIP events over "
                        "loop_steps iterations, no host sync; *_over_step = against the mean "
                        "of the same loop without appends just before and after (the step "
                        "grows with the local window); bulk = median wall time of 3 appends of "
                        "bulk_tokens (their K/V made contiguous before timing), incl. host sync "
                        "(*_each_us: every append in order; *_call_us: the append call alone, "
                        "before the sync)",
            }

    sl_bytes, top_bytes = kv_gather_bytes(top_gpu, p)
    phases = None if args.no_gather_phases else gather_phases(k, v, index, q, steps=50)
    nbytes = kernel_bytes(status, p, nc)
    total_bytes = sum(nbytes.values())
    dominant = max(alone_ms, key=alone_ms.get)
    dom_us = alone_ms[dominant] * 1e3
    dom_gbs = nbytes.get(dominant, 0) / (alone_ms[dominant] * 1e-3) / 1e9
    per_kernel = {
        name: {"us": round(alone_ms[name] * 1e3, 2),
               "in_step_us": round(kernel_ms[name] * 1e3, 2),
               "bytes": int(nbytes.get(name, 0)),
               "GB/s": round(nbytes.get(name, 0) / max(alone_ms[name], 1e-9) / 1e6, 1)}
        for name in names
    }

    cpu = None
    match = None
    dense_err = None
    dense_bytes = G_KV * p.context * 512  # every FP8 [V || K] record once
    if not args.no_cpu_baseline:
        cpu, match, out_ref, dense_ref, prefill = cpu_baseline(index, k, v, q, top_gpu,
                                                               args.cpu_budget)
        if ref_entry is not None:
            reference_profile_check(ref_entry, ref_indexes, q, prefill)
        err = np.abs(out_gpu - out_ref).max()
        cos = min(
            float(out_gpu[j] @ out_ref[j] / (np.linalg.norm(out_gpu[j]) * np.linalg.norm(out_ref[j])))
            for j in range(16)
        )
        log(f"oracle: top-100 match {match:.4f}, output max-abs {err:.3g}, min cosine {cos:.6f}")
        dense_err = float(np.abs(dense_gpu - dense_ref).max())
        log(f"dense FP8 decode vs oracle: max-abs {dense_err:.3g}")

    result = {
        "metric": METRIC,
        "value": round(ms_per_step * 1e3, 2),
        "unit": "µs/step",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8-mfma scores / fp8-e4m3 attention",
        "data": "synthetic: seeded 4096-component Gaussian-mixture K with RoPE, N(0,1) V",
        "config": {
            "workload": f"{args.config}: {workload_name(args.config)} (T={p.context}, 4 KV x 16 Q heads, "
                        f"d=256, nc={nc}, nprobe={p.nprobe}, top-100, sink "
                        f"{p.sink}, local {p.local}, FP8 K/V records)",
            "context": p.context,
            "n_centroids": nc,
            "nprobe": p.nprobe,
            "kv_heads": 4,
            "q_heads": 16,
            "head_dim": 256,
        },
        "step_hbm_bytes": int(total_bytes),
        "step_hbm_GBps": round(total_bytes / (ms_per_step * 1e-3) / 1e9, 1),
        "value_cold": round(cold_ms * 1e3, 2),
        "cold_instances": N_COLD,
        "top100_match": match,
        "host_inclusive_us": round(host_us["run"], 2),
        "bind_enqueue_us": round(host_us["bind_enqueue"], 2),
        "roofline": {
            "bound": "hbm",
            "kernel": dominant,
            "achieved": round(dom_gbs, 1),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(dom_gbs / HBM_PEAK_GBS, 4),
            "traffic": measured_traffic(dominant, args.config),
            "kernel_us": round(dom_us, 2),
            "bytes_per_launch": int(nbytes.get(dominant, 0)),
        },
        "kernels": per_kernel,
        "kv_gather": kv_gather_entry(sl_bytes, top_bytes, phases, alone_ms),
        "dense_fp8": {
            "us": round(dn_ms * 1e3, 2),
            "kernel_us": round(dn_kernel_ms * 1e3, 2),
            "merge_us": round(dn_merge_ms * 1e3, 2),
            "bytes": int(dense_bytes),
            "GB/s": round(dense_bytes / (dn_kernel_ms * 1e-3) / 1e9, 1),
            "frac": round(dense_bytes / (dn_kernel_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
            "traffic": measured_traffic("dense_fp8", args.config),
            "max_abs_vs_oracle": dense_err,
            "sparse_over_dense": round(ms_per_step / dn_ms, 3),
        },
        "append": append,
        "paged": paged_entry,
        "profiled_steps": n_prof,
        "stage_sizes": {k_: status[k_] for k_ in ("survivors", "selected", "pool", "u1", "u2")},
        "cpu_baseline": cpu,
        "reference_profile": ref_entry,
        "reference_published": {
            "value": 518, "unit": "µs/layer", "hardware": "Tenstorrent Blackhole p150a",
            "note": "reference README 128K profile at its own centroid count (32672/head); "
                    "measured here on that profile in reference_profile (vs_published); "
                    "`value` is config 2 (8192 centroids/head), so vs_baseline is null",
        },
    }
    print(json.dumps(result), flush=True)
    attn.close()
    return 0


if __name__ == "__main__":
    sys.exit(main())
