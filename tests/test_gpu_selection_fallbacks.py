"""Selections whose first path does not fit, against the oracle and through
the status bits that record them.

Centroid lists held in registers (8K-32K centroids): ``octn_top`` counts only
the items above the P-th largest thread maximum.  It cannot serve a probe
budget past the 1024 threads, a selection whose items lie in fewer than P
threads' octets, or a P-th score 4095 or more BF16 steps above that maximum;
the two-pass selection of the same registers has to take those.  Each KV head
of a runtime gets a cell that reaches one of them."""

from __future__ import annotations

import dataclasses
import types

import numpy as np
import pytest
import torch

from oracle import arith
from oracle import decode as od
from seoulkv_amd import SeoulKV4Index, _hip
from seoulkv_amd.synthetic import make_cache
from tests.helpers import bits, case, cosine, oracle_inputs

pytestmark = pytest.mark.gpu

THRESH, FINE = 1, 2  # status bits
THREADS, MAX_TIES, STEPS = 1024, 1024, 4095

LONG = {
    "nc10240": dict(context=40960, components=1024, nc=10240, nprobe=256, seed_shift=5),
    "nc24576": dict(context=98304, components=2048, nc=24576, nprobe=256, seed_shift=9),
}


def _top_misses(scores, k, ties_by_id):
    """Whether the k best of the ordered ``scores`` (0: excluded) are out of
    the register shortcut's reach (the bound and its bin as the kernel's)."""
    if k > THREADS:
        return True
    maxima = np.zeros(THREADS, dtype=np.int64)
    np.maximum.at(maxima, (np.arange(len(scores)) // 8) % THREADS, scores)
    bound = np.sort(maxima)[::-1][k - 1]
    if bound == 0:
        return True
    kth = np.sort(scores)[::-1][k - 1]
    if kth - max(bound >> 4 << 4, 1) >= STEPS:
        return True
    ties = int((scores == kth).sum())
    need = k - int((scores > kth).sum())
    return ties_by_id and need < ties and ties > MAX_TIES


def _expected_bits(cell, qp):
    lower, upper = (arith.ordered16(x).astype(np.int64) for x in od.coarse(cell, qp))
    fine = arith.ordered16(od.fine_scores(cell, qp, np.arange(len(cell.upper)))).astype(np.int64)
    out = 0
    for h in range(4):
        thr = np.sort(lower[h])[::-1][cell.p - 1]
        out |= THRESH * _top_misses(lower[h], cell.p, False)
        out |= FINE * _top_misses(np.where(upper[h] >= thr, fine[h], 0), cell.p, True)
    return out


def _lam_with_few_positive_bounds(cell, qb, scales, p):
    """A lambda at which some head has at least p positive lower bounds, in
    the octets of fewer than p threads: the p-th score lies above zero and the
    p-th thread maximum below."""
    lo, hi = 0.0, 8.0
    for _ in range(60):
        lam = (lo + hi) / 2
        qp = od.prepare_query(qb, scales, lam)
        lower = arith.ordered16(od.coarse(dataclasses.replace(cell, lam=lam), qp)[0])
        positive = lower > 0x8000
        threads = [len(np.unique((np.flatnonzero(r) // 8) % THREADS)) for r in positive]
        counts = positive.sum(axis=-1)
        if any(c >= p > t for c, t in zip(counts, threads)):
            return float(np.float32(lam))
        if min(threads) >= p:  # a larger margin leaves fewer positive bounds
            lo = lam
        else:
            hi = lam
    raise AssertionError("no such lambda")


@pytest.mark.parametrize("name", list(LONG))
def test_long_lists_past_the_register_shortcut(name):
    p = LONG[name]
    index, k, v, qs = case(**p)
    cells, code8, scales, k8, v8 = oracle_inputs(**p)
    q = qs[0]
    qb = bits(q).reshape(16, 256)
    gap_lam = _lam_with_few_positive_bounds(dataclasses.replace(cells[2], p=512), qb[8:12],
                                            scales[2], 512)
    changes = [dict(p=2048),             # a budget past the thread count
               dict(p=512, lam=1e-6),    # eligible centroids in fewer than 512 octets
               dict(p=512, lam=gap_lam),  # a wide gap below the 512th lower bound
               dict(p=p["nc"])]          # every centroid
    cells = [dataclasses.replace(c, **ch) for c, ch in zip(cells, changes)]
    device = types.SimpleNamespace(
        cells=tuple({**c, **ch} for c, ch in zip(index.cells, changes)), zones=index.zones)
    want = [_expected_bits(c, od.prepare_query(qb[4 * g:4 * g + 4], scales[g], c.lam))
            for g, c in enumerate(cells)]
    assert want[0] == THRESH | FINE and want[1] & FINE and want[2] & THRESH and want[3]
    print(f"[gpu] {name}: runtime with p 2048 / 512 / 512 / nc", flush=True)
    rt = _hip.Runtime(0, k, v, device, pool_min=0, pool_capacity=None, debug=True)
    try:
        for kind, x in (("real", q), ("zero", torch.zeros_like(q))):
            xb = bits(x).reshape(16, 256)
            if kind == "zero":  # every fine score ties
                want = [THRESH | FINE, FINE, FINE, THRESH | FINE]
            print(f"[gpu] {name} query {kind}", flush=True)
            rt.bind_query(x)
            rt.enqueue()
            status = rt.synchronize()
            assert status["err"] == [0, 0, 0, 0]
            assert [b & (THRESH | FINE) for b in status["full_select"]] == want, kind
            traces, out = od.decode_step(cells, code8, scales, k8, v8, xb, sink=128, local=256)
            for g, tr in enumerate(traces):
                for stage, ref in (("thresh", tr.thr), ("selected", tr.selected),
                                   ("pool", tr.pool), ("top", tr.top100)):
                    np.testing.assert_array_equal(rt.read_stage(stage, g), ref,
                                                  err_msg=f"{kind} g{g} {stage}")
            got = rt.read_output().float().numpy().reshape(16, 256)
            for j in range(16):
                assert np.abs(got[j] - out[j]).max() <= 2e-2, f"{kind} head {j} max-abs"
                assert cosine(got[j], out[j]) >= 0.999, f"{kind} head {j} cosine"
    finally:
        rt.close()


# ---------------------------------------------------------------- tiled rows
# Pools past the register selections are cut from a 4096-item sample, and the
# tiles that reach the cut are selected in registers.  The k-th score may lie
# far above the cut, or tie with more items than are ranked by comparison.
M15 = 1600


def _sampled_cut(scores, k):
    """``fs_cut`` of n > 4096 ordered scores: the score that about
    k + 4 sqrt(k) + 8 items reach, from every n/4096-th item."""
    n = len(scores)
    sample = np.sort(scores[(np.arange(4096, dtype=np.int64) * n) >> 12])[::-1]
    e = k * 4096 / n
    return int(sample[int(np.ceil(e + 4 * np.sqrt(e) + 8)) - 1])


def _split_keys(kind, context, sink, local, gen):
    """K [4, context, 256] of four directions (q of a KV head: its direction):
    ``gap``: 1650 retrieval keys along it, the rest against it; ``ties``: 1000
    along it, 2500 copies of one key, the rest against it."""
    retrieval = torch.arange(sink, context - local)
    k = 0.25 * torch.randn(4, context, 256, generator=gen)
    directions = torch.randn(4, 256, generator=gen)
    for g in range(4):
        sign = -torch.ones(context)
        pick = retrieval[torch.randperm(len(retrieval), generator=gen)]
        sign[pick[:1650 if kind == "gap" else 1000]] = 1.0
        k[g] += sign[:, None] * directions[g]
        if kind == "ties":
            k[g][pick[1000:3500]] = 0.4 * directions[g]
    return k.bfloat16(), directions


@pytest.mark.parametrize("kind", ["gap", "ties"])
def test_tiled_top1600_far_above_the_cut_and_tied(kind):
    context, sink, local, nc = 20000, 40, 200, 512
    gen = torch.Generator().manual_seed(77)
    k, directions = _split_keys(kind, context, sink, local, gen)
    v = torch.randn(4, context, 256, generator=gen).bfloat16()
    q = directions.repeat_interleave(4, 0) + 0.05 * torch.randn(16, 256, generator=gen)
    q = q.bfloat16().reshape(1, 1, 16, 256)
    built = SeoulKV4Index.build(k, v, sink=sink, local=local, nprobe=512, n_centroids=nc)
    code8, scales = od.key_codec(bits(k))
    k8, v8 = od.fp8_records(bits(k), bits(v))
    cells = [od.GroupCell.from_cell(c) for c in built.cells]
    traces, out = od.decode_step(cells, code8, scales, k8, v8, bits(q).reshape(16, 256),
                                 sink=sink, local=local)
    for tr in traces:  # every list is probed: the pool is the retrieval region
        assert len(tr.pool) == context - sink - local
        for row in arith.ordered16(tr.s2).astype(np.int64):
            cut, kth = _sampled_cut(row, M15), np.sort(row)[::-1][M15 - 1]
            above, ties = int((row > kth).sum()), int((row == kth).sum())
            if kind == "gap":
                assert kth - cut >= STEPS
            else:
                assert kth - cut < STEPS and ties > MAX_TIES and above + ties > M15
    print(f"[gpu] tiled top-1600 {kind}", flush=True)
    rt = _hip.Runtime(0, k, v, built, pool_min=0, pool_capacity=None, debug=True)
    try:
        rt.bind_query(q)
        rt.enqueue()
        status = rt.synchronize()
        assert status["err"] == [0, 0, 0, 0]
        assert all(b & 4 == 0 for b in status["full_select"])
        for g, tr in enumerate(traces):
            for stage, ref in (("pool", tr.pool), ("u1", tr.u1), ("u2", tr.u2),
                               ("top", tr.top100)):
                np.testing.assert_array_equal(rt.read_stage(stage, g), ref,
                                              err_msg=f"g{g} {stage}")
        got = rt.read_output().float().numpy().reshape(16, 256)
        assert np.abs(got - out).max() <= 2e-2
    finally:
        rt.close()


def test_tiled_fine_selection_ties_past_32k_centroids():
    """nc > 32768: the fine selection is a tiled row; the zero query ties every
    centroid, so the P lowest centroid IDs win."""
    context, nc = 98304, 33792
    k, v, qs = make_cache(context, 2048, n_queries=1)
    built = SeoulKV4Index.build(k, v, nprobe=384, n_centroids=nc, build_device="cuda")
    code8, scales = od.key_codec(bits(k))
    k8, v8 = od.fp8_records(bits(k), bits(v))
    cells = [od.GroupCell.from_cell(c) for c in built.cells]
    print("[gpu] nc 33792: real and zero query", flush=True)
    rt = _hip.Runtime(0, k, v, built, pool_min=0, pool_capacity=None, debug=True)
    try:
        for q in (qs[0], torch.zeros_like(qs[0])):
            rt.bind_query(q)
            rt.enqueue()
            status = rt.synchronize()
            assert status["err"] == [0, 0, 0, 0] and all(b & 2 == 0 for b in status["full_select"])
            traces, _ = od.decode_step(cells, code8, scales, k8, v8, bits(q).reshape(16, 256),
                                       sink=128, local=256)
            for g, tr in enumerate(traces):
                for stage, ref in (("thresh", tr.thr), ("selected", tr.selected),
                                   ("pool", tr.pool), ("top", tr.top100)):
                    np.testing.assert_array_equal(rt.read_stage(stage, g), ref,
                                                  err_msg=f"g{g} {stage}")
    finally:
        rt.close()
