"""``skv_run``: a step whose host query rides with the front kernel's arguments.

The result must equal bind + enqueue bit for bit, the query must be bound
afterwards (repeated steps, the dense decode, kernel timing read it from device
memory), queued steps must each keep their own query, and the calls that need
an upload (folded appends, captured steps) must take one.
"""

from __future__ import annotations

import pytest
import torch

from seoulkv_amd import _hip
from seoulkv_amd.result import _DeviceArray
from tests.helpers import case

SMALL = dict(context=8192, components=256, nc=512, nprobe=64)  # one pass of the front grid
LOOPED = dict(context=81920, components=64, nc=16640, nprobe=128, seed_shift=40)  # looped front


def test_run_rejects_a_null_handle():
    assert _hip.load_library().skv_run(None, None) == 6


def _runtime(p, stream=None, append=0):
    index, k, v, qs = case(**p)
    return _hip.Runtime(0, k, v, index, pool_min=0, pool_capacity=None, debug=False,
                        stream=stream, append_capacity=append), qs


@pytest.mark.gpu
@pytest.mark.parametrize("p", [SMALL, LOOPED], ids=["small", "looped"])
def test_run_equals_bind_and_enqueue(p):
    a, qs = _runtime(p)
    b, _ = _runtime(p)
    try:
        for q in (qs[0], qs[1], torch.zeros_like(qs[0]), qs[0]):
            a.run(q)
            b.bind_query(q)
            b.enqueue()
            assert torch.equal(a.read_output(), b.read_output())
            assert torch.equal(a.debug_ids(), b.debug_ids())
            out = a.read_output()
            a.enqueue()  # the query is bound: a later step repeats it
            assert torch.equal(a.read_output(), out)
        a.dense_decode()
        b.dense_decode()
        assert torch.equal(a.read_dense_output(), b.read_dense_output())
        a.time_kernel(0, 2)
        assert torch.equal(a.read_output(), out)
    finally:
        a.close()
        b.close()


@pytest.mark.gpu
def test_queued_runs_keep_their_queries():
    stream = torch.cuda.Stream()
    rt, qs = _runtime(SMALL, stream.cuda_stream)
    try:
        gen = torch.Generator().manual_seed(5)
        queries = [qs[0], qs[1]] + [torch.randn(1, 1, 16, 256, generator=gen).bfloat16()
                                    for _ in range(6)]
        want = []
        for q in queries:
            rt.bind_query(q)
            rt.enqueue()
            want.append(rt.read_output())
        out = torch.as_tensor(_DeviceArray(rt.output_device_ptr(), (16, 256), "<i2", rt),
                              device="cuda:0")
        got = torch.zeros(200, 16, 256, dtype=torch.int16, device="cuda:0")
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            for i in range(200):  # no host wait between the steps
                rt.run(queries[(3 * i) % 8])
                got[i].copy_(out)
        torch.cuda.synchronize()
        for i in range(200):
            w = want[(3 * i) % 8].reshape(16, 256).view(torch.int16)
            assert torch.equal(got[i].cpu(), w), i
    finally:
        rt.close()


@pytest.mark.gpu
def test_run_with_appends_and_captured_steps():
    a, qs = _runtime(SMALL, append=64)
    b, _ = _runtime(SMALL, append=64)
    try:
        a.run(qs[0])
        b.bind_query(qs[0])
        b.enqueue()
        gen = torch.Generator().manual_seed(9)
        for i, n in enumerate((1, 3, 20)):  # folded, folded, packed by its own kernel
            k, v = (torch.randn(4, n, 256, generator=gen).bfloat16() for _ in range(2))
            q = qs[i % 2]
            a.append(k, v)
            a.run(q)
            b.append(k, v)
            b.bind_query(q)
            b.enqueue()
            assert torch.equal(a.read_output(), b.read_output()), n
        a.graph_mode(True)
        for q in (qs[1], qs[0], qs[1]):
            a.run(q)
            b.bind_query(q)
            b.enqueue()
            assert torch.equal(a.read_output(), b.read_output())
        a.graph_mode(False)
        a.run(qs[0])
        b.bind_query(qs[0])
        b.enqueue()
        assert torch.equal(a.read_output(), b.read_output())
    finally:
        a.close()
        b.close()
