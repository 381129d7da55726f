"""Device views of a result keep the memory they alias: dropping the last
reference to the instance (without ``close()``) must not free the output
buffer under a tensor that ``device_tensors`` returned."""

from __future__ import annotations

import gc
import weakref

import pytest
import torch

from seoulkv_amd import SeoulKV4, SeoulKV4Config
from seoulkv_amd.result import _DeviceArray
from tests.helpers import case


class _Owner:
    pass


def test_wrapper_holds_its_owner():
    owner = _Owner()
    alive = weakref.ref(owner)
    view = _DeviceArray(0x1000, (4,), "<i2", owner)
    del owner
    gc.collect()
    assert alive() is not None
    del view
    gc.collect()
    assert alive() is None


@pytest.mark.gpu
def test_views_outlive_a_dropped_instance():
    index, k, v, qs = case()
    attn = SeoulKV4(device="cuda:0", k=k, v=v, index=index,
                    config=SeoulKV4Config(stage15_capacity=None))
    result = attn.run(qs[0])
    want = result.to_torch().reshape(4, 4, 256)
    views = result.device_tensors
    runtime = weakref.ref(attn._state)
    del attn, result
    gc.collect()
    assert runtime() is not None  # checked before the views are read
    for g in range(4):
        got = torch.stack([views[g][0, h, h] for h in range(4)]).cpu()
        assert torch.equal(got, want[g])
    del views
    gc.collect()
    assert runtime() is None
