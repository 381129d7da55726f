"""The dense decode at the edges of its tiles, pairs and block shares.

Contexts around one key, one 16-key tile, one 32-key pair, one pair per block
(64 blocks per KV head) and one pass of a block's 12 waves (12 x 64 pairs),
in a record buffer whose rows past the context hold NaN records (a key read
past the end poisons the output), against a float64 softmax over the same FP8
records.  Tolerance as in ``test_gpu_dense.py``: the output is a BF16 rounding
(half an ulp <= 2^-8 relative) of FP32 sums; the sums of up to 25000 exact
products of probabilities that add up to 1 and |v| < 8 are within
8 x 25000 x 2^-24 = 1.2e-2 in the worst order and within 8 x sqrt(25000) x
2^-24 < 1e-4 for rounding errors that do not line up.  The logits add a term
that grows with the query: a matrix core sums the 128 FP8 products of a step
aligned to the largest, so a logit is good to about 2^-20 of the sum of its
products' magnitudes (2^-19 is allowed), S = sum |q k| / 16, and a logit error
of d moves an output by at most 2 d max |v|.
"""

from __future__ import annotations

import pytest
import torch

from seoulkv_amd import _hip

pytestmark = pytest.mark.gpu

PAIR, BLOCKS, WAVES = 32, 64, 12


def _records(context, spare, seed, spread):
    gen = torch.Generator("cuda").manual_seed(seed)
    kv8 = torch.full((4, context + spare, 512), 0x7f, dtype=torch.uint8, device="cuda")
    x = torch.randn(4, context, 512, generator=gen, device="cuda")
    kv8[:, :context] = x.to(torch.float8_e4m3fn).view(torch.uint8)
    q = (spread * torch.randn(16, 256, generator=gen, device="cuda")).bfloat16()
    return kv8, q


def _tolerance(kv8, context, q, ref):
    both = kv8[:, :context].view(torch.float8_e4m3fn).float().abs()
    x = q.float().abs().reshape(4, 4, 256)
    s = max(float((x[g] @ both[g, :, 256:].T.contiguous()).max()) / 16 for g in range(4))
    return ref.abs() * 2.0**-8 + 1e-4 + 2 * 2.0**-19 * s * float(both[..., :256].max())


def _reference(kv8, context, q):
    both = kv8[:, :context].view(torch.float8_e4m3fn).double()
    k, v = both[..., 256:], both[..., :256]
    x = q.double().reshape(4, 4, 256)
    out = []
    for g in range(4):
        p = torch.softmax(x[g] @ k[g].T.contiguous() / 16, -1)
        out.append(p @ v[g].contiguous())
    return torch.cat(out)


@pytest.mark.parametrize("spread", [0.05, 1.0, 30.0])  # near-uniform .. one key takes all
@pytest.mark.parametrize("context", [
    1, 15, 16, 17, 31, 32, 33, 63,
    BLOCKS * PAIR - 1, BLOCKS * PAIR, BLOCKS * PAIR + 1, BLOCKS * PAIR + 17,
    WAVES * BLOCKS * PAIR - 16, WAVES * BLOCKS * PAIR + 33])
def test_dense_decode_at_tile_edges(context, spread):
    print(f"[gpu] dense tiles context {context} spread {spread}", flush=True)
    kv8, q = _records(context, 5, context, spread)
    out = torch.empty_like(q)
    _hip.dense_decode_static(kv8, context, q, out)
    got, ref = out.double(), _reference(kv8, context, q)
    assert torch.isfinite(got).all()
    err = (got - ref).abs()
    assert not (err > _tolerance(kv8, context, q, ref)).any(), float(err.max())


def test_dense_decode_propagates_a_nan_value_and_ignores_masked_rows():
    """A NaN V element reaches its dimension's outputs of its KV head only; a
    NaN key reaches every output of its KV head."""
    kv8, q = _records(1000, 5, 3, 1.0)
    ref = _reference(kv8, 1000, q)
    tol = _tolerance(kv8, 1000, q, ref)
    kv8[1, 700, 37] = 0x7f
    kv8[2, 999, 256] = 0xff
    out = torch.empty_like(q)
    _hip.dense_decode_static(kv8, 1000, q, out)
    bad = torch.isnan(out).reshape(4, 4, 256)
    want = torch.zeros_like(bad)
    want[1, :, 37] = True
    want[2] = True
    assert torch.equal(bad, want)
    fine = ~want.reshape(16, 256)
    assert not ((out.double() - ref).abs() > tol)[fine].any()
