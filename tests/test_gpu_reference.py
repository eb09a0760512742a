"""The fused routes' fixed softmax reference: a key whose exact score lies far above its row's far-field maximum,
from well inside the range of row totals to past it (the tile is then redone), with values small
enough and too large for the outputs at such a total, against the oracle at the operator's tolerance.
"""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from helpers import bits, rel_l2
from htrc_amd import htrc_flat, workloads
from oracle import flat_i8

pytestmark = pytest.mark.gpu
OUT_REL_L2 = 1e-2
LOGZ_ABS = 1e-3


@pytest.mark.parametrize("store,heads", [("int8", 1), ("int8", 8), ("bf16", 1), ("fp8", 1)])
@pytest.mark.parametrize("mag,vexp", [(20, 0), (27, 0), (32, 0), (34, 0), (27, 60), (32, 90)])
def test_scores_far_above_the_reference(device, store, heads, mag, vexp):
    """mag^2 / sqrt(128) nats above zero: 51, 93, 131 and 147 octaves, on both sides of the range's end."""
    if store == "fp8" and vexp:
        pytest.skip("the fp8 state's fp16 weights do not hold such value scales")
    n, leaf, ex, row = 1024, 64, 4, 5
    q, k, v = workloads.clustered_runs(n=n * 4, runs=n // 16, heads=heads, seed=17)
    q, k = ((x.float() * 0.3).to(torch.bfloat16) for x in (q, k))
    v = (v.float() * 2.0 ** vexp).to(torch.bfloat16)
    q[:, row], k[:, 3] = 0, 0
    q[:, row, 0], k[:, 3, 0] = mag, mag
    out, logz = htrc_flat.flat_attention(q.to(device), k.to(device), v.to(device), backend="hip", store=store, dot="bf16",
                                         leaf=leaf, exact_leaves=ex, tile_chunk=None, sink_leaves=1, return_logz=True)
    torch.cuda.synchronize()
    h = heads - 1
    ref = flat_i8.flat_i8(bits(q[h, :64]), bits(k[h]), bits(v[h]), tile=64, leaf=leaf, exact_leaves=ex, sink_leaves=1,
                          splits=1, bn=64, store=store)
    assert ref["logz"][row] > 0.9 * mag * mag / math.sqrt(128)
    s = 2.0 ** -vexp
    assert rel_l2(out[h, :64].cpu().numpy() * s, np.asarray(ref["out"]) * s) <= OUT_REL_L2
    assert np.abs(logz[h, :64].cpu().numpy() - ref["logz"]).max() <= LOGZ_ABS


@pytest.mark.parametrize("heads,n,m,sink,far,chunk", [
    (1, 4096, 4096, 8, 7, None),      # four key parts: the two keys in the first and the last
    (6, 4096, 4096, 8, 7, None),      # two key parts
    (8, 4096, 4096, 8, 7, None),      # one key part
    (1, 33000, 8192, 66, 40, None),   # four segments in turn: the two keys in the first and the third
    (1, 33000, 8192, 66, 40, 128)])   # the segments as workgroups of their own
def test_sums_over_parts_that_overflow(device, heads, n, m, sink, far, chunk):
    """Two near keys of one weight (121 octaves) in different parts of the tile's key stream, their value 1.5 * 2^e: at one
    e of the sweep each part's output is finite and their sum is not.  Their common value is the
    row's output (every other weight is below 2^-90 of theirs), up to the weights' bf16 rounding."""
    leaf, row, mag = 64, 5, 30.75
    q, k, v = (x.to(device) for x in workloads.clustered_runs(n=max(n, m), runs=max(n, m) // 64, heads=heads, seed=19))
    q, k = ((x.float() * 0.3).to(torch.bfloat16) for x in (q[:, :n], k[:, :m]))
    v = v[:, :m].contiguous()
    keys = [3, far * leaf + 3]
    q[:, row], k[:, keys] = 0, 0
    q[..., 0], k[..., 0] = 0, 0           # dim 0 is theirs alone: no other row's centre or leaf mean points at them
    q[:, row, 0] = mag
    k[:, keys, 0] = mag
    ws = {}
    for e in range(72):
        v[:, keys] = 1.5 * 2.0 ** e
        out, logz = htrc_flat.flat_attention(q, k, v, backend="hip", store="int8", dot="bf16", leaf=leaf, exact_leaves=0,
                                             sink_leaves=sink, tile_chunk=chunk, ws=ws, return_logz=True)
        finite = bool(torch.isfinite(out).all()) and bool(torch.isfinite(logz).all())
        assert finite, e
        assert float((out[:, row] * (2.0 ** -e / 1.5) - 1).abs().max()) <= 1e-2, e


@pytest.mark.parametrize("store,heads", [("int8", 1), ("int8", 6), ("int8", 8), ("bf16", 1)])
@pytest.mark.parametrize("vexp", [-60, -90, -100, -110])
def test_small_values(device, store, heads, vexp):
    """Values scaled by a power of two scale the outputs by it, in every dim or in half of them: a row's weights lie near
    1 or above, so outputs of 2^-110 are sums whose roundings, 2^-150 each where they fall below the normal range,
    are 4096 keys * 2^-40 of them at most.  (The statistics' own roundings move by 4e-7 under the scale.)"""
    n, leaf, ex = 4096, 64, 4
    q, k, v = (x.to(device) for x in workloads.clustered_runs(n=n, runs=n // 64, heads=heads, seed=23))
    kw = dict(backend="hip", store=store, dot="bf16", leaf=leaf, exact_leaves=ex, tile_chunk=None)
    want = htrc_flat.flat_attention(q, k, v, **kw)
    s = 2.0 ** vexp
    for dims in (slice(0, 128), slice(64, 128)):
        small = v.clone()
        small[..., dims] *= s
        got = htrc_flat.flat_attention(q, k, small, **kw)
        rel = rel_l2((got[..., dims] / s).cpu().numpy(), want[..., dims].cpu().numpy())
        assert rel <= 2e-6, (dims, rel)


@pytest.mark.parametrize("store,heads,n,m,leaf,near,chunk", [
    ("int8", 1, 4096, 4096, 64, 8, None), ("int8", 6, 4096, 4096, 64, 8, None), ("int8", 8, 4096, 4096, 64, 8, None),
    ("bf16", 2, 4096, 4096, 64, 8, None), ("fp8", 2, 4096, 4096, 64, 8, None),
    ("int8", 1, 33000, 8192, 64, 66, None), ("int8", 1, 33000, 8192, 64, 66, 128)])     # segments in turn, apart
def test_a_value_that_is_not_finite_stays_in_its_dim(device, store, heads, n, m, leaf, near, chunk):
    """A NaN among the values makes its dim NaN and leaves the others' bits: tiles within the ordinary range of totals
    are not redone (at another reference) for it."""
    q, k, v = (x.to(device) for x in workloads.clustered_runs(n=max(n, m), runs=-(-max(n, m) // 64), heads=heads, seed=29))
    q, k, v = q[:, :n].contiguous(), k[:, :m].contiguous(), v[:, :m].contiguous()
    kw = dict(backend="hip", store=store, dot="bf16", leaf=leaf, exact_leaves=near, tile_chunk=chunk)
    want = htrc_flat.flat_attention(q, k, v, **kw)
    v[:, 100, 7] = float("nan")
    got = htrc_flat.flat_attention(q, k, v, **kw)
    dims = [i for i in range(128) if i != 7]
    assert bool(torch.isnan(got[..., 7]).all())
    assert torch.equal(got[..., dims], want[..., dims])
