"""The native window loop (htrc_windows_i8 / _16 / _f32, what flat_attention runs without checks) against the
stage-by-stage loop of the same call (what it runs when ``state`` collects the stages): the same launches in the same
order per window, so the same bits, for one and several windows over one to three streams.
"""
from __future__ import annotations

import pytest
import torch

from htrc_amd import htrc_flat, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(store="int8", dot="bf16"), dict(store="fp8", dot="bf16"), dict(store="bf16", dot="bf16"),
                                dict(store="int8", dot="bf16", precision="tf32", exact_leaves=0),
                                dict(store="fp32", dot="tf32"), dict(store="bf16", dot="tf32", precision="tf32", splits=3),
                                dict(store="fp32", dot="tf32", splits=1)])
@pytest.mark.parametrize("chunk,streams,group,ws", [(None, 2, 1, True), (4, 2, 1, False), (4, 1, 2, True), (3, 3, 1, True)])
def test_native_windows_equal_the_stage_loop(device, kw, chunk, streams, group, ws):
    q, k, v = (x.to(device) for x in workloads.clustered_runs(n=1130, runs=18, heads=2, seed=5))
    k, v = k[:, :1088].contiguous(), v[:, :1088].contiguous()
    kw = {"leaf": 32, "exact_leaves": 6, **kw, "backend": "hip", "tile_chunk": chunk, "sink_leaves": 1,
          "kern": {"window_streams": streams, "group": group}, "return_logz": True}
    want = [x.clone() for x in htrc_flat.flat_attention(q, k, v, state={}, **kw)]
    space = {} if ws else None
    for _ in range(2):                                  # the workspace's first and a later call
        got = htrc_flat.flat_attention(q, k, v, ws=space, **kw)
        torch.cuda.synchronize()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("kw", [dict(store="int8", dot="bf16"), dict(store="fp32", dot="tf32")])
def test_host_values_are_refused(device, kw):
    q, k, v = workloads.clustered_runs(n=256, runs=4, heads=1, seed=1)
    with pytest.raises(ValueError):
        htrc_flat.flat_attention(q.to(device), k.to(device), v, backend="hip", leaf=32, exact_leaves=2, tile_chunk=2, **kw)
