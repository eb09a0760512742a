"""The native window loop (htrc_windows_i8 / _16 / _f32, what flat_attention runs without checks) against the
stage-by-stage loop of the same call (what it runs when ``state`` collects the stages): the same launches in the same
order per window, so the same bits, for one and several windows over one to three streams.
"""
from __future__ import annotations

import pytest
import torch

from htrc_amd import htrc_flat, htrc_flat_hip as hip, htrc_flat_runner, workloads

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


@pytest.mark.parametrize("heads,n,order,group,ws", [(2, 17000, "seq", 1, True), (2, 17000, "kmeans", 1, False),
                                                     (3, 11000, "seq", 2, True), (3, 11000, "kmeans", 2, False)])
def test_segmented_layers_of_several_heads(device, heads, n, order, group, ws):
    """Layers of 532 and 516 (head, tile) pairs of 129 key blocks: one window (the segments in turn), small windows (as workgroups
    of their own, the last one shorter) and windows of more than 384 pairs before a short one (both forms
    in one call): the same bits from every one, natively and stage by stage."""
    q, k, v = (x.to(device) for x in workloads.clustered_runs(n=n, runs=-(-n // 64), heads=heads, seed=heads))
    k, v = k[:, :4128].contiguous(), v[:, :4128].contiguous()
    nt = -(-n // 64)
    assert 512 < heads * nt <= 1024 and htrc_flat_runner.route_segments(heads * nt, heads * 60, 258, 240, 16) == 4
    kw = dict(backend="hip", store="int8", dot="bf16", leaf=16, exact_leaves=240, order=order, kern={"group": group},
              return_logz=True)
    want = [x.clone() for x in htrc_flat.flat_attention(q, k, v, tile_chunk=None, **kw)]
    space = {} if ws else None
    for chunk in (400 // heads, 60):
        staged = htrc_flat.flat_attention(q, k, v, tile_chunk=chunk, state={}, **kw)
        native = htrc_flat.flat_attention(q, k, v, tile_chunk=chunk, ws=space, **kw)
        torch.cuda.synchronize()
        for got in (staged, native):
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), chunk


@pytest.mark.parametrize("kw", [dict(store="int8", dot="bf16"), dict(store="fp32", dot="tf32")])
def test_host_values_are_refused(device, kw):
    q, k, v = workloads.clustered_runs(n=256, runs=4, heads=1, seed=1)
    with pytest.raises(ValueError):
        htrc_flat.flat_attention(q.to(device), k.to(device), v, backend="hip", leaf=32, exact_leaves=2, tile_chunk=2, **kw)


@pytest.mark.parametrize("d", [1, 3, 32, 64, 80, 127])
@pytest.mark.parametrize("kinds", [("bf16", "bf16", "bf16"), ("fp32", "fp32", "bf16"), ("fp32", "bf16", "fp32")])
def test_pad_dims_equals_torch(device, d, kinds):
    """One launch for q, k, v: the rows' values (fp32 keys rounded to bf16 as torch rounds them, infinities and NaN kept),
    zeros past d in a buffer that held other values."""
    dt = {"bf16": torch.bfloat16, "fp32": torch.float32}
    g = torch.Generator().manual_seed(d)
    xs = [(torch.randn((2, n, d), generator=g) * 3).to(dt[k]).to(device) for n, k in zip((7, 33, 33), kinds)]
    xs[1][0, 0, 0], xs[1][0, 1, 0], xs[2][1, 2, d - 1] = float("inf"), float("nan"), -float("inf")
    outs_dt = (xs[0].dtype, torch.bfloat16, torch.bfloat16)
    ws = {n: torch.full((2, x.shape[1], 128), 9.0, device=device, dtype=t) for n, x, t in zip("abc", xs, outs_dt)}
    outs = hip.pad_dims(xs, ws, tuple("abc"), outs_dt)
    for x, o, t in zip(xs, outs, outs_dt):
        assert torch.equal(o[..., :d].nan_to_num(123.0), x.to(t).nan_to_num(123.0))
        assert bool((o[..., d:] == 0).all())


@pytest.mark.parametrize("d", [1, 31, 64, 96, 127])
@pytest.mark.parametrize("kinds", [("bf16", "bf16"), ("fp32", "bf16"), ("fp32", "fp32"), ("bf16", "fp32")])
def test_pad_dims_of_rows_off_a_16_byte_boundary(device, d, kinds):
    """1 to 1500 rows (whole workgroups of 32 and a remainder) that start 0, 4, 8 and 12 bytes past such a boundary."""
    dt = {"bf16": torch.bfloat16, "fp32": torch.float32}
    src, dst = (dt[k] for k in kinds)
    for rows in (1, 32, 33, 1500):
        for off in (0, 4, 8, 12):
            raw = torch.randn((rows * d + 8,), device=device).to(src)
            x = raw[off // raw.element_size():][:rows * d].view(1, rows, d)
            assert x.data_ptr() % 16 == off
            (o,) = hip.pad_dims((x,), {"a": torch.full((1, rows, 128), 9.0, device=device, dtype=dst)}, ("a",), (dst,))
            assert torch.equal(o[..., :d], x.to(dst)) and bool((o[..., d:] == 0).all())


def test_odd_address_keys_take_the_copying_path(device):
    """Rows of 31 bf16 values at an address that is not a multiple of four: the same result."""
    q, k, v = (x[..., :31].contiguous().to(device) for x in workloads.clustered_runs(n=256, runs=4, heads=1, seed=2))
    kw = dict(store="int8", dot="bf16", backend="hip", leaf=32, exact_leaves=2)
    want = htrc_flat.flat_attention(q, k, v, **kw).clone()
    raw = torch.empty((k.numel() + 1,), dtype=torch.bfloat16, device=device)
    k2 = raw[1:].view(k.shape)
    k2.copy_(k)
    assert k2.data_ptr() % 4 == 2 and hip.pad_dims((k2,), None, ("a",), (torch.bfloat16,)) is None
    assert torch.equal(htrc_flat.flat_attention(q, k2, v, **kw), want)
