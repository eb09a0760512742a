"""Long tiles of the fused int8 route (more than 128 blocks of 32 keys): the segments of a tile run as
workgroups of their own, run in turn by one workgroup (no partial-sum workspace) and the whole-tile
kernel of htrc_route on the same state.  The first two add the same sums in the same order: bit for
bit.  Against the whole tile only the grouping of the fp32 sums differs: at most keys roundings of
2^-24 each, measured 1e-6.
"""
from __future__ import annotations

import math

import pytest
import torch

from htrc_amd import htrc_flat_hip as hip, htrc_flat_runner, workloads
from htrc_amd._lib import call, ptr, stream_handle

pytestmark = pytest.mark.gpu


def _route(device, n, m, leaf, kx, tile, heads, group, spike):
    q, k, v = workloads.clustered_runs(n=max(n, m), runs=-(-max(n, m) // 64), heads=heads, seed=leaf + tile)
    q, k, v = q[:, :n].clone(), k[:, :m].contiguous(), v[:, :m].contiguous().to(device)
    if spike:                             # key 3 (leaf 0, always near) far above row 5's far-field maximum
        q, k = (q.float() * 0.3).to(torch.bfloat16), (k.float() * 0.3).to(torch.bfloat16)
        q[:, 5], k[:, 3] = 0, 0
        q[:, 5, 0], k[:, 3, 0] = 64, 64
    q, k = q.to(device), k.to(device)
    mu, q8, sq, dq8, sdq = hip.pack_q(q, tile=tile, group=group)
    k8, ks = hip.pack_k(k)
    nb, nt, scale = m // leaf, -(-n // tile), 1 / math.sqrt(128)
    g8, lz, vb, sg, _ = hip.leaf_stats(mu, k, v, nb, scale, leaf=leaf)
    ng = int(mu.shape[1])
    kxe = min(kx, nb)
    segs = hip.library().htrc_route_segments(heads, n, m, leaf, kx, tile, group, 0, ng)
    assert segs == htrc_flat_runner.route_segments(heads * nt, nb, kxe, leaf)
    outs = []
    for entry, parts in (("htrc_route_seg", True), ("htrc_route_seg", False), ("htrc_route", None)):
        out, lzr = torch.full((heads, n, 128), 7.0, device=device), torch.full((heads, n), 7.0, device=device)
        idx = torch.empty((heads, ng, kxe), dtype=torch.int32, device=device)
        rowmax = torch.empty((heads, nt * tile), device=device)
        buf = torch.empty((heads * nt * segs * tile * 129,), device=device) if parts and segs > 1 else None
        extra = () if parts is None else (ptr(buf),)
        call(entry, *[ptr(t) for t in (q8, sq, dq8, sdq, g8, sg, lz, vb, k8, ks, v)], heads, n, m, leaf, 128, kx,
             int(spike), 1, tile, group, 0, ng, None, scale, ptr(out), ptr(lzr), ptr(idx), ptr(rowmax), None, *extra,
             stream_handle(device))
        outs.append((out, lzr))
    torch.cuda.synchronize()
    return segs, outs


@pytest.mark.parametrize("n,m,leaf,kx,tile,heads,group,spike,segs", [
    (200, 4128, 16, 240, 64, 1, 1, False, 4),       # 9 + 120 blocks: the shortest segmented tile
    (200, 4112, 16, 239, 64, 1, 1, False, 4),       # 9 + 119.5 blocks: a half-empty last block
    (193, 2048, 16, 128, 64, 1, 1, False, 1),       # 4 + 64 blocks: whole tiles
    (200, 4128, 32, 129, 32, 2, 1, False, 4),       # 5 + 129 blocks, 32-row tiles
    (1000, 40752, 16, 256, 64, 1, 2, False, 4),     # 80 + 128 blocks, shared centres
    (130, 33024, 128, 100, 64, 1, 1, False, 4),     # 9 + 400 blocks, a partial last tile
    (4160, 8192, 64, 66, 32, 4, 1, False, 1),       # 4 + 132 blocks, 520 tiles: in turn, no workspace
    (500, 8192, 16, 300, 64, 1, 1, True, 4),        # a row whose reference misses: the tile is redone
    (500, 8192, 64, 64, 32, 1, 1, True, 4)])
def test_segmented_route(device, n, m, leaf, kx, tile, heads, group, spike, segs):
    got, ((o1, z1), (o2, z2), (o3, z3)) = _route(device, n, m, leaf, kx, tile, heads, group, spike)
    assert got == segs
    assert torch.equal(o1, o2) and torch.equal(z1, z2)
    assert bool(torch.isfinite(o1).all()) and bool(torch.isfinite(z1).all())
    assert float((o1 - o3).norm() / o3.norm()) <= 1e-5
    assert float(((z1 - z3).abs() / z3.abs().clamp_min(1.0)).max()) <= 1e-5
