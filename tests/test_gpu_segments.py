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


def _route(device, n, m, leaf, kx, tile, group, g0, gn, spike):
    """The window [g0, g0 + gn) of tile groups of one head through the three forms -> (segments, outputs of its rows)."""
    q, k, v = workloads.clustered_runs(n=max(n, m), runs=-(-max(n, m) // 64), heads=1, seed=leaf + tile)
    q, k, v = q[:, :n].clone(), k[:, :m].contiguous(), v[:, :m].contiguous().to(device)
    if spike:                             # key 3 (leaf 0, always near) far above row 5's far-field maximum
        q, k = (q.float() * 0.3).to(torch.bfloat16), (k.float() * 0.3).to(torch.bfloat16)
        q[:, 5], k[:, 3] = 0, 0
        q[:, 5, 0], k[:, 3, 0] = 64, 64
    q, k = q.to(device), k.to(device)
    mu, q8, sq, dq8, sdq = hip.pack_q(q, tile=tile, group=group)
    k8, ks = hip.pack_k(k)
    nb, nt, scale = m // leaf, -(-n // tile), 1 / math.sqrt(128)
    units = min(nt, (g0 + gn) * group) - g0 * group
    rows = slice(g0 * group * tile, min(n, (g0 * group + units) * tile))
    g8, lz, vb, sg, _ = hip.leaf_stats(mu, k, v, nb, scale, leaf=leaf, c0=g0, cn=gn)
    kxe = min(kx, nb)
    segs = hip.library().htrc_route_segments(1, n, m, leaf, kx, tile, group, g0, gn)
    assert segs == htrc_flat_runner.route_segments(nt, units, nb, kxe, leaf)
    outs = []
    for entry, parts in (("htrc_route_seg", True), ("htrc_route_seg", False), ("htrc_route", None)):
        out, lzr = torch.full((1, n, 128), 7.0, device=device), torch.full((1, n), 7.0, device=device)
        idx = torch.empty((1, gn, kxe), dtype=torch.int32, device=device)
        rowmax = torch.empty((1, nt * tile), device=device)
        buf = torch.empty((units * segs * tile * 129,), device=device) if parts and segs > 1 else None
        extra = () if parts is None else (ptr(buf),)
        call(entry, *[ptr(t) for t in (q8, sq, dq8, sdq, g8, sg, lz, vb, k8, ks, v)], 1, n, m, leaf, 128, kx,
             int(spike), 1, tile, group, g0, gn, None, scale, ptr(out), ptr(lzr), ptr(idx), ptr(rowmax), None, *extra,
             stream_handle(device))
        outs.append((out[0, rows], lzr[0, rows]))
        # no other row is written
        assert bool((out[0, : rows.start] == 7).all()) and bool((out[0, rows.stop:] == 7).all())
    torch.cuda.synchronize()
    return segs, outs


@pytest.mark.parametrize("n,m,leaf,kx,tile,group,g0,gn,spike,segs", [
    (33000, 4128, 16, 240, 64, 1, 513, 3, False, 4),    # 9 + 120 blocks: the shortest segmented tile; a partial last tile
    (33000, 4112, 16, 239, 64, 1, 0, 4, False, 4),      # 9 + 119.5 blocks: a half-empty last block
    (33000, 2048, 16, 128, 64, 1, 0, 3, False, 1),      # 4 + 64 blocks: whole tiles
    (32768, 4128, 16, 240, 64, 1, 0, 3, False, 1),      # 512 tiles in the layer: whole tiles
    (65600, 4128, 16, 240, 64, 1, 0, 3, False, 1),      # 1025 tiles
    (65536, 4128, 16, 240, 64, 1, 0, 3, False, 4),      # 1024 tiles
    (17000, 4128, 32, 129, 32, 1, 5, 6, False, 4),      # 5 + 129 blocks, 32-row tiles
    (33000, 40752, 16, 256, 64, 2, 100, 8, False, 4),   # 80 + 128 blocks, shared centres
    (33000, 33024, 128, 100, 64, 1, 0, 3, False, 4),    # 9 + 400 blocks
    (33000, 8192, 64, 66, 64, 1, 0, 384, False, 4),     # the largest launch that runs segments apart
    (33000, 8192, 64, 66, 64, 1, 0, 385, False, 1),     # in turn, no workspace
    (33000, 16128, 64, 124, 64, 1, 0, 512, False, 4),   # 8 + 248 = 256 blocks: two tiles a CU apart
    (33000, 16128, 64, 124, 64, 1, 0, 513, False, 1),
    (33000, 16128, 64, 123, 64, 1, 0, 385, False, 1),   # 254 blocks
    (33000, 8192, 16, 300, 64, 1, 0, 8, True, 4),       # a row whose reference misses: the tile is redone
    (17000, 8192, 64, 64, 32, 1, 0, 8, True, 4)])
def test_segmented_route(device, n, m, leaf, kx, tile, group, g0, gn, spike, segs):
    got, ((o1, z1), (o2, z2), (o3, z3)) = _route(device, n, m, leaf, kx, tile, group, g0, gn, spike)
    assert got == segs
    assert torch.equal(o1, o2) and torch.equal(z1, z2)
    assert bool(torch.isfinite(o1).all()) and bool(torch.isfinite(z1).all())
    assert float((o1 - o3).norm() / o3.norm()) <= 1e-5
    assert float(((z1 - z3).abs() / z3.abs().clamp_min(1.0)).max()) <= 1e-5


@pytest.mark.parametrize("groups,nb,kx,sink,group", [
    (300, 1008, 64, 0, 1), (40, 2547, 256, 0, 1), (40, 2547, 476, 220, 1), (300, 300, 128, 3, 1), (40, 130, 129, 0, 2),
    (300, 1500, 49, 0, 1), (300, 1500, 48, 0, 1),
    (600, 500, 57, 0, 1), (600, 1008, 56, 0, 1), (3, 12000, 100, 0, 1), (3, 11264, 129, 0, 1), (20, 257, 128, 0, 1),
    (20, 66, 60, 0, 1),
    (128, 2100, 64, 0, 1), (129, 2100, 64, 0, 1), (256, 2100, 49, 3, 1), (257, 2100, 64, 0, 1), (256, 1024, 48, 0, 1),
    (256, 1023, 64, 0, 1), (200, 1500, 49, 0, 1)])
@pytest.mark.parametrize("ties", [False, True])
def test_route_select_wave_counts(device, groups, nb, kx, sink, group, ties):
    """route_select's launches of 4, 8 and 16 waves per tile group (more than 256, 129 to 256, fewer groups; heads of
    fewer than 1024 and 2048 leaves, and those whose keys leave no room for 16 rings), and its top-k at and beside
    each bound of its methods: index sets equal to the stage select and top-k on the same state, row maxima to the
    largest of the row's scores in 64 bits (four roundings of 2^-24 of at most 127^2 * 128 * 1e-4 + 5 here: 5e-5)."""
    torch.manual_seed(nb + kx)
    nbp, nt = -(-nb // 32) * 32, groups * group
    dq8 = torch.randint(-127, 128, (1, nt * 64, 128), device=device, dtype=torch.int8)
    sdq = torch.rand((1, nt * 64), device=device) * 1e-4
    g8 = torch.randint(-127, 128, (1, groups, nbp, 128), device=device, dtype=torch.int8)
    sg, lz = torch.rand((1, groups, nbp), device=device), torch.randn((1, groups, nbp), device=device)
    if ties:
        g8.zero_()
        lz = torch.round(lz)
    sg[..., nb:], lz[..., nb:] = 0, -math.inf
    g8[..., nb:, :] = 0
    packed = {"dq8": dq8, "sdq": sdq, "k8": torch.empty((1, nb * 16, 128), device=device, dtype=torch.int8)}
    state = {"g8": g8, "sg": sg, "lz": lz}
    idx, rowmax = hip.route_select(packed, state, nq=nt * 64, leaf=16, kx=kx, sink=sink, group=group)
    sel = hip.rowmax_select(g=g8, lz=lz, sg=sg, nb=nb, dq8=dq8, sdq=sdq, group=group)
    want, _ = hip.topk_excl(sel, nb, kx, sink)
    assert torch.equal(idx, want)
    rows, step = 64 * group, max(1, 1 << 22 >> nbp.bit_length())
    q64, s64, m64 = dq8.view(groups, rows, 128).double(), sdq.view(groups, rows, 1).double(), rowmax.view(groups, rows)
    for g in range(0, groups, max(1, step // rows)):
        e = min(groups, g + max(1, step // rows))
        dots = torch.bmm(q64[g:e], g8[0, g:e, :nb].double().transpose(1, 2).contiguous())
        best = (dots * s64[g:e] * sg[0, g:e, None, :nb].double() + lz[0, g:e, None, :nb].double()).amax(2)
        assert float((best - m64[g:e]).abs().max()) <= 5e-5
    # the same groups inside a window: the launch's first groups alone
    few = min(groups, 2)
    part = {k: x[:, :few].contiguous() for k, x in state.items()}
    idx2, rowmax2 = hip.route_select(packed, part, nq=nt * 64, leaf=16, kx=kx, sink=sink, group=group)
    rows = few * group * 64
    assert torch.equal(idx2, idx[:, :few]) and torch.equal(rowmax2[:, :rows], rowmax[:, :rows])
