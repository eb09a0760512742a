"""The order in which a call of several tile windows allocates, waits, launches and drops its buffers, on the host: streams and
launches are stand-ins that write down what happens, tensors live in host memory.  The window buffers are used on the
side streams and may belong to the caller's stream, which other threads may share.  So a side stream has to wait for
the caller's stream after the last of its buffers is allocated (the block may be one that another thread freed while
its kernels still run), and the caller's stream for the side streams before the first is dropped (the next owner's
kernels wait for the caller's stream alone).
"""
from __future__ import annotations

import contextlib
import weakref

import pytest
import torch

from htrc_amd import htrc_flat, htrc_flat_hip as hip

WINDOW = {"mu_terms", "g", "g_fp8", "g_bf16", "g_f32", "vb", "vb_fp8", "vb_f32", "lz", "sg", "sv", "idx", "sel", "excl", "pm",
          "pl", "pacc", "parts", "route_keys"}


class _Stream:
    def __init__(self, name, events):
        self.name, self.events, self.cuda_stream = name, events, 64 + len(name)

    def wait_stream(self, other):
        self.events.append(("wait", self.name, other.name))


@pytest.fixture
def events(monkeypatch):
    log = []
    cur, side = _Stream("cur", log), tuple(_Stream(f"side{i}", log) for i in range(3))
    buf = hip._buf

    owner = ["cur"]

    @contextlib.contextmanager
    def on(stream):
        before, owner[0] = owner[0], stream.name
        yield
        owner[0] = before

    def traced(ws, name, shape, dtype, device):
        held = ws is not None and name in ws
        t = buf(ws, name, shape, dtype, device)
        if name in WINDOW and not held:
            log.append(("alloc", name, owner[0]))
            weakref.finalize(t, log.append, ("drop", name))
        return t

    def launch(name, *args):
        log.append(("call", name))
        if name.startswith("htrc_windows") and "fail" in log:
            raise ValueError("refused")

    monkeypatch.setattr(hip, "_buf", traced)
    monkeypatch.setattr(hip, "_need", lambda *a: None)
    monkeypatch.setattr(hip, "call", launch)
    monkeypatch.setattr(hip, "stream_handle", lambda *a: 0)
    monkeypatch.setattr(hip, "_cus", lambda dev: 256)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: cur)
    monkeypatch.setattr(torch.cuda, "stream", on)
    monkeypatch.setattr(torch.cuda, "device", lambda *a: contextlib.nullcontext())
    monkeypatch.setattr(htrc_flat, "_window_streams", lambda dev, n: side[:n])
    return log


@pytest.mark.parametrize("kw", [dict(store="int8", dot="bf16"), dict(store="fp8", dot="bf16"), dict(store="bf16", dot="bf16"),
                                dict(store="fp32", dot="tf32"), dict(store="bf16", dot="tf32", splits=3)])
@pytest.mark.parametrize("streams,ws,refused", [(2, False, False), (3, False, False), (2, True, False), (2, False, True)])
def test_side_streams_are_ordered_around_the_buffers(events, kw, streams, ws, refused):
    q, k, v = (torch.zeros((2, n, 128), dtype=torch.bfloat16) for n in (700, 512, 512))
    if refused:
        events.append("fail")
    space = {} if ws else None
    with pytest.raises(ValueError) if refused else contextlib.nullcontext():
        htrc_flat.flat_attention(q, k, v, backend="hip", leaf=32, exact_leaves=4, tile_chunk=2, ws=space,
                                 kern={"window_streams": streams}, **kw)
    at = next(i for i, e in enumerate(events) if e[0] == "call" and e[1].startswith("htrc_windows"))
    allocs = [i for i, e in enumerate(events) if e[0] == "alloc"]
    drops = [i for i, e in enumerate(events) if e[0] == "drop"]
    assert allocs and max(allocs) < at
    for s in range(streams):
        forks = [i for i, e in enumerate(events) if e == ("wait", f"side{s}", "cur")]
        joins = [i for i, e in enumerate(events) if e == ("wait", "cur", f"side{s}")]
        assert [i for i in forks if max(allocs) < i < at], "a side stream does not wait for its buffers' stream"
        assert joins and at < max(joins)
        assert all(i > max(joins) for i in drops), "a buffer is dropped before the streams are joined"
    assert ws or refused or len(drops) == len(allocs)
    # a new workspace's blocks are the side streams', so that the next one, of whatever stream, takes them up again
    assert {e[2] for e in events if e[0] == "alloc"} == ({f"side{s}" for s in range(streams)} if ws else {"cur"})
    if ws:                                # a kept one allocates nothing
        del events[:]
        htrc_flat.flat_attention(q, k, v, backend="hip", leaf=32, exact_leaves=4, tile_chunk=2, ws=space,
                                 kern={"window_streams": streams}, **kw)
        assert not [e for e in events if e[0] == "alloc"]


@pytest.mark.parametrize("store,chunk", [("int8", 2), ("int8", None), ("fp8", 2), ("bf16", None)])
def test_fused_routes_do_not_look_at_the_split_knobs(events, store, chunk):
    q, k, v = (torch.zeros((n, 128), dtype=torch.bfloat16) for n in (300, 256, 256))
    htrc_flat.flat_attention(q, k, v, backend="hip", store=store, dot="bf16", leaf=32, exact_leaves=2, tile_chunk=chunk,
                             splits=None, kern={"tile_bn": None})
    assert [e for e in events if e[0] == "call" and e[1].startswith("htrc_windows")]


def test_unsplit_windows_do_not_look_at_splits(events):
    q, k = torch.zeros((2, 65536, 128), dtype=torch.bfloat16), torch.zeros((2, 512, 128), dtype=torch.bfloat16)
    htrc_flat.flat_attention(q, k, k, backend="hip", leaf=128, exact_leaves=1, tile_chunk=None, splits=None)
    assert ("call", "htrc_windows_f32") in events
