"""The calls that a user of the flat-HTRC operator makes, as measurable cases.

One case is one pass through a public entry point: ``flat_attention`` (one head or a whole layer), the
production configuration ``flat_attention_prod``, or a ``FlatRunner`` replaying its recorded graph over a
list of per-head jobs.  A case's fields:

  entry             "flat" (flat_attention), "prod" (flat_attention_prod), "runner" (FlatRunner.run)
  data              "runs" (64-token runs around shared centroids), "video" (regions of a t x y x latent
                    grid, raster order), "h3" (low-rank mixtures plus noise)
  heads, queries, keys, dim    sizes; ``tail`` keys past the last full leaf, attended exactly
  leaf, near        tokens per leaf and exact leaves per tile (``near`` 0 in a runner: the mode's own)
  store, dot, precision        state type, product type and statistics operands of flat_attention
  tile, group, stride, order   rows per tile, tiles per shared centre, select stride, query order
  chunk             tiles per window (0: the whole layer in one window)
  mode, batch, sink            the runner's quality mode, heads per replay, leading leaves always near
  qdtype            "bf16" or "fp32" queries
"""
from __future__ import annotations

import math

import torch

from htrc_amd import htrc_flat, htrc_flat_runner, workloads

_BASE = {"entry": "flat", "data": "runs", "heads": 1, "queries": 16384, "keys": 16384, "dim": 128, "tail": 0,
         "leaf": 64, "near": 16, "store": "int8", "dot": "bf16", "precision": "fp32", "tile": 64, "group": 1,
         "stride": 1, "order": "seq", "chunk": 0, "mode": "", "batch": 1, "sink": 0, "qdtype": "bf16"}
_MODES = {"fast": (256, "seq", 64), "balanced": (512, "seq", 64), "accurate": (1024, "kmeans", 64),
          "max": (1024, "kmeans", 32)}


def _case(name=None, **over):
    case = {**_BASE, **over}
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # The smallest call: the NumPy teaching model's shape (1024 queries, 4096 keys, 64 dims).
        _case("small_d64", queries=1024, keys=4096, dim=64),
        # One head of a 16 k sequence in one window, called again and again: launches and host time count.
        _case("head_16k"),
        # A video diffusion layer, 16 x 48 x 84 latent patches, 24 heads, in one window (the benchmark's layer).
        _case("layer_64k", data="video", heads=24, queries=64512, keys=64512, near=32),
        # The same layer for a clip of twice the length: 31 x 48 x 84 patches.
        _case("layer_125k", data="video", heads=24, queries=124992, keys=124992, near=32),
        # The production setting as it stands (leaf 16, 256 near leaves, windows of 128 tiles) on one head of
        # the live video shape: 40759 queries, 40752 leaf keys and 7 tail keys.
        _case("prod_head_h3", entry="prod", data="h3", queries=40759, keys=40752, tail=7, leaf=16, near=256,
              precision="tf32", chunk=128, qdtype="fp32"),
        # The runner in mode "fast" with the text tokens (220 leaves) always near, six heads a replay.
        _case("runner_fast_h3", entry="runner", data="h3", heads=6, queries=40759, keys=40752, tail=7, leaf=16,
              near=0, precision="tf32", chunk=128, mode="fast", batch=6, sink=220, qdtype="fp32"),
        # The runner's quality modes, one head a replay: k-means order and 1024 near leaves, 64-row tiles ...
        _case("runner_accurate_h3", entry="runner", data="h3", heads=2, queries=40759, keys=40752, tail=7, leaf=16,
              near=0, precision="tf32", chunk=256, mode="accurate", qdtype="fp32"),
        # ... and 32-row tiles, on a shorter clip.
        _case("runner_max_20k", entry="runner", data="h3", heads=2, queries=20011, keys=20000, tail=11, leaf=16,
              near=0, precision="tf32", chunk=256, mode="max", qdtype="fp32"),
        # flat_attention with every knob but the backend at its default: fp32 state and dots, leaf 16, 64 near
        # leaves, windows of 32 tiles.
        _case("default_fp32", data="h3", queries=12345, keys=12336, leaf=16, near=64, store="fp32", dot="tf32",
              chunk=32, qdtype="fp32"),
        # The fp32 path over a group of heads in one window.
        _case("layer_fp32", heads=6, queries=32768, keys=32768, near=32, store="fp32", dot="tf32", qdtype="fp32"),
        # The fp8 state store over a layer of a shorter clip, leaf 32.
        _case("layer_fp8", heads=12, queries=32256, keys=32256, leaf=32, near=64, store="fp8"),
        # The bf16 state store, ragged query count, leaf 128, two tiles sharing a centre.
        _case("layer_bf16_ragged", heads=24, queries=20001, keys=20096, leaf=128, near=12, store="bf16", group=2),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        leaf = rng.choice((16, 16, 32, 64, 64, 128))
        queries = log(700, 70000)
        keys = max(leaf * 8, int(queries * rng.choice((1, 1, 1, rng.uniform(0.4, 1.6)))) // leaf * leaf)
        heads = log(1, 24)
        kind = rng.choice(("int8", "int8", "int8", "prod", "runner", "fp8", "bf16", "fp32"))
        over = {"heads": heads, "queries": queries, "keys": keys, "leaf": leaf}
        nb = keys // leaf
        over["near"] = min(nb // 2, max(1, log(8, 64) * 64 // max(leaf, 32)))
        if kind == "prod":
            over.update(entry="prod", precision="tf32", chunk=128, qdtype="fp32", near=min(256, nb), tail=rng.choice((0, 5)))
        elif kind == "runner":
            mode = rng.choice(tuple(_MODES))
            over.update(entry="runner", data="h3", precision="tf32", chunk=rng.choice((128, 256, 1024)), mode=mode, near=0,
                        tile=_MODES[mode][2], order=_MODES[mode][1], leaf=16, keys=keys // 16 * 16, qdtype="fp32",
                        sink=rng.choice((0, keys // 16 // 12)), tail=rng.choice((0, 7)), heads=min(heads, 6))
            over["batch"] = rng.choice((1, over["heads"]))
        elif kind == "fp32":
            over.update(data="h3", store="fp32", dot="tf32", precision=rng.choice(("fp32", "fp32", "tf32")), qdtype="fp32",
                        chunk=rng.choice((0, 32)))
        else:
            over.update(store=kind, precision=rng.choice(("fp32", "tf32")), chunk=rng.choice((0, 0, 128)),
                        dim=rng.choice((128, 128, 128, 64)), group=rng.choice((1, 1, 1, 2)),
                        stride=rng.choice((1, 1, 2)), tail=rng.choice((0, 0, 9)))
        case = _case(**over)
        if _flops(case) <= 2.0e12 and heads * (queries / case["tile"]) * (keys / case["leaf"]) <= 2.4e7:
            return case


def _inputs(case, seed):
    """q, k, v [heads, n, dim] (k, v bf16) and the tail keys / values fp32 (or None)."""
    h, nq, nk, d, tail = (case[x] for x in ("heads", "queries", "keys", "dim", "tail"))
    dev = "cuda"
    if case["data"] == "h3":
        q, k, v, tk, tv = workloads.h3_live(n=nq, keys=nk, tail=max(tail, 1), d=d, heads=h, seed=seed, device=dev)
    elif case["data"] == "video":
        q, k, v = workloads.video_regions(t=nq // (48 * 84), y=48, x=84, d=d, heads=h, seed=seed, device=dev)
    else:
        n = max(nq, nk)
        q, k, v = workloads.clustered_runs(n=n, runs=-(-n // 64), run=64, d=d, heads=h, seed=seed, device=dev)
        q, k, v = (x[:, :m].contiguous() for x, m in ((q, nq), (k, nk), (v, nk)))
    if not tail:
        tk = tv = None
    elif case["data"] != "h3":
        g = torch.Generator(device=dev).manual_seed(seed + (1 << 20))
        tk, tv = (torch.randn((h, tail, d), generator=g, device=dev) for _ in range(2))
    if case["qdtype"] == "fp32":
        q = q.float()
    return q, k, v, (None if tk is None else (tk, tv))


def prepare(case, seed):
    q, k, v, tail = _inputs(case, seed)
    if case["entry"] == "runner":
        jobs = [(h, q[h], k[h], v[h], *((() if tail is None else ((tail[0][h], tail[1][h]),)))) for h in range(case["heads"])]
        runner = htrc_flat_runner.FlatRunner(case["queries"], case["keys"], mode=case["mode"], dim=case["dim"],
                                             tile_chunk=case["chunk"], heads=case["batch"], sink_leaves=case["sink"],
                                             tail_rows=case["tail"], leaf=case["leaf"])
        return {"runner": runner, "jobs": jobs}
    if case["heads"] == 1:
        q, k, v = q[0], k[0], v[0]
        tail = None if tail is None else (tail[0][0], tail[1][0])
    kw = {"leaf": case["leaf"], "exact_leaves": case["near"], "tail": tail, "ws": {}, "return_logz": True}
    if case["entry"] == "prod":
        return {"fn": htrc_flat.flat_attention_prod, "args": (q, k, v), "kw": kw}
    kw.update(backend="triton", store=case["store"], dot=case["dot"], precision=case["precision"], tile=case["tile"],
              sel_stride=case["stride"], order=case["order"], sink_leaves=case["sink"],
              tile_chunk=case["chunk"] or None)
    if case["group"] > 1:
        kw["kern"] = {"group": case["group"]}
    return {"fn": htrc_flat.flat_attention, "args": (q, k, v), "kw": kw}


def run(state):
    if "runner" in state:
        return state["runner"].run(state["jobs"])
    return state["fn"](*state["args"], **state["kw"])


def _shape(case):
    """near leaves, query order and rows per tile as the case's entry resolves them."""
    near, order, tile = _MODES[case["mode"]] if case["entry"] == "runner" else (case["near"], case["order"], case["tile"])
    return min(near + case["sink"], case["keys"] // case["leaf"]), order, tile


def _flops(case):
    kx, order, tile = _shape(case)
    nq, nk, d = case["queries"], case["keys"], case["dim"]
    nb = nk // case["leaf"]
    ng = -(-(-(-nq // tile)) // case["group"])
    # statistics (centre scores, key and value means), far scores and values, near scores and values, tail
    f = 6 * ng * nk * d + 4 * nq * nb * d + 4 * nq * (kx * case["leaf"] + case["tail"]) * d
    if order == "kmeans":
        f += 3 * 32 * d * (nq + 8 * min(4096, nq))
    return case["heads"] * f


def work(case):
    nq, nk, d = case["queries"], case["keys"], case["dim"]
    logz = 4 * nq if case["entry"] != "runner" else 0
    qb = 4 if case["qdtype"] == "fp32" else 2
    per_head = qb * nq * d + 2 * 2 * nk * d + 2 * 4 * case["tail"] * d + 4 * nq * d + logz
    return {"bytes": case["heads"] * per_head, "flops": _flops(case)}


def tolerance(case):
    """Measured with every leaf's keys and values in reverse order (the same sums in another order), and, for fp32,
    against the same products on another matrix instruction.  fp32 state: rel 3e-6, max 1e-5 with IEEE operands;
    rel 1.7e-4, max 1.3e-3 with TF32 ones (a weight at a rounding point rounds either way).  The other stores: rel up
    to 1.6e-4, max 0.02 where every tile keeps its near leaves; where two leaves tie for a tile's last near place the
    other one is as right, and that tile's rows differ by up to a few times the output's own size (rel 1.6e-3 and
    4.4e-3 over calls with one or two such tiles)."""
    if case["store"] == "fp32":
        return {"rel": 7e-4, "max": 1e-2} if case["precision"] == "tf32" else {"rel": 1e-5, "max": 1e-3}
    return {"rel": 5e-3, "max": 0.99}


def _kmeans(q, clusters=32, sample=4096, iters=8):
    n = q.shape[0]
    at = torch.linspace(0, n - 1, min(sample, n), device=q.device).round().long()
    s = q[at]
    c = s[torch.linspace(0, s.shape[0] - 1, min(clusters, s.shape[0]), device=q.device).round().long()].clone()
    for _ in range(iters):
        near = torch.cdist(s, c).argmin(1)
        total = torch.zeros_like(c).index_add_(0, near, s)
        count = torch.bincount(near, minlength=c.shape[0]).to(c.dtype)
        c = torch.where(count[:, None] > 0, total / count.clamp_min(1)[:, None], c)
    return torch.argsort(torch.cdist(q, c).argmin(1), stable=True)


def _exact_head(case, q, k, v, tail):
    """The operator's definition in 64 bits: every leaf's log-mass, tilted key mean and value mean at the tile's
    centre, the near leaves by the largest far score of the tile's rows, one softmax over both."""
    kx, order, tile = _shape(case)
    d, leaf, G, stride = case["dim"], case["leaf"], case["group"], case["stride"]
    nq, nk = q.shape[0], k.shape[0]
    nb, scale = nk // leaf, 1.0 / math.sqrt(d)
    q, k, v = q.double(), k.double(), v.double()
    perm = _kmeans(q) if order == "kmeans" else torch.arange(nq, device=q.device)
    qp = q[perm]
    nt = -(-nq // tile)
    rows = torch.cat([qp, qp[-1:].expand(nt * tile - nq, d)]).view(nt, tile, d)
    if G == 1:
        mu = rows.mean(1)
        last = nq - (nt - 1) * tile
        mu[-1] = rows[-1, :last].mean(0)
    else:
        ng = -(-nt // G)
        mu = torch.cat([rows, rows[-1:].expand(ng * G - nt, tile, d)]).view(ng, G * tile, d).mean(1)
    kl, vl = k.view(nb, leaf, d), v.view(nb, leaf, d)
    out = torch.empty((nt, tile, d), dtype=torch.float64, device=q.device)
    logz = torch.empty((nt, tile), dtype=torch.float64, device=q.device)
    step = max(1, min(64, int(3e8 / (kx * leaf * d + 2 * nb * d + tile * nb))))      # groups a window
    for c in range(0, mu.shape[0], step):
        m = mu[c:c + step]
        a = ((m @ k.t()) * scale).view(-1, nb, leaf)
        lz = a.logsumexp(2)
        w = (a - lz[..., None]).exp().transpose(0, 1)                                # [nb, centres, leaf]
        g = (w @ kl).transpose(0, 1) * scale                                         # [centres, nb, d]
        vb = (w @ vl).transpose(0, 1)
        for i in range(m.shape[0]):
            t0, t1 = (c + i) * G, min(nt, (c + i + 1) * G)
            r = rows[t0:t1].reshape(-1, d)
            s = (r - m[i]) @ g[i].t() + lz[i]                                        # far scores
            score = s[::stride].amax(0)
            score[:case["sink"]] = math.inf
            idx = score.topk(kx).indices
            if kx:
                s[:, idx] = -math.inf
            parts, vals = [s], [vb[i]]
            if kx:
                parts.append((r @ kl[idx].reshape(-1, d).t()) * scale)
                vals.append(vl[idx].reshape(-1, d))
            if tail is not None:
                parts.append((r @ tail[0].double().t()) * scale)
                vals.append(tail[1].double())
            z = torch.cat(parts, 1)
            lse = z.logsumexp(1)
            p = (z - lse[:, None]).exp()
            out[t0:t1] = (p @ torch.cat(vals)).view(t1 - t0, tile, d)
            logz[t0:t1] = lse.view(t1 - t0, tile)
    res, lzr = torch.empty_like(q), q.new_empty(nq)
    res[perm] = out.view(-1, d)[:nq]
    lzr[perm] = logz.view(-1)[:nq]
    return res, lzr


def exact(case, seed):
    if _flops(case) > 4e12:
        return None                                                                  # over 20 seconds in 64 bits
    q, k, v, tail = _inputs(case, seed)
    got = [_exact_head(case, q[h], k[h], v[h], None if tail is None else (tail[0][h], tail[1][h]))
           for h in range(case["heads"])]
    if case["entry"] == "runner":
        return [o for o, _ in got]
    if case["heads"] == 1:
        return got[0]
    return torch.stack([o for o, _ in got]), torch.stack([z for _, z in got])
