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
    """mag^2 / sqrt(128) nats above zero: 51, 93, 131 and 147 octaves (the last past the range)."""
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
