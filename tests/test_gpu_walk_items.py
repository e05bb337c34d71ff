"""The fp32 path's walk over item blocks (pass_c_walk_x6.hip) at the shapes where
its work split can go wrong: one to five (head, P slab) items per B/C group
(blocks of four with one to four live items; up to two take their waves a SIMD
each), slabs and d_state short of their tiles, ragged last chunks, runs of one
chunk and of several, and the state carried through the groups of a small
scratch. Against the fp64 oracle at the fp32 per-element bound of the parity
suite (rel 5e-6, abs 5e-7)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from helix_amd.desc import HELIX_BACKEND_SGMMA
from gpu_harness import F32_ABS, F32_REL, ctx_for, run

pytestmark = pytest.mark.gpu

# (L, S, H, P, N, G, label), knobs
SHAPES = [
    ((700, 1, 4, 64, 128, 4), {}),                      # one item per group
    ((333, 2, 2, 128, 128, 2), {}),                     # one head of two slabs
    ((449, 1, 6, 64, 64, 2), {}),                       # three items
    ((513, 1, 5, 72, 120, 1), {}),                      # ten items, an 8-channel last slab
    ((1025, 1, 5, 64, 96, 1), {"HELIX_WALK_LEN": 8, "HELIX_SEG_LEN": 4}),   # five items, runs of 4 or 8, one token last
    ((640, 1, 4, 64, 128, 1), {"HELIX_WALK_LEN": 3, "HELIX_SEG_LEN": 1}),   # runs of 1 to 3 over ten chunks
    ((1500, 2, 3, 64, 128, 1), {"HELIX_SCRATCH_MB": 1}),                    # carried through several groups
]


@pytest.mark.parametrize("shape,knobs", SHAPES, ids=["x".join(map(str, s)) + ("k" if k else "") for s, k in SHAPES])
def test_item_blocks(gpu, shape, knobs):
    p = po.problem_harness(*shape, 515, "long")
    p.s0 = (np.random.default_rng(5).standard_normal(p.s0.shape) * 0.2).astype(np.float32)
    y_ref, s_ref = po.scan(p, use_ids=False)
    ctx = ctx_for(gpu, HELIX_F32_WALK="1", **knobs)
    d = p.d.copy()
    d.backend, d.multipass = HELIX_BACKEND_SGMMA, True
    assert b"helix_scan_walk_x6_n" in ctx.plan_info(d).kernel_c
    _, y, s1 = run(ctx, p, d)
    assert po.allclose_ratio(y, y_ref, F32_REL, F32_ABS) <= 1.0
    assert po.allclose_ratio(s1, s_ref, F32_REL, F32_ABS) <= 1.0
