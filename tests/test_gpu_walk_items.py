"""The walk over item blocks (pass_c_walk_x6.hip) at the shapes where its work
split can go wrong: one to five (head, P slab) items per B/C group
(blocks of four with one to four live items; up to two take their waves a SIMD
each), slabs and d_state short of their tiles, ragged last chunks, runs of one
chunk and of several, and the state carried through the groups of a small
scratch. Against the fp64 oracle at the fp32 per-element bound of the parity
suite (rel 5e-6, abs 5e-7)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import pyoracle as po
from helix_amd.desc import HELIX_BACKEND_MPP, HELIX_BACKEND_SGMMA, HELIX_BF16, HELIX_F16, HELIX_OK, HELIX_TENSOR_NULL
from gpu_harness import BF16_ABS, BF16_REL, F32_ABS, F32_REL, T, ctx_for, run
from test_gpu_io import TORCH, U, check, rounded, run_io

pytestmark = pytest.mark.gpu

# (L, S, H, P, N, G, label), knobs
SHAPES = [
    ((700, 1, 4, 64, 128, 4), {}),                      # one item per group
    ((333, 2, 2, 128, 128, 2), {}),                     # one head of two slabs
    ((449, 1, 6, 64, 64, 2), {}),                       # three items
    ((513, 1, 5, 72, 120, 1), {}),                      # ten items, an 8-channel last slab
    ((1025, 1, 5, 64, 96, 1), {"HELIX_WALK_LEN": 8, "HELIX_SEG_LEN": 4}),   # five items, runs of 8, one token last
    ((640, 1, 4, 64, 128, 1), {"HELIX_WALK_LEN": 3, "HELIX_SEG_LEN": 1}),   # runs of 3 over ten chunks, the last of 1
    ((1500, 2, 3, 64, 128, 1), {"HELIX_SCRATCH_MB": 1}),                    # carried through several groups
]


# Items per workgroup: four, and two as a small grid has by default.
ITEMS = pytest.mark.parametrize("items", ["4", "2"], ids=["four", "two"])


@ITEMS
@pytest.mark.parametrize("shape,knobs", SHAPES, ids=["x".join(map(str, s)) + ("k" if k else "") for s, k in SHAPES])
def test_item_blocks(gpu, shape, knobs, items):
    p = po.problem_harness(*shape, 515, "long")
    p.s0 = (np.random.default_rng(5).standard_normal(p.s0.shape) * 0.2).astype(np.float32)
    y_ref, s_ref = po.scan(p, use_ids=False)
    ctx = ctx_for(gpu, HELIX_F32_WALK="1", HELIX_WALK_ITEMS=items, **knobs)
    d = p.d.copy()
    d.backend, d.multipass = HELIX_BACKEND_SGMMA, True
    assert ctx.run_info(d).run_items == int(items)
    assert b"helix_scan_walk_x6_n" in ctx.plan_info(d).kernel_c
    assert ctx.run_info(d).run_len == knobs.get("HELIX_WALK_LEN", 1)
    _, y, s1 = run(ctx, p, d)
    assert po.allclose_ratio(y, y_ref, F32_REL, F32_ABS) <= 1.0
    assert po.allclose_ratio(s1, s_ref, F32_REL, F32_ABS) <= 1.0


@ITEMS
@pytest.mark.parametrize("copies", ["0", "1"], ids=["rows", "copies"])
@pytest.mark.parametrize("shape,knobs", SHAPES, ids=["x".join(map(str, s)) + ("k" if k else "") for s, k in SHAPES])
def test_item_blocks_bf16(gpu, shape, knobs, copies, items):
    """The bf16 path's instantiations, on the caller's rows of B and C and on Pass A's bf16 copies."""
    p = po.problem_harness(*shape, 515, "long")
    p.s0 = (np.random.default_rng(5).standard_normal(p.s0.shape) * 0.2).astype(np.float32)
    y_ref, s_ref = po.scan(p, use_ids=False)
    ctx = ctx_for(gpu, HELIX_WALK_BCCOPY=copies, HELIX_WALK_ITEMS=items, **knobs)
    d = p.d.copy()
    d.backend, d.multipass = HELIX_BACKEND_MPP, True
    assert (b"helix_scan_walk16_bf16_bc_n" if copies == "1" else b"helix_scan_walk16_bf16_n") in ctx.plan_info(d).kernel_c
    assert ctx.run_info(d).run_len == knobs.get("HELIX_WALK_LEN", 1)
    _, y, s1 = run(ctx, p, d)
    assert po.allclose_ratio(y, y_ref, BF16_REL, BF16_ABS) <= 1.0
    assert po.allclose_ratio(s1, s_ref, F32_REL, F32_ABS) <= 1.0


# 16-bit storage on the fp32 path: Pass A and the walk on one (bf16) or two
# (f16) exact planes of B and C past the lengths that run as one launch.
IO_SHAPES = [
    ((513, 1, 5, 72, 120, 1), 0),       # ten items, an 8-channel last slab, one token last
    ((449, 2, 6, 64, 64, 2), 0),        # three items per group, d_state 64
    ((450, 1, 64, 64, 128, 8), 6),      # B and C inside wider rows
]


@pytest.mark.parametrize("io", [HELIX_BF16, HELIX_F16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape,pad", IO_SHAPES, ids=["x".join(map(str, s)) for s, _ in IO_SHAPES])
def test_16bit_storage(gpu, shape, pad, io):
    """Against the oracle fed the rounded inputs: y within the fp32 bound plus
    its own rounding to the storage type, s1 within the fp32 bound. Without
    scratch, or with y in x's place, the one-launch single pass serves the
    call, to the same bounds."""
    p = rounded(po.problem_harness(*shape, 616, "long"), io)
    p.s0 = (np.random.default_rng(6).standard_normal(p.s0.shape) * 0.2).astype(np.float32)
    y_ref, s_ref = po.scan(p, use_ids=False)
    L, S, H, P, N, G = shape
    d = p.d.copy()
    d.io_dtype, d.backend, d.multipass = io, HELIX_BACKEND_SGMMA, True
    for k in (d.s_b, d.s_c):
        k[0], k[1] = G * (N + pad), N + pad
    d.seq_b = d.seq_c = L * G * (N + pad)
    info = gpu.plan_info(d)
    assert b"helix_scan_walk_x6_" in info.kernel_c and info.total_bytes == gpu.scratch_size(d) > 0

    def up(a, width=0):
        t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
        return torch.nn.functional.pad(t, (0, width))

    x, B, C = up(p.x).to(TORCH[io]), up(p.B, pad).to(TORCH[io]), up(p.C, pad).to(TORCH[io])
    dt, A, s0 = up(p.dt), up(p.A), up(p.s0)
    scratch = torch.empty(info.total_bytes, dtype=torch.uint8, device="cuda")
    for route in ("passes", "no scratch", "in place"):
        y = x.clone() if route == "in place" else torch.full_like(x, float("nan"))
        s1 = torch.full_like(s0, float("nan"))
        rc = gpu.encode(torch.cuda.current_stream().cuda_stream, d, T(s0), T(y if route == "in place" else x), T(dt), T(A),
                        T(B), T(C), HELIX_TENSOR_NULL, T(y), T(s1), T(None if route == "no scratch" else scratch))
        assert rc == HELIX_OK, gpu.last_error()
        torch.cuda.synchronize()
        assert po.allclose_ratio(y.float().cpu().numpy(), y_ref, F32_REL + U[io], F32_ABS) <= 1.0, route
        assert po.allclose_ratio(s1.cpu().numpy(), s_ref, F32_REL, F32_ABS) <= 1.0, route


# Pass A segments and walk runs of several chunks: state carried from chunk to
# chunk in both, planes and records staged for a next chunk, runs of one and of
# two segments, ragged last chunks of one token and of four.
RUNS = [
    ((1025, 1, 5, 72, 120, 1), {"HELIX_WALK_LEN": 6, "HELIX_SEG_LEN": 3}),
    ((900, 2, 6, 64, 64, 2), {"HELIX_WALK_LEN": 4, "HELIX_SEG_LEN": 4}),
]


@ITEMS
@pytest.mark.parametrize("io", [HELIX_BF16, HELIX_F16], ids=["bf16", "f16"])
@pytest.mark.parametrize("backend", [HELIX_BACKEND_SGMMA, HELIX_BACKEND_MPP], ids=["fp32", "bf16"])
@pytest.mark.parametrize("shape,knobs", RUNS, ids=["x".join(map(str, s)) for s, _ in RUNS])
def test_16bit_storage_runs(gpu, shape, knobs, backend, io, items):
    p = rounded(po.problem_harness(*shape, 617, "long"), io)
    p.s0 = (np.random.default_rng(6).standard_normal(p.s0.shape) * 0.2).astype(np.float32)
    y_ref, s_ref = po.scan(p, use_ids=False)
    ctx = ctx_for(gpu, HELIX_WALK_ITEMS=items, **knobs)
    d = p.d.copy()
    d.io_dtype, d.backend, d.multipass = io, backend, True
    assert ctx.run_info(d).run_len == knobs["HELIX_WALK_LEN"] and ctx.plan_info(d).seg_len == knobs["HELIX_SEG_LEN"]
    desc, y, s1 = run_io(ctx, p, io, backend, True)
    check(io, desc, y, s1, y_ref, s_ref)


# Folded runs about the line between the two orders of workgroups: two and three
# runs, seven and eight sequences, grids past a multiple of eight.
ORDERS = [(1, 1, 2), (1, 1, 3), (2, 2, 4), (7, 1, 3), (8, 1, 3), (3, 2, 5)]   # sequences, chunks per run, runs


@ITEMS
@pytest.mark.parametrize("backend", [HELIX_BACKEND_SGMMA, HELIX_BACKEND_MPP], ids=["fp32", "bf16"])
@pytest.mark.parametrize("S,run_len,runs", ORDERS, ids=["x".join(map(str, o)) for o in ORDERS])
def test_folded_run_order(gpu, S, run_len, runs, backend, items):
    p = po.problem_harness(64 * run_len * runs - 5, S, 6, 72, 72, 2, 619, "long")
    p.s0 = (np.random.default_rng(7).standard_normal(p.s0.shape) * 0.2).astype(np.float32)
    y_ref, s_ref = po.scan(p, use_ids=False)
    ctx = ctx_for(gpu, HELIX_WALK_LEN=run_len, HELIX_SEG_LEN=run_len, HELIX_FUSE_B="1", HELIX_F32_WALK="1",
                  HELIX_WALK_ITEMS=items)
    d = p.d.copy()
    d.backend, d.multipass = backend, True
    info = ctx.run_info(d)
    assert info.kernel_b is None and (info.run_len, info.runs_per_group) == (run_len, runs)
    _, y, s1 = run(ctx, p, d)
    rel, ab = (BF16_REL, BF16_ABS) if backend == HELIX_BACKEND_MPP else (F32_REL, F32_ABS)
    assert po.allclose_ratio(y, y_ref, rel, ab) <= 1.0
    assert po.allclose_ratio(s1, s_ref, F32_REL, F32_ABS) <= 1.0


@ITEMS
@pytest.mark.parametrize("backend", [HELIX_BACKEND_SGMMA, HELIX_BACKEND_MPP], ids=["fp32", "bf16"])
@pytest.mark.parametrize("N", [136, 256])
def test_state_block_runs(gpu, N, backend, items):
    """The walk that adds into y, over runs of several chunks."""
    p = po.problem_harness(1025, 1, 5, 72, N, 1, 618, "long")
    p.s0 = (np.random.default_rng(6).standard_normal(p.s0.shape) * 0.2).astype(np.float32)
    y_ref, s_ref = po.scan(p, use_ids=False)
    ctx = ctx_for(gpu, HELIX_WALK_LEN=6, HELIX_SEG_LEN=3, HELIX_F32_WALK="1", HELIX_WALK_ITEMS=items)
    d = p.d.copy()
    d.backend, d.multipass = backend, True
    assert ctx.plan_info(d).state_blocks == 2 and ctx.run_info(d).run_len == 6
    _, y, s1 = run(ctx, p, d)
    rel, ab = (BF16_REL, BF16_ABS) if backend == HELIX_BACKEND_MPP else (F32_REL, F32_ABS)
    assert po.allclose_ratio(y, y_ref, rel, ab) <= 1.0
    assert po.allclose_ratio(s1, s_ref, F32_REL, F32_ABS) <= 1.0


@pytest.mark.parametrize("io", [HELIX_BF16, HELIX_F16], ids=["bf16", "f16"])
def test_16bit_storage_lent_little(gpu, io):
    """A tensor too small for the passes, lent to ssd_scan: the single pass's bits, as without scratch; a path
    that needs its scratch still refuses it."""
    from helix_amd import scan
    p = po.problem_harness(513, 1, 5, 72, 120, 1, 616, "long")
    x, dt, A, B, C = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (p.x, p.dt, p.A, p.B, p.C))
    x, B, C = (t.to(TORCH[io]) for t in (x, B, C))
    little = torch.empty(64, dtype=torch.uint8, device="cuda")
    want = scan.ssd_scan(x, dt, A, B, C, backend="fp32", multipass=False)
    got = scan.ssd_scan(x, dt, A, B, C, backend="fp32", scratch=little)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    with pytest.raises(ValueError):
        scan.ssd_scan(x, dt, A, B, C, backend="bf16", scratch=little)


def test_16bit_storage_past_fixed_scratch(gpu):
    """helix_scan_encode_noalloc where one chunk per group exceeds its scratch: the single pass's bits."""
    from helix_amd import scan
    S, L, H, P, N = 65, 65, 64, 64, 128
    g = torch.Generator(device="cuda").manual_seed(9)
    x, B, C = (torch.randn(S, L, k, n, generator=g, device="cuda").to(torch.bfloat16) for k, n in ((H, P), (1, N), (1, N)))
    dt = torch.randn(S, L, H, generator=g, device="cuda")
    A = -1.0 - torch.rand(H, generator=g, device="cuda")
    s0 = torch.randn(S, H, P, N, generator=g, device="cuda")
    y, s1 = torch.empty_like(x), torch.empty_like(s0)
    d = scan.make_desc(x, dt, B, C, s0, y, A, backend="fp32")
    rc = gpu.encode_noalloc(torch.cuda.current_stream().cuda_stream, d, *map(T, (s0, x, dt, A, B, C, None, y, s1)))
    assert rc == HELIX_OK, gpu.last_error()
    want = scan.ssd_scan(x, dt, A, B, C, s0, backend="fp32", multipass=False)
    assert torch.equal(y, want[0]) and torch.equal(s1, want[1])


# Short scans: at the limit of the one-launch route on each path (caps.cpp,
# one_launch_scan) and one chunk past it, with the passes that a tuning
# override keeps (HELIX_STATE_BLOCKS=1, the default's value).
SHORT = [
    ((257, 1, 8, 64, 64, 1), True), ((321, 1, 8, 64, 64, 1), False),     # d_state 64: 5 / 6 chunks, fp32 path
    ((384, 1, 64, 64, 128, 8), True), ((385, 1, 64, 64, 128, 8), False),
    ((64, 3, 40, 72, 96, 1), False),                                     # four rounds of workgroups of one chunk
    ((40, 3, 27, 72, 96, 1), True),                                      # three rounds of a ragged chunk
    ((200, 1, 4, 64, 256, 1), True),                                     # two blocks of state indices
]


@pytest.mark.parametrize("shape,one", SHORT, ids=["x".join(map(str, s)) for s, _ in SHORT])
def test_short_scan(gpu, shape, one):
    p = po.problem_harness(*shape, 717, "long")
    p.s0 = (np.random.default_rng(7).standard_normal(p.s0.shape) * 0.2).astype(np.float32)
    y_ref, s_ref = po.scan(p, use_ids=False)
    d = p.d.copy()
    d.backend, d.multipass = HELIX_BACKEND_SGMMA, True
    results = {}
    for name, ctx, multipass in (("default", gpu, True), ("passes", ctx_for(gpu, HELIX_STATE_BLOCKS="1"), True),
                                 ("one launch", ctx_for(gpu, HELIX_1PASS_Y="0"), False)):
        d.multipass = multipass
        _, y, s1 = results[name] = run(ctx, p, d)
        assert po.allclose_ratio(y, y_ref, F32_REL, F32_ABS) <= 1.0, name
        assert po.allclose_ratio(s1, s_ref, F32_REL, F32_ABS) <= 1.0, name
    same = all(np.array_equal(a, b) for a, b in zip(results["default"][1:], results["one launch" if one else "passes"][1:]))
    assert same


@pytest.mark.parametrize("over", ["C", "dt", "x"])
def test_short_scan_y_over_input(gpu, over):
    """A short scan whose y lies over C or dt runs the passes, which have read both before y is written (C as Pass A's
    bf16 copy); over x, in x's strides, the one launch. Bits of the same route with a y of its own."""
    from helix_amd import scan
    L, S, H, P, N, G = 300, 1, 16, 64, 128, 1
    p = po.problem_harness(L, S, H, P, N, G, 929, "long")
    x, dt, A, B, C, s0 = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (p.x, p.dt, p.A, p.B, p.C, p.s0))
    route = gpu if over == "x" else ctx_for(gpu, HELIX_WALK_BCCOPY="1")
    d = p.d.copy()
    d.backend, d.multipass = HELIX_BACKEND_MPP, True
    _, y_want, s_want = run(route, p, d)
    y = x.clone() if over == "x" else torch.full_like(x, float("nan"))
    if over == "x":
        x = y
    elif over == "C":       # the first N columns of y's rows
        C = y.view(S, L, 1, H * P)[..., :N].copy_(C)
    else:                   # a column of H of them
        dt = y.view(S, L, H * P)[..., :H].copy_(dt)
    _, s1 = scan.ssd_scan(x, dt, A, B, C, s0, backend="bf16", y=y)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), y_want) and np.array_equal(s1.cpu().numpy(), s_want)


@pytest.mark.parametrize("shape", [(900, 2, 9, 64, 128, 1), (700, 1, 5, 136, 64, 1), (900, 1, 4, 64, 256, 2)],
                         ids=["nine items", "three slabs", "state blocks"])
def test_copy_plan_runs_without_copies(gpu, shape):
    """Plans with bf16 copies of B and C: the bits of the plan without them."""
    p = po.problem_harness(*shape, 919, "long")
    d = p.d.copy()
    d.backend, d.multipass = HELIX_BACKEND_MPP, True
    assert gpu.plan_info(d).bccopy_bytes > 0
    _, y, s1 = run(gpu, p, d)
    _, y0, s0 = run(ctx_for(gpu, HELIX_WALK_BCCOPY="0"), p, d)
    assert np.array_equal(y, y0) and np.array_equal(s1, s0)
    y_ref, s_ref = po.scan(p, use_ids=False)
    assert po.allclose_ratio(y, y_ref, BF16_REL, BF16_ABS) <= 1.0
    assert po.allclose_ratio(s1, s_ref, F32_REL, F32_ABS) <= 1.0


NO_STATE = [   # (shape, multipass, backend, knobs): every place that reads s0
    ((700, 1, 64, 64, 128, 8), True, "fp32", {}),                      # Pass B
    ((1500, 1, 8, 64, 64, 1), True, "bf16", {"HELIX_SCRATCH_MB": 1}),  # Pass B, many groups
    ((1024, 4, 40, 64, 128, 1), True, "bf16", {}),                     # the bf16 walk's prologue
    ((1024, 4, 40, 64, 128, 1), True, "fp32", {}),                     # the fp32 walk's
    ((600, 1, 16, 64, 128, 2), False, "auto", {"HELIX_1PASS_Y": "1"}),  # state tiles in y
    ((100, 2, 8, 72, 256, 1), True, "auto", {}),                       # one launch per block of state indices
]


@pytest.mark.parametrize("shape,multipass,backend,knobs", NO_STATE, ids=range(len(NO_STATE)))
def test_ssd_scan_without_state(gpu, shape, multipass, backend, knobs, monkeypatch):
    """ssd_scan without s0 gives the bits of a state of zeros, with and without ids, twice on one scratch."""
    from helix_amd import scan
    p = po.problem_harness(*shape, 818, "long")
    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (p.x, p.dt, p.A, p.B, p.C)]
    monkeypatch.setitem(scan._contexts, torch.cuda.current_device(), ctx_for(gpu, **knobs))
    zeros = torch.zeros(p.s0.shape, device="cuda")
    ids = torch.arange(shape[1], dtype=torch.int32, device="cuda").flip(0).contiguous()
    want = scan.ssd_scan(*t, zeros, backend=backend, multipass=multipass)
    for i in (None, ids, None):
        got = scan.ssd_scan(*t, None, i, backend=backend, multipass=multipass)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
