"""Inputs at the edge of what the walks (pass_c_walk_x6.hip) take: x and y with
tokens inside channels, padded with NaN, and a ragged last chunk, on every
route; decays whose sums leave fp32's range, at fp32 accuracy. Against the fp64 oracle, to the bounds of the parity and storage suites:
y on the fp32 path at the fp32 per-element bound (plus its rounding to 16-bit
storage), on the bf16 path at the bf16 bound, s1 at the fp32 bound."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import pyoracle as po
from helix_amd.desc import HELIX_BF16, HELIX_F16, HELIX_F32
from helix_amd import scan
from helix_amd.scan import make_desc, ssd_scan
from gpu_harness import BF16_ABS, BF16_REL, F32_ABS, F32_REL, ctx_for
from test_gpu_io import TORCH, U, rounded

pytestmark = pytest.mark.gpu

TORCH = {HELIX_F32: torch.float32, **TORCH}
U = {HELIX_F32: 0.0, **U}
IDS = {HELIX_F32: "f32", HELIX_BF16: "bf16", HELIX_F16: "f16"}


def up(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dtype)


@pytest.fixture
def gpu(gpu, monkeypatch):
    """ssd_scan on a context that keeps the form the route names (HELIX_1PASS_Y=1: tiles in y)."""
    ctx = ctx_for(gpu, HELIX_1PASS_Y="1")
    monkeypatch.setitem(scan._contexts, torch.cuda.current_device(), ctx)
    return ctx


def check(p, y, s1, io, bf16):
    y_ref, s_ref = po.scan(p, use_ids=False)
    rel, ab = (BF16_REL, BF16_ABS) if bf16 else (F32_REL + U[io], F32_ABS)
    y, s1 = y.float().cpu().numpy(), s1.cpu().numpy()
    assert np.all(np.isfinite(s1)) and po.allclose_ratio(s1, s_ref, F32_REL, F32_ABS) <= 1.0
    assert np.all(np.isfinite(y)) and po.allclose_ratio(y, y_ref, rel, ab) <= 1.0


# (route, backend, multipass, storage, d_state): the walks of both paths, by
# storage type; blocks of state indices (the second adds into y); state tiles
# in y; the one-launch single pass.
ROUTES = [("fp32", "fp32", True, HELIX_F32, 128), ("fp32", "fp32", True, HELIX_BF16, 128),
          ("fp32", "fp32", True, HELIX_F16, 64), ("bf16", "auto", True, HELIX_F32, 128),
          ("bf16", "auto", True, HELIX_F32, 64), ("bf16", "auto", True, HELIX_BF16, 128),
          ("bf16", "auto", True, HELIX_F16, 128), ("blocks", "fp32", True, HELIX_F32, 256),
          ("blocks", "auto", True, HELIX_F32, 256), ("tiles in y", "auto", False, HELIX_F32, 128),
          ("one launch", "auto", False, HELIX_BF16, 128)]


@pytest.mark.parametrize("route", ROUTES, ids=[f"{r[0]}-{r[1]}-{IDS[r[3]]}-n{r[4]}" for r in ROUTES])
def test_tokens_inside_channels(gpu, route):
    """x [S, H, P, L + 27] seen as [S, L, H, P], its padding NaN; y likewise, its padding left alone."""
    label, backend, multipass, io, N = route
    S, L, H, P, pad = 2, 714, 16, 128 if label == "tiles in y" else 72, 27
    p = po.problem_harness(L, S, H, P, N, 1, 1234, "long")
    p = rounded(p, io) if io != HELIX_F32 else p
    xb = torch.full((S, H, P, L + pad), float("nan"), device="cuda", dtype=TORCH[io])
    x = xb[..., :L].permute(0, 3, 1, 2)
    x.copy_(up(p.x))
    yb = torch.full_like(xb, float("nan"))
    # State tiles in y take a dense y.
    dense = label == "tiles in y"
    y = torch.empty((S, L, H, P), device="cuda") if dense else yb[..., :L].permute(0, 3, 1, 2)
    dt, A, s0 = up(p.dt), up(p.A), up(p.s0)
    B, C = up(p.B, TORCH[io]), up(p.C, TORCH[io])
    d = make_desc(x, dt, B, C, s0, y, A, backend=backend, multipass=multipass)
    info = gpu.run_info(d)
    assert b"walk" in info.kernel_c if label != "one launch" else info.kernel_c is None
    _, s1 = ssd_scan(x, dt, A, B, C, s0, backend=backend, multipass=multipass, y=y)
    torch.cuda.synchronize()
    check(p, y, s1, io, backend == "auto" and multipass)
    assert dense or torch.isnan(yb[..., L:]).all()


@pytest.mark.parametrize("route", [r for r in ROUTES if r[1] == "fp32" or not r[2]],
                         ids=lambda r: f"{r[0]}-{r[1]}-{IDS[r[3]]}-n{r[4]}")
def test_lowest_decay(gpu, route):
    """Heads without memory between ordinary ones: the sums of dt A over a chunk pass fp32's range from the first
    tokens on (A at the lowest float), in the chunk's later tokens only (-1e37), or not at all (-1e30)."""
    label, backend, multipass, io, N = route
    S, L, H, P = 2, 714, 16, 128 if label == "tiles in y" else 72
    p = po.problem_harness(L, S, H, P, N, 1, 4321, "long")
    p = rounded(p, io) if io != HELIX_F32 else p
    p.A[::4] = np.finfo(np.float32).min
    p.A[1::4] = -1e37
    p.A[2::4] = -1e30
    p.dt += 6.0     # dt of about 0.6
    x, B, C = up(p.x, TORCH[io]), up(p.B, TORCH[io]), up(p.C, TORCH[io])
    d = make_desc(x, up(p.dt), B, C, up(p.s0), x, up(p.A), backend=backend, multipass=multipass)
    info = gpu.run_info(d)
    assert b"walk" in info.kernel_c if label != "one launch" else info.kernel_c is None
    y, s1 = ssd_scan(x, up(p.dt), up(p.A), B, C, up(p.s0), backend=backend, multipass=multipass)
    torch.cuda.synchronize()
    check(p, y, s1, io, False)
