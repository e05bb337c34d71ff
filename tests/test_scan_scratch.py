"""ssd_scan's own scratch (helix_amd/scan.py): calls that may run at the same
time never share a buffer, one that is replaced goes back to its own stream, and
a captured graph keeps memory that no later call touches."""
from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

from helix_amd import scan
from oracle import pyoracle as po


@pytest.fixture
def host_scratch(monkeypatch):
    """_scratch_for on host memory, in a pool of its own; the streams it allocates under, in order."""
    empty, under = torch.empty, []
    monkeypatch.setattr(scan, "_scratch", threading.local())
    monkeypatch.setattr(torch, "empty", lambda n, dtype, device: empty(n, dtype=dtype))
    monkeypatch.setattr(scan, "_under", lambda device, st, stream: under.append((device, st)) or scan.contextlib.nullcontext())
    return under


def test_scratch_per_stream(host_scratch):
    a = scan._scratch_for(0, 11, 64)
    b = scan._scratch_for(0, 22, 64)
    c = scan._scratch_for(1, 11, 64)
    assert len({t.data_ptr() for t in (a, b, c)}) == 3
    assert scan._scratch_for(0, 11, 0) is a and scan._scratch_for(0, 11, 64) is a and scan._scratch_for(0, 33, 0) is None
    grown = scan._scratch_for(0, 11, 65)
    assert grown.numel() >= 65 and scan._scratch_for(0, 11, 1) is grown and scan._scratch_for(0, 22, 1) is b
    assert host_scratch == [(0, 11), (0, 22), (1, 11), (0, 11)]


def test_scratch_is_bounded(host_scratch):
    keep = scan._scratch_for(0, 1, 8)
    for st in range(2, 3 * scan.SCRATCH_STREAMS):
        scan._scratch_for(0, st, 8)
        assert scan._scratch_for(0, 1, 0) is keep     # used last but one: never the oldest
    assert len(scan._scratch.pool) == scan.SCRATCH_STREAMS
    other = []
    th = threading.Thread(target=lambda: other.append(scan._scratch_for(0, 1, 8)))
    th.start()
    th.join()
    assert other[0] is not keep


def _inputs(L, seed, dtype):
    p = po.problem_harness(L, 1, 16, 64, 128, 2, seed, "long")
    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (p.x, p.dt, p.A, p.B, p.C)]
    return [t[0].to(dtype), t[1], t[2], t[3].to(dtype), t[4].to(dtype)]


@pytest.mark.gpu
@pytest.mark.parametrize("explicit", [False, True], ids=["current stream", "stream argument"])
@pytest.mark.parametrize("dtype,backend", [(torch.bfloat16, "fp32"), (torch.float32, "auto")], ids=["bf16 storage", "f32"])
def test_two_streams(gpu, dtype, backend, explicit):
    """Calls of one thread in flight on two streams, of growing sizes, give the bits of the same calls one by one."""
    work = [[_inputs(L, 10 * i + L, dtype) for L in (500, 1500, 700, 2600)] for i in range(2)]
    want = [[[t.clone() for t in scan.ssd_scan(*w, backend=backend)] for w in ws] for ws in work]
    streams = [torch.cuda.Stream() for _ in work]
    got = [[], []]
    torch.cuda.synchronize()
    for k in range(len(work[0])):
        for i, st in enumerate(streams):
            if explicit:
                got[i].append(scan.ssd_scan(*work[i][k], backend=backend, stream=st))
            else:
                with torch.cuda.stream(st):
                    got[i].append(scan.ssd_scan(*work[i][k], backend=backend))
    torch.cuda.synchronize()
    for gs, ws in zip(got, want):
        for g, w in zip(gs, ws):
            assert all(torch.equal(a, b) for a, b in zip(g, w))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,backend", [(torch.bfloat16, "fp32"), (torch.float32, "auto")], ids=["bf16 storage", "f32"])
def test_captured_scratch(gpu, dtype, backend):
    """Replays of a captured call, with longer eager calls on the same stream between them, give the eager bits."""
    t = _inputs(1500, 3, dtype)
    longer = _inputs(4000, 4, dtype)
    want = [a.clone() for a in scan.ssd_scan(*t, backend=backend)]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        y, s1 = scan.ssd_scan(*t, backend=backend)
    for _ in range(3):
        with torch.cuda.stream(side):
            y.fill_(float("nan"))
            s1.fill_(float("nan"))
            scan.ssd_scan(*longer, backend=backend)
            g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want[0]) and torch.equal(s1, want[1])
