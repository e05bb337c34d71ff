"""What a user of this framework has it do, as cases that can be timed and checked.

Every case is one call of helix_amd.scan.ssd_scan, the torch-facing operator over the C ABI, with
tensors in HBM, as a Mamba-2 layer's prefill makes it: x, dt, A, B, C, the carried state where there is
one, and y and the final state back. The shapes are the workloads that bench.py reports, the shapes of the
parity and storage tests, or ragged ones between them; the values are drawn as bench.py draws them
(x ~ N(0, 1); dt before softplus ~ N(mu, sigma); A = -exp(U(0, ln 16)); B, C ~ N(0, 1) / sqrt(d_state)).

Options of a case: S sequences of L tokens, H heads of P channels, d_state N, G B/C groups; `store`, the
storage type of x, B, C and y; `backend` and `multipass` as ssd_scan takes them; `carry`, whether a state is
carried in; `packed`, whether x, B and C are column ranges of one projected row per token (as a layer's
causal convolution leaves them) and not tensors of their own; `mu` and `sigma` of dt.
"""
import math

import torch

from helix_amd.scan import ssd_scan

STORE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _case(name, S, L, H, P, N, G, backend="auto", store="f32", multipass=True, carry=False, packed=False, mu=-1.0,
          sigma=0.5):
    return {"name": name, "S": S, "L": L, "H": H, "P": P, "N": N, "G": G, "backend": backend, "store": store,
            "multipass": multipass, "carry": carry, "packed": packed, "mu": mu, "sigma": sigma}


def listed():
    return [
        # A short prompt through a small layer, at fp32 accuracy: all launches and host work.
        _case("short prompt, fp32 path", 1, 256, 8, 64, 64, 1, backend="fp32"),
        # The next user turn of a running conversation, just past the length from which the llama.cpp hook
        # takes a call: two chunks, the second ragged, the state carried in.
        _case("chat turn of 67 tokens", 1, 67, 64, 64, 128, 8, carry=True),
        # An ordinary prompt through a 64-head layer, by a caller that wants fp32 accuracy.
        _case("2k prompt, fp32 path", 1, 2048, 64, 64, 128, 8, backend="fp32"),
        # The same prompt by a bf16 model that wants the scan itself at fp32 accuracy.
        _case("2k prompt, bf16 storage, fp32 path", 1, 2048, 64, 64, 128, 8, backend="fp32", store="bf16"),
        # The headline workload: a long prompt, on the bf16 path and on the fp32 path.
        _case("8k prompt", 1, 8192, 64, 64, 128, 8),
        _case("8k prompt, fp32 path", 1, 8192, 64, 64, 128, 8, backend="fp32"),
        # The long prompt in a bf16 model: x, B and C are column ranges of the convolution's output.
        _case("8k prompt, bf16 storage", 1, 8192, 64, 64, 128, 8, store="bf16", packed=True),
        # A ragged batch of prompts with a wide head, long memory and carried states, at fp32 accuracy.
        _case("ragged batch, fp32 path", 4, 1000, 32, 128, 128, 1, backend="fp32", carry=True, mu=-2.0, sigma=1.0),
        # Where the caller has no memory to lend: the operator's form without scratch.
        _case("4k prompt without scratch", 1, 4096, 64, 64, 128, 8, multipass=False),
        # A model with d_state 256.
        _case("4k prompt, d_state 256", 1, 4096, 64, 64, 256, 8),
        # The largest: batched prefill in serving, many heads on one B/C group; and an odd number of heads of
        # three channel slabs each.
        _case("batch of 8, 80 heads", 8, 4096, 80, 64, 128, 1, carry=True),
        _case("batch of 8, 27 heads of 192", 8, 4096, 27, 192, 128, 1, carry=True),
    ]


def _cost(c):
    """About how much a case costs: tokens x channels, more where the scan is at fp32 accuracy or wider."""
    slow = 1.0
    if c["backend"] == "fp32" or not c["multipass"]:
        slow = 2.5 if c["store"] == "f32" else 8.0
    return c["S"] * c["L"] * c["H"] * c["P"] * max(1.0, c["N"] / 128) * slow


def draw(rng):
    most = _cost(_case("", 8, 4096, 80, 64, 128, 1)) * 0.8
    while True:
        heads, group = rng.choice([(8, 1), (16, 2), (24, 1), (27, 1), (32, 1), (32, 4), (48, 1), (64, 8), (64, 1), (80, 1)])
        c = _case("", rng.choice([1, 1, 1, 2, 3, 4, 8]), int(round(math.exp(rng.uniform(math.log(64), math.log(8192))))),
                  heads, rng.choice([64, 64, 64, 128, 192, 80]), rng.choice([64, 128, 128, 128, 96, 256]), group,
                  backend=rng.choice(["auto", "auto", "fp32"]), store=rng.choice(["f32", "f32", "bf16", "f16"]),
                  multipass=rng.random() < 0.85, carry=rng.random() < 0.5, packed=rng.random() < 0.4,
                  mu=rng.choice([-1.0, -2.0]), sigma=rng.choice([0.5, 1.0]))
        if not c["multipass"] or c["backend"] == "fp32":
            # At most the longest of these that is listed.
            c["L"] = min(c["L"], 4096 if c["N"] <= 128 else 2048)
        if _cost(c) <= most:
            del c["name"]
            return c


def prepare(case, seed):
    S, L, H, P, N, G = (case[k] for k in "SLHPNG")
    g = torch.Generator(device="cuda").manual_seed(seed)
    dev, st = "cuda", STORE[case["store"]]

    def normal(*shape, dtype=torch.float32):
        return torch.randn(*shape, generator=g, device=dev, dtype=dtype)

    if case["packed"]:
        # One row per token: x of every head, then B and C of every group.
        row = torch.empty(S, L, H * P + 2 * G * N, device=dev, dtype=st)
        row[..., :H * P] = normal(S, L, H * P)
        row[..., H * P:] = normal(S, L, 2 * G * N) / math.sqrt(N)
        x = row[..., :H * P].unflatten(-1, (H, P))
        B = row[..., H * P:H * P + G * N].unflatten(-1, (G, N))
        C = row[..., H * P + G * N:].unflatten(-1, (G, N))
    else:
        x = normal(S, L, H, P).to(st)
        B = (normal(S, L, G, N) / math.sqrt(N)).to(st)
        C = (normal(S, L, G, N) / math.sqrt(N)).to(st)
    dt = case["mu"] + case["sigma"] * normal(S, L, H)
    A = -torch.exp(torch.rand(H, generator=g, device=dev) * math.log(16.0))
    s0 = 0.1 * normal(S, H, P, N) if case["carry"] else None
    return {"x": x, "dt": dt, "A": A, "B": B, "C": C, "s0": s0, "backend": case["backend"],
            "multipass": case["multipass"]}


def run(state):
    y, s1 = ssd_scan(state["x"], state["dt"], state["A"], state["B"], state["C"], state["s0"],
                     backend=state["backend"], multipass=state["multipass"])
    return {"y": y, "s1": s1}


def work(case):
    """Every input read once and every output written once; the products of the scan in chunks of 64 tokens
    (the triangle of C B^T and of its product with dt x, the state's part of y and the state's advance)."""
    S, L, H, P, N, G = (case[k] for k in "SLHPNG")
    es = 4 if case["store"] == "f32" else 2
    states = (2 if case["carry"] else 1) * S * H * P * N
    nbytes = es * (2 * S * L * H * P + 2 * S * L * G * N) + 4 * (S * L * H + H + states)
    tri = 0.5 * 64 * 65
    flops = 2.0 * S * (L / 64) * (G * tri * N + H * tri * P + 2 * 64 * H * N * P)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # The bf16 path rounds the products' operands to bf16 (measured against 64 bits: 3.4e-3 of y's norm).
    if case["backend"] == "auto" and case["multipass"]:
        return {"rel": 1e-2}
    # The fp32 path and the form without scratch, stored in fp32 (measured 1.7e-7) ...
    if case["store"] == "f32":
        return {"rel": 1e-6, "max": 1e-4}
    # ... or with y rounded once to 16 bits, where a sum that lies between two values may go either way.
    return {"rel": 1e-3, "max": 1e-2} if case["store"] == "bf16" else {"rel": 2e-4, "max": 2e-3}


def exact(case, seed):
    st = prepare(case, seed)
    S, L, H, P, N, G = (case[k] for k in "SLHPNG")
    x, B, C = st["x"], st["B"], st["C"]
    v = st["dt"].double()
    dt = torch.where(v > 20, v, torch.log1p(torch.exp(v.clamp(max=20))))
    lam = dt * st["A"].double()
    R = st["s0"].double() if case["carry"] else torch.zeros(S, H, P, N, device="cuda", dtype=torch.float64)
    y = torch.empty(S, L, H, P, device="cuda", dtype=torch.float64)
    for t0 in range(0, L, 64):
        t1 = min(L, t0 + 64)
        n = t1 - t0
        # [S, H, t, .] in 64 bits
        xd = (x[:, t0:t1].double() * dt[:, t0:t1, :, None]).permute(0, 2, 1, 3).contiguous()
        b = B[:, t0:t1].double().permute(0, 2, 1, 3).repeat_interleave(H // G, 1).contiguous()
        c = C[:, t0:t1].double().permute(0, 2, 1, 3).repeat_interleave(H // G, 1).contiguous()
        cs = lam[:, t0:t1].permute(0, 2, 1).cumsum(-1)
        low = torch.ones(n, n, device="cuda", dtype=torch.bool).tril()
        decay = torch.exp(torch.where(low, cs[..., :, None] - cs[..., None, :], -math.inf))
        m = torch.matmul(c, b.transpose(-1, -2).contiguous()) * decay
        o = torch.matmul(m, xd) + torch.exp(cs)[..., None] * torch.matmul(c, R.transpose(-1, -2).contiguous())
        y[:, t0:t1] = o.permute(0, 2, 1, 3)
        w = torch.exp(cs[..., -1:] - cs)
        R = R * torch.exp(cs[..., -1])[..., None, None] + torch.matmul((xd * w[..., None]).transpose(-1, -2).contiguous(), b)
    return {"y": y, "s1": R}
