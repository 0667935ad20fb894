"""Performance cases of the MoC framework: what a user's program has it do,
through the public entry points (``moc.MoC``, ``moc.MoCGroup``,
``moc.moc_triton``), from one decode token to a full training step.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare(case, seed)`` makes the layers and inputs on the GPU, ``run(state)``
is one pass, ``exact(case, seed)`` the same results in 64-bit torch.

A case's ``kind``:

  step     ``MoC.step``: one decode token per sequence, cache updated in place
  forward  ``MoC.forward`` without gradients, final state returned (a prompt)
  prefill  ``MoC.forward`` without gradients, continuing from a cache
  train    ``MoC.forward`` and the gradients of x, z, router and basis
  func     ``moc_triton`` on given routing weights, forward and gradients
  group    ``MoCGroup`` over one z (the QKV pattern), forward and gradients

``tokens`` > 0 (train, func, group) packs sequences of uneven lengths behind
``cu_seqlens``; otherwise the batch is ``batch`` x ``time``.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "mixture-of-convolutions_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import moc  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, kind, batch, time, dim, z, k, s, dtype="bf16", act="silu", route="softmax",
          std=0.0, tokens=0, shortest=0, longest=0, dim2=0, dim3=0):
    """std 0: the layer's own fan-in initialisation of the basis."""
    c = {"kind": kind, "batch": batch, "time": time, "dim": dim, "z": z, "k": k, "s": s,
         "dtype": dtype, "act": act, "route": route, "std": std, "tokens": tokens,
         "shortest": shortest, "longest": longest, "dim2": dim2, "dim3": dim3}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one user's token-by-token generation: the smallest call, all latency
        _case("step_one", "step", 1, 1, 2048, 2048, 16, 4),
        # a serving batch of the decode benchmark: 256 sequences, one token each
        _case("step_batch", "step", 256, 1, 2048, 2048, 16, 4, std=0.002),
        # decode of a layer kept in 32 bits, a middling batch
        _case("step_fp32", "step", 48, 1, 1024, 1024, 16, 4, dtype="fp32"),
        # prompts of a serving batch: 1024 tokens each, the cache kept for decode
        _case("prompt", "forward", 8, 1024, 2048, 2048, 16, 4, std=0.002),
        # chunked prefill of ragged prompts continuing from their caches; sizes
        # off every tile
        _case("chunk_ragged", "prefill", 3, 777, 1544, 1536, 12, 3, route="exp"),
        # the small fp32 layer of the CPU reference configuration, as a training
        # step: launches and host time
        _case("train_small_fp32", "train", 2, 512, 256, 256, 4, 4, dtype="fp32", act=""),
        # the benchmark's layer step (README shape), with a gradient of its own
        # for every output as a model above the layer hands one down
        _case("train_layer", "train", 4, 4096, 2048, 2048, 16, 4, std=0.002),
        # packed sequences of 16 to 4096 tokens, exp routing, no activation
        _case("train_packed", "train", 0, 0, 4096, 2048, 16, 4, act="", route="exp",
              std=0.002, tokens=32768, shortest=16, longest=4096),
        # an fp32 training step of a middling layer
        _case("train_fp32", "train", 4, 2048, 1024, 1024, 16, 4, dtype="fp32"),
        # odd token count, channel count off the tiles, few taps
        _case("train_ragged", "train", 3, 1021, 1130, 1152, 12, 3, route="exp"),
        # weights from a router of the user's own: the functional call, packed,
        # longer kernels
        _case("func_long", "func", 0, 0, 2048, 0, 16, 8, std=0.002, tokens=8191, shortest=32,
              longest=2048),
        # q, k and v convolutions of one attention layer on a shared z: the largest
        _case("group_qkv", "group", 2, 8192, 4096, 4096, 32, 8, act="", route="exp",
              dim2=1024, dim3=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A channel count: mostly multiples of 64, the rest even or anything."""
    n, p = _log_int(rng, lo, hi), rng.random()
    if p < 0.6:
        return max(64, n // 64 * 64)
    return n // 2 * 2 if p < 0.9 else n


def draw(rng):
    kind = rng.choice(["step", "step", "forward", "prefill", "train", "train", "train", "func",
                       "group"])
    dtype = "fp32" if kind != "group" and rng.random() < 0.25 else "bf16"
    act, route = rng.choice(["silu", ""]), rng.choice(["softmax", "exp"])
    z = max(64, _log_int(rng, 128, 4096) // 64 * 64) if rng.random() < 0.85 else _log_int(rng, 128, 2048)
    k = rng.choice([4, 8, 12, 16, 16, 16, 24, 32])
    s = rng.choice([2, 3, 4, 4, 4, 4, 5, 6, 8])
    std = rng.choice([0.0, 0.002])
    if kind == "step":
        return _case("", kind, _log_int(rng, 1, 512), 1, _width(rng, 256, 4096), z, k, s, dtype,
                     act, route, std)
    dim = _width(rng, 128, 4096)
    most = 16384 if dtype == "bf16" else 8192
    n = _log_int(rng, 64, min(most, max(64, (1 << 26) // dim)))
    b = min(_log_int(rng, 1, 8), n // 16)
    if kind == "group":
        k, dim2 = rng.choice([8, 16, 16, 32]), max(128, dim // 4 // 2 * 2)
        z = max(64, z // 64 * 64)
        return _case("", kind, b, n // b, dim, z, k, s, dtype, act, route, std, dim2=dim2,
                     dim3=dim2)
    if kind in ("train", "func") and rng.random() < 0.35:
        return _case("", kind, 0, 0, dim, z, k, s, dtype, act, route, std, tokens=n,
                     shortest=rng.choice([1, 8, 16]), longest=max(32, n // rng.choice([2, 4, 8])))
    return _case("", kind, b, max(n // b, 2), dim, z, k, s, dtype, act, route, std)


# ---------------------------------------------------------------------------
# inputs

def _lengths(case, gen):
    """Uneven lengths that add up to ``tokens``."""
    left, out = case["tokens"], []
    while left:
        n = int(torch.randint(case["shortest"], case["longest"] + 1, (1,), generator=gen))
        out.append(min(n, left))
        left -= out[-1]
    return out


def _dims(case):
    return [d for d in (case["dim"], case["dim2"], case["dim3"]) if d]


def _routes(case):
    """exp for q and k, softmax for v in a group; one layer: its own."""
    n = len(_dims(case))
    return [case["route"]] * n if n == 1 else [case["route"]] * (n - 1) + ["softmax"]


def _make(case, seed):
    """Parameters and inputs as a dict of tensors on the GPU (the layer's dtype)."""
    dev, dt = torch.device("cuda"), _DTYPES[case["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(seed)
    k, s, z = case["k"], case["s"], case["z"]
    bound = (case["std"] or math.sqrt(k / (3 * s))) * math.sqrt(3)  # MoC's fan-in rule

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    t = {"basis": [((torch.rand(k, s, d, generator=gen, device=dev) * 2 - 1) * bound).to(dt)
                   for d in _dims(case)]}
    if case["tokens"]:
        lens = _lengths(case, torch.Generator().manual_seed(seed))
        lead = (case["tokens"],)
        t["longest"] = max(lens)
        t["cu"] = torch.tensor([0] + lens).cumsum(0).to(dev, torch.int32)
    else:
        lead = (case["batch"], case["time"])
    t["x"] = [normal(*lead, d).to(dt) for d in _dims(case)]
    if case["kind"] == "func":
        t["alpha"] = torch.softmax(normal(*lead, k), -1).to(dt)
    else:
        t["router"] = [(normal(k, z) * 0.02).to(dt) for _ in _dims(case)]
        t["z"] = normal(*lead, z).to(dt)
    if case["kind"] in ("step", "prefill"):
        t["cache"] = normal(case["batch"], case["dim"], s).to(dt)
    if case["kind"] in ("train", "func", "group"):
        t["dy"] = [normal(*lead, d).to(dt) for d in _dims(case)]
    return t


def prepare(case, seed):
    t = _make(case, seed)
    dt, act = _DTYPES[case["dtype"]], case["act"] or None
    st = {"case": case, "t": t, "act": act}
    grad = case["kind"] in ("train", "func", "group")
    if case["kind"] != "func":
        layers = []
        for d, route, basis, router in zip(_dims(case), _routes(case), t["basis"], t["router"]):
            m = moc.MoC(d, case["z"], case["s"], case["k"], activation=act,
                        router_activation=route).to("cuda", dt)
            with torch.no_grad():
                m.conv_bases.copy_(basis)
                m.router.copy_(router)
            layers.append(m)
        st["layers"] = layers
        st["m"] = moc.MoCGroup(*layers) if case["kind"] == "group" else layers[0]
    if grad:
        for x in t["x"]:
            x.requires_grad_()
        if "z" in t:
            t["z"].requires_grad_()
    if case["kind"] == "func":
        t["alpha"].requires_grad_()
        t["basis"][0].requires_grad_()
    st["packed"] = {"cu_seqlens": t["cu"], "max_seqlen": t["longest"]} if case["tokens"] else {}
    return st


def run(state):
    t, kind = state["t"], state["case"]["kind"]
    if kind == "step":
        with torch.no_grad():
            y, cache = state["m"].step(t["x"][0], t["z"], cache=t["cache"], output_final_state=True)
        return {"y": y, "cache": cache}
    if kind in ("forward", "prefill"):
        with torch.no_grad():
            y, last = state["m"](t["x"][0], t["z"], cache=t.get("cache"), output_final_state=True)
        return {"y": y, "state": last}
    if kind == "func":
        y, _ = moc.moc_triton(t["x"][0], t["alpha"], t["basis"][0], activation=state["act"],
                              **state["packed"])
        wrt = [t["x"][0], t["alpha"], t["basis"][0]]
        return {"y": y, "grads": list(torch.autograd.grad(y, wrt, t["dy"][0]))}
    if kind == "train":
        m = state["m"]
        y, _ = m(t["x"][0], t["z"], **state["packed"])
        wrt = [t["x"][0], t["z"], m.router, m.conv_bases]
        return {"y": y, "grads": list(torch.autograd.grad(y, wrt, t["dy"][0]))}
    ys = [y for y, _ in state["m"](t["x"], t["z"], **state["packed"])]
    wrt = [*t["x"], t["z"], *(p for m in state["layers"] for p in (m.router, m.conv_bases))]
    return {"y": ys, "grads": list(torch.autograd.grad(ys, wrt, t["dy"]))}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what it gives in 64 bits

def work(case):
    """Inputs read once, outputs written once; the products of the layer."""
    e = 2 if case["dtype"] == "bf16" else 4
    n = case["tokens"] or case["batch"] * case["time"]
    k, s, z = case["k"], case["s"], case["z"]
    dims = _dims(case)
    d, g = sum(dims), len(dims)
    params = k * s * d + g * k * z
    nbytes, flops = 2 * n * d + n * z + params, 2 * n * d * s * (k + 1) + 2 * g * n * k * z
    if case["kind"] == "func":
        nbytes += n * k
    if case["kind"] in ("step", "prefill"):
        nbytes += 2 * case["batch"] * d * s
    if case["kind"] == "forward":
        nbytes += case["batch"] * d * s
    if case["kind"] in ("train", "func", "group"):
        nbytes += 2 * n * d + n * z + params + (n * k if case["kind"] == "func" else 0)
        flops += n * d * s * (4 * k + 3) + 4 * g * n * k * z
    return {"bytes": e * nbytes, "flops": flops}


def tolerance(case):
    """About four times the relative (2-norm) error of the outputs against
    ``exact`` as measured: bf16 data round the logits, the weights and every
    output to 8 bits (0.002 to 0.007); fp32 data differ in the order of sums
    only (up to 9e-7; the longest sums of the ranges get twice that)."""
    return {"rel": 1.5e-2} if case["dtype"] == "bf16" else {"rel": 1e-5}


def _conv64(case, x, a, basis, cache, cu):
    """sum_s (a . basis[:, s]) * x[t - (S-1-s)] per sequence, in 64 bits."""
    k, s, d = basis.shape
    lead = x.shape[:-1]
    a2 = a.reshape(-1, k)
    if cu is not None:
        n = x.shape[0]
        at = torch.arange(n, device=x.device)
        start = cu.long()[torch.searchsorted(cu.long(), at, right=True) - 1]
    else:
        head = cache.transpose(1, 2)[:, 1:] if cache is not None else x.new_zeros(lead[0], s - 1, d)
        xx = torch.cat((head, x), 1)
    p = None
    for j in range(s):
        back = s - 1 - j
        if cu is None:
            xs = xx[:, j:j + lead[1]]
        else:
            xs = torch.cat((x.new_zeros(back, d), x[:n - back]), 0) * (at - back >= start)[:, None]
        q = (a2 @ basis[:, j]).reshape(*lead, d) * xs
        p = q if p is None else p + q
    return torch.nn.functional.silu(p) if case["act"] else p


def exact(case, seed):
    t = _make(case, seed)
    grad = case["kind"] in ("train", "func", "group")

    def f64(v):
        return v.double().requires_grad_(grad)

    xs, bases = [f64(x) for x in t["x"]], [f64(b) for b in t["basis"]]
    cu, cache = t.get("cu"), t["cache"] if "cache" in t else None
    if case["kind"] == "func":
        alphas, shared, routers = [f64(t["alpha"])], None, []
    else:
        shared, routers = f64(t["z"]), [f64(r) for r in t["router"]]
        logits = [(shared.reshape(-1, case["z"]) @ r.T).reshape(*shared.shape[:-1], -1)
                  for r in routers]
        alphas = [v.softmax(-1) if r == "softmax" else v.exp()
                  for v, r in zip(logits, _routes(case))]
    ys = [_conv64(case, x, a, b, None if cache is None else cache.double(), cu)
          for x, a, b in zip(xs, alphas, bases)]
    if grad:
        dys = [v.double() for v in t["dy"]]
        if case["kind"] == "func":
            return {"y": ys[0].detach(),
                    "grads": list(torch.autograd.grad(ys, [xs[0], alphas[0], bases[0]], dys))}
        params = [p for pair in zip(routers, bases) for p in pair]
        grads = list(torch.autograd.grad(ys, [*xs, shared, *params], dys))
        y = [v.detach() for v in ys]
        return {"y": y if case["kind"] == "group" else y[0], "grads": grads}
    if cache is not None:
        seq = torch.cat((cache.double(), xs[0].transpose(1, 2)), -1)
    else:
        pad = xs[0].new_zeros(case["batch"], case["dim"], case["s"])
        seq = torch.cat((pad, xs[0].transpose(1, 2)), -1)
    return {"y": ys[0], "cache" if case["kind"] == "step" else "state": seq[..., -case["s"]:]}
