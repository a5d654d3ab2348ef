"""The work this package is measured on: calls a program makes through its public entry points.

Four kinds of call:

* ``readout``: ``softmax_readout`` without gradients (generation, where O is fed back as the next
  input, and evaluation);
* ``grad``: ``softmax_readout`` inside a model, with cotangents of O and LSE arriving from later
  layers; gradients of every parameter, or of h alone when the head and the embedding are frozen;
* ``mse``: a training step of ``softmax_readout_mse``, returning the loss and every gradient;
* ``fp8``: the opt-in e4m3 readout for evaluation, with the weights quantised once beforehand.

A case is a dict: ``dtype`` is the parameters' and h's storage dtype, or "autocast" (fp32 parameters
and activations under bf16 autocast); h is ``[tokens, K]``, or ``[rows, tokens, K]`` when ``rows`` is
not 0; ``weight`` is the per-token loss weight (none, Bernoulli(0.9), or a ragged tail of padding per
row); ``spread`` is the standard deviation of the logits (1: an untrained head, 3: a trained one).
"""
import math

import torch

import swvr_amd
from swvr_amd import fp8

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "autocast": torch.float32}
RAGGED_TAIL = 0.25   # a ragged row's padding: uniform in 0 .. a quarter of the row


def _case(name, kind, dtype, tokens, K, V, D, *, rows=0, bias=True, weight="none", z=0.0, spread=1.0, wrt="all"):
    c = dict(kind=kind, dtype=dtype, rows=rows, tokens=tokens, K=K, V=V, D=D, bias=bias, weight=weight, z=z,
             spread=spread, wrt=wrt)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one decoding step of one sequence: the smallest call on a full vocabulary
        _case("readout_one_token", "readout", "bf16", 1, 2560, 151936, 64, spread=3.0),
        # one decoding step of a batch of 48 sequences
        _case("readout_decode_batch", "readout", "bf16", 48, 4096, 128256, 128, spread=3.0),
        # an evaluation batch onto 300-wide word vectors, in fp16: more columns than one pass holds
        _case("readout_eval_fp16_d300", "readout", "fp16", 2500, 768, 50021, 300, bias=False, spread=3.0),
        # evaluation through the e4m3 readout, the weights quantised once
        _case("readout_eval_fp8", "fp8", "bf16", 8192, 2560, 151936, 64, spread=3.0),
        # the plumbing-size training step in fp32: a call of a few launches
        _case("train_small_fp32", "mse", "fp32", 512, 256, 4096, 16),
        # a model trained in fp32, a few sequences of odd length
        _case("train_fp32", "mse", "fp32", 333, 768, 30001, 100, rows=4, weight="ragged"),
        # a microbatch of a model with a mid-size vocabulary
        _case("train_microbatch", "mse", "bf16", 125, 1024, 32000, 64, rows=4, weight="bernoulli", z=1e-4),
        # fp32 parameters under bf16 autocast
        _case("train_autocast", "mse", "autocast", 512, 2048, 65536, 128, rows=4, weight="ragged", z=1e-4),
        # gradients of h alone, through a frozen head and embedding
        _case("frozen_head_fp16", "grad", "fp16", 2048, 1024, 151936, 16, spread=3.0, wrt="h"),
        # the headline training step
        _case("train_headline", "mse", "bf16", 16384, 2560, 151936, 64, weight="bernoulli", z=1e-4),
        # the training step of a wider model, half the tokens, D = 128
        _case("train_d128", "mse", "bf16", 8192, 4096, 128256, 128),
        # the largest step: a batch of padded sequences, D = 256 and the largest vocabulary
        _case("train_d256_large", "mse", "bf16", 4096, 4096, 256000, 256, rows=8, weight="ragged", z=1e-4),
    ]


# A drawn case does at most this many FLOPs (about the headline's step; fp32 has a sixteenth of the
# matrix rate of the 2-byte types).
DRAW_FLOPS = {"bf16": 50e12, "fp16": 50e12, "autocast": 50e12, "fp32": 2e12}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["readout", "readout", "grad", "mse", "mse", "mse", "fp8"])
    dtype = "bf16" if kind == "fp8" else rng.choice(["bf16", "bf16", "fp16", "autocast", "fp32"])
    if kind == "mse" and dtype == "fp16":
        dtype = "bf16"   # a mean loss's fp16 gradients need a loss scale, which is the grad kind
    lo_n = 512 if kind == "fp8" else 1 if kind == "readout" else 128
    while True:
        tokens, K, V = _log(rng, lo_n, 16384), _log(rng, 256, 4096), _log(rng, 4096, 256000)
        D = _log(rng, 16, 128 if kind == "fp8" else 300)
        if rng.random() < 0.75:
            K = K // 64 * 64   # hidden sizes are mostly multiples of 64; others are padded by the call
        rows = rng.choice([0, 0, 2, 3, 8])
        if rows:
            tokens = max(1, tokens // rows)
        weight = rng.choice(["none", "bernoulli", "ragged"] if rows else ["none", "bernoulli"])
        c = _case(None, kind, dtype, tokens, K, V, D, rows=rows, bias=rng.random() < 0.75,
                  weight=weight if kind == "mse" else "none", z=rng.choice([0.0, 1e-4]) if kind == "mse" else 0.0,
                  spread=1.0 if kind == "mse" else 3.0, wrt=rng.choice(["all", "h"]) if kind == "grad" else "all")
        if work(c)["flops"] <= DRAW_FLOPS[dtype]:
            return c


def _inputs(case, seed):
    """The call's tensors, on the GPU: h, W, b, E, the loss's target and weight or the cotangents."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    K, V, D = case["K"], case["V"], case["D"]
    lead = (case["rows"], case["tokens"]) if case["rows"] else (case["tokens"],)

    def r(*s, sc=1.0):
        return torch.randn(*s, device=DEVICE, generator=g).mul_(sc)

    t = {"h": r(*lead, K).to(dt), "W": r(V, K, sc=case["spread"] * K ** -0.5).to(dt)}
    t["b"] = r(V, sc=0.5 if case["spread"] > 1 else 0.02).to(dt) if case["bias"] else None
    t["E"] = r(V, D).to(dt)
    if case["kind"] == "mse":
        t["target"] = r(*lead, D)
        t["weight"] = None
        if case["weight"] == "bernoulli":
            t["weight"] = (torch.rand(*lead, device=DEVICE, generator=g) >= 0.1).float()
        elif case["weight"] == "ragged":
            n = lead[1]
            tails = torch.randint(0, max(1, int(RAGGED_TAIL * n)) + 1, (lead[0], 1), device=DEVICE, generator=g)
            t["weight"] = (torch.arange(n, device=DEVICE)[None, :] < n - tails).float()
    elif case["kind"] == "grad":
        # cotangents under a loss scale of 256: inside fp16's normal range
        t["gO"], t["glse"] = r(*lead, D, sc=256.0), r(*lead, sc=256.0)
    return t


def _params(case, t):
    if case["kind"] == "grad" and case["wrt"] == "h":
        return ["h"]
    return ["h", "W", "E"] + (["b"] if t["b"] is not None else [])


def prepare(case, seed):
    t = _inputs(case, seed)
    state = {"case": case, **t}
    if case["kind"] in ("mse", "grad"):
        state["params"] = [t[k].requires_grad_(True) for k in _params(case, t)]
    elif case["kind"] == "fp8":
        state["w_q"] = fp8.quantize_rows(t["W"])
    return state


def run(state):
    case = state["case"]
    h, W, E, b = state["h"], state["W"], state["E"], state["b"]
    if case["kind"] == "fp8":
        with torch.no_grad():
            return fp8.softmax_readout_fp8(h, W, E, b, w_q=state["w_q"])
    amp = case["dtype"] == "autocast"
    if case["kind"] == "readout":
        with torch.no_grad(), torch.autocast(DEVICE, dtype=torch.bfloat16, enabled=amp):
            return swvr_amd.softmax_readout(h, W, E, b)
    with torch.autocast(DEVICE, dtype=torch.bfloat16, enabled=amp):
        if case["kind"] == "grad":
            O, lse = swvr_amd.softmax_readout(h, W, E, b)
        else:
            loss = swvr_amd.softmax_readout_mse(h, W, E, state["target"], b, weight=state["weight"],
                                                z_loss_weight=case["z"])
    if case["kind"] == "grad":
        return (O.detach(), lse.detach(), *torch.autograd.grad((O, lse), state["params"], (state["gO"], state["glse"])))
    return (loss.detach(), *torch.autograd.grad(loss, state["params"]))


def work(case):
    """Each input read and each output written once; the products of the forward, one recompute of
    the scores in the backward (they are never stored) and the gradients' products, over the tokens
    of non-zero weight."""
    N = max(1, case["rows"]) * case["tokens"]
    K, V, D = case["K"], case["V"], case["D"]
    e = 4 if case["dtype"] in ("fp32", "autocast") else 2
    active = N * {"none": 1.0, "bernoulli": 0.9, "ragged": 1.0 - RAGGED_TAIL / 2}[case["weight"]]
    nb = V if case["bias"] else 0
    if case["kind"] == "fp8":
        return {"bytes": e * (N * K + V * D + nb) + V * K + 4 * V + 4 * N * (D + 1), "flops": 2.0 * N * V * (K + D)}
    params = e * (N * K + V * K + V * D + nb)
    if case["kind"] == "readout":
        return {"bytes": params + 4 * N * (D + 1), "flops": 2.0 * N * V * (K + D)}
    if case["wrt"] == "h":   # forward, scores, dP, dh
        return {"bytes": params + e * N * K + 4 * N * 2 * (D + 1), "flops": 2.0 * N * V * (3 * K + 2 * D)}
    io = 4 * N * 2 * (D + 1) if case["kind"] == "grad" else 4 * N * (D + (case["weight"] != "none"))
    return {"bytes": 2 * params + io, "flops": 2.0 * active * V * (4 * K + 3 * D)}


def tolerance(case):
    # about four times the largest distance from 64 bits of any output, over listed and drawn cases:
    # fp32 2.0e-6; readouts 3e-4 (bf16, e4m3 against its dequantised operands) and 4e-5 (fp16), whose
    # rounded P averages out; gradients 2.9e-3 (bf16) and 3.7e-4 (fp16); autocast 7.4e-3, the rounding
    # of the fp32 parameters included
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["dtype"] == "autocast":
        return {"rel": 3e-2}
    if case["kind"] in ("readout", "fp8"):
        return {"rel": 1.5e-3 if case["dtype"] == "bf16" else 2e-4}
    return {"rel": 1.2e-2 if case["dtype"] == "bf16" else 1.5e-3}


EXACT_FLOPS = 60e12          # above this the 64-bit result takes over about 20 seconds
EXACT_BYTES = 4 << 30        # one block of 64-bit scores


def _quantised(x, per_row):
    """x as its e4m3 rounding holds it: scale = amax / 448, one per row or one for the matrix."""
    x = x.float()
    amax = x.abs().amax(dim=-1, keepdim=True) if per_row else x.abs().amax()
    scale = amax.clamp_min(1e-30) / 448
    return (x / scale).to(torch.float8_e4m3fn).double() * scale.double()


def exact(case, seed):
    """The same outputs in 64 bits with plain torch, row block by row block (rows are independent;
    the gradients of W, E and b are sums over the rows)."""
    if work(case)["flops"] > EXACT_FLOPS:
        return None
    t = _inputs(case, seed)
    K, D, V = case["K"], case["D"], case["V"]
    lead = t["h"].shape[:-1]
    h, W, E = t["h"].reshape(-1, K).double(), t["W"].double(), t["E"].double()
    if case["kind"] == "fp8":
        h, W = _quantised(t["h"].reshape(-1, K), False), _quantised(t["W"], True)
    b = t["b"].double() if t["b"] is not None else None
    N = h.shape[0]
    O = torch.empty(N, D, dtype=torch.float64, device=DEVICE)
    lse = torch.empty(N, dtype=torch.float64, device=DEVICE)
    grads = case["kind"] in ("mse", "grad")
    names = _params(case, t) if grads else []
    if grads:
        gh = torch.empty_like(h)
        gW = torch.zeros_like(W) if "W" in names else None
        gE = torch.zeros_like(E) if "E" in names else None
        gb = torch.zeros_like(b) if "b" in names else None
    if case["kind"] == "mse":
        target = t["target"].reshape(N, D).double()
        w = t["weight"].reshape(N).double() if t["weight"] is not None else torch.ones_like(lse)
        total = w.sum()
        loss = torch.zeros((), dtype=torch.float64, device=DEVICE)
    elif case["kind"] == "grad":
        all_gO, all_glse = t["gO"].reshape(N, D).double(), t["glse"].reshape(N).double()
    step = max(1, EXACT_BYTES // (8 * V))
    for n0 in range(0, N, step):
        s = slice(n0, min(N, n0 + step))
        S = h[s] @ W.t()
        if b is not None:
            S += b
        lse[s] = torch.logsumexp(S, dim=1)
        P = S.sub_(lse[s, None]).exp_()
        O[s] = P @ E
        if not grads:
            continue
        if case["kind"] == "mse":
            diff = O[s] - target[s]
            loss += (w[s] * (diff.pow(2).mean(dim=1) + case["z"] * lse[s].pow(2))).sum() / total
            gO = diff * (w[s] * 2 / (D * total))[:, None]
            glse = w[s] * 2 * case["z"] * lse[s] / total
        else:
            gO, glse = all_gO[s], all_glse[s]
        if gE is not None:
            gE += P.t() @ gO
        dS = gO @ E.t()
        dS -= ((O[s] * gO).sum(dim=1) - glse)[:, None]
        dS *= P
        del P, S
        gh[s] = dS @ W
        if gW is not None:
            gW += dS.t() @ h[s]
        if gb is not None:
            gb += dS.sum(dim=0)
        del dS
    if not grads:
        return O.view(*lead, D), lse.view(lead)
    out = {"h": gh.view(*lead, K), "W": gW, "E": gE, "b": gb}
    first = (loss,) if case["kind"] == "mse" else (O.view(*lead, D), lse.view(lead))
    return (*first, *[out[k] for k in names])
