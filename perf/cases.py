"""The work a user of this package has it do, as cases that can be timed and checked.

A layer-wise quantisation run makes three kinds of call for every linear of a model: it sums the
saliency-weighted Hessians over chunks of calibration activations (``add_batch`` /
``add_batch_shared``, then ``finalize_hessian``), it quantises the weight (``find_params`` and
``fasterquant``), and it stores the codes (``export_packed``, read back by ``dequantize_packed``).
The cases below take each of them through the public classes: alone at the sizes of an 8B decoder
layer's linears (4096 and 14336 wide, 16 x 2048 tokens a chunk), and all together on small and
ragged linears, where launches and host work count.

A case is a dict of plain values.  Its "kind" is one of

  accum    construct, add the chunks, finalize: H and act_square of 1-3 modules on one input
  quant    find_params and fasterquant on finished Hessians
  linear   construct, add the chunks, finalize, fasterquant: one linear from start to end
  classic  the same for the classic GPTQ class (one Hessian, no saliency)
  packed   export_packed and dequantize_packed of a quantised linear
"""
from __future__ import annotations

import numpy as np
import torch

from gptq_plus_mp_quant_amd import (GPTQ, GPTQPlus, WeightQuantizer, add_batch_shared, dequantize_packed,
                                    export_packed)

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BLOCK = 128          # fasterquant's block size, the reference's default
PERCDAMP = 0.01

# what fasterquant and the quantizer are asked for, by name
DEFAULTS = dict(dtype="fp16", G=4, modules=1, chunks=1, samples=16, seq=2048, bits=4, sym=False, mse=False,
                groupsize=-1, static=False, atomic=False, actorder=True, alpha=0.0, ref_loss=0.0,
                gmode="frozen", outliers=8)


def _case(kind, name=None, **kw):
    c = dict(DEFAULTS, kind=kind, **kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # A toy linear, as in a first try or a unit test: launches and host work are all there is.
        _case("linear", "linear_tiny", R=128, C=256, G=2, chunks=2, samples=2, seq=64),
        # A ragged linear (columns, tokens and rows off every tile size) in bf16, symmetric.
        _case("linear", "linear_ragged", R=1026, C=1365, G=3, chunks=3, samples=5, seq=501, dtype="bf16", sym=True),
        # Hessians of q/k/v, which read one input: 12 targets from one chunk of an 8B layer's run.
        _case("accum", "accum_qkv", R=1024, C=4096, modules=3),
        # Hessians of down_proj, the widest input of that layer; half a chunk.
        _case("accum", "accum_down", R=1024, C=14336, samples=8),
        # One saliency group: a single target on a chunk in bf16.
        _case("accum", "accum_one_group", R=1024, C=4096, G=1, dtype="bf16"),
        # Activations that the calibration run keeps in fp32.
        _case("accum", "accum_fp32", R=1024, C=4096, dtype="fp32", samples=8),
        # Quantising q_proj with four groups, w4 asymmetric per channel, act_order: the common call.
        _case("quant", "quant_q", R=4096, C=4096),
        # Quantising down_proj: the longest Cholesky chain and block loop of the layer.
        _case("quant", "quant_down", R=4096, C=14336, samples=8),
        # The GPTQ+ first-order term on, static 128-column groups, bf16 weights.
        _case("quant", "quant_gptqplus", R=4096, C=4096, alpha=0.05, ref_loss=50.0, groupsize=128, static=True,
              dtype="bf16"),
        # A rotated gate_proj: symmetric, scales found again per 128-column block, blocks solved at once.
        _case("quant", "quant_rotated", R=14336, C=4096, sym=True, groupsize=128, atomic=True, outliers=0),
        # Classic GPTQ on k_proj with the quantizer's clip search, static groups.
        _case("classic", "classic_kproj", R=1024, C=4096, G=1, chunks=2, samples=4, sym=True, mse=True,
              groupsize=128, static=True),
        # Storing gate_proj's codes and reading them back.
        _case("packed", "packed_gate", R=14336, C=4096, G=4, samples=1, seq=64),
    ]


def _log(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def _width(rng, lo, hi):
    """A width between lo and hi: a multiple of 128 or of 8 as model widths are, or any number."""
    c = _log(rng, lo, hi)
    m = rng.choice((128, 128, 8, 1))
    return max(lo, c // m * m)


def draw(rng):
    kind = rng.choice(("accum", "accum", "quant", "quant", "linear", "classic", "packed"))
    dtype = rng.choice(("fp16", "fp16", "bf16", "bf16", "fp32"))
    sym = rng.random() < 0.5
    c = dict(sym=sym, bits=rng.choice((4, 4, 8)), actorder=rng.random() < 0.8)
    if kind in ("quant", "linear"):
        group = rng.choice(("channel", "channel", "static", "dynamic"))
        c.update(groupsize=-1 if group == "channel" else BLOCK, static=group == "static",
                 atomic=rng.random() < 0.25, mse=rng.random() < 0.15,
                 dtype=rng.choice(("fp16", "bf16")), outliers=rng.choice((0, 8)))
        if rng.random() < 0.3:
            c.update(alpha=0.05, ref_loss=50.0, gmode=rng.choice(("frozen", "frozen", "surrogate_online")))
    if kind == "accum":
        C, G, modules = _width(rng, 256, 14336), rng.choice((1, 2, 4)), rng.choice((1, 1, 2, 3))
        flops = 1.3e13 if dtype != "fp32" else 2e12
        tokens = min(32768, int(flops / (G * modules * C * C)))
        seq = max(1, min(_log(rng, 64, 2048), tokens))
        samples = max(1, min(16, tokens // seq))
        return _case(kind, R=64 * G, C=C, G=G, modules=modules, samples=samples, seq=seq, dtype=dtype,
                     chunks=1, outliers=rng.choice((0, 8)))
    if kind == "quant":
        G = rng.choice((1, 2, 4))
        return _case(kind, R=G * max(16, _width(rng, 64, 14336) // G), C=_width(rng, 256, 6144), G=G, samples=8, **c)
    if kind == "linear":
        G = rng.choice((1, 2, 4))
        return _case(kind, R=G * max(8, _width(rng, 64, 2048) // G), C=_width(rng, 64, 2048), G=G,
                     chunks=rng.choice((1, 2, 4)), samples=rng.randint(1, 8), seq=_log(rng, 32, 1024), **c)
    if kind == "classic":
        group = rng.choice((-1, 64, BLOCK))
        return _case(kind, R=_width(rng, 64, 4096), C=_width(rng, 64, 4096), G=1, chunks=rng.choice((1, 2)),
                     samples=rng.randint(1, 8), seq=_log(rng, 64, 2048), dtype=rng.choice(("fp16", "bf16")),
                     groupsize=group, static=rng.random() < 0.5, mse=rng.random() < 0.25, **c)
    return _case(kind, R=_width(rng, 64, 14336), C=_width(rng, 256, 4096), G=1, samples=1, seq=64,
                 dtype=rng.choice(("fp16", "bf16")), groupsize=rng.choice((-1, BLOCK)), static=True, **c)


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _weight_dtype(case):
    return torch.float16 if case["dtype"] == "fp32" else DTYPES[case["dtype"]]


def _inputs(case, seed, tokens=True):
    """X in chunks of [samples, seq, C] (normal, a few channels twenty times larger), per module a
    saliency [N, seq, G] (log-normal, clipped at its 0.99 quantile), weight (normal, 0.02) and
    gradient (normal, 1e-4)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kw = dict(device="cuda", generator=g)
    C, R, G = case["C"], case["R"], case["G"]
    N = case["samples"] * case["chunks"]
    wide = torch.randperm(C, **kw)[:case["outliers"]]
    X = []
    for _ in range(case["chunks"] if tokens else 0):
        x = torch.randn((case["samples"], case["seq"], C), **kw)
        x[:, :, wide] *= 20.0
        X.append(x.to(DTYPES[case["dtype"]]))
    mods = []
    for _ in range(case["modules"]):
        s = torch.randn((N, case["seq"], G), **kw).exp_()
        flat = s.reshape(-1, G)
        top = flat.sort(dim=0).values[int(0.99 * (flat.shape[0] - 1))]
        s = torch.minimum(s, top)
        W = (torch.randn((R, C), **kw) * 0.02).to(_weight_dtype(case))
        grad = torch.randn((R, C), **kw) * 1e-4
        mods.append((s, W, grad))
    return X, mods


def _layer(W):
    layer = torch.nn.Linear(W.shape[1], W.shape[0], bias=False, device="meta")
    layer.weight = torch.nn.Parameter(W, requires_grad=False)
    return layer


def _quantizer(case):
    q = WeightQuantizer()
    q.configure(case["bits"], perchannel=True, sym=case["sym"], mse=case["mse"])
    return q


def _gptqplus(case, layer, s, grad):
    return GPTQPlus(layer, saliency=s, gradient=grad, num_groups=case["G"], alpha=case["alpha"],
                    reference_loss=case["ref_loss"])


def _hessians(case, X, s):
    """sum of s x x^T per group over the chunks, divided by the tokens, and sum of x^2 divided by the
    tokens of a sample, in 32 bits: the Hessians that a quantising call starts from."""
    C, G = case["C"], case["G"]
    H = torch.zeros((G, C, C), device="cuda")
    act = torch.zeros(C, device="cuda")
    ntok = 0
    for k, x in enumerate(X):
        n = x.shape[0]
        sk = s[k * n:(k + 1) * n].reshape(-1, G)
        x2 = x.reshape(-1, C).float()
        for g in range(G):
            H[g].addmm_((x2 * sk[:, g:g + 1]).t(), x2)
        act += (x2 * x2).sum(0)
        ntok += x2.shape[0]
    H = 0.5 * (H + H.transpose(1, 2)) / ntok
    return H, act / case["seq"]


def _finished(case, seed, hessians=_hessians):
    """A GPTQPlus whose Hessians are finished, as fasterquant finds it, and its weight."""
    X, mods = _inputs(case, seed)
    s, W, grad = mods[0]
    H, act = hessians(case, X, s)
    layer = _layer(W)
    g = _gptqplus(case, layer, s, grad)
    g.add_batch(X[0][:1], None)
    g.finalize_hessian()
    g.H.copy_(H)
    g.act_square.copy_(act)
    return g, layer, W


def _unit_hessians(case, X, s):
    """Hessians under which every code is its weight rounded to nearest."""
    H = torch.eye(case["C"], device="cuda").expand(case["G"], -1, -1)
    return H, X[0].float().square().sum(dim=(0, 1))


def _fasterquant(case, g):
    g.quantizer = _quantizer(case)
    g.fasterquant(blocksize=BLOCK, percdamp=PERCDAMP, groupsize=case["groupsize"], actorder=case["actorder"],
                  static_groups=case["static"], g_update_mode=case["gmode"], block_atomic_quant=case["atomic"])


def prepare(case, seed):
    if case["kind"] == "quant":
        g, layer, W = _finished(case, seed)
        return {"case": case, "g": g, "layer": layer, "W": W}
    if case["kind"] == "packed":
        g, _, _ = _finished(case, seed, _unit_hessians)
        _fasterquant(case, g)
        return {"case": case, "g": g}
    X, mods = _inputs(case, seed)
    return {"case": case, "X": X, "mods": mods, "layers": [_layer(W) for _, W, _ in mods]}


# ---------------------------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------------------------
def _accumulate(state):
    case = state["case"]
    gs = [_gptqplus(case, layer, s, grad) for layer, (s, _, grad) in zip(state["layers"], state["mods"])]
    for x in state["X"]:
        if len(gs) > 1:
            add_batch_shared(gs, x)
        else:
            gs[0].add_batch(x, None)
    for g in gs:
        g.finalize_hessian()
    return gs


def run(state):
    case = state["case"]
    if case["kind"] == "accum":
        gs = _accumulate(state)
        return {"H": [g.H for g in gs], "act": [g.act_square for g in gs]}
    if case["kind"] == "quant":
        g, layer = state["g"], state["layer"]
        layer.weight.data = state["W"]
        _fasterquant(case, g)
        return _quantised(g, layer)
    if case["kind"] == "linear":
        layer = state["layers"][0]
        layer.weight.data = state["mods"][0][1]
        g = _accumulate(state)[0]
        _fasterquant(case, g)
        return dict(_quantised(g, layer), H=g.H, act=g.act_square)
    if case["kind"] == "classic":
        layer = state["layers"][0]
        layer.weight.data = state["mods"][0][1]
        g = GPTQ(layer)
        for x in state["X"]:
            g.add_batch(x, None)
        g.quantizer = _quantizer(case)
        g.fasterquant(blocksize=BLOCK, percdamp=PERCDAMP, groupsize=case["groupsize"], actorder=case["actorder"],
                      static_groups=case["static"])
        return _quantised(g, layer)
    entry = export_packed(state["g"])
    return {"qweight": entry["qweight"], "scales": entry["scales"], "g_idx": entry["g_idx"],
            "weight": dequantize_packed(entry)}


def _quantised(g, layer):
    out = {"weight": layer.weight.data, "scale": g.quantizer.scale}
    if g.perm is not None:
        out["perm"] = g.perm
    return out


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def work(case):
    C, R, G, T = case["C"], case["R"], case["G"], case["modules"]
    n = case["samples"] * case["seq"] * case["chunks"]
    xb, wb = DTYPES[case["dtype"]].itemsize, _weight_dtype(case).itemsize
    if case["kind"] == "packed":
        nbits = case["bits"] + (0 if case["sym"] else 1)
        return {"bytes": R * C * (2 + 2 * nbits / 8 + wb), "flops": 0}
    # X once, the saliencies once, each Hessian written once; the upper triangles' multiply-adds
    acc = {"bytes": n * C * xb + 4 * n * G * T + 4.0 * T * G * C * C, "flops": 1.0 * T * G * n * C * (C + 1)}
    # the Hessians and the weight once, the weight written; factor and inverse of the factor
    # (2/3 C^3 in 64 bits), each column's error into the columns after it, the first-order products
    term = case["alpha"] > 0 and case["kind"] != "classic"
    qnt = {"bytes": 4.0 * G * C * C + R * C * (2.0 * wb + (4 if term else 0)),
           "flops": G * 2 * C ** 3 / 3 + 1.0 * R * C * C * (3 + 2 if term else 1)}
    if case["kind"] == "accum":
        return acc
    if case["kind"] == "quant":
        return qnt
    return {"bytes": acc["bytes"] + qnt["bytes"] - 4.0 * G * C * C, "flops": acc["flops"] + qnt["flops"]}


def tolerance(case):
    if case["kind"] == "accum":
        # 32-bit sums of up to 32768 products in another order
        return {"rel": 4e-6}
    if case["kind"] == "packed":
        return "exact"
    # A weight's code is decided by rounding: where it lies within the 32-bit error of a midpoint
    # it may move by one step, which the rest of its row follows.  One code in 20000 that moves
    # by a step of about half the weights' root mean square is 2e-3 of the weight's norm, and one
    # row of R with three codes in ten moved is 0.27 / sqrt(R).
    return {"rel": min(0.03, max(1e-2 if case["C"] <= 4096 else 2e-2, 0.27 / case["R"] ** 0.5)), "max": 0.99}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits, without this package's code
# ---------------------------------------------------------------------------------------------
def _exact_accum(case, X, s):
    C, G = case["C"], case["G"]
    H = torch.zeros((G, C, C), device="cuda", dtype=torch.float64)
    act = torch.zeros(C, device="cuda", dtype=torch.float64)
    ntok = 0
    for k, x in enumerate(X):
        n = x.shape[0]
        sk = s[k * n:(k + 1) * n].reshape(-1, G).double()
        x2 = x.reshape(-1, C).double()
        for g in range(G):
            H[g].addmm_((x2 * sk[:, g:g + 1]).t(), x2)
        act += (x2 * x2).sum(0)
        ntok += x2.shape[0]
    return H / ntok, act / case["seq"]


def _scale64(w, bits, sym):
    """Per-row step of the range that includes 0 (w [..., n])."""
    lo, hi = w.amin(-1).clamp(max=0.0), w.amax(-1).clamp(min=0.0)
    if sym:
        return torch.maximum(lo.abs(), hi).clamp(min=1e-5) / (2 ** (bits - 1) - 1)
    none = (lo == 0) & (hi == 0)
    lo, hi = torch.where(none, -1.0, lo), torch.where(none, 1.0, hi)
    return (hi - lo).clamp(min=1e-5) / (2 ** bits - 1)


def _exact_quant(case, g, W):
    """fasterquant in 64 bits on the object's Hessians: the weight, and its scale."""
    C, R, G, bits, sym = case["C"], case["R"], case["G"], case["bits"], case["sym"]
    maxq = 2 ** (bits - 1) - 1 if sym else 2 ** bits - 1
    Wd = W.double()
    chan = _scale64(Wd, bits, sym).reshape(-1, 1)
    perm = torch.arange(C)
    if case["actorder"]:
        perm = torch.argsort(g.act_square.cpu(), descending=True)
    perm = perm.to(W.device)
    gs = case["groupsize"]
    table = None
    if gs != -1 and case["static"]:
        table = torch.stack([_scale64(Wd[:, i:i + gs], bits, sym) for i in range(0, C, gs)], 1)
    out = torch.empty_like(Wd)
    rs = R // G
    w, u, z, gh = [], [], [], []
    for k in range(G):
        H = g.H[k].double()
        dead = torch.diagonal(H) == 0
        H[dead, dead] = 1.0
        H = H[perm][:, perm]
        Wk = Wd[k * rs:(k + 1) * rs].clone()
        Wk[:, dead] = 0
        H.diagonal().add_(PERCDAMP * torch.diagonal(H).mean())
        Hi = torch.cholesky_inverse(torch.linalg.cholesky(H))
        U = torch.linalg.cholesky(Hi, upper=True)
        Gk = g.gradients[k * rs:(k + 1) * rs].double()[:, perm]
        beta = torch.zeros(rs, device=W.device, dtype=torch.float64)
        if case["alpha"] > 0:
            gi = Gk @ Hi
            c = (Gk * gi).sum(1) - (gi * gi / torch.diagonal(Hi)).mean(1)
            target = 2 * case["alpha"] / (R * C) * case["ref_loss"]
            beta = 1 - torch.sqrt(1 - (target / c.clamp(min=target)).clamp(0, 1))
        w.append(Wk[:, perm])
        u.append(U)
        z.append((Gk @ U.t()) * beta[:, None])
        gh.append(z[-1] @ U)
    w, u, z, gh = (torch.stack(t) for t in (w, u, z, gh))
    chan3 = chan.reshape(G, rs, 1)
    Q = torch.empty_like(w)
    for i1 in range(0, C, BLOCK):
        i2 = min(i1 + BLOCK, C)
        n = i2 - i1
        w1, g1 = w[:, :, i1:i2].clone(), gh[:, :, i1:i2].clone()
        if gs == -1:
            s = chan3.expand(G, rs, n)
        elif case["static"]:
            s = table[:, perm[i1:i2] // gs].reshape(G, rs, n)
        else:
            s = _scale64(w1, bits, sym)[..., None].expand(G, rs, n)
        u1 = u[:, i1:i2, i1:i2]
        err = torch.empty_like(w1)
        if case["atomic"] and i2 < C:
            Q[:, :, i1:i2] = s * torch.clamp(torch.round(w1 / s), -(maxq + 1), maxq)
            err = torch.linalg.solve_triangular(u1, w1 - Q[:, :, i1:i2] - g1, upper=True, left=False)
        else:
            for i in range(n):
                q = s[:, :, i] * torch.clamp(torch.round(w1[:, :, i] / s[:, :, i]), -(maxq + 1), maxq)
                Q[:, :, i1 + i] = q
                e = (w1[:, :, i] - q - g1[:, :, i]) / u1[:, None, i, i]
                err[:, :, i] = e
                w1[:, :, i:] -= e[:, :, None] * u1[:, None, i, i:] + g1[:, :, i:]
                g1[:, :, i:] -= z[:, :, i1 + i, None] * u1[:, None, i, i:]
        if i2 < C:
            tail = u[:, i1:i2, i2:]
            z1 = z[:, :, i1:i2]
            left = torch.arange(n - 1, -1, -1, device=W.device, dtype=torch.float64)
            w[:, :, i2:] -= err @ tail + n * gh[:, :, i2:] - (z1 * left) @ tail
            gh[:, :, i2:] -= z1 @ tail
    out[:, perm] = Q.reshape(R, C)
    return out.to(W.dtype).double(), chan


def exact(case, seed):
    """The Hessians have a value in 64 bits.  So has the quantised weight where its Hessians are given
    and nothing but rounding stands between; with a search over clipped ranges, with a weight so
    small that single codes decide, or where the width would take minutes, it has none here."""
    if case["kind"] == "accum":
        X, mods = _inputs(case, seed)
        found = [_exact_accum(case, X, s) for s, _, _ in mods]
        return {"H": [h for h, _ in found], "act": [a for _, a in found]}
    if case["kind"] == "linear":
        X, mods = _inputs(case, seed)
        H, act = _exact_accum(case, X, mods[0][0])
        return {"H": H, "act": act, "weight": None, "scale": None, "perm": None}
    if case["kind"] == "quant" and not case["mse"] and case["gmode"] == "frozen":
        if case["C"] > 8192 or case["R"] * case["C"] < 4_000_000:
            return None
        g, _, W = _finished(case, seed)
        Q, chan = _exact_quant(case, g, W)
        return {"weight": Q, "scale": chan, "perm": None}
    return None
