"""The work a user of this framework has it do, as cases to be timed and checked.

Every case goes through the public entry points of ``myelin_amd`` with the
shapes of this repository's own workloads (``bench.py``) or generic ones of
the same ranges, odd sizes among them:

  lif           fused-time LIF inference
  lif_packed    LIF inference that emits bitpacked spikes only
  surrogate_lif, surrogate_alif
                a neuron layer's training step over given currents: forward
                and reverse-time surrogate backward
  layer         a dense synapse streamed into LIF, training step (spikes,
                kept packed, and the gradients of weight, bias and, for an
                inner layer, input)
  layer_packed  the same layer's inference with bitpacked output
  classifier    hidden layer + rate readout, training step on its rates
  long_rate     the packed-hidden two-layer rate network, training step
  codec         pack, unpack, per-neuron counts over time, per-sample rates
"""

from __future__ import annotations

import math

import torch

import myelin_amd as myelin

DEV = "cuda:0"
SURROGATES = ("fast_sigmoid", "atan", "superspike")
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "u8": torch.uint8}


def listed():
    return [
        # the smallest workload: a 64 x 1024 population over 100 steps, some
        # microseconds of GPU time, so launches and host work count
        {"name": "lif_inference", "kind": "lif", "T": 100, "B": 64, "N": 1024},
        # spikes kept packed between layers; 3000 is no multiple of the 32-bit word
        {"name": "lif_packed_ragged", "kind": "lif_packed", "T": 200, "B": 48, "N": 3000},
        # training a neuron layer of odd sizes (no vector width divides B * N)
        {"name": "surrogate_lif_odd", "kind": "surrogate_lif", "T": 150, "B": 37, "N": 2051, "surrogate": "atan"},
        # the headline training step: adaptive LIF [256, 128, 4096]
        {"name": "surrogate_alif_headline", "kind": "surrogate_alif", "T": 256, "B": 128, "N": 4096,
         "surrogate": "fast_sigmoid"},
        # the hidden layer 784 -> 2048 over Poisson-coded input at the default
        # fp32 synapse, and the same layer at the bf16 option
        {"name": "layer_fp32", "kind": "layer", "T": 50, "B": 256, "F": 784, "N": 2048, "surrogate": "atan",
         "precision": "fp32", "checkpoint": "none", "inputs": "spikes", "inner": False},
        {"name": "layer_bf16", "kind": "layer", "T": 50, "B": 256, "F": 784, "N": 2048, "surrogate": "atan",
         "precision": "bf16", "checkpoint": "none", "inputs": "spikes", "inner": False},
        # an inner layer over real-valued features of ragged widths,
        # checkpointed, with the gradient of its input
        {"name": "layer_analog_inner", "kind": "layer", "T": 100, "B": 64, "F": 700, "N": 1000,
         "surrogate": "fast_sigmoid", "precision": "fp32", "checkpoint": "balanced", "inputs": "analog",
         "inner": True},
        # deployment: spikes of a 1024 -> 2048 layer straight to packed words
        {"name": "layer_packed_inference", "kind": "layer_packed", "T": 100, "B": 128, "F": 1024, "N": 2048},
        # the small classifier: 784 -> 256 -> 10, batch 128, 25 steps; tens of
        # launches of a few microseconds each
        {"name": "classifier_small", "kind": "classifier", "T": 25, "B": 128, "F": 784, "H": 256, "O": 10},
        # the long horizon: 2000 steps, 1024 -> 4096 -> 20, hidden spikes packed
        {"name": "long_rate_packed", "kind": "long_rate", "T": 2000, "B": 32, "F": 1024, "H": 4096, "O": 20,
         "checkpoint": 45},
        # the spike codec on a large raster, and on ragged byte rasters as
        # event data and bool comparisons give them
        {"name": "codec_large", "kind": "codec", "T": 512, "B": 64, "N": 8192, "dtype": "f32"},
        {"name": "codec_ragged_bytes", "kind": "codec", "T": 300, "B": 50, "N": 2312, "dtype": "u8"},
    ]


# ------------------------------------------------------------------- ranges
def _log(rng, lo, hi):
    """Sizes spread over the logarithm of their range, odd ones among them."""

    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """Layer widths: two in three a multiple of 64 or 8, the rest as drawn."""

    n = _log(rng, lo, hi)
    step = rng.choice((64, 8, 1))
    return max(lo, min(hi, n // step * step))


def _cost(case):
    """Rough seconds of a pass, to keep drawn cases below the largest listed one."""

    w = work(case)
    bf16 = case.get("precision") == "bf16" or case["kind"] == "long_rate"
    return w["bytes"] / 3e12 + w["flops"] / (4e14 if bf16 else 1e14)


def _cells(case):
    return case["T"] * case["B"] * max(case.get(k, 1) for k in ("F", "N", "H"))


def draw(rng):
    while True:
        kind = rng.choice(("lif", "lif_packed", "surrogate_lif", "surrogate_alif", "layer", "layer", "layer",
                           "layer_packed", "classifier", "long_rate", "codec"))
        c = {"kind": kind}
        if kind in ("lif", "lif_packed", "surrogate_lif", "surrogate_alif"):
            c.update(T=_log(rng, 10, 512), B=_log(rng, 1, 256), N=_width(rng, 32, 8192))
            if kind.startswith("surrogate"):
                c["surrogate"] = rng.choice(SURROGATES)
        elif kind in ("layer", "layer_packed"):
            c.update(T=_log(rng, 10, 400), B=_log(rng, 8, 512), F=_width(rng, 64, 2048), N=_width(rng, 64, 4096))
            if kind == "layer":
                c.update(surrogate=rng.choice(SURROGATES), precision=rng.choice(("fp32", "fp32", "bf16")),
                         checkpoint=rng.choice(("none", "balanced")), inputs=rng.choice(("spikes", "spikes", "analog")),
                         inner=rng.random() < 0.5)
        elif kind == "classifier":
            c.update(T=_log(rng, 10, 100), B=_log(rng, 16, 256), F=_width(rng, 64, 1024), H=_width(rng, 64, 2048),
                     O=_log(rng, 2, 32))
        elif kind == "long_rate":
            c.update(T=_log(rng, 300, 2000), B=_log(rng, 4, 32), F=_width(rng, 128, 1024), H=_width(rng, 256, 4096),
                     O=_log(rng, 2, 32), checkpoint=_log(rng, 20, 100))
        else:
            c.update(T=_log(rng, 16, 512), B=_log(rng, 1, 64), N=_width(rng, 64, 8192),
                     dtype=rng.choice(("f32", "f32", "bf16", "u8")))
        if 1 << 16 <= _cells(c) <= 1 << 28 and _cost(c) <= _cost(listed()[9]):
            return c


# ------------------------------------------------------------------- inputs
def _bernoulli_raster(g, T, B, N):
    """0/1 spikes, each unit with a rate of its own in [0, 0.2)."""

    rate = 0.2 * torch.rand(N, generator=g, device=DEV)
    return (torch.rand((T, B, N), generator=g, device=DEV) < rate).float()


def _weight(g, fan_in, fan_out):
    """Kaiming-uniform [in, out]."""

    bound = math.sqrt(6.0 / fan_in)
    return (2.0 * torch.rand((fan_in, fan_out), generator=g, device=DEV) - 1.0) * bound


def _bias(g, n):
    return 0.02 * torch.randn(n, generator=g, device=DEV)


def _inputs(case, seed):
    """All tensors of a case, made on the GPU from the seed alone."""

    g = torch.Generator(device=DEV).manual_seed(seed)
    k, T, B = case["kind"], case["T"], case["B"]
    d = {}
    if k in ("lif", "lif_packed", "surrogate_lif", "surrogate_alif"):
        N = case["N"]
        d["x"] = 0.25 + 0.6 * torch.randn((T, B, N), generator=g, device=DEV)
        d["m0"] = torch.rand((B, N), generator=g, device=DEV) * 0.5
        if k == "surrogate_alif":
            d["a0"] = torch.rand((B, N), generator=g, device=DEV) * 0.2
        if k.startswith("surrogate"):
            d["gs"] = torch.randn((T, B, N), generator=g, device=DEV)
    elif k in ("layer", "layer_packed"):
        F, N = case["F"], case["N"]
        if case.get("inputs", "spikes") == "spikes":
            d["x"] = _bernoulli_raster(g, T, B, F)
        else:
            d["x"] = 0.35 * torch.randn((T, B, F), generator=g, device=DEV)
        d["w"], d["b"] = _weight(g, F, N), _bias(g, N)
        if k == "layer":
            d["gs"] = torch.randn((T, B, N), generator=g, device=DEV)
    elif k in ("classifier", "long_rate"):
        F, H, O = case["F"], case["H"], case["O"]
        d["x"] = _bernoulli_raster(g, T, B, F)
        d["wh"], d["bh"] = _weight(g, F, H), _bias(g, H)
        d["wo"], d["bo"] = _weight(g, H, O), _bias(g, O)
        d["gr"] = torch.randn((B, O), generator=g, device=DEV)
    else:
        N = case["N"]
        rate = torch.exp(-3.0 + torch.randn(N, generator=g, device=DEV)).clamp(0.0, 1.0)
        d["x"] = (torch.rand((T, B, N), generator=g, device=DEV) < rate).to(DTYPES[case["dtype"]])
    return d


LIF = myelin.LIFParams(tau_mem=20.0, threshold=1.0, reset=0.0)
ALIF = myelin.ALIFParams(tau_mem=20.0, tau_adaptation=50.0, threshold=1.0, reset=0.0, beta=1.8)
SLOPE = 10.0
LAYER_SLOPE = 5.0  # of the classifier and the layers in it
FNS = {"fast_sigmoid": myelin.fast_sigmoid_surrogate, "atan": myelin.atan_surrogate,
       "superspike": myelin.superspike_surrogate}


def _set(synapse, w, b):
    with torch.no_grad():
        synapse.weight.copy_(w)
        synapse.bias.copy_(b)


def prepare(case, seed):
    d = _inputs(case, seed)
    k = case["kind"]
    st = {"case": case, "x": d["x"]}
    if k in ("lif", "lif_packed", "surrogate_lif"):
        st["state"] = myelin.LIFState(membrane=d["m0"])
    elif k == "surrogate_alif":
        st["state"] = myelin.ALIFState(membrane=d["m0"], adaptation=d["a0"])
    if k.startswith("surrogate"):
        st["x"].requires_grad_()
        st["gs"] = d["gs"]
    if k == "layer":
        ck = None if case["checkpoint"] == "none" else case["checkpoint"]
        layer = myelin.LinearSurrogateLIF(case["F"], case["N"], LIF, surrogate=FNS[case["surrogate"]],
                                          surrogate_slope=LAYER_SLOPE, stream_synapse=True, checkpoint_size=ck,
                                          synapse_precision=case["precision"]).to(DEV)
        _set(layer.synapse, d["w"], d["b"])
        st["layer"], st["gs"] = layer, d["gs"]
        st["wrt"] = list(layer.parameters())
        if case["inner"]:
            st["wrt"].append(st["x"].requires_grad_())
    elif k == "layer_packed":
        layer = myelin.LinearSurrogateLIFPacked(case["F"], case["N"], LIF).to(DEV)
        _set(layer.synapse, d["w"], d["b"])
        st["layer"] = layer
    elif k == "classifier":
        net = myelin.RateReadoutClassifier(case["F"], case["H"], case["O"], LIF, checkpoint_size="balanced").to(DEV)
        _set(net.hidden.synapse, d["wh"], d["bh"])
        _set(net.output.synapse, d["wo"], d["bo"])
        st["net"], st["gr"], st["wrt"] = net, d["gr"], list(net.parameters())
    elif k == "long_rate":
        st["wrt"] = [d[n].requires_grad_() for n in ("wh", "bh", "wo", "bo")]
        st["gr"] = d["gr"]
    return st


def run(st):
    c, x = st["case"], st["x"]
    k = c["kind"]
    if k == "lif":
        out, spikes = myelin.lif_forward(x, st["state"], LIF)
        return [out.membrane, spikes]
    if k == "lif_packed":
        out, packed = myelin.lif_forward_packed_spikes(x, st["state"], LIF)
        return [out.membrane, packed.data]
    if k == "surrogate_lif":
        out, spikes = myelin.surrogate_lif_forward(x, st["state"], LIF, surrogate=c["surrogate"],
                                                   surrogate_slope=SLOPE)
        return [out.membrane, spikes, *torch.autograd.grad(spikes, [x], st["gs"])]
    if k == "surrogate_alif":
        out, spikes = myelin.surrogate_alif_forward(x, st["state"], ALIF, surrogate=c["surrogate"],
                                                    surrogate_slope=SLOPE)
        return [out.membrane, out.adaptation, spikes, *torch.autograd.grad(spikes, [x], st["gs"])]
    if k == "layer":
        # the raster is kept packed, as a program that stores or sends it does
        spikes = st["layer"](x)
        return [myelin.pack_spikes(spikes.detach()).data, *torch.autograd.grad(spikes, st["wrt"], st["gs"])]
    if k == "layer_packed":
        with torch.no_grad():
            return [st["layer"](x).data]
    if k == "classifier":
        rates = st["net"](x)
        return [rates, *torch.autograd.grad(rates, st["wrt"], st["gr"])]
    if k == "long_rate":
        wh, bh, wo, bo = st["wrt"]
        rates = myelin.two_layer_surrogate_lif_rate_packed_hidden_forward(
            x, wh, bh, wo, bo, LIF, surrogate="superspike", surrogate_slope=SLOPE, checkpoint_size=c["checkpoint"])
        return [rates, *torch.autograd.grad(rates, st["wrt"], st["gr"])]
    packed = myelin.pack_spikes(x)
    return [packed.data, myelin.unpack_spikes(packed, dtype=x.dtype), myelin.packed_spike_count(packed, dim=0),
            myelin.packed_spike_rate(packed, dim=(0, -1))]


# --------------------------------------------------------- bytes, operations
def work(case):
    k, T, B = case["kind"], case["T"], case["B"]
    if k in ("lif", "lif_packed", "surrogate_lif", "surrogate_alif"):
        n = T * B * case["N"]
        per = {"lif": 8, "lif_packed": 4 + 1 / 8, "surrogate_lif": 20, "surrogate_alif": 20}[k]
        return {"bytes": n * per, "flops": n * {"lif": 4, "lif_packed": 4}.get(k, 20)}
    if k in ("layer", "layer_packed"):
        F, N = case["F"], case["N"]
        macs, wb = T * B * F * N, 4 * F * N
        if k == "layer_packed":
            return {"bytes": T * B * (4 * F + N / 8) + wb, "flops": 2 * macs}
        inner = 1 if case["inner"] else 0
        # x, W read; spikes written, dense and packed; dL/dspikes read; dW (and dX) written
        return {"bytes": T * B * (4 * F + 8 * N + N / 8 + 4 * F * inner) + 2 * wb, "flops": 2 * macs * (2 + inner)}
    if k in ("classifier", "long_rate"):
        F, H, O = case["F"], case["H"], case["O"]
        # the hidden synapse and its dW; the readout's currents, dS and dW
        return {"bytes": 4 * T * B * F + 8 * (F * H + H * O), "flops": 2 * T * B * (2 * F * H + 3 * H * O)}
    n = T * B * case["N"]
    size = DTYPES[case["dtype"]].itemsize
    return {"bytes": n * (2 * size + 1 / 8) + 8 * B * case["N"], "flops": n}


# ---------------------------------------------------------------- tolerances
def tolerance(case):
    """About four times what the start's outputs differ by from ``exact``.

    A neuron whose membrane meets the threshold within the sum's rounding
    spikes a step earlier or later in another order of the sum: a few spikes
    in 10^7, of which each changes one neuron's chain of gradients by its
    whole size (measured over seeds and drawn sizes: none to 7e-3 of the
    gradients' 2-norm for a layer, to 1e-3 for the networks, and to 0.8 of
    the root mean square at single elements).  bf16 operands: 1.3e-3 to
    2.7e-3."""

    k = case["kind"]
    if k in ("lif", "lif_packed", "codec"):
        return "exact"  # elementwise fp32 in a stated order, and integers
    if k in ("surrogate_lif", "surrogate_alif"):
        return {"rel": 1e-5, "max": 1e-3}  # spikes exact, fp32 adjoint
    # one flipped spike in a small raster is 1e-3 of its words
    rel = 2.5e-2 if k == "layer" and case["precision"] == "fp32" else 1e-2
    return {"rel": rel, "max": 0.95, "differ": 1e-3}


# ------------------------------------------------------------- 64-bit oracle
def _derivative(name, c):
    if name == "fast_sigmoid":
        return 0.5 / (1.0 + c.abs()) ** 2
    if name == "superspike":
        return 1.0 / (1.0 + c.abs()) ** 2
    return 0.5 / (1.0 + (0.5 * math.pi * c) ** 2)


def _unroll(cur, m, p, a=None):
    """(m', threshold distance, spikes, final m, final a) of the unroll; a: ALIF."""

    pre, dist, spikes = torch.empty_like(cur), torch.empty_like(cur), torch.empty_like(cur)
    for t in range(cur.shape[0]):
        mp = m * p.decay + cur[t]
        d = mp - p.threshold if a is None else mp - (p.threshold + p.beta * a)
        s = (d >= 0).double()
        pre[t], dist[t], spikes[t] = mp, d, s
        m = mp * (1.0 - s) + p.reset * s
        if a is not None:
            a = a * p.adaptation_decay + s
    return pre, dist, spikes, m, a


def _adjoint(pre, dist, spikes, gs, p, surrogate, slope=SLOPE, alif=False):
    """dL/d(current) from dL/dspikes (a tensor [T, B, N], or [B, N] at every step)."""

    g = torch.empty_like(pre)
    gm = torch.zeros_like(pre[0])
    ga = torch.zeros_like(gm)
    for t in range(pre.shape[0] - 1, -1, -1):
        q = gm * (p.reset - pre[t]) + (gs[t] if gs.ndim == 3 else gs) + ga
        gc = q * slope * _derivative(surrogate, slope * dist[t])
        g[t] = gm * (1.0 - spikes[t]) + gc
        if alif:
            ga = ga * p.adaptation_decay - p.beta * gc
        gm = g[t] * p.decay
    return g


def exact(case, seed):
    k, T, B = case["kind"], case["T"], case["B"]
    if k == "layer_packed":
        return None  # words only
    raw = _inputs(case, seed)
    d = {n: t.double() for n, t in raw.items()}
    if k in ("lif", "lif_packed"):
        _, _, s, m, _ = _unroll(d["x"], d["m0"], LIF)
        return [m, s if k == "lif" else None]
    if k in ("surrogate_lif", "surrogate_alif"):
        alif = k == "surrogate_alif"
        p = ALIF if alif else LIF
        pre, dist, s, m, a = _unroll(d["x"], d["m0"], p, d.get("a0"))
        g = _adjoint(pre, dist, s, d["gs"], p, case["surrogate"], alif=alif)
        return [m, a, s, g] if alif else [m, s, g]
    if k == "layer":
        x, w, F = d["x"], d["w"], case["F"]
        if case["precision"] == "bf16":  # the option rounds the products' operands
            x, w = raw["x"].bfloat16().double(), raw["w"].bfloat16().double()
        cur = (x.reshape(T * B, F) @ w + d["b"]).reshape(T, B, -1)
        pre, dist, s, _, _ = _unroll(cur, torch.zeros_like(cur[0]), LIF)
        g = _adjoint(pre, dist, s, d["gs"], LIF, case["surrogate"], LAYER_SLOPE).reshape(T * B, -1)
        out = [None, x.reshape(T * B, F).t() @ g, g.sum(0)]
        return out + [(g @ w.t()).reshape(T, B, F)] if case["inner"] else out
    if k in ("classifier", "long_rate"):
        F, H = case["F"], case["H"]
        # RateReadoutClassifier's defaults, and what run() passes
        sg, slope = ("fast_sigmoid", LAYER_SLOPE) if k == "classifier" else ("superspike", SLOPE)
        x2 = d["x"].reshape(T * B, F)
        cur = (x2 @ d["wh"] + d["bh"]).reshape(T, B, H)
        pre, dist, s, _, _ = _unroll(cur, torch.zeros_like(cur[0]), LIF)
        del cur
        s2 = s.reshape(T * B, H)
        cur_o = (s2 @ d["wo"] + d["bo"]).reshape(T, B, -1)
        pre_o, dist_o, s_o, _, _ = _unroll(cur_o, torch.zeros_like(cur_o[0]), LIF)
        g_o = _adjoint(pre_o, dist_o, s_o, d["gr"] / T, LIF, sg, slope).reshape(T * B, -1)
        g_h = _adjoint(pre, dist, s, (g_o @ d["wo"].t()).reshape(T, B, H), LIF, sg, slope).reshape(T * B, H)
        return [s_o.mean(0), x2.t() @ g_h, g_h.sum(0), s2.t() @ g_o, g_o.sum(0)]
    counts = raw["x"].long()
    return [None, d["x"] if DTYPES[case["dtype"]].is_floating_point else None, None,
            counts.sum((0, 2)).double() / (T * case["N"])]
