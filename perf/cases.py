"""Workloads a user of this framework runs, for timing it over its real range.

A case is one call of a user's program on one LTC layer: a training step
(forward and backward through the module, or through the function-level entry
point), a captured training step, or inference (training-mode module without
grad, or the eval-mode module). `listed()` names the fixed ones, `draw(rng)`
gives more of the same ranges, `prepare` makes what the program holds before
the call, `run` is the call, `exact` the same outputs from plain torch in
float64.

Keys of a case:
  mode      "train"     module in training mode: forward, backward, all gradients
            "captured"  the same as one replayed HIP graph (ltc_cuda.CapturedStep)
            "boundary"  ltc_cuda.ltc_cuda_forward on the 13 boundary tensors, with
                        the gradients of all of them
            "infer"     module in training mode under no_grad
            "eval"      module in eval mode under no_grad (cached transforms)
  B T D H U batch rows, time steps, inputs, neurons, ODE unfolds per step
  density   Bernoulli density of the recurrent and the sensory mask (1.0: dense)
  x         "normal" N(0,1), "uniform" U(-3,3), "strided" every second input of a
            tensor twice as wide
  loss      training modes: "sum" of the outputs, "mse" against a target, or
            "upstream" (the layer inside a network: a given dL/dout, and dL/dx back)
  h0        whether an initial state is given (else the module's zero state)
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "ltc-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ltc  # noqa: E402
import ltc_cuda  # noqa: E402

DEV = "cuda"
DT = 1.0 / 30.0
EPS = 1e-8

LEAVES = ("w", "erev", "mu", "sigma", "sensory_w", "sensory_erev", "sensory_mu",
          "sensory_sigma", "gleak", "vleak", "cm", "input_w", "input_b",
          "input_norm.weight", "input_norm.bias")
MASKS = ("sparsity_mask", "sensory_sparsity_mask")
# The function-level entry point's parameters, in its argument order.
BOUNDARY = ("w_pos", "w_erev", "mu", "sigma", "sensory_mu", "sensory_sigma", "sensory_erev",
            "sensory_w_pos", "cm_t", "gleak_pos", "vleak")


def _case(name, mode, B, T, D, H, U=6, density=0.5, x="normal", loss="upstream", h0=False):
    return {"name": name, "mode": mode, "B": B, "T": T, "D": D, "H": H, "U": U,
            "density": density, "x": x, "loss": loss, "h0": h0}


def listed():
    return [
        # One control tick of a deployed policy: one robot, one frame, the state
        # carried by the caller. Latency and launches are all there is.
        _case("eval_tick_b1", "eval", 1, 1, 128, 64, h0=True),
        # The headline step (24 windows of 8 frames), as a user who minds host
        # time runs it: one graph replay per batch.
        _case("train_captured_b24", "captured", 24, 8, 128, 64, loss="sum"),
        # An ordinary eager training step of a middle-sized layer.
        _case("train_b32_h128", "train", 32, 16, 128, 128, loss="sum"),
        # The same kind of layer inside a network, a larger batch, sizes that
        # are not multiples of 64.
        _case("train_b128_h100", "train", 128, 25, 100, 100, h0=True),
        # The reference's production input width (224) with a layer between the
        # powers of two.
        _case("train_b64_h192", "train", 64, 32, 224, 192),
        # Long-sequence training batch.
        _case("train_b256_h256", "train", 256, 64, 256, 256, loss="mse"),
        # A wide layer with the default half-dense wiring.
        _case("train_b64_h512", "train", 64, 32, 256, 512),
        # Dense wiring, inputs that push the gates to saturation: the largest.
        _case("train_dense_b128_h512", "train", 128, 32, 512, 512, density=1.0, x="uniform",
              loss="sum"),
        # The function-level entry point with autograd (a program that keeps its
        # own parameter transforms), many short windows through a small layer.
        _case("boundary_b1024_h64", "boundary", 1024, 16, 64, 64, h0=True),
        # Streaming inference over many streams, input sliced in place.
        _case("infer_b4096_h64", "infer", 4096, 4, 64, 64, x="strided"),
        # Batch scoring with a wider layer.
        _case("infer_b1024_h256", "infer", 1024, 8, 128, 256),
        # Offline rollout of a trained layer over long recordings, odd sizes.
        _case("eval_rollout_h320", "eval", 8, 100, 33, 320, h0=True),
    ]


def _synapses(c):
    return c["B"] * c["T"] * (c["D"] * c["H"] + c["U"] * c["H"] ** 2)


def _trains(c):
    return c["mode"] in ("train", "captured", "boundary")


def draw(rng):
    """A case of the same ranges; sizes spread over their logarithm, at most a
    quarter of the largest listed case's synapse evaluations."""

    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    cap = 0.25 * 3.2 * 128 * 32 * (512 * 512 + 6 * 512 * 512)
    while True:
        mode = rng.choice(["train", "train", "train", "infer", "eval", "boundary", "captured"])
        c = {"mode": mode, "B": logint(1, 4096 if mode in ("infer", "boundary") else 1024),
             "T": logint(1, 100), "D": logint(8, 512), "H": logint(16, 768),
             "U": rng.choice([6, 6, 6, 3, 10]),
             "density": rng.choice([0.5, 0.5, 0.5, 0.3, 1.0]),
             "x": rng.choice(["normal", "normal", "uniform", "strided"]),
             "loss": rng.choice(["upstream", "upstream", "sum", "mse"]),
             "h0": rng.random() < 0.5}
        if mode == "captured":
            # what the capture is for: steps bound by the host
            c["B"] = min(c["B"], 64)
            c["T"] = min(c["T"], 32)
            c["H"] = min(c["H"], 128)
        if (3.2 if _trains(c) else 1.0) * _synapses(c) <= cap:
            return c


# ------------------------------------------------------------------------- inputs


def _wiring(rows, H, density, g):
    """Bernoulli mask with no empty column, and +/-1 reversal signs, as the layer's own."""
    if density >= 1.0:
        mask = torch.ones(rows, H)
    else:
        mask = (torch.rand(rows, H, generator=g) < density).float()
        for col in (mask.sum(0) == 0).nonzero().flatten().tolist():
            mask[int(torch.randint(0, rows, (1,), generator=g)), col] = 1.0
    sign = torch.where(torch.rand(rows, H, generator=g) < 0.8, 1.0, -1.0)
    return mask, sign * mask


def _inputs(c, seed):
    """Leaves (the layer's init ranges, LayerNorm and affine as after some
    training), x, h0, target and dL/dout of a seed, on the host in float32."""
    g = torch.Generator().manual_seed(seed * 1000003 + 17)
    B, T, D, H = c["B"], c["T"], c["D"], c["H"]

    def uni(lo, hi, *shape):
        return torch.rand(*shape, generator=g) * (hi - lo) + lo

    p = {"w": uni(0.001, 1.0, H, H), "mu": uni(0.3, 0.8, H, H), "sigma": uni(3.0, 8.0, H, H)}
    p["sparsity_mask"], p["erev"] = _wiring(H, H, c["density"], g)
    p["sensory_w"] = uni(0.001, 1.0, D, H)
    p["sensory_mu"], p["sensory_sigma"] = uni(0.3, 0.8, D, H), uni(3.0, 8.0, D, H)
    p["sensory_sparsity_mask"], p["sensory_erev"] = _wiring(D, H, c["density"], g)
    p["gleak"], p["vleak"] = uni(0.001, 1.0, H), uni(-0.2, 0.2, H)
    p["cm"] = uni(0.4, 0.6, H)
    p["input_w"], p["input_b"] = uni(0.9, 1.1, D), uni(-0.1, 0.1, D)
    p["input_norm.weight"], p["input_norm.bias"] = uni(0.9, 1.1, D), uni(-0.1, 0.1, D)
    wide = 2 * D if c["x"] == "strided" else D
    if c["x"] == "uniform":
        x = uni(-3.0, 3.0, B, T, D)
    else:
        x = torch.randn(B, T, wide, generator=g)
    h0 = torch.randn(B, H, generator=g) * 0.2 if c["h0"] else None
    target = grad = None
    if _trains(c) and c["loss"] == "mse":
        target = torch.randn(B, T, H, generator=g)
    if _trains(c) and c["loss"] == "upstream":
        grad = torch.randn(B, T, H, generator=g)
    return p, x, h0, target, grad


def _transforms(p, U):
    """The boundary parameters of the leaves (ltc.py:259-288), in p's precision."""
    w_pos = F.softplus(p["w"]) * p["sparsity_mask"]
    return {"w_pos": w_pos, "w_erev": w_pos * p["erev"], "mu": p["mu"], "sigma": p["sigma"],
            "sensory_mu": p["sensory_mu"], "sensory_sigma": p["sensory_sigma"],
            "sensory_erev": p["sensory_erev"],
            "sensory_w_pos": F.softplus(p["sensory_w"]) * p["sensory_sparsity_mask"],
            "cm_t": F.softplus(p["cm"]) / (DT / U), "gleak_pos": F.softplus(p["gleak"]),
            "vleak": p["vleak"]}


def _normalise(p, x):
    xn = F.layer_norm(x, x.shape[-1:], p["input_norm.weight"], p["input_norm.bias"], 1e-5)
    return xn * p["input_w"] + p["input_b"]


def _loss(c, out, target):
    return out.sum() if c["loss"] == "sum" else F.mse_loss(out, target)


def prepare(case, seed):
    c = case
    p, x, h0, target, grad = _inputs(c, seed)
    st = {"case": c}
    x = x.to(DEV)
    if c["x"] == "strided":
        x = x[:, :, 0::2]
    st["target"] = None if target is None else target.to(DEV)
    st["grad"] = None if grad is None else grad.to(DEV)
    st["h0"] = None if h0 is None else h0.to(DEV)
    if c["mode"] == "boundary":
        # A program with its own transforms: it holds the 13 tensors.
        dp = {k: v.to(DEV) for k, v in p.items()}
        bp = _transforms(dp, c["U"])
        st["x"] = _normalise(dp, x).detach().requires_grad_(True)
        h = torch.zeros(c["B"], c["H"], device=DEV) if h0 is None else st["h0"]
        st["h0"] = h.requires_grad_(True)
        st["params"] = [bp[k].detach().clone().requires_grad_(True) for k in BOUNDARY]
        return st
    m = ltc.TrueLiquidTimeConstant(c["D"], c["H"], dt=DT, ode_unfolds=c["U"], sparsity=1.0,
                                   sensory_sparsity=1.0, epsilon=EPS)
    m.load_state_dict(p)
    m = m.to(DEV)
    st["module"] = m
    if c["mode"] == "eval":
        m.eval()
    if c["mode"] == "train" and c["loss"] == "upstream":
        x = x.detach().requires_grad_(True)
    st["x"] = x
    if c["mode"] == "captured":
        hs = None if st["h0"] is None else (st["h0"], st["h0"])
        tgt, up = st["target"], st["grad"]

        def loss_fn(o):
            return (o[0] * up).sum() if up is not None else _loss(c, o[0], tgt)

        args = (x.clone(),) if hs is None else (x.clone(), hs)
        st["step"] = ltc_cuda.CapturedStep(m, args, loss_fn)
    return st


def run(state):
    c = state["case"]
    if c["mode"] == "captured":
        step = state["step"]
        step.inputs[0].copy_(state["x"])
        step.replay()
        return [step.outputs[0], step.outputs[1][0], *step.grads]
    x, h0 = state["x"], state["h0"]
    if c["mode"] == "boundary":
        leaves = [x, h0, *state["params"]]
        out, h = ltc_cuda.ltc_cuda_forward(x, h0, *state["params"], c["U"], EPS)
        if c["loss"] == "upstream":
            grads = torch.autograd.grad(out, leaves, state["grad"])
        else:
            grads = torch.autograd.grad(_loss(c, out, state["target"]), leaves)
        return [out.detach(), h.detach(), *grads]
    m = state["module"]
    hs = None if h0 is None else (h0, h0)
    if c["mode"] in ("infer", "eval"):
        with torch.no_grad():
            out, (h, _) = m(x, hs)
        return [out, h]
    m.zero_grad()
    out, (h, _) = m(x, hs)
    grads = []
    if c["loss"] == "upstream":
        x.grad = None
        out.backward(state["grad"])
        grads.append(x.grad)
    else:
        _loss(c, out, state["target"]).backward()
    return [out.detach(), h.detach(), *grads, *[q.grad for q in m.parameters()]]


# ------------------------------------------------------------- what a pass must do


def work(case):
    """Inputs read once and outputs written once. Operations: per synapse that
    the masks leave, 10 for a forward evaluation (gate 6, two products and two
    sums 4) and 22 more for its backward."""
    c = case
    B, T, D, H, U = c["B"], c["T"], c["D"], c["H"], c["U"]
    n = c["density"] * _synapses(c)
    params = 4 * H * H + 4 * D * H + 3 * H
    masks = 0
    if c["mode"] != "boundary":
        params += 4 * D
        masks = H * H + D * H
    floats = B * T * D + params + masks + B * T * H + B * H + (B * H if c["h0"] else 0)
    flops = 10.0 * n
    if _trains(c):
        # dL/dout, every parameter's gradient, and dL/dx (dL/dh0) where asked
        floats += (B * T * H if c["loss"] != "sum" else 0) + params
        if c["mode"] == "boundary" or c["loss"] == "upstream" and c["mode"] == "train":
            floats += B * T * D
        if c["mode"] == "boundary":
            floats += B * H
        flops += 22.0 * n
    return {"bytes": 4.0 * floats, "flops": flops}


def tolerance(case):
    """About four times the largest error against `exact` over the listed and
    some 80 drawn cases: outputs 1e-6 (2-norm) and 5e-6 (largest, over the
    root mean square) in small sparse layers over many unfolds, gradients
    4.4e-6 and 8e-5 (those of weights and mu, where large terms cancel)."""
    if _trains(case):
        return {"rel": 2e-5, "max": 3e-4}
    return {"rel": 4e-6, "max": 2e-5}


# ------------------------------------------------------------------------- exact


def _step(xt, v, q, U):
    """One time step of the boundary equations (ltc.py:42-63)."""
    gate = torch.sigmoid(q["sensory_sigma"] * (xt.unsqueeze(-1) - q["sensory_mu"]))
    cond = q["sensory_w_pos"] * gate
    sn, sd = (cond * q["sensory_erev"]).sum(1), cond.sum(1)
    for _ in range(U):
        gate = torch.sigmoid(q["sigma"] * (v.unsqueeze(-1) - q["mu"]))
        num = (gate * q["w_erev"]).sum(1) + sn
        den = (gate * q["w_pos"]).sum(1) + sd
        v = ((q["cm_t"] * v + q["gleak_pos"] * q["vleak"] + num)
             / (q["cm_t"] + q["gleak_pos"] + den + EPS))
    return v


def _chunks(c):
    """Batch rows at a time, so that one (rows, H, H) tensor stays near 64 MB."""
    per = max(1, (1 << 23) // max(c["H"] ** 2, c["D"] * c["H"]))
    return [(b, min(c["B"], b + per)) for b in range(0, c["B"], per)]


def exact(case, seed):
    c = case
    dev = DEV if torch.cuda.is_available() else "cpu"
    if dev == "cpu" and _synapses(c) > 2e8:
        return None
    B, T, U, H = c["B"], c["T"], c["U"], c["H"]
    p, x, h0, target, grad = _inputs(c, seed)

    def dbl(t):
        return None if t is None else t.to(dev).double()

    if c["x"] == "strided":
        x = x[:, :, 0::2]
    train, boundary = _trains(c), c["mode"] == "boundary"
    if boundary:
        # the float32 tensors that prepare hands to the entry point
        p32 = {k: v.to(dev) for k, v in p.items()}
        bp = {k: v.double() for k, v in _transforms(p32, U).items()}
        xa = _normalise(p32, x.to(dev)).double()
    else:
        p = {k: dbl(v).requires_grad_(train and k in LEAVES) for k, v in p.items()}
        x = dbl(x).requires_grad_(train)
        bp = _transforms(p, U)
        xa = _normalise(p, x)
    q = {k: v.detach().clone().requires_grad_(train) for k, v in bp.items()}
    h0 = torch.zeros(B, H, device=dev, dtype=torch.float64) if h0 is None else dbl(h0)
    xd = xa.detach()
    # v[t]: the state before step t; rows are independent
    v = torch.empty(T + 1, B, H, device=dev, dtype=torch.float64)
    with torch.no_grad():
        for b0, b1 in _chunks(c):
            s = h0[b0:b1]
            for t in range(T):
                v[t, b0:b1] = s
                s = _step(xd[b0:b1, t], s, q, U)
            v[T, b0:b1] = s
    out = v[1:].transpose(0, 1).contiguous()
    h = v[T].clone()
    if not train:
        return [out, h]
    if c["loss"] == "upstream":
        g_out = dbl(grad)
    elif c["loss"] == "sum":
        g_out = torch.ones_like(out)
    else:
        g_out = 2.0 * (out - dbl(target)) / out.numel()
    gxa, gh0 = torch.zeros_like(xd), torch.zeros_like(h0)
    for b0, b1 in _chunks(c):
        g = torch.zeros(b1 - b0, H, device=dev, dtype=torch.float64)
        for t in range(T - 1, -1, -1):
            vin = v[t, b0:b1].detach().requires_grad_(True)
            xt = xd[b0:b1, t].detach().requires_grad_(True)
            with torch.enable_grad():
                _step(xt, vin, q, U).backward(g + g_out[b0:b1, t])
            g = vin.grad
            gxa[b0:b1, t] = xt.grad
        gh0[b0:b1] = g
    if boundary:
        return [out, h, gxa, gh0, *[q[k].grad for k in BOUNDARY]]
    outs = [xa, *[bp[k] for k in BOUNDARY]]
    gos = [gxa, *[q[k].grad for k in BOUNDARY]]
    torch.autograd.backward(outs, gos)
    # in the module's parameter order
    order = ("w", "mu", "sigma", "erev", "sensory_w", "sensory_mu", "sensory_sigma",
             "sensory_erev", "gleak", "vleak", "cm", "input_w", "input_b",
             "input_norm.weight", "input_norm.bias")
    lead = [x.grad] if c["loss"] == "upstream" and c["mode"] == "train" else []
    return [out, h, *lead, *[p[k].grad for k in order]]
