"""The workloads whose speed is watched, one pass of each through the public
entry points, with their float64 values for comparison.

A case is a dict. `kind` says which part of a user's program it stands for:

  prefill     DeltaInput.run over a prompt, no gradients
  train       DeltaInput.run and the backward of its output through autograd
  step        delta_step, one decode token, the state updated in place
  recurrent   DeltaInput.run(DeltaPath.recurrent()): a decode token of several
              Householder micro-steps
  block       a block between in_proj and out_proj over a prompt:
              QkvProjection.forward_projected, DeltaInput.run, OutNorm.forward
  block_step  the same for one decode token: block_step, in place

Sizes: B sequences of T tokens, H heads of K key and V value channels; `dtype`
is that of q, k, v and the output (gates and states are float32); `gate` is
the width of the forget gate and, for "channel", of the erase and write gates
too; `neg` doubles beta (allow_neg_eigval); `u` counts micro-steps a token.
"""

import importlib
import math

import torch
import torch.nn.functional as F

pkg = importlib.import_module("burn-deltanet_amd")

DEVICE = "cuda"
CONV = 4  # short convolution length of the block cases


def _case(name, kind, B, T, H, K, V, dtype, gate="head", neg=False, u=1):
    case = {"kind": kind, "B": B, "T": T, "H": H, "K": K, "V": V, "dtype": dtype, "gate": gate,
            "neg": neg, "u": u}
    return {"name": name, **case} if name else case


def listed():
    return [
        # A batch of long prompts of a Gated DeltaNet layer: the headline workload.
        _case("prefill_8x4096", "prefill", 8, 4096, 16, 128, 256, "bf16"),
        # One user's prompt, of no round length: few sequences, latency counts.
        _case("prefill_1x1531", "prefill", 1, 1531, 16, 128, 256, "bf16"),
        # DeltaProduct, two micro-steps a token folded into the sequence, beta in (0, 2).
        _case("prefill_product_4x8192", "prefill", 4, 8192, 16, 128, 128, "bf16", neg=True, u=2),
        # The smallest forward: a single sequence in float32.
        _case("prefill_f32_1x512", "prefill", 1, 512, 4, 64, 64, "f32"),
        # Training of a Gated DeltaNet layer.
        _case("train_8x2048", "train", 8, 2048, 16, 128, 256, "bf16"),
        # Training of a GDN-2 layer (every gate per channel) on long sequences: the largest.
        _case("train_channel_2x16384", "train", 2, 16384, 16, 128, 128, "bf16", gate="channel"),
        # Training in float32 at the size of the layer benchmark.
        _case("train_f32_2x256", "train", 2, 256, 4, 64, 64, "f32"),
        # Training in float32 at an ordinary size, ragged.
        _case("train_f32_4x1000", "train", 4, 1000, 8, 128, 128, "f32"),
        # Decode of a large batch, bound by the state's traffic.
        _case("step_256", "step", 256, 1, 16, 128, 256, "f32"),
        # Decode of a DeltaProduct layer for a middling batch.
        _case("recurrent_u2_48", "recurrent", 48, 1, 16, 128, 256, "f32", neg=True, u=2),
        # A whole block over a few prompts of no round length.
        _case("block_3x2000", "block", 3, 2000, 16, 128, 256, "bf16"),
        # Decode of a whole block for a few users: latency.
        _case("block_step_4", "block_step", 4, 1, 16, 128, 256, "bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kinds = ("prefill", "prefill", "prefill", "train", "train", "train", "step", "recurrent",
             "block", "block_step")
    most = max(_weight(c) for c in listed())
    while True:
        kind = rng.choice(kinds)
        H = rng.choice((2, 4, 8, 12, 16))
        if kind in ("step", "recurrent", "block_step"):
            u = 2 if kind == "recurrent" else 1
            dtype = "bf16" if kind == "block_step" else rng.choice(("f32", "bf16"))
            case = _case(None, kind, _log_int(rng, 1, 256), 1, H, rng.choice((64, 128, 256)),
                         rng.choice((64, 128, 256)), dtype, neg=u == 2, u=u)
        elif kind == "block":
            case = _case(None, kind, _log_int(rng, 1, 8), _log_int(rng, 64, 4096), H,
                         rng.choice((64, 128)), rng.choice((64, 128, 256)), "bf16")
        else:
            f32 = rng.random() < 0.4
            gate = rng.choice(("head", "head", "head", "channel", "none"))
            # float32 runs where models are small; bfloat16 over the whole range.
            T = _log_int(rng, 16, 2048) if f32 else _log_int(rng, 64, 16384)
            B = _log_int(rng, 1, 8)
            K = rng.choice((32, 64, 96, 128) if f32 else (64, 128, 128, 256))
            V = rng.choice((32, 64, 96, 128, 256) if f32 else (64, 128, 192, 256))
            if gate == "channel" and K == 256:
                K = 128
            u = 2 if gate == "head" and kind == "prefill" and rng.random() < 0.25 else 1
            case = _case(None, kind, B, T, H, K, V, "f32" if f32 else "bf16", gate, u == 2, u)
        if _weight(case) <= most:
            return case


# -- inputs ----------------------------------------------------------------------


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _inputs(case, seed):
    """Everything a pass reads, made from the seed alone: q and k L2-normalised
    N(0, 1), v ~ N(0, 1), write gates sigmoid(N(0, 1)), log forget gates
    -0.05 softplus(N(0, 1))."""
    B, T, H, K, V, u = (case[n] for n in "BTHKVu")
    kind, S = case["kind"], case["T"] * case["u"]
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    randn = lambda *shape: torch.randn(shape, generator=gen, device=DEVICE)
    l2 = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
    forget = lambda *shape: F.softplus(randn(*shape)) * -0.05
    dt = _dtype(case)
    x = {}
    if kind in ("block", "block_step"):
        conv_dim = H * (2 * K + V)
        x["projected"] = randn(B, T, conv_dim + H + H * V).to(dt)
        x["conv_weight"] = randn(conv_dim, CONV) * 0.5
        # A prompt starts from an empty window, a decode token from the last inputs.
        x["window"] = (randn(B, conv_dim, CONV) if kind == "block_step"
                       else torch.zeros(B, conv_dim, CONV, device=DEVICE)).to(dt)
        x["norm_weight"] = 1 + 0.1 * randn(V)
        x["g"] = forget(B, T, H, 1)
    else:
        q = l2(randn(B, T, H, K))
        if u > 1:  # q on the last micro-step of a token, the forget gate on the first
            q = F.pad(q.unsqueeze(2), (0, 0, 0, 0, u - 1, 0)).reshape(B, S, H, K)
        x["q"] = q.to(dt)
        x["k"] = l2(randn(B, S, H, K)).to(dt)
        x["v"] = randn(B, S, H, V).to(dt)
        top = 2.0 if case["neg"] else 1.0
        if case["gate"] == "channel":
            x["erase"] = top * torch.sigmoid(randn(B, S, H, K))
            x["write"] = torch.sigmoid(randn(B, S, H, V))
        else:
            x["beta"] = top * torch.sigmoid(randn(B, S, H))
        if case["gate"] != "none":
            g = forget(B, T, H, K if case["gate"] == "channel" else 1)
            if u > 1:
                g = F.pad(g.unsqueeze(2), (0, 0, 0, 0, 0, u - 1)).reshape(B, S, H, -1)
            x["g"] = g
    if kind == "train":
        x["dy"] = randn(B, S, H, V).to(dt)
    # A prompt starts from an empty state, a decode token from a filled one.
    x["state"] = (randn(B, H, K, V) * 0.02 if kind in ("step", "recurrent", "block_step")
                  else torch.zeros(B, H, K, V, device=DEVICE))
    return x


def _leaves(case):
    gates = ("erase", "write") if case["gate"] == "channel" else ("beta",)
    return ("q", "k", "v") + gates + (() if case["gate"] == "none" else ("g",))


def prepare(case, seed):
    x = _inputs(case, seed)
    state = {"case": case, "x": x}
    if case["kind"] in ("block", "block_step"):
        state["proj"] = pkg.QkvProjection(
            nheads=case["H"], head_k_dim=case["K"], head_v_dim=case["V"], has_gate=True,
            conv=pkg.ShortConv(x["conv_weight"]))
        state["norm"] = pkg.OutNorm(x["norm_weight"])
    if case["kind"] == "train":
        for n in _leaves(case):
            x[n].requires_grad_()
    if case["kind"] in ("step", "block_step"):
        for n in set(x) - {"state", "window", "conv_weight", "norm_weight"}:
            x[n] = x[n][:, 0].contiguous()
    return state


def _delta_input(x, state):
    erase, write = (x["erase"], x["write"]) if "erase" in x else pkg.beta_gates(x["beta"])
    return pkg.DeltaInput(x["q"], x["k"], x["v"], erase, write, x.get("g"), state)


def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "train":
        y, s = _delta_input(x, x["state"]).run()
        leaves = _leaves(case)
        grads = torch.autograd.grad(y, [x[n] for n in leaves], x["dy"])
        return {"y": y.detach(), "state": s.detach(),
                **{"d_" + n: d for n, d in zip(leaves, grads)}}
    with torch.no_grad():
        if kind == "prefill":
            y, s = _delta_input(x, x["state"]).run()
            return {"y": y, "state": s}
        if kind == "recurrent":
            y, s = _delta_input(x, x["state"]).run(pkg.DeltaPath.recurrent())
            return {"y": y, "state": s}
        if kind == "step":
            erase, write = pkg.beta_gates(x["beta"])
            y, s = pkg.delta_step(x["q"], x["k"], x["v"], erase, write, x["g"], x["state"],
                                  1.0 / math.sqrt(case["K"]), in_place=True)
            return {"y": y, "state": s}
        if kind == "block_step":
            out, window, s = pkg.block_step(state["proj"], state["norm"], x["projected"],
                                            x["window"], x["g"], x["state"], in_place=True)
            return {"out": out, "window": window, "state": s}
        qkv, window = state["proj"].forward_projected(x["projected"], x["window"])
        y, s = pkg.DeltaInput(qkv.q_bshk, qkv.k_bShk, qkv.v_bShv, qkv.erase_bShK,
                              qkv.write_bShV, x["g"], x["state"]).run()
        return {"out": state["norm"].forward(y, qkv.gate_bshv), "window": window, "state": s}


# -- what a pass cannot do without -----------------------------------------------


def work(case):
    B, T, H, K, V, u = (case[n] for n in "BTHKVu")
    kind, S, el = case["kind"], case["T"] * case["u"], 2 if case["dtype"] == "bf16" else 4
    rows = B * S * H
    if case["gate"] == "channel":
        gates = rows * (2 * K + V) * 4
    else:
        gates = rows * 4 * (1 if case["gate"] == "none" else 2)
    state = 2 * B * H * K * V * 4
    nbytes = rows * (2 * K + 2 * V) * el + gates + state
    # One pass over the state per token: two contractions and a rank-one update.
    flops = rows * 6.0 * K * V
    if kind in ("prefill", "train", "block"):
        # The chunkwise form with chunks of 64 tokens, per chunk and head.
        L, chunks = 64, rows / 64
        flops = chunks * (6 * L * L * K + 4 * L * L * V + 6 * L * K * V + L ** 3 / 3)
    if kind == "train":
        # The backward reads the inputs and dy again and writes the gradients.
        nbytes += rows * (4 * K + 3 * V) * el + 2 * gates
        flops += chunks * (18 * L * K * V + 10 * L * L * V + 18 * L * L * K + 4.33 * L ** 3)
    if kind in ("block", "block_step"):
        conv_dim = H * (2 * K + V)
        nbytes = (B * T * (conv_dim + H + 2 * H * V) * el + 2 * B * conv_dim * CONV * el
                  + conv_dim * CONV * 4 + V * 4 + B * T * H * 4 + state)
        flops += B * T * (2.0 * CONV * conv_dim + 8.0 * H * (2 * K + 2 * V))
    return {"bytes": float(nbytes), "flops": float(flops)}


def _weight(case):
    # Bytes at 5 TB/s and flops on the matrix units of the case's type, in seconds.
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / (1e15 if case["dtype"] == "bf16" else 1e14)


def tolerance(case):
    # About four times the distance to the float64 values, which is that of
    # 32-bit sums (2e-7 to 5e-7 through a chunk's inverse, 1e-7 for one token),
    # of bf16 outputs alone (1.7e-3), or of bf16 operands in a chunk's products
    # too (3e-3 to 3.8e-3).
    one_token = case["kind"] in ("step", "recurrent", "block_step")
    if case["dtype"] == "f32":
        return {"rel": 5e-7 if one_token else 2e-6}
    return {"rel": 7e-3 if one_token else 1.5e-2}


# -- the same values in 64 bits, token by token ------------------------------------


def _recurrence(x, scale):
    """The delta rule over float64 inputs, one token after the other:
    S <- a S; u = w v - S^T (e k); S <- S + k u^T; y = scale S^T q. The states
    entering each 64-token segment are kept for the backward."""
    q, k, v = x["q"], x["k"], x["v"]
    B, S, H, K = q.shape
    V = v.shape[3]
    by_time = lambda t: t.transpose(0, 1).reshape(S, B * H, -1).contiguous()
    q, k, v, e, w = (by_time(t) for t in (q * scale, k, v, x["erase"], x["write"]))
    a = by_time(x["g"].exp()) if "g" in x else None
    ke, vw = k * e, v * w
    s = x["state"].reshape(B * H, K, V).clone()
    y = torch.empty_like(v)
    starts = []
    for t in range(S):
        if t % 64 == 0:
            starts.append(s.clone())
        if a is not None:
            s *= a[t].unsqueeze(-1)
        r = torch.bmm(ke[t].unsqueeze(1), s)
        s.baddbmm_(k[t].unsqueeze(2), vw[t].unsqueeze(1) - r)
        torch.bmm(q[t].unsqueeze(1), s, out=y[t].unsqueeze(1))
    back = lambda t, n: t.reshape(S, B, H, n).transpose(0, 1)
    return {"y": back(y, V), "state": s.reshape(B, H, K, V)}, (q, k, v, e, w, a, ke, vw, starts)


def _recurrence_grads(x, dy, kept, scale):
    """The gradients of sum(y dy), by the reverse recurrence."""
    q, k, v, e, w, a, ke, vw, starts = kept
    B, S, H, K = x["q"].shape
    dy = dy.transpose(0, 1).reshape(S, B * H, -1)
    dq, dk, dke, dvw = (torch.empty_like(t) for t in (q, k, ke, vw))
    da = None if a is None else torch.empty_like(a)
    ds = torch.zeros_like(starts[0])
    for n in range(len(starts) - 1, -1, -1):
        lo, hi = 64 * n, min(64 * n + 64, S)
        held = [starts[n]]  # the states entering the segment's tokens
        for t in range(lo, hi):
            s = held[-1] if a is None else held[-1] * a[t].unsqueeze(-1)
            r = torch.bmm(ke[t].unsqueeze(1), s)
            held.append(torch.baddbmm(s, k[t].unsqueeze(2), vw[t].unsqueeze(1) - r))
        for t in range(hi - 1, lo - 1, -1):
            col = lambda z: z[t].unsqueeze(2)
            row = lambda z: z[t].unsqueeze(1)
            before, after = held[t - lo], held[t + 1 - lo]
            torch.bmm(after, col(dy), out=col(dq))
            ds.baddbmm_(col(q), row(dy))
            s = before if a is None else before * a[t].unsqueeze(-1)
            u = row(vw) - torch.bmm(row(ke), s)
            torch.bmm(ds, u.transpose(1, 2), out=col(dk))
            torch.bmm(row(k), ds, out=row(dvw))
            torch.bmm(s, col(dvw), out=col(dke))
            ds.baddbmm_(col(ke), row(dvw), alpha=-1)
            if a is not None:
                gate = (ds * before).sum(-1)
                da[t] = gate if a.shape[-1] > 1 else gate.sum(-1, keepdim=True)
                ds *= a[t].unsqueeze(-1)
    dke = -dke
    de, dw = dke * k, dvw * v
    back = lambda t: t.reshape(S, B, H, -1).transpose(0, 1)
    narrow = lambda t, to: t if to.shape[-1] > 1 else t.sum(-1, keepdim=True)
    out = {"q": dq * scale, "k": dk + dke * e, "v": dvw * w, "erase": narrow(de, e),
           "write": narrow(dw, w)}
    if a is not None:
        out["g"] = da * a
    return {n: back(t) for n, t in out.items()}


def _front(case, x):
    """Short convolution, SiLU, the q/k L2 norm and the write gate of a block."""
    B, T, H, K, V = (case[n] for n in "BTHKV")
    p = x["projected"]
    n = H * (2 * K + V)
    padded = torch.cat((x["window"][:, :, 1:], p[:, :, :n].transpose(1, 2)), 2)
    z = sum(x["conv_weight"][:, j, None] * padded[:, :, j:j + T] for j in range(CONV))
    z = F.silu(z).transpose(1, 2)
    q, k, v = z.split((H * K, H * K, H * V), 2)
    l2 = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    beta = torch.sigmoid(p[:, :, n:n + H]).unsqueeze(-1)
    made = {"q": l2(q.reshape(B, T, H, K)), "k": l2(k.reshape(B, T, H, K)),
            "v": v.reshape(B, T, H, V), "erase": beta, "write": beta, "g": x["g"],
            "state": x["state"]}
    return made, p[:, :, n + H:].reshape(B, T, H, V), padded[:, :, T - 1:]


def exact(case, seed):
    x = {n: t.double() for n, t in _inputs(case, seed).items()}
    scale = 1.0 / math.sqrt(case["K"])
    with torch.no_grad():
        if case["kind"] in ("block", "block_step"):
            made, gate, window = _front(case, x)
            out, _ = _recurrence(made, scale)
            y = out["y"]
            y = y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-5) * x["norm_weight"]
            y = y * F.silu(gate)
            if case["kind"] == "block_step":
                y = y[:, 0]
            return {"out": y, "window": window, "state": out["state"]}
        if "beta" in x:
            x["erase"] = x["write"] = x["beta"].unsqueeze(-1)
        out, kept = _recurrence(x, scale)
        if case["kind"] == "step":
            out["y"] = out["y"][:, 0]
        if case["kind"] == "train":
            d = _recurrence_grads(x, x["dy"], kept, scale)
            if "beta" in x:
                d["beta"] = (d["erase"] + d["write"]).squeeze(-1)
            out.update({"d_" + n: d[n] for n in _leaves(case)})
        return out
