"""Performance cases of the Hyena long-convolution ops: what is timed, on which inputs, and what the results are.

A case is one call of a public op (``pass`` "fwd": under ``no_grad``, as in inference) or one forward and backward
("train": the output and the gradient of every operand).  Inputs follow the distributions of the repository's
benchmark workloads: activations N(0, 1), filters decaying from their first tap (causal) or their centre (N-d).
"""

import math

import torch


DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
DEVICE = "cuda:0"


def listed():
    return [
        # A short causal conv of an inference step: two rows of 4096 samples, where launches and latency count.
        {"name": "conv1d-small-fwd", "op": "conv1d", "pass": "fwd", "dtype": "f32", "B": 2, "H": 128, "L": 4096,
         "K": 4096},
        # The ordinary training step of a causal Hyena layer, 8K context, filter as long as the sequence.
        {"name": "conv1d-train", "op": "conv1d", "pass": "train", "dtype": "bf16", "B": 4, "H": 1024, "L": 8192,
         "K": 8192},
        # The long-context training step, 256K samples by 4096 channels (the repository's headline workload).
        {"name": "conv1d-long-train", "op": "conv1d", "pass": "train", "dtype": "bf16", "B": 1, "H": 4096,
         "L": 262144, "K": 262144},
        # A depthwise causal conv layer with its activation, medium filter (128 taps), training.
        {"name": "short-conv-train", "op": "short", "pass": "train", "dtype": "bf16", "B": 4, "C": 4096, "L": 8192,
         "K": 128, "act": "silu"},
        # The striped-Hyena block, projection conv -> gate -> mixer conv -> gate: prefill, and a training step.
        {"name": "b2b-fwd", "op": "b2b", "pass": "fwd", "dtype": "bf16", "B": 4, "C": 4096, "L": 8192, "Kp": 3,
         "Km": 128},
        {"name": "b2b-train", "op": "b2b", "pass": "train", "dtype": "bf16", "B": 2, "C": 2048, "L": 8192, "Kp": 3,
         "Km": 128},
        # A 2D Hyena layer over a 128 x 128 image, inference.
        {"name": "conv2d-fwd", "op": "nd", "pass": "fwd", "dtype": "bf16", "B": 16, "H": 384, "S0": 128, "S1": 128,
         "S2": 0, "K0": 128, "K1": 128, "K2": 0, "film": False},
        # A 2D Hyena layer of an image classifier, 14 x 14 tokens with a 27 x 27 filter, training.
        {"name": "conv2d-tokens-train", "op": "nd", "pass": "train", "dtype": "bf16", "B": 64, "H": 384, "S0": 14,
         "S1": 14, "S2": 0, "K0": 27, "K1": 27, "K2": 0, "film": False},
        # A field on a channel, periodic along x and bounded along y (64 x 16 tokens), training.
        {"name": "mixed2d-train", "op": "mixed", "pass": "train", "dtype": "bf16", "B": 64, "H": 384, "S0": 64,
         "S1": 16, "K0": 64, "K1": 31},
        # A 3D Hyena layer over a 64^3 volume, training.
        {"name": "conv3d-train", "op": "nd", "pass": "train", "dtype": "bf16", "B": 2, "H": 128, "S0": 64, "S1": 64,
         "S2": 64, "K0": 64, "K1": 64, "K2": 64, "film": False},
        # The gated 2D Hyena operator (gate, conv, gate) over a 128 x 128 image, training.
        {"name": "gated2d-train", "op": "gated", "pass": "train", "dtype": "bf16", "B": 16, "H": 384, "S0": 128,
         "S1": 128, "K0": 128, "K1": 128},
        # The Hyena operator's tail: gate, RMSNorm over channels, channels-last layout, training.
        {"name": "output-norm-train", "op": "norm", "pass": "train", "dtype": "bf16", "B": 16, "C": 384, "S": 16384},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _dtype(rng):
    return rng.choice(["bf16", "bf16", "bf16", "f32", "f16"])


def draw(rng):
    op = rng.choice(["conv1d", "conv1d", "short", "b2b", "nd", "nd", "mixed", "gated", "norm"])
    c = {"op": op, "pass": rng.choice(["fwd", "train", "train"]), "dtype": _dtype(rng)}
    if op == "conv1d":
        L = _log_int(rng, 200, 262144)
        K = L if rng.random() < 0.6 else _log_int(rng, max(2, L // 8), L)
        H = _log_int(rng, 32, max(33, min(2048, (1 << 26) // L)))
        B = _log_int(rng, 1, max(1, min(16, (1 << 26) // (L * H))))
        c.update(B=B, H=H, L=L, K=K)
    elif op == "short":
        C, L = _log_int(rng, 64, 4096), _log_int(rng, 512, 16384)
        c.update(B=_log_int(rng, 1, max(1, min(8, (1 << 26) // (C * L)))), C=C, L=L, K=_log_int(rng, 3, 256),
                 act=rng.choice(["identity", "silu"]))
    elif op == "b2b":
        C, L = _log_int(rng, 64, 4096), _log_int(rng, 512, 16384)
        c.update(B=_log_int(rng, 1, max(1, min(4, (1 << 25) // (C * L)))), C=C, L=L, Kp=rng.choice([3, 3, 4]),
                 Km=rng.choice([7, 16, 64, 128, _log_int(rng, 7, 128)]))
    elif op == "nd":
        if rng.random() < 0.65:
            S = [_log_int(rng, 7, 192) for _ in range(2)]
        else:
            S = [_log_int(rng, 7, 64) for _ in range(3)]
        K = [rng.choice([s, 2 * s - 1, max(3, s // 2) | 1]) for s in S]
        H = _log_int(rng, 32, 512)
        c.update(B=_log_int(rng, 1, max(1, min(64, (1 << 24) // (H * math.prod(S))))), H=H,
                 film=len(S) == 2 and rng.random() < 0.15)
        S, K = (S + [0])[:3], (K + [0])[:3]
        c.update(S0=S[0], S1=S[1], S2=S[2], K0=K[0], K1=K[1], K2=K[2])
    elif op == "mixed":
        S0, S1 = rng.choice([16, 32, 64, 128]), _log_int(rng, 8, 128)
        H = _log_int(rng, 32, 512)
        c.update(B=_log_int(rng, 1, max(1, min(64, (1 << 24) // (H * S0 * S1)))), H=H, S0=S0, S1=S1,
                 K0=rng.choice([S0, S0 - 1, S0 // 2 + 1]), K1=rng.choice([S1, 2 * S1 - 1]))
    elif op == "gated":
        S = [_log_int(rng, 12, 128) for _ in range(2)]
        H = _log_int(rng, 32, 512)
        K = [rng.choice([s, 2 * s - 1]) for s in S]
        c.update(B=_log_int(rng, 1, max(1, min(64, (1 << 24) // (H * S[0] * S[1])))), H=H, S0=S[0], S1=S[1], K0=K[0],
                 K1=K[1])
    else:
        C, S = _log_int(rng, 64, 1536), _log_int(rng, 196, 16384)
        c.update(B=_log_int(rng, 1, max(1, min(64, (1 << 25) // (C * S)))), C=C, S=S)
    return c


def _dims(case, letter):
    return [case[letter + i] for i in "012" if case.get(letter + i)]


def _randn(gen, *shape):
    return torch.randn(*shape, device=DEVICE, generator=gen)


def _causal_filter(gen, H, K):
    """N(0, 1) * exp(-a t / K) with a ~ U(1, 50) per channel."""
    k = _randn(gen, H, K)
    a = torch.empty(H, 1, device=DEVICE).uniform_(1.0, 50.0, generator=gen)
    return k.mul_(torch.exp(-a * torch.arange(K, device=DEVICE).view(1, K) / K))


def _centred_filter(gen, n, K):
    """N(0, 1) * exp(-r / sigma) with r the distance from the centre, sigma ~ U(1/32, 1/2) of the longest axis."""
    axes = torch.meshgrid(*[torch.arange(s, device=DEVICE).float() - s // 2 for s in K], indexing="ij")
    r = torch.sqrt(sum(a * a for a in axes))
    sig = torch.empty(n, device=DEVICE).uniform_(1 / 32, 1 / 2, generator=gen) * max(K)
    return _randn(gen, n, *K).mul_(torch.exp(-r[None] / sig.view(-1, *[1] * len(K))))


def _inputs(case, seed):
    """The operands of a case in the order of its op's arguments, and the upstream gradient."""
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    dt, op = DTYPES[case["dtype"]], case["op"]
    B = case["B"]

    def act(*shape):
        return _randn(gen, *shape).to(dt)

    if op == "conv1d":
        H, L = case["H"], case["L"]
        return [act(B, H, L), _causal_filter(gen, H, case["K"]).unsqueeze(0), act(H)], act(B, H, L)
    if op == "short":
        C, K = case["C"], case["K"]
        return [act(B, C, case["L"]), _randn(gen, C, K) / K ** 0.5, _randn(gen, C)], act(B, C, case["L"])
    if op == "b2b":
        C, L, Kp, Km = case["C"], case["L"], case["Kp"], case["Km"]
        return [act(B, 3 * C, L), _randn(gen, 3 * C, Kp) / Kp ** 0.5, _randn(gen, C, Km) / Km ** 0.5,
                _randn(gen, C)], act(B, C, L)
    if op == "norm":
        C = case["C"]
        return [act(B, C, case["S"]), act(B, C, case["S"]), 1 + 0.1 * _randn(gen, C)], act(B, case["S"], C)
    H, S, K = case["H"], _dims(case, "S"), _dims(case, "K")
    kb = B if case.get("film") else 1
    k = _centred_filter(gen, kb * H, K).view(kb, H, *K)
    first = 3 if op == "gated" else 1
    return [*(act(B, H, *S) for _ in range(first)), k, act(H)], act(B, H, *S)


def prepare(case, seed):
    args, g = _inputs(case, seed)
    if case["pass"] == "fwd":
        return {"case": case, "args": args, "g": None}
    return {"case": case, "args": [a.requires_grad_(True) for a in args], "g": g}


def _call(case, args):
    op = case["op"]
    if op == "conv1d":
        from nvsubquadratic_amd.fftconv_hip import causal_fftconv1d_bhl

        return causal_fftconv1d_bhl(*args)
    if op == "short":
        from nvsubquadratic_amd.causal_conv1d_hip import causal_conv1d

        return causal_conv1d(*args, activation=case["act"])
    if op == "b2b":
        from nvsubquadratic_amd.causal_conv1d_hip import b2b_causal_conv1d

        return b2b_causal_conv1d(*args)
    if op == "norm":
        from nvsubquadratic_amd.norm_hip import hyena_output_norm

        return hyena_output_norm(*args)
    if op == "mixed":
        from nvsubquadratic_amd.mixed_fftconv_hip import mixed_fftconv2d_fp32_bhl

        x, k, s = args
        return mixed_fftconv2d_fp32_bhl(x, k, (True, False), s)
    if op == "gated":
        from nvsubquadratic_amd.gated_fftconv_hip import hyena_gated_fftconv2d_bhl

        return hyena_gated_fftconv2d_bhl(*args, "silu")
    from nvsubquadratic_amd import fftconv_hip

    return (fftconv_hip.fftconv3d_bhl if case["S2"] else fftconv_hip.fftconv2d_bhl)(*args)


def run(state):
    case, args = state["case"], state["args"]
    if case["pass"] == "fwd":
        with torch.no_grad():
            return {"y": _call(case, args)}
    y = _call(case, args)
    grads = torch.autograd.grad(y, args, state["g"])
    return {"y": y.detach(), **{"g%d" % i: t for i, t in enumerate(grads)}}


def _sizes(case):
    """(elements of one activation tensor, activations read / written forward and backward, weight elements)."""
    op, B = case["op"], case["B"]
    if op == "conv1d":
        return B * case["H"] * case["L"], (2, 3), case["H"] * case["K"]
    if op == "short":
        return B * case["C"] * case["L"], (2, 3), case["C"] * case["K"]
    if op == "b2b":
        return B * case["C"] * case["L"], (4, 7), case["C"] * (3 * case["Kp"] + case["Km"])
    if op == "norm":
        return B * case["C"] * case["S"], (3, 5), case["C"]
    E = B * case["H"] * math.prod(_dims(case, "S"))
    w = (B if case.get("film") else 1) * case["H"] * math.prod(_dims(case, "K"))
    return E, ((4, 7) if op == "gated" else (2, 3)), w


def work(case):
    E, (fwd, bwd), W = _sizes(case)
    item = DTYPES[case["dtype"]].itemsize
    train = case["pass"] == "train"
    nbytes = (fwd + (bwd if train else 0)) * E * item + (3 if train else 1) * 4 * W
    op = case["op"]
    if op == "norm":
        return {"bytes": nbytes, "flops": E * (30 if train else 10)}
    if op in ("short", "b2b"):
        taps = case["K"] if op == "short" else 3 * case["Kp"] + case["Km"]
        return {"bytes": nbytes, "flops": 2 * E * taps * (3 if train else 1)}
    # one real transform of F points costs 2.5 F log2 F
    if op == "conv1d":
        F, rows, filters = case["L"] + case["K"], case["B"] * case["H"], case["H"]
    else:
        S, K = _dims(case, "S"), _dims(case, "K")
        F = math.prod(s if op == "mixed" and d == 0 else min(s + (k + 1) // 2, 2 * s)
                      for d, (s, k) in enumerate(zip(S, K)))
        rows = case["B"] * case["H"]
        filters = rows if case.get("film") else case["H"]
    transforms = 2 * rows + filters + ((2 * rows + filters) if train else 0)
    return {"bytes": nbytes, "flops": 2.5 * F * math.log2(F) * transforms}


def tolerance(case):
    # 32-bit inputs, sums and outputs against results rounded once to 16 bits (some ops round twice).  "max" bounds
    # single values, relative to the output's RMS or to the value where that is larger.
    return {"f32": {"rel": 2e-5, "max": 1e-3}, "bf16": {"rel": 1e-2, "max": 0.1},
            "f16": {"rel": 2e-3, "max": 2e-2}}[case["dtype"]]


# ---------------------------------------------------------------------------
# The same results from torch in 64 bits
# ---------------------------------------------------------------------------
def _conv64(x, k, periodic, causal):
    """The linear (causal or "same") or per-axis periodic convolution over the trailing axes, by FFT."""
    nd = x.dim() - 2
    S, K = x.shape[2:], k.shape[2:]
    F = [S[d] if periodic[d] else S[d] + K[d] for d in range(nd)]
    dims = tuple(range(2, 2 + nd))
    y = torch.fft.irfftn(torch.fft.rfftn(x, s=F, dim=dims) * torch.fft.rfftn(k, s=F, dim=dims), s=F, dim=dims)
    for d in range(nd):
        if periodic[d]:
            y = torch.roll(y, -((K[d] - 1) // 2), dims=2 + d)
        else:
            y = y.narrow(2 + d, 0 if causal else K[d] // 2, S[d])
    return y


def _taps64(x, w):
    """Depthwise causal taps of [B, C, L] with [C, K]: y[n] = sum_j w[j] x[n - K + 1 + j]."""
    return _conv64(x, w.flip(-1).unsqueeze(0), (False,), True)


def _exact_op(case, a):
    op = case["op"]

    def ch(t, nd):
        return t.view(1, -1, *[1] * nd)

    if op == "short":
        x, w, b = a
        p = _taps64(x, w) + ch(b, 1)
        return p * torch.sigmoid(p) if case["act"] == "silu" else p
    if op == "b2b":
        x, wp, wm, skip = a  # x and wp as [B, 3, C, L] and [3, C, Kp]
        q, k, v = (_taps64(x[:, i], wp[i]) for i in range(3))
        z = k * v
        return q * (_taps64(z, wm) + ch(skip, 1) * z)
    if op == "norm":
        y, v, w = a
        u = y * torch.sigmoid(v)
        return (ch(w, 1) * u * torch.rsqrt((u * u).mean(1, keepdim=True) + 1e-6)).transpose(1, 2)
    if op == "gated":
        q, kg, v, k, s = a
        z = q * torch.nn.functional.silu(kg)
        return (_conv64(z, k, (False, False), False) + ch(s, 2) * z) * torch.nn.functional.silu(v)
    x, k, s = a
    nd = x.dim() - 2
    periodic = (op == "mixed",) + (False,) * (nd - 1)
    return _conv64(x, k, periodic, op == "conv1d") + ch(s, nd) * x


# the axis of each operand, and of the output, along which a case's channels lie
_CHANNEL_AXES = {"conv1d": ((1, 1, 0), 1), "short": ((1, 0, 0), 1), "b2b": ((2, 1, 0, 0), 1), "nd": ((1, 1, 0), 1),
                 "mixed": ((1, 1, 0), 1), "gated": ((1, 1, 1, 1, 0), 1)}


def exact(case, seed):
    args, g = _inputs(case, seed)
    op, train = case["op"], case["pass"] == "train"
    if op == "b2b":
        B, C = case["B"], case["C"]
        args = [args[0].view(B, 3, C, -1), args[1].view(3, C, -1), args[2], args[3]]
    if op == "norm":  # channels are normalised together: batch rows one by one
        axes, out_axis, n, chunk = (0, 0, None), 0, case["B"], 1
    else:
        axes, out_axis = _CHANNEL_AXES[op]
        n = case["C"] if op in ("short", "b2b") else case["H"]
        if op in ("short", "b2b"):
            points = case["L"] + 128
        else:
            points = math.prod(s + k for s, k in zip(_dims(case, "S"), _dims(case, "K"))) if op != "conv1d" else (
                case["L"] + case["K"])
        chunk = max(1, min(n, (1 << 26) // (case["B"] * points)))
    outs, grads = [], [[] for _ in args]
    for at in range(0, n, chunk):
        m = min(chunk, n - at)
        part = [(a if ax is None else a.narrow(ax, at, m)).double() for a, ax in zip(args, axes)]
        if not train:
            with torch.no_grad():
                outs.append(_exact_op(case, part))
            continue
        part = [p.requires_grad_(True) for p in part]
        y = _exact_op(case, part)
        for into, t in zip(grads, torch.autograd.grad(y, part, g.narrow(out_axis, at, m).double())):
            into.append(t)
        outs.append(y.detach())
    result = {"y": torch.cat(outs, out_axis)}
    if train:
        for i, (ts, ax) in enumerate(zip(grads, axes)):
            t = torch.stack(ts).sum(0) if ax is None else torch.cat(ts, ax)
            if op == "b2b" and i < 2:
                t = t.reshape(case["B"], 3 * case["C"], -1) if i == 0 else t.reshape(3 * case["C"], -1)
            result["g%d" % i] = t
    return result
