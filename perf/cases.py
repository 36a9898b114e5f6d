"""Performance cases of the dynamic short convolutions: what a program that uses them calls, over the
range of sizes, types and options that it calls them with.

A case is a dict:
    op      "headwise", "lowrank", or "qkv" (the grouped lowrank module: proj_in, then the q, k and v
            convolutions of one attention layer, README.md:57-110)
    pass    "train": forward and backward through autograd, every gradient returned;
            "infer": the forward under torch.no_grad()
    B, T, D, W, dtype, static, residual
    hs      head size (headwise)
    R       dynamic rank (lowrank, qkv): R, or R + 1 with a static filter, is a power of two
    hd      head dim of the qkv module's [B, D / hd, T, hd] outputs

Sizes are those of this repository's benchmark and tests (D 256-4096, T up to 8192, W 2-16, head
sizes 1-64, kernel ranks 8-64) and ragged ones between them.  Distributions are the benchmark's:
x, z, dy ~ N(0, 1), headwise weights ~ N(0, 1/W), U ~ N(0, 1/(kernel rank * W)), static filter uniform
in +-1/sqrt(W).
"""

import math

import torch

from headwise import headwise_dynamic_convolution
from lowrank import GroupedLowRankDynamicShortConvolution, lowrank_dynamic_convolution

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
GROUPS = 3  # q, k, v


def listed():
    hw = dict(op="headwise", dtype="bf16", W=4, static=True, residual=True)
    lr = dict(op="lowrank", dtype="bf16", W=4, static=True, residual=True)
    big = dict(B=4, T=4096, D=2048)
    return [
        # one decoding step of 8 sequences: the convolution over each sequence's last W tokens
        {"name": "lr_decode", **lr, "pass": "infer", "B": 8, "T": 4, "D": 2048, "R": 15},
        # the smallest training shapes that the tests and the CPU baseline use
        {"name": "lr_train_small", **lr, "pass": "train", "B": 2, "T": 512, "D": 256, "R": 15},
        {"name": "hw_train_fp32_small", "op": "headwise", "pass": "train", "dtype": "fp32", "B": 2, "T": 1024, "D": 512,
         "W": 4, "hs": 1, "static": False, "residual": False},
        # ragged lengths and a width off the powers of two, as packed batches of a small model have
        {"name": "lr_train_fp16_ragged", **lr, "pass": "train", "dtype": "fp16", "B": 3, "T": 1537, "D": 1000, "R": 7,
         "W": 3},
        # prefill of one long prompt
        {"name": "hw_prefill_fp16", **hw, "pass": "infer", "dtype": "fp16", "B": 1, "T": 8191, "D": 4096, "hs": 16},
        # the three training shapes of the headline benchmark
        {"name": "hw_train_hs1", **hw, "pass": "train", **big, "hs": 1},
        {"name": "hw_train_hs32", **hw, "pass": "train", **big, "hs": 32},
        {"name": "lr_train_r16", **lr, "pass": "train", **big, "R": 16, "static": False},
        # long filters and high ranks at the same shape, and the fp32 tier
        {"name": "lr_train_W8", **lr, "pass": "train", **big, "R": 15, "W": 8},
        {"name": "lr_train_r64", **lr, "pass": "train", **big, "R": 63},
        {"name": "lr_train_fp32", **lr, "pass": "train", "dtype": "fp32", **big, "R": 15},
        # the q, k and v convolutions of one layer with their input projection, outputs laid out for attention
        {"name": "qkv_train", "op": "qkv", "pass": "train", "dtype": "bf16", "B": 2, "T": 8192, "D": 4096, "R": 31,
         "W": 4, "hd": 128, "static": True, "residual": True},
    ]


def draw(rng):
    """One case of the same ranges: sizes over their logarithms, ragged ones among them."""
    while True:
        op = rng.choice(["headwise"] * 9 + ["lowrank"] * 9 + ["qkv"] * 2)
        c = {
            "op": op,
            "pass": rng.choice(["train", "train", "train", "infer"]),
            "dtype": rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"]),
            "B": rng.choice([1, 1, 2, 3, 4, 8]),
            "W": rng.choice([2, 3, 4, 4, 4, 4, 6, 8, 12, 16]),
            "static": rng.random() < 0.6,
            "residual": rng.random() < 0.6,
        }
        # sequences of a training batch are long; a forward call may be one decoding step
        shortest = 256 if c["pass"] == "train" else 4
        c["T"] = int(round(math.exp(rng.uniform(math.log(shortest), math.log(8192)))))
        if rng.random() < 0.4:
            c["T"] = 1 << max(2, round(math.log2(c["T"])))
        d = math.exp(rng.uniform(math.log(256), math.log(4096)))
        # most models' widths are multiples of 128; some are only multiples of 8
        c["D"] = 8 * round(d / 8) if rng.random() < 0.2 else 128 * max(2, round(d / 128))
        if op == "headwise":
            c["hs"] = rng.choice([h for h in (1, 1, 4, 8, 16, 32, 64) if c["D"] % h == 0])
        else:
            if op == "qkv":
                c.update({"static": True, "residual": True, "D": 128 * max(2, round(d / 128)), "hd": 128})
                c["dtype"] = rng.choice(["bf16", "bf16", "fp16"])
                c["W"] = rng.choice([2, 3, 4, 4, 4])
            rank = rng.choice([8, 16, 16, 16, 32, 32] + ([64] if op == "lowrank" else []))
            c["R"] = rank - 1 if c["static"] else rank
        # within the largest listed case: its bytes, and its operations (an eighth of them in fp32,
        # whose products run on slower units); long filters on ragged widths come in small batches
        most, w = work(listed()[-1]), work(c)
        if c["dtype"] == "fp32":
            most["flops"] /= 8
        if c["W"] > 8 and c["D"] % 128:
            most["bytes"] /= 16
        if w["bytes"] <= most["bytes"] and w["flops"] <= most["flops"]:
            return c


def prepare(case, seed):
    """The tensors (and for "qkv" the module) that a program holds before the call."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    B, T, D, W = case["B"], case["T"], case["D"], case["W"]
    train = case["pass"] == "train"

    def normal(*shape, scale=1.0, grad=train):
        return (torch.randn(*shape, generator=g, device=dev) * scale).to(dt).requires_grad_(grad)

    def uniform(*shape):
        return ((torch.rand(*shape, generator=g, device=dev) * 2 - 1) / math.sqrt(W)).to(dt).requires_grad_(train)

    state = {"case": case}
    if case["op"] == "qkv":
        R, hd = case["R"], case["hd"]
        m = GroupedLowRankDynamicShortConvolution(D, R, W, groups=GROUPS, head_dim=hd).to(device=dev, dtype=dt)
        with torch.no_grad():
            m.proj_in.weight.copy_(normal(GROUPS * R, D, scale=1 / math.sqrt(D), grad=False))
            m.proj_out.copy_(normal(GROUPS, R, W * D, scale=1 / math.sqrt((R + 1) * W), grad=False))
            m.proj_out_bias.copy_(uniform(GROUPS, W, D))
        state["module"] = m
        state["x"], state["pre_z"] = normal(B, T, GROUPS * D), normal(B, T, D)
        state["leaves"] = [state["x"], state["pre_z"], m.proj_in.weight, m.proj_out, m.proj_out_bias]
        if train:
            state["dy"] = tuple(normal(B, D // hd, T, hd, grad=False) for _ in range(GROUPS))
        return state
    state["x"] = normal(B, T, D)
    if case["op"] == "headwise":
        state["weight"] = normal(B, T, D // case["hs"], W, scale=1 / math.sqrt(W))
        args = [state["x"], state["weight"]]
    else:
        rank = case["R"] + (1 if case["static"] else 0)
        state["z"] = normal(B, T, case["R"])
        state["U"] = normal(case["R"], W * D, scale=1 / math.sqrt(rank * W))
        args = [state["x"], state["z"], state["U"]]
    state["static_w"] = uniform(W, D) if case["static"] else None
    state["leaves"] = args + ([state["static_w"]] if case["static"] else [])
    if train:
        state["dy"] = normal(B, T, D, grad=False)
    return state


def _call(s):
    c = s["case"]
    if c["op"] == "qkv":
        return s["module"](s["x"], s["pre_z"])
    if c["op"] == "headwise":
        return headwise_dynamic_convolution(s["x"], s["weight"], static_w=s["static_w"], residual=c["residual"])
    return lowrank_dynamic_convolution(s["x"], s["z"], s["U"], static_w=s["static_w"], residual=c["residual"])


def run(state):
    """One pass: the outputs, and for "train" the gradients of every leaf."""
    if state["case"]["pass"] == "infer":
        with torch.no_grad():
            return {"y": _call(state)}
    y = _call(state)
    return {"y": y, "grads": torch.autograd.grad(y, state["leaves"], state["dy"])}


def work(case):
    """Bytes and operations of one pass: each call (forward, backward) reads each of its inputs once
    and writes each of its outputs once; the products and sums of the formulas, 2 a multiply-add."""
    e = 4 if case["dtype"] == "fp32" else 2
    B, T, D, W = case["B"], case["T"], case["D"], case["W"]
    BT, train = B * T, case["pass"] == "train"
    x, sw = BT * D, (W * D if case["static"] else 0)
    conv = 2 * BT * D * W  # one multiply-add per tap and element
    if case["op"] == "headwise":
        w = BT * (D // case["hs"]) * W
        n = 2 * x + w + sw + (3 * x + 2 * w + 2 * sw if train else 0)
        return {"bytes": e * n, "flops": conv * (3 if train else 1)}  # y; dx and dweight
    R, G = case["R"], GROUPS if case["op"] == "qkv" else 1
    rank = R + (1 if case["static"] else 0)
    z, U = BT * R, R * W * D
    n = 2 * x + z + U + sw + (3 * x + 2 * z + 2 * U + 2 * sw if train else 0)
    gen = 2 * BT * D * W * rank  # one contraction over (rank or rows or channels)
    # forward: z @ U and the taps; backward: z @ U again, dU, dz, dy * x and dx
    f = gen + conv + (3 * gen + 2 * conv if train else 0)
    n, f = G * n, G * f
    if case["op"] == "qkv":  # proj_in: z = pre_z W_in^T; d pre_z = dz W_in, dW_in = dz^T pre_z
        w_in, zs = G * R * D, G * z
        n += x + w_in + zs + (2 * x + 2 * w_in + zs if train else 0)
        f += 2 * BT * D * G * R * (3 if train else 1)
    return {"bytes": e * n, "flops": f}


def tolerance(case):
    """About four times what two correct computations differ by: one rounding of each output, and in
    16 bits the roundings of z and of dy * x before the matrix products; in fp32 the order of the sums."""
    if case["dtype"] == "fp32":
        return {"rel": 2e-6, "max": 1e-4}
    if case["dtype"] == "fp16":
        return {"rel": 1.2e-3, "max": 0.05}
    return {"rel": 1.2e-2, "max": 0.3}


def _shift(t, k):
    """Row t of the result is row t - k of t (rows before 0 are zero); k < 0 looks ahead."""
    if k == 0:
        return t
    out = torch.zeros_like(t)
    if abs(k) < t.shape[1]:
        if k > 0:
            out[:, k:] = t[:, :-k]
        else:
            out[:, :k] = t[:, -k:]
    return out


def _exact_headwise(x, weight, sw, residual, hs, dy):
    W = weight.shape[-1]
    B, T, D = x.shape
    taps = [weight[..., k].repeat_interleave(hs, dim=2) + (0 if sw is None else sw[k]) for k in range(W)]
    y = sum(taps[k] * _shift(x, k) for k in range(W)) + (x if residual else 0)
    if dy is None:
        return y, None
    dx = sum(_shift(dy * taps[k], -k) for k in range(W)) + (dy if residual else 0)
    dw, dsw = torch.empty_like(weight), None if sw is None else torch.empty_like(sw)
    for k in range(W):
        p = dy * _shift(x, k)
        dw[..., k] = p.view(B, T, D // hs, hs).sum(-1)
        if sw is not None:
            dsw[k] = p.sum((0, 1))
    return y, [dx, dw] + ([dsw] if sw is not None else [])


def _exact_lowrank(x, z, U, sw, residual, dy):
    B, T, D = x.shape
    R, W = z.shape[-1], U.shape[-1] // D
    z2 = z.reshape(B * T, R)

    def tap(k):
        K = (z2 @ U[:, k * D:(k + 1) * D].contiguous()).view(B, T, D)
        return K if sw is None else K + sw[k]

    y = x.clone() if residual else torch.zeros_like(x)
    for k in range(W):
        y += tap(k) * _shift(x, k)
    if dy is None:
        return y, None
    dx = dy.clone() if residual else torch.zeros_like(dy)
    dz, dU, dsw = torch.zeros_like(z2), torch.empty_like(U), None if sw is None else torch.empty_like(sw)
    for k in range(W):
        dx += _shift(dy * tap(k), -k)
        p = (dy * _shift(x, k)).view(B * T, D)
        dz += p @ U[:, k * D:(k + 1) * D].t().contiguous()
        dU[:, k * D:(k + 1) * D] = z2.t().contiguous() @ p
        if sw is not None:
            dsw[k] = p.sum(0)
    return y, [dx, dz.view_as(z), dU] + ([dsw] if sw is not None else [])


def exact(case, seed):
    """run()'s outputs from the same inputs in 64 bits, by the formulas of the operators."""
    s = prepare(case, seed)
    train = case["pass"] == "train"

    def wide(t):
        return None if t is None else t.detach().double()

    with torch.no_grad():
        if case["op"] != "qkv":
            dy = wide(s.get("dy"))
            if case["op"] == "headwise":
                y, grads = _exact_headwise(wide(s["x"]), wide(s["weight"]), wide(s["static_w"]), case["residual"],
                                           case["hs"], dy)
            else:
                y, grads = _exact_lowrank(wide(s["x"]), wide(s["z"]), wide(s["U"]), wide(s["static_w"]),
                                          case["residual"], dy)
            return {"y": y, "grads": tuple(grads)} if train else {"y": y}
        B, T, D, R, hd = case["B"], case["T"], case["D"], case["R"], case["hd"]
        m, H = s["module"], D // hd
        pre, w_in = wide(s["pre_z"]).view(B * T, D), wide(m.proj_in.weight)
        ys, dz, dU, dsw = [], [], [], []
        dx = torch.empty(B, T, GROUPS * D, dtype=torch.float64, device=pre.device) if train else None
        for g in range(GROUPS):
            z = (pre @ w_in[g * R:(g + 1) * R].t().contiguous()).view(B, T, R)
            dy = wide(s["dy"][g]).transpose(1, 2).reshape(B, T, D) if train else None
            y, grads = _exact_lowrank(wide(s["x"][..., g * D:(g + 1) * D]), z, wide(m.proj_out[g]),
                                      wide(m.proj_out_bias[g]), True, dy)
            ys.append(y.view(B, T, H, hd).transpose(1, 2).contiguous())
            if train:
                dx[..., g * D:(g + 1) * D] = grads[0]
                dz.append(grads[1].view(B * T, R))
                dU.append(grads[2])
                dsw.append(grads[3])
        if not train:
            return {"y": tuple(ys)}
        dz = torch.cat(dz, dim=1)
        dpre = (dz @ w_in).view(B, T, D)
        return {"y": tuple(ys), "grads": (dx, dpre, dz.t().contiguous() @ pre, torch.stack(dU), torch.stack(dsw))}
