"""The work that programs using this library give it, as cases that can be timed and checked.

Every case goes through the public entry points of kunlunk200_lib_amd. Sizes are the
Llama-2-7B projections that bench.py and the tests use (K4096 with N4096, N11008, N12288
and N32000, K11008 with N4096), the rowwise INT8 bench shape, and ragged ones.

`call` of a case:
  matmul   one matmul() of [n, k] weights of `type`, X [batch, k]
  step     the Q4_0 projections of `layers` decoder layers for `batch` tokens, then the
           LM head (n_head rows; 0: none), the way a decode loop submits them
  mlp      a Q4_0 feed-forward block with its norm and residual, for `batch` prompt tokens
  native   one native_q4_matmul()
  common   one common_q4_matmul() of `batch` rows
"""
import torch

import kunlunk200_lib_amd as kl

DEV = 0
EPS = 1e-5


def listed():
    return [
        # the smallest call of the bench's rowwise INT8 set: launch and call cost
        {"name": "i8_k1024_n512_b4", "call": "matmul", "type": "rowwise_i8", "k": 1024, "n": 512, "batch": 4},
        # single-user decoding: every weight read once from HBM for one token
        {"name": "q4_step_b1", "call": "step", "k": 4096, "ffn": 11008, "n_head": 32000, "layers": 2, "batch": 1},
        # a few users, or a short speculative window
        {"name": "q4_step_b8", "call": "step", "k": 4096, "ffn": 11008, "n_head": 0, "layers": 1, "batch": 8},
        # continuous batching: tens of sequences per decode step
        {"name": "q4_step_b32", "call": "step", "k": 4096, "ffn": 11008, "n_head": 0, "layers": 1, "batch": 32},
        # the bench's prefill GEMM
        {"name": "q4_gemm_b512", "call": "matmul", "type": "q4_0", "k": 4096, "n": 11008, "batch": 512},
        # a long prompt through a whole feed-forward block: the largest case
        {"name": "q4_mlp_b2048", "call": "mlp", "k": 4096, "ffn": 11008, "batch": 2048},
        # the last chunk of a prompt on a matrix with odd sizes (K % 64 != 0, N odd)
        {"name": "q4_ragged_b77", "call": "matmul", "type": "q4_0", "k": 5600, "n": 2999, "batch": 77},
        # prefill on half-precision weights
        {"name": "f16_gemm_b512", "call": "matmul", "type": "f16", "k": 4096, "n": 4096, "batch": 512},
        # full-precision weights over a batch
        {"name": "f32_b64", "call": "matmul", "type": "f32", "k": 4096, "n": 4096, "batch": 64},
        # prefill on rowwise INT8 weights, activations quantized on the way
        {"name": "i8_gemm_b512", "call": "matmul", "type": "rowwise_i8", "k": 4096, "n": 4096, "batch": 512},
        # the native Q4 layout for a few tokens (a call that completes before it returns)
        {"name": "native_b4", "call": "native", "k": 4096, "n": 11008, "batch": 4, "f16": False},
        # the common Q4 ABI on a prompt chunk (completes before it returns)
        {"name": "common_m512", "call": "common", "k": 4096, "n": 11008, "batch": 512, "f16": False},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def _k(rng, lo, hi):
    """A row length: mostly multiples of 256, and any multiple of 32."""
    step = rng.choice([256, 256, 64, 32])
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    call = rng.choice(["step", "matmul", "matmul", "matmul", "matmul", "mlp", "native", "common"])
    if call == "step":
        return {"call": call, "k": _k(rng, 1024, 5120), "ffn": _k(rng, 2048, 14336), "n_head": rng.choice([0, 0, 32000]),
                "layers": 1, "batch": _log(rng, 1, 48)}
    if call == "mlp":
        return {"call": call, "k": _k(rng, 1024, 4096), "ffn": _k(rng, 2048, 11008), "batch": _log(rng, 64, 2048)}
    if call == "native":
        return {"call": call, "k": _k(rng, 1024, 11008), "n": _log(rng, 65, 11008), "batch": _log(rng, 1, 16),
                "f16": rng.random() < 0.5}
    if call == "common":
        return {"call": call, "k": _k(rng, 1024, 11008), "n": _log(rng, 65, 11008), "batch": _log(rng, 1, 512),
                "f16": rng.random() < 0.5}
    kind = rng.choice(["q4_0", "q4_0", "f16", "f32", "rowwise_i8"])
    most_b, most_w = {"q4_0": (2048, 1 << 27), "f16": (2048, 1 << 27), "f32": (256, 1 << 24),
                      "rowwise_i8": (1024, 48 << 20)}[kind]
    k = _k(rng, 256, 11008)
    n = min(_log(rng, 65, 32000), most_w // k)
    # one prompt's worth of work at most; ragged rows (K % 64 != 0) at small batch on small matrices
    batch = min(_log(rng, 1, most_b), max(1, (1 << 36) // (k * n)))
    if k % 64 and batch < 64:
        n = min(n, 4096)
    return {"call": call, "type": kind, "k": k, "n": n, "batch": batch}


# --- inputs ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _gauss(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * scale


def _q4(w):
    """F32 [n, k] -> Q4_0 blocks [n, k/32*18] (the ggml closed form)."""
    n, k = w.shape
    b = w.view(n, k // 32, 32)
    m = b.gather(2, b.abs().argmax(2, keepdim=True))
    d = m / -8.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    q = (b * inv + 8.5).trunc().clamp(max=15).to(torch.uint8)
    out = torch.empty(n, k // 32, 18, dtype=torch.uint8, device=w.device)
    out[..., :2] = d.half().view(torch.uint8).view(n, k // 32, 2)
    out[..., 2:] = q[..., :16] | (q[..., 16:] << 4)
    return out.view(n, k // 32 * 18)


def _q4_weight(g, k, n):
    """Q4_0 rows of N(0, 0.02) weights."""
    out = torch.empty(n, k // 32 * 18, dtype=torch.uint8, device="cuda")
    for r in range(0, n, 8192):
        out[r:r + 8192] = _q4(_gauss(g, min(8192, n - r), k, scale=0.02))
    return out


def _weight(g, case, k, n):
    if case["type"] == "q4_0":
        return _q4_weight(g, k, n)
    w = _gauss(g, n, k, scale=0.02)
    return w.half() if case["type"] == "f16" else w


def _step_inputs(case, seed):
    g, k, f, b = _gen(seed), case["k"], case["ffn"], case["batch"]
    layers = [{"qkv": _q4_weight(g, k, 3 * k), "o": _q4_weight(g, k, k), "gate": _q4_weight(g, k, f),
               "up": _q4_weight(g, k, f), "down": _q4_weight(g, f, k), "attn": _gauss(g, b, k)}
              for _ in range(case["layers"])]
    head = _q4_weight(g, k, case["n_head"]) if case["n_head"] else None
    return {"x": _gauss(g, b, k), "layers": layers, "head": head}


def _mlp_inputs(case, seed):
    g, k, f, b = _gen(seed), case["k"], case["ffn"], case["batch"]
    return {"gate": _q4_weight(g, k, f), "up": _q4_weight(g, k, f), "down": _q4_weight(g, f, k),
            "norm": 1 + _gauss(g, k, scale=0.1), "x": _gauss(g, b, k)}


def _product_inputs(case, seed):
    g, k, n, b = _gen(seed), case["k"], case["n"], case["batch"]
    if case["call"] == "matmul":
        return {"w": _weight(g, case, k, n), "x": _gauss(g, b, k)}
    x = _gauss(g, b, k)
    return {"w": _q4_weight(g, k, n), "x": x.half() if case["f16"] else x}


def _inputs(case, seed):
    return {"step": _step_inputs, "mlp": _mlp_inputs}.get(case["call"], _product_inputs)(case, seed)


def _out(*shape):
    return torch.zeros(*shape, device="cuda")


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    k, b, call = case["k"], case["batch"], case["call"]
    if call == "step":
        for layer in s["layers"]:
            layer["y"] = {"qkv": _out(b, 3 * k), "o": _out(b, k), "act": _out(b, case["ffn"]), "down": _out(b, k)}
        s["logits"] = _out(b, case["n_head"]) if case["n_head"] else None
        s["kernel"] = kl.Kernel()
    elif call == "mlp":
        s["h"], s["act"], s["y"] = _out(b, k), _out(b, case["ffn"]), _out(b, k)
        s["kernel"] = kl.Kernel()
    else:
        n = case["n"]
        s["y"] = _out(b, n)
        if call == "matmul":
            s["kernel"] = kl.Kernel()
            if case["type"] == "rowwise_i8":
                packed = torch.zeros(kl.packed_i8_size(k, n), dtype=torch.uint8, device="cuda")
                rows = s.pop("w").cpu().numpy()
                torch.cuda.synchronize()
                kl.upload_i8_rows(DEV, packed.data_ptr(), k, n, 0, n, rows)
                s["w"] = packed
                s["scales"] = kl.packed_i8_scales(packed.data_ptr(), k, n)
                s["maxima"] = kl.packed_i8_maxima(packed.data_ptr(), k, n)
        else:
            q4 = s.pop("w").cpu().numpy()
            torch.cuda.synchronize()
            if call == "native":
                s["w"] = torch.zeros(kl.native_q4_size(k, n), dtype=torch.uint8, device="cuda")
                torch.cuda.synchronize()
                kl.upload_native_q4(DEV, s["w"].data_ptr(), q4, k, n)
                s["workspace"] = kl.NativeQ4Workspace()
            else:
                s["w"] = kl.CommonQ4Weight(DEV, k, n)
                s["w"].upload(q4)
                s["workspace"] = kl.CommonQ4Workspace()
    torch.cuda.synchronize()
    return s


# --- one pass -------------------------------------------------------------------------

def _run_step(s):
    case, kernel = s["case"], s["kernel"]
    k, f, b, q4 = case["k"], case["ffn"], case["batch"], kl.WeightType.q4_0
    x = s["x"]
    out = []
    for layer in s["layers"]:
        y = layer["y"]
        kl.matmul(kernel, DEV, y["qkv"].data_ptr(), layer["qkv"].data_ptr(), x.data_ptr(), k, 3 * k, b, q4)
        kl.matmul(kernel, DEV, y["o"].data_ptr(), layer["o"].data_ptr(), layer["attn"].data_ptr(), k, k, b, q4)
        kl.matmul_swiglu(kernel, DEV, y["act"].data_ptr(), layer["gate"].data_ptr(), layer["up"].data_ptr(),
                         y["o"].data_ptr(), k, f, b, q4)
        kl.matmul(kernel, DEV, y["down"].data_ptr(), layer["down"].data_ptr(), y["act"].data_ptr(), f, k, b, q4)
        x = y["down"]
        out.append(y)
    if s["head"] is not None:
        kl.matmul(kernel, DEV, s["logits"].data_ptr(), s["head"].data_ptr(), x.data_ptr(), k, case["n_head"], b, q4)
        out.append(s["logits"])
    return out


def _run_mlp(s):
    case, kernel, op = s["case"], s["kernel"], kl.ElementwiseOp
    k, f, b, q4 = case["k"], case["ffn"], case["batch"], kl.WeightType.q4_0
    x, h, act, y = s["x"].data_ptr(), s["h"].data_ptr(), s["act"].data_ptr(), s["y"].data_ptr()
    kl.elementwise(kernel, DEV, h, x, x, b * k, k, b * k, op.rms_norm, EPS)
    kl.elementwise(kernel, DEV, h, h, s["norm"].data_ptr(), b * k, k, k, op.multiply)
    kl.matmul_swiglu(kernel, DEV, act, s["gate"].data_ptr(), s["up"].data_ptr(), h, k, f, b, q4)
    kl.matmul(kernel, DEV, y, s["down"].data_ptr(), act, f, k, b, q4)
    kl.elementwise(kernel, DEV, y, y, x, b * k, k, b * k, op.add)
    return {"h": s["h"], "act": s["act"], "y": s["y"]}


def run(state):
    case = state["case"]
    call = case["call"]
    if call == "step":
        return _run_step(state)
    if call == "mlp":
        return _run_mlp(state)
    k, n, b, y, x = case["k"], case["n"], case["batch"], state["y"], state["x"]
    if call == "matmul":
        kl.matmul(state["kernel"], DEV, y.data_ptr(), state["w"].data_ptr(), x.data_ptr(), k, n, b,
                  kl.WeightType[case["type"]], state.get("scales"), state.get("maxima"))
    else:
        t = kl.InputType.f16 if case["f16"] else kl.InputType.f32
        if call == "native":
            kl.native_q4_matmul(state["workspace"], DEV, y.data_ptr(), state["w"].data_ptr(), x.data_ptr(), k, n, b, t)
        else:
            kl.common_q4_matmul(state["workspace"], DEV, y.data_ptr(), state["w"], x.data_ptr(), b, t)
    return y


# --- what a pass cannot do without ------------------------------------------------------

def _cost(weight_bytes, k, n, b, x_bytes=4):
    return weight_bytes + x_bytes * k * b + 4 * n * b, 2 * k * n * b


def _q4_bytes(k, n):
    return k // 32 * 18 * n


def work(case):
    k, b, call = case["k"], case["batch"], case["call"]
    if call == "step":
        f = case["ffn"]
        parts = [_cost(_q4_bytes(k, 3 * k), k, 3 * k, b), _cost(_q4_bytes(k, k), k, k, b),
                 _cost(2 * _q4_bytes(k, f), k, f, b), (0, 2 * k * f * b), _cost(_q4_bytes(f, k), f, k, b)]
        parts *= case["layers"]
        if case["n_head"]:
            parts.append(_cost(_q4_bytes(k, case["n_head"]), k, case["n_head"], b))
    elif call == "mlp":
        f = case["ffn"]
        # h, act and y are outputs of the pass, written once and read by the next call
        parts = [(8 * b * k, 0), (8 * b * k, 0), _cost(2 * _q4_bytes(k, f), k, f, b), (0, 2 * k * f * b),
                 _cost(_q4_bytes(f, k), f, k, b), (12 * b * k, 0)]
    else:
        n = case["n"]
        if call == "matmul":
            weights = {"q4_0": _q4_bytes(k, n), "f16": 2 * k * n, "f32": 4 * k * n, "rowwise_i8": k * n + 4 * n}
            parts = [_cost(weights[case["type"]], k, n, b)]
        else:
            parts = [_cost(_q4_bytes(k, n), k, n, b, 2 if case["f16"] else 4)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    # fp16 matrix products (batch 64 and up): both operands are rounded to 11 bits
    if case["call"] == "mlp" or (case["call"] == "matmul" and case["type"] in ("q4_0", "f16") and case["batch"] >= 64):
        return {"rel": 1.5e-3}
    # 32-bit sums, and 32-bit combinations of exact integer sums
    return {"rel": 1e-5}


# --- the same in 64 bits ----------------------------------------------------------------

def _decode(q4, k):
    n = q4.shape[0]
    b = q4.view(n, k // 32, 18)
    d = b[..., :2].contiguous().view(torch.float16).double()
    v = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], 2).double() - 8
    return (v * d).view(n, k)


def _times(x, q4):
    """X W^T in 64 bits for Q4_0 rows, a slab of rows at a time."""
    x = x.double()
    return torch.cat([x @ _decode(w, x.shape[1]).T for w in q4.split(4096)], 1)


def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def _i8_rows(w):
    """The codes that rows of weights are stored as, times their scales."""
    scale = w.abs().amax(1, keepdim=True) / 127
    v = w / torch.where(scale > 0, scale, torch.ones_like(scale))
    return ((v.abs() + 0.5).floor() * v.sign()).double() * scale.double()


def exact(case, seed):
    s = _inputs(case, seed)
    call = case["call"]
    if call == "step":
        x, out = s["x"], []
        for layer in s["layers"]:
            o = _times(layer["attn"], layer["o"])
            act = _silu_mul(_times(o, layer["gate"]), _times(o, layer["up"]))
            down = _times(act, layer["down"])
            out.append({"qkv": _times(x, layer["qkv"]), "o": o, "act": act, "down": down})
            x = down
        if s["head"] is not None:
            out.append(_times(x, s["head"]))
        return out
    if call == "mlp":
        x = s["x"].double()
        h = x / (x.square().mean(1, keepdim=True) + EPS).sqrt() * s["norm"].double()
        act = _silu_mul(_times(h, s["gate"]), _times(h, s["up"]))
        return {"h": h, "act": act, "y": _times(act, s["down"]) + x}
    if call != "matmul" or case["type"] == "q4_0":
        return _times(s["x"], s["w"])
    w = _i8_rows(s["w"]) if case["type"] == "rowwise_i8" else s["w"].double()
    return s["x"].double() @ w.T
