"""The work whose speed is followed: calls of the packed-weight linears at the sizes users run them.

Each case is one or several linears through qlin's public ops, on inputs made on the GPU from a seed.
A case is a dict: `op` (gguf, int8, a8 or train), `m` activation rows, `layers` ("KxN" joined by "+",
for gguf with the block type in front, a trailing "r" asks for a residual), `dtype`, `bias`, and per
op the ConvRot group `g`, weight `bits`, scale group `gs`, `codebook` and LoRA rank `lora`.
Consecutive layers with the same K share their activation, as projections of one block do.
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mac-kernels-public_amd"))

import qlin  # noqa: E402

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BLOCK = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210),
         "IQ4_NL": (32, 18), "IQ4_XS": (256, 136)}
IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
CODEBOOK = (-0.980602, -0.794529, -0.638165, -0.500986, -0.377321, -0.263187, -0.155210, -0.050720,
            0.052541, 0.156985, 0.265284, 0.379533, 0.502636, 0.638953, 0.794876, 0.980671)


def listed():
    return [
        # one projection of a language model's decode step, one token
        {"name": "gguf_decode", "op": "gguf", "m": 1, "layers": "Q4_K:4096x4096", "dtype": "fp16", "bias": False},
        # gate, up and down of a decode step; mixed files keep the down projection at 6 bits
        {"name": "gguf_decode_mlp", "op": "gguf", "m": 1, "layers": "Q4_K:5120x13824+Q4_K:5120x13824+Q6_K:13824x5120",
         "dtype": "bf16", "bias": False},
        # a small decode batch
        {"name": "gguf_batch", "op": "gguf", "m": 8, "layers": "Q8_0:4096x4096", "dtype": "fp16", "bias": False},
        # a text encoder on a prompt of 77 tokens
        {"name": "gguf_prompt", "op": "gguf", "m": 77, "layers": "Q5_K:4096x4096", "dtype": "bf16", "bias": True},
        # the MLP of a diffusion transformer from a GGUF file, 4608 image and text tokens
        {"name": "gguf_image_mlp", "op": "gguf", "m": 4608, "layers": "Q4_K:3072x12288+Q6_K:12288x3072", "dtype": "bf16",
         "bias": True},
        # a modulation projection: one vector per step
        {"name": "int8_vector", "op": "int8", "m": 1, "layers": "3072x3072", "dtype": "fp16", "bias": True, "g": 128,
         "lora": 0},
        # the text stream of a diffusion transformer
        {"name": "int8_text", "op": "int8", "m": 256, "layers": "3072x3072", "dtype": "fp16", "bias": True, "g": 128,
         "lora": 0},
        # the four linears of a diffusion transformer block, residuals on the two that end a branch
        {"name": "int8_block", "op": "int8", "m": 4608, "layers": "3072x9216+3072x3072r+3072x12288+12288x3072r",
         "dtype": "fp16", "bias": True, "g": 128, "lora": 0},
        # an attention projection with an unmerged LoRA
        {"name": "int8_lora", "op": "int8", "m": 4608, "layers": "6144x6144", "dtype": "bf16", "bias": True, "g": 256,
         "lora": 64},
        # one frozen MLP layer in LoRA training: forward and the gradient of its input, 1056 tokens
        {"name": "int8_train", "op": "train", "m": 1056, "layers": "6144x16384", "dtype": "bf16", "bias": True, "g": 256},
        # W4A8 MLP up projection
        {"name": "w4a8_image_up", "op": "a8", "m": 4096, "layers": "3072x12288", "dtype": "fp16", "bias": True, "g": 128,
         "bits": 4, "gs": 128, "codebook": False},
        # W6A8 MLP of a video model, 9504 tokens: up and down
        {"name": "w6a8_video_mlp", "op": "a8", "m": 9504, "layers": "5120x13824+13824x5120", "dtype": "bf16", "bias": True,
         "g": 256, "bits": 6, "gs": 64, "codebook": False},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One call of the ranges above: decode and small batches, prompts, image- and video-sized rows."""
    op = rng.choice(("gguf", "gguf", "gguf", "int8", "int8", "int8", "a8", "a8", "train"))
    lo, hi = rng.choice(((1, 16), (17, 512), (513, 9504)))
    if op == "train":
        lo, hi = 64, 4608
    m = _log(rng, lo, hi)
    while True:
        k = 256 * max(4, _log(rng, 4, 64))
        n = _log(rng, 512, 16384)
        if rng.random() < 0.8:
            n = n // 64 * 64
        if 2 * m * n * k <= 1.5e12:
            break
    case = {"op": op, "m": m, "layers": "%dx%d" % (k, n), "dtype": rng.choice(("fp16", "bf16", "bf16", "fp16", "fp32")),
            "bias": rng.random() < 0.7}
    if op == "gguf":
        case["layers"] = rng.choice(sorted(BLOCK)) + ":" + case["layers"]
        return case
    case["g"] = rng.choice((128, 256))
    if op == "int8":
        case["lora"] = rng.choice((0, 0, 16, 64)) if m > 1 else 0
        if not case["lora"] and m > 16 and rng.random() < 0.3:
            case["layers"] += "r"
    elif op == "a8":
        case["bits"] = rng.choice((4, 6))
        case["gs"] = rng.choice((64, 128))
        case["codebook"] = case["bits"] == 4 and rng.random() < 0.5
    return case


def _layers(case):
    for text in case["layers"].split("+"):
        qtype, _, size = text.rpartition(":")
        k, n = size.rstrip("r").split("x")
        yield qtype, int(k), int(n), size.endswith("r")


# ------------------------------------------------------------------------------------------ inputs

def _activation(gen, m, k, dtype):
    """Gaussian rows with unequal channels, one channel in a hundred 10 times larger."""
    gain = torch.exp(0.3 * torch.randn(k, generator=gen, device=DEV))
    gain = torch.where(torch.rand(k, generator=gen, device=DEV) < 0.01, 10 * gain, gain)
    return (torch.randn(m, k, generator=gen, device=DEV) * gain).to(dtype)


def _f16(d):
    """fp16 scales as (their two bytes, their value)."""
    h = d.half()
    return h.unsqueeze(-1).view(torch.uint8), h.float()


def _nearest(v, levels):
    t = torch.tensor(levels, device=DEV)
    return torch.bucketize(v, (t[1:] + t[:-1]) / 2)


def _absmax_signed(v):
    return v.gather(-1, v.abs().argmax(-1, keepdim=True)).squeeze(-1)


def _div(a, b):
    return a / torch.where(b == 0, 1.0, b)


def _k_scales(sc, mn):
    """Eight 6-bit scales and minima in the K-quants' 12 bytes."""
    return torch.cat([(sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6), (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6),
                      (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1).byte()


def _gguf_weight(gen, qtype, n, k):
    """N(0, 0.02) weights in blocks of `qtype`: uint8 [n, row bytes]."""
    qk, ts = BLOCK[qtype]
    x = (torch.randn(n * (k // qk), qk, generator=gen, device=DEV)) * 0.02
    nb = x.shape[0]
    if qtype == "Q8_0":
        db, d = _f16(x.abs().amax(-1) / 127)
        out = [db, _div(x, d[:, None]).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)]
    elif qtype in ("Q4_0", "IQ4_NL"):
        db, d = _f16(_absmax_signed(x) / (-8 if qtype == "Q4_0" else -127))
        v = _div(x, d[:, None])
        q = ((v.round() + 8).clamp(0, 15) if qtype == "Q4_0" else _nearest(v, IQ4)).to(torch.uint8)
        out = [db, q[:, :16] | (q[:, 16:] << 4)]
    elif qtype in ("Q4_K", "Q5_K"):
        top = 15 if qtype == "Q4_K" else 31
        s = x.view(nb, 8, 32)
        low = s.amin(-1).clamp(max=0)
        scale, mins = (s.amax(-1) - low) / top, -low
        db, d = _f16(scale.amax(-1) / 63)
        mb, dm = _f16(mins.amax(-1) / 63)
        sc, mc = (_div(a, b[:, None]).round().clamp(0, 63) for a, b in ((scale, d), (mins, dm)))
        q = _div(s + (dm[:, None] * mc)[..., None], (d[:, None] * sc)[..., None]).round().clamp(0, top).to(torch.uint8)
        p = (q & 15).view(nb, 4, 2, 32)
        out = [db, mb, _k_scales(sc.to(torch.int32), mc.to(torch.int32))]
        if qtype == "Q5_K":
            out.append(((q >> 4).int() << torch.arange(8, device=DEV)[None, :, None]).sum(1).byte())
        out.append((p[:, :, 0] | (p[:, :, 1] << 4)).reshape(nb, 128))
    elif qtype == "Q6_K":
        s = x.view(nb, 16, 16)
        sub = _absmax_signed(s) / -32
        db, d = _f16(sub.abs().amax(-1) / 127)
        sc = _div(sub, d[:, None]).round().clamp(-128, 127)
        q = (_div(s, (d[:, None] * sc)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8).view(nb, 2, 4, 32)
        ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], -1)
        qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        out = [ql.reshape(nb, 128), qh.reshape(nb, 64), sc.to(torch.int8).view(torch.uint8), db]
    else:  # IQ4_XS
        s = x.view(nb, 8, 32)
        sub = _absmax_signed(s) / -127
        db, d = _f16(sub.abs().amax(-1) / 32)
        ls = (_div(sub, d[:, None]).round() + 32).clamp(0, 63).to(torch.int32)
        q = _nearest(_div(s, (d[:, None] * (ls - 32))[..., None]), IQ4).to(torch.uint8)
        sh = ((ls >> 4) << (2 * torch.arange(8, device=DEV))).sum(1)
        out = [db, torch.stack([sh & 255, sh >> 8], 1).byte(), ((ls[:, 0::2] & 15) | ((ls[:, 1::2] & 15) << 4)).byte(),
               (q[..., :16] | (q[..., 16:] << 4)).reshape(nb, 128)]
    return torch.cat(out, 1).view(n, k // qk * ts)


def _int8_weight(gen, n, k, scale_dtype):
    """Gaussian int8 rows (a rotated weight is close to Gaussian) and their scales."""
    q = (torch.randn(n, k, generator=gen, device=DEV) * 34).round_().clamp_(-127, 127).to(torch.int8)
    return q, ((0.7 + 0.6 * torch.rand(n, generator=gen, device=DEV)) * 0.02 / 34).to(scale_dtype)


def _a8_weight(gen, n, k, bits, gs, codebook):
    """Gaussian weights as 4- or 6-bit codes per group: (packed codes, s_rel, s_channel, codebook)."""
    w = torch.randn(n, k // gs, gs, generator=gen, device=DEV) * 0.02
    amax = w.abs().amax(-1)
    top = (1 << (bits - 1)) - 1
    if codebook:
        c = _nearest(w / amax[..., None], CODEBOOK)
        step = amax
    else:
        step = amax / top
        c = (w / step[..., None]).round().clamp(-top, top) + (1 << (bits - 1))
    c = c.to(torch.uint8).view(n, k)
    s_channel = amax.amax(-1) / 127
    packed = c[:, 0::2] & 15 | (c[:, 1::2] & 15) << 4
    if bits == 6:
        h = c >> 4
        packed = torch.cat([packed, h[:, 0::4] | h[:, 1::4] << 2 | h[:, 2::4] << 4 | h[:, 3::4] << 6], 1)
    cb = torch.tensor(CODEBOOK, device=DEV) if codebook else None
    return packed.contiguous().view(torch.int8), (step / s_channel[:, None]).half(), s_channel, cb


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    dtype, m, op = DTYPES[case["dtype"]], case["m"], case["op"]
    calls, x = [], None
    for qtype, k, n, residual in _layers(case):
        if x is None or x.shape[1] != k:
            x = _activation(gen, m, k, dtype)
        c = {"x": x, "n": n, "k": k}
        if op == "gguf":
            c["w"], c["qtype"] = _gguf_weight(gen, qtype, n, k), qtype
        elif op == "a8":
            c["w"] = _a8_weight(gen, n, k, case["bits"], case["gs"], case["codebook"])
        else:
            c["w"] = _int8_weight(gen, n, k, torch.float16 if dtype == torch.float16 else torch.float32)
        c["bias"] = (0.1 * torch.randn(n, generator=gen, device=DEV)).to(dtype) if case["bias"] else None
        c["more"] = {}
        if residual:
            c["more"]["residual"] = torch.randn(m, n, generator=gen, device=DEV).to(dtype)
        if case.get("lora"):
            r = case["lora"]
            c["more"].update(lora_down=(torch.randn(r, k, generator=gen, device=DEV) * k ** -0.5).to(dtype),
                             lora_up=(torch.randn(n, r, generator=gen, device=DEV) * 0.1).to(dtype), lora_scale=0.8)
        if op == "train":
            c["x"] = x.detach().requires_grad_(True)
            c["dy"] = (torch.randn(m, n, generator=gen, device=DEV) * 1e-3).to(dtype)
        calls.append(c)
    return {"case": dict(case), "calls": calls}


def run(state):
    case, out = state["case"], []
    for c in state["calls"]:
        if case["op"] == "gguf":
            out.append(qlin.gguf_linear(c["x"], c["w"], c["qtype"], (c["n"], c["k"]), c["bias"]))
        elif case["op"] == "int8":
            q, s = c["w"]
            out.append(qlin.int8_linear(c["x"], q, s, c["bias"], convrot=True, convrot_groupsize=case["g"], **c["more"]))
        elif case["op"] == "a8":
            q, s_rel, s_channel, cb = c["w"]
            out.append(qlin.w4a8_int8_linear(c["x"], q, s_rel, s_channel, cb, None, c["bias"], case["gs"], case["g"]))
        else:
            q, s = c["w"]
            y = qlin.int8_linear_trainable(c["x"], q, s, c["bias"], True, case["g"])
            out.append(y.detach())
            out += torch.autograd.grad(y, c["x"], c["dy"])
    return out


def work(case):
    nbytes = flops = 0
    es, m, seen = (4 if case["dtype"] == "fp32" else 2), case["m"], None
    for qtype, k, n, residual in _layers(case):
        if case["op"] == "gguf":
            nbytes += n * (k // BLOCK[qtype][0]) * BLOCK[qtype][1]
        elif case["op"] == "a8":
            nbytes += n * k * case["bits"] // 8 + n * (k // case["gs"]) * 2 + 4 * n
        else:
            nbytes += n * k + 4 * n
        nbytes += es * (m * n + (m * k if seen != k else 0) + (n if case["bias"] else 0) + (m * n if residual else 0))
        flops += 2 * m * n * k
        if case.get("lora"):
            nbytes += es * case["lora"] * (n + k)
            flops += 2 * m * case["lora"] * (n + k)
        if case["op"] == "train":
            nbytes += es * m * (n + k)
            flops += 2 * m * n * k
        seen = k
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # one rounding to the output type (fp16 2.1e-4, bf16 1.7e-3 of a normal result), the operand rounded to
    # fp16 in the weight-only paths (2e-4 to 4e-4), for A8 an int8 code that a rounding of the rotation moves
    return {"rel": {"fp16": 2e-3, "bf16": 8e-3, "fp32": 2e-3}[case["dtype"]]}


# ----------------------------------------------------------------------------- the results in 64 bits

def _half(b):
    return b.contiguous().view(torch.float16).double()


def _gguf_values(raw, qtype, n, k):
    qk, ts = BLOCK[qtype]
    b = raw.reshape(-1, ts)
    nb = b.shape[0]

    def nibbles(q):  # [.., 16] bytes: 32 values, low halves first
        return torch.cat([q & 15, q >> 4], -1).long()

    levels = torch.tensor(IQ4, device=DEV, dtype=torch.float64)
    if qtype == "Q8_0":
        w = _half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif qtype == "Q4_0":
        w = _half(b[:, :2]) * (nibbles(b[:, 2:]) - 8)
    elif qtype == "IQ4_NL":
        w = _half(b[:, :2]) * levels[nibbles(b[:, 2:])]
    elif qtype in ("Q4_K", "Q5_K"):
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, -128:].reshape(nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(nb, 8, 32).int()
        if qtype == "Q5_K":
            q = q + (((b[:, None, 16:48].int() >> torch.arange(8, device=DEV)[None, :, None]) & 1) << 4)
        w = (_half(b[:, :2]) * sc)[..., None] * q - (_half(b[:, 2:4]) * mn)[..., None]
    elif qtype == "Q6_K":
        ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (lo | (hi << 4)).reshape(nb, 16, 16).double() - 32
        w = (_half(b[:, 208:]) * b[:, 192:208].contiguous().view(torch.int8).double())[..., None] * q
    else:
        sh = b[:, 2].int() | (b[:, 3].int() << 8)
        sl = torch.stack([b[:, 4:8] & 15, b[:, 4:8] >> 4], -1).reshape(nb, 8).int()
        ls = sl | (((sh[:, None] >> (2 * torch.arange(8, device=DEV))) & 3) << 4)
        w = (_half(b[:, :2]) * (ls - 32))[..., None] * levels[nibbles(b[:, 8:].reshape(nb, 8, 16))]
    return w.reshape(n, k)


def _rotate(x, g):
    """x times the block Hadamard: the Kronecker power of the 4 x 4 one (an H2 factor in front for 2 * 4^p)."""
    h4 = torch.ones(4, 4, dtype=torch.float64, device=DEV) - 2 * torch.eye(4, dtype=torch.float64, device=DEV).flip(0)
    h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    while h.shape[0] * 4 <= g:
        h = torch.kron(h, h4)
    if h.shape[0] < g:
        h = torch.kron(torch.tensor([[1.0, 1.0], [1.0, -1.0]], dtype=torch.float64, device=DEV), h)
    return (x.double().reshape(-1, g) @ (h / g ** 0.5)).reshape(x.shape)


def _a8_rows(x, g):
    """Per-token int8 of the rotated rows, with the rounding steps of the activation's type."""
    r = _rotate(x, g).to(x.dtype)
    scale = (r.float().abs().amax(1, keepdim=True) / 127).clamp(min=1e-30)
    q = (r.float() / scale.to(x.dtype).float()).to(x.dtype).float().round().clamp(-128, 127)
    return q.double(), scale.double()


def _a8_grid(w, k, bits, gs):
    packed, s_rel, s_channel, cb = w
    p = packed.view(torch.uint8)
    n = p.shape[0]
    low = p[:, :k // 2]
    c = torch.stack([low & 15, low >> 4], -1).reshape(n, k)
    if bits == 6:
        hi = p[:, k // 2:]
        c = c | (torch.stack([(hi >> s) & 3 for s in (0, 2, 4, 6)], -1).reshape(n, k) << 4)
    level = cb[c.long()] if cb is not None else c.float() - (1 << (bits - 1))
    grid = (level * s_rel.float().repeat_interleave(gs, 1)).round().clamp(-127, 127)
    return grid.double(), s_channel.double()


def exact(case, seed):
    out = []
    for c in prepare(case, seed)["calls"]:
        x = c["x"].detach()
        if case["op"] == "gguf":
            y = x.double() @ _gguf_values(c["w"], c["qtype"], c["n"], c["k"]).T
        elif case["op"] == "a8":
            q, sx = _a8_rows(x, case["g"])
            grid, s_channel = _a8_grid(c["w"], c["k"], case["bits"], case["gs"])
            y = q @ grid.T * sx * s_channel
        else:
            q, s = c["w"][0].double(), c["w"][1].double()
            y = _rotate(x, case["g"]) @ q.T * s
        if c["bias"] is not None:
            y = y + c["bias"].double()
        more = c["more"]
        if "lora_down" in more:
            y = y + more["lora_scale"] * (x.double() @ more["lora_down"].double().T) @ more["lora_up"].double().T
        if "residual" in more:
            y = y + more["residual"].double()
        out.append(y)
        if case["op"] == "train":
            out.append(_rotate((c["dy"].double() * s) @ q, case["g"]))
    return out
