"""The work this library is used for, as measurable cases.

Each case is one call, or one short chain of calls, that a program using the
library makes per layer: W8A8 linears (opcode 15), packed-F16 products with
their epilogues (opcodes 1/16), quantized-weight products (opcodes 2/3/4),
model auxiliary ops (opcode 19), and one transformer block sent as a message
of nine requests (opcodes 19, 12 and 15).  Weights are packed once in
prepare(), as a serving program does; inputs and outputs live in HBM.

exact() restates the same mathematics in 64-bit torch without the library:
the quantization of activations to int8 and the conversion of activations to
fp16 are part of what these ops are defined to compute, so they are applied
there too (in 32 bits, as defined); products, sums and everything after them
are in 64 bits.
"""
import ctypes
import math
import os
import struct
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "htp-ops-lib-sd.cpp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import htp_ops as h  # noqa: E402

# ---- the cases ------------------------------------------------------------------


def listed():
    return [
        # one token through an MLP up projection: the decode step, bound by the weights' bytes
        {"name": "w8a8 decode 1x4096x14336", "op": "w8a8", "m": 1, "k": 4096, "n": 14336, "gelu": False},
        # a text encoder's linear over its 77 tokens: the smallest calls, latency and launches
        {"name": "w8a8 text 77x768x3072", "op": "w8a8", "m": 77, "k": 768, "n": 3072, "gelu": False},
        # a diffusion transformer's MLP up projection over 64x64 latent patches
        {"name": "w8a8 dit 4096x1536x6144", "op": "w8a8", "m": 4096, "k": 1536, "n": 6144, "gelu": False},
        # fused Q/K/V projection (4096 + 1024 + 1024 columns) of a 2048-token prefill
        {"name": "w8a8 prefill 2048x4096x6144", "op": "w8a8", "m": 2048, "k": 4096, "n": 6144, "gelu": False},
        # a text encoder's MLP: up with QuickGELU, then down, 77 tokens, two dependent calls
        {"name": "f16 text mlp 77x768x3072", "op": "mlp", "m": 77, "d": 768, "f": 3072, "mode": 2},
        # a diffusion transformer's F16 MLP over 4096 image and 77 text tokens: a ragged row count
        {"name": "f16 dit mlp 4173x1536x6144", "op": "mlp", "m": 4173, "d": 1536, "f": 6144, "mode": 1},
        # a VAE decoder's 3x3 convolution at 256x256, 256 channels, as an im2col product (channel-major out)
        {"name": "f16 vae conv 65536x2304x256", "op": "conv", "m": 65536, "k": 2304, "c": 256},
        # a UNet's 3x3 convolution at 32x32, 640 channels: few output tiles, a long sum
        {"name": "f16 unet conv 1024x5760x640", "op": "conv", "m": 1024, "k": 5760, "c": 640},
        # one token through 4-bit weights
        {"name": "q4_0 decode 1x4096x14336", "op": "qk0", "m": 1, "k": 4096, "n": 14336, "type": h.GGML_Q4_0},
        # a 333-token prompt through 8-bit block weights (dequantized once into the F16 image)
        {"name": "q8_0 prefill 333x4096x14336", "op": "qk0", "m": 333, "k": 4096, "n": 14336, "type": h.GGML_Q8_0},
        # the group norm and SiLU before a VAE decoder's last convolutions, 128 channels at 512x512
        {"name": "group norm 128x262144", "op": "aux", "what": "group norm", "rows": 128, "width": 262144},
        # one joint-attention block as one message: norm, Q/K/V, out projection, gate, norm, MLP, gate
        {"name": "dit block 256+4096 tokens", "op": "block", "image": 256, "text": 4096, "heads": 24},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of step between lo and hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    op = rng.choice(["w8a8", "w8a8", "w8a8", "mlp", "mlp", "conv", "conv", "qk0", "qk0", "aux", "block"])
    if op == "w8a8":
        # decode to image-token scale; any column count the format takes (multiples of 64), any row length (of 32)
        k, n = _log(rng, 512, 14336, 32), _log(rng, 512, 14336, 64)
        most = int(min(4608, 2048 * 4096 * 6144 / (k * n)))
        m = _log(rng, 1, max(1, most))
        return {"op": op, "m": m, "k": k, "n": n, "gelu": m > 16 and rng.random() < 0.3}
    if op == "mlp":
        d = _log(rng, 512, 2048, 64)
        f = 4 * d
        return {"op": op, "m": _log(rng, 16, int(min(4608, 4173 * 1536 * 6144 / (d * f)))), "d": d, "f": f,
                "mode": rng.choice([1, 2])}
    if op == "conv":
        # 3x3 convolutions from 1280 channels at 8x8 to 128 channels at 512x512, any aspect ratio
        cin, c = _log(rng, 128, 1280, 32), _log(rng, 64, 1280, 32)
        m = _log(rng, 64, int(min(131072, 65536 * 2304 * 256 / (9 * cin * c), 65536 * 2304 / (9 * cin))))
        return {"op": op, "m": m, "k": 9 * cin, "c": c}
    if op == "qk0":
        k, n = _log(rng, 1024, 8192, 256), _log(rng, 1024, 14336, 64)
        m = rng.choice([1, 1, rng.randint(2, 16), _log(rng, 17, int(min(512, 333 * 4096 * 14336 / (k * n))))])
        return {"op": op, "m": m, "k": k, "n": n, "type": rng.choice([h.GGML_Q4_0, h.GGML_Q8_0, h.GGML_IQ4_NL])}
    if op == "aux":
        what = rng.choice(["group norm", "layer norm", "rms norm", "swiglu", "gelu", "rope", "transpose"])
        if what == "group norm":
            rows = 32 * rng.randint(4, 20)
            return {"op": op, "what": what, "rows": rows, "width": _log(rng, 256, 128 * 262144 // rows)}
        if what == "rope":
            return {"op": op, "what": what, "rows": _log(rng, 77, 4352), "width": 64 * rng.choice([24, 30, 38])}
        return {"op": op, "what": what, "rows": _log(rng, 77, 4352), "width": _log(rng, 640, 3072, 4)}
    return {"op": op, "image": 32 * rng.randint(1, 8), "text": _log(rng, 77, 4096 if rng.random() < 0.5 else 1024),
            "heads": 24}


# ---- buffers and inputs ---------------------------------------------------------


class _Buf:
    """A torch tensor under the names the library's wrappers use."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


class _Rpc(h.RpcBuffer):
    """An rpcmem buffer in HBM with a torch view of its memory."""

    def __init__(self, shape, dtype=torch.float32):
        n = math.prod(shape)
        super().__init__(n * torch.empty(0, dtype=dtype).element_size(), device=True)
        kind = {torch.float32: "<f4", torch.float16: "<f2", torch.uint8: "|u1"}[dtype]
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (self.ptr, False),
                                         "version": 2}
        self.t = torch.as_tensor(self, device="cuda")

    @classmethod
    def of(cls, t):
        b = cls(tuple(t.shape), t.dtype)
        b.t.copy_(t)
        return b


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def _uniform(g, lo, hi, *shape):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _w8a8_tensors(g, k, n):
    """A constants blob: int8 weights uniform in [-127, 127] in the blob's tile order, their column sums,
    scales that give outputs near one, and a smoothing vector."""
    tiles = torch.randint(-127, 128, (n // 64, k // 32, 2, 8, 32, 4), generator=g, device="cuda", dtype=torch.int8)
    sums = tiles.sum(dim=(1, 3, 5), dtype=torch.int32).reshape(n)
    sw = _uniform(g, 5e-5, 5e-4, n)
    inv = _uniform(g, 0.5, 1.5, k)
    w_end = 128 + k * n
    header = struct.pack("<10IQ80x", 0x38574D48, 1, k, n, 128, w_end, w_end + 4 * n, w_end + 8 * n,
                         w_end + 8 * n + 4 * k, 0, 0)
    head = torch.frombuffer(bytearray(header), dtype=torch.uint8).cuda()
    blob = torch.cat([head, tiles.reshape(-1).view(torch.uint8), sw.view(torch.uint8), sums.view(torch.uint8),
                      inv.view(torch.uint8)])
    return blob, tiles, sw, inv


def _w8a8_input(g, m, k):
    """Normal activations, 1% of the channels twenty times as large (the outliers a transformer has)."""
    x = _normal(g, m, k)
    loud = torch.randperm(k, generator=g, device="cuda")[: max(1, k // 100)]
    x[:, loud] *= 20.0
    return x


def _f16_tensors(g, k, n):
    """Permuted fp16 weights whose products with unit inputs have a variance near one."""
    return (_normal(g, n // 32, k // 32, 16, 32, 2) * (k ** -0.5)).half()


def _qk0_tensors(g, k, n, kind):
    """Super-blocks of 256 weights: 8 fp16 scales, then the codes, which are uniform."""
    raw = torch.randint(0, 256, (k * n // 256, h.lib().hb_qk0_block_bytes(kind)), generator=g, device="cuda",
                        dtype=torch.uint8)
    spread = {h.GGML_Q4_0: 4.6, h.GGML_Q8_0: 74.0, h.GGML_IQ4_NL: 66.0}[kind]
    scales = (_uniform(g, 0.5, 1.5, raw.shape[0], 8) * (k ** -0.5 / spread)).half()
    raw[:, :16] = scales.view(torch.uint8)
    return raw


def _inputs(case, seed):
    """Every tensor of the case, made from the seed alone; prepare() and exact() both start here."""
    g, op = _gen(seed), case["op"]
    if op == "w8a8":
        m, k, n = case["m"], case["k"], case["n"]
        blob, tiles, sw, inv = _w8a8_tensors(g, k, n)
        return {"x": _w8a8_input(g, m, k), "blob": blob, "tiles": tiles, "sw": sw, "inv": inv}
    if op == "mlp":
        m, d, f = case["m"], case["d"], case["f"]
        return {"x": _normal(g, m, d), "w1": _f16_tensors(g, d, f), "w2": _f16_tensors(g, f, d),
                "b1": _normal(g, f, std=0.1), "b2": _normal(g, d, std=0.1)}
    if op == "conv":
        m, k, c = case["m"], case["k"], case["c"]
        x = _normal(g, m, k)
        return {"x": torch.nn.functional.silu(x), "w": _f16_tensors(g, k, c), "b": _normal(g, c, std=0.1)}
    if op == "qk0":
        m, k, n = case["m"], case["k"], case["n"]
        return {"x": _normal(g, m, k), "blocks": _qk0_tensors(g, k, n, case["type"])}
    if op == "aux":
        what, r, w = case["what"], case["rows"], case["width"]
        x = _normal(g, r, 2 * w if what == "swiglu" else w) + 0.3
        if what == "rope":
            angle = _uniform(g, -3.1, 3.1, r, 32)
            p = torch.stack([angle.cos(), -angle.sin(), angle.sin(), angle.cos()], -1)
            return {"x": x, "w": p, "b": None}
        n = r if what == "group norm" else w
        has = what in ("group norm", "layer norm", "rms norm")
        return {"x": x, "w": _normal(g, n, std=0.2) if has else None,
                "b": _normal(g, n, std=0.2) if has and what != "rms norm" else None}
    t, d, hd = case["image"] + case["text"], case["heads"] * 64, 64
    made = {"x": _normal(g, t, d), "attn": _normal(g, t, d), "zero": None}
    for name in ("shift1", "scale1", "gate1", "shift2", "scale2", "gate2"):
        made[name] = _normal(g, d, std=0.3)
    for part in ("image", "text"):
        made[part + "_w"] = _f16_tensors(g, d, 3 * d)
        made[part + "_b"] = _normal(g, 3 * d, std=0.1)
        made[part + "_qn"], made[part + "_kn"] = _uniform(g, 0.5, 1.5, hd), _uniform(g, 0.5, 1.5, hd)
    angle = _uniform(g, -3.1, 3.1, t, hd // 2)
    made["pe"] = torch.stack([angle.cos(), -angle.sin(), angle.sin(), angle.cos()], -1)
    made["o"], made["up"] = _w8a8_tensors(g, d, d), _w8a8_tensors(g, d, 4 * d)
    made["down"] = _w8a8_tensors(g, 4 * d, d)
    return made


# ---- prepare and run ------------------------------------------------------------


def _aux_args(case):
    """Arguments of opcode 19 for the case: mode, count, and the shape it takes."""
    r, w = case["rows"], case["width"]
    return {
        "group norm": dict(mode=2, count=r * w, width=w, channels=r, spatial=w, groups=32, other_count=r,
                           activation=1, eps=1e-6),
        "layer norm": dict(mode=9, count=r * w, width=w, spatial=r, other_count=w, eps=1e-6),
        "rms norm": dict(mode=1, count=r * w, width=w, other_count=w, eps=1e-6),
        "swiglu": dict(mode=12, count=r * w, width=w, channels=2 * w, spatial=r, activation=1),
        "gelu": dict(mode=6, count=r * w, width=w),
        "rope": dict(mode=11, count=r * w, width=64, channels=w // 64, spatial=r, groups=1, other_count=128 * r),
        "transpose": dict(mode=8, count=r * w, width=w, spatial=r),
    }[case["what"]]


def _empty(nbytes):
    return _Buf(torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device="cuda"))


def _out(*shape):
    return _Buf(torch.empty(shape, device="cuda"))


def _f16_image(t, k, n):
    """The weight image made once per weight (hb_f16_prepack) from the permuted fp16 weight."""
    image = _empty(h.lib().hb_f16_packed_bytes(k, n))
    h.check(h.lib().hb_f16_prepack(image.ptr, t.data_ptr(), k, n, None), "hb_f16_prepack")
    return image


def prepare(case, seed):
    h.init(0)
    made = _inputs(case, seed)
    torch.cuda.synchronize()  # the library has a stream of its own
    op = case["op"]
    if op == "w8a8":
        m, k, n = case["m"], case["k"], case["n"]
        packed = _empty(h.w8a8_packed_bytes(k, n))
        h.check(h.lib().hb_w8a8_prepack(packed.ptr, made["blob"].data_ptr(), k, n, None), "hb_w8a8_prepack")
        state = {"x": _Buf(made["x"]), "packed": packed, "y": _out(m, n), "m": m, "k": k, "n": n,
                 "ws": _empty(h.w8a8_linear_workspace_bytes(m, k, n)),
                 "epilogue": h.EPI_SCALE_GELU if case["gelu"] else h.EPI_SCALE}
    elif op == "mlp":
        m, d, f = case["m"], case["d"], case["f"]
        state = {"x": _Buf(made["x"]), "w1": _f16_image(made["w1"], d, f), "w2": _f16_image(made["w2"], f, d),
                 "b1": _Buf(made["b1"]), "b2": _Buf(made["b2"]), "h": _out(m, f), "y": _out(m, d), "m": m, "d": d,
                 "f": f, "mode": case["mode"],
                 "ws": _empty(max(h.f16_workspace_bytes(m, d, f), h.f16_workspace_bytes(m, f, d)))}
    elif op == "conv":
        m, k, c = case["m"], case["k"], case["c"]
        state = {"x": _Buf(made["x"]), "w": _f16_image(made["w"], k, c), "b": _Buf(made["b"]), "y": _out(c, m),
                 "m": m, "k": k, "c": c, "ws": _empty(h.f16_workspace_bytes(m, k, c))}
    elif op == "qk0":
        m, k, n = case["m"], case["k"], case["n"]
        state = {"x": _Buf(made["x"]), "y": _out(m, n), "m": m, "k": k, "n": n, "type": case["type"],
                 "ws": _empty(h.f16_workspace_bytes(m, k, n))}
        if m <= 16:  # few rows multiply the blocks themselves
            state["blocks"] = _Buf(made["blocks"])
        else:
            state["image"] = _empty(h.lib().hb_f16_packed_bytes(k, n))
            h.check(h.lib().hb_qk0_prepack(state["image"].ptr, made["blocks"].data_ptr(), k, n, case["type"], None),
                    "hb_qk0_prepack")
    elif op == "aux":
        a = _aux_args(case)
        ws = h.model_aux_workspace_bytes(a["mode"], a.get("channels", 1), a.get("spatial", 1), a.get("groups", 1), 1)
        state = {"x": _Buf(made["x"]), "w": _Buf(made["w"]) if made["w"] is not None else None,
                 "b": _Buf(made["b"]) if made["b"] is not None else None, "args": a,
                 "y": _out(a["count"]), "ws": _empty(ws) if ws else None}
    else:
        state = _prepare_block(case, made)
    state["op"] = op
    torch.cuda.synchronize()
    return state


def _prepare_block(case, made):
    """The block's tensors in rpcmem buffers and the message of its nine requests."""
    t, d, heads, hd = case["image"] + case["text"], case["heads"] * 64, case["heads"], 64
    tiles = (t + 31) // 32
    buf = {name: _Rpc.of(v) for name, v in made.items() if torch.is_tensor(v)}
    for name in ("o", "up", "down"):
        buf[name] = _Rpc.of(made[name][0])
    for name, shape in (("h1", (t, d)), ("ao", (t, d)), ("x1", (t, d)), ("h2", (t, d)), ("u", (t, 4 * d)),
                        ("a", (t, 4 * d)), ("dn", (t, d)), ("out", (t, d))):
        buf[name] = _Rpc(shape)
    for name in ("q", "k", "v"):
        buf[name] = _Rpc((heads * tiles * hd * 32,), torch.float16)
    at = {name: (b.fd, 0) for name, b in buf.items()}

    def aux(out, x, w, b, **kw):
        a = dict(mode=10, count=t * d, width=d, channels=1, spatial=t, groups=1, batch=1, other_count=d, activation=0,
                 eps=1e-6)
        a.update(kw)
        return 19, h.aux_params(at[out], at[x], at[w] if w else (-1, 0), at[b] if b else (-1, 0), **a)

    def qkv_part(part, first):
        return (at["h1"][0], first * d * 4), at[part + "_w"], at[part + "_b"], at[part + "_qn"], at[part + "_kn"]

    def linear(out, x, w, k, n):
        return h.OP_MAT_MUL_NATIVE_W8A8, h.w8a8_params(at[out], at[x], at[w], t, k, n)

    requests = [
        aux("h1", "x", "scale1", "shift1", mode=9),
        (h.OP_QKV_MUL_RMS_PACKED_DUAL_ROPE,
         h.qkv_dual_rope_params(at["q"], at["k"], at["v"], qkv_part("image", 0), qkv_part("text", case["image"]),
                                at["pe"], case["image"], case["text"], d, heads, hd, 0, case["image"])),
        linear("ao", "attn", "o", d, d),
        aux("x1", "ao", "gate1", "x"),
        aux("h2", "x1", "scale2", "shift2", mode=9),
        linear("u", "h2", "up", d, 4 * d),
        aux("a", "u", None, None, mode=6, count=4 * t * d, width=4 * d, other_count=0),
        linear("dn", "a", "down", 4 * d, d),
        aux("out", "dn", "gate2", "x1"),
    ]
    msg, offsets = h.build_message([(h.REQUEST_TYPE_OP_COMPUTE, h.compute_request(op, raw)) for op, raw in requests],
                                   4096)
    raw = (ctypes.c_uint8 * len(msg)).from_buffer(msg)
    return {"buf": buf, "msg": msg, "raw": raw, "address": ctypes.addressof(raw), "offsets": offsets,
            "count": len(requests)}


def run(state):
    op = state["op"]
    if op == "w8a8":
        h.w8a8_linear(state["y"], state["x"], state["packed"], state["m"], state["k"], state["n"], state["ws"],
                      state["epilogue"])
        return state["y"].t
    if op == "mlp":
        m, d, f = state["m"], state["d"], state["f"]
        h.f16_gemm(state["h"], state["x"], state["w1"], state["b1"], m, d, f, f, state["mode"], workspace=state["ws"])
        h.f16_gemm(state["y"], state["h"], state["w2"], state["b2"], m, f, d, d, 0, workspace=state["ws"])
        return [state["h"].t, state["y"].t]
    if op == "conv":
        h.f16_gemm(state["y"], state["x"], state["w"], state["b"], state["m"], state["k"], state["c"], state["c"], 3,
                   workspace=state["ws"])
        return state["y"].t
    if op == "qk0":
        m, k, n = state["m"], state["k"], state["n"]
        if m <= 16:
            h.qk0_gemm(state["y"], state["x"], state["blocks"], m, k, n, state["type"], state["ws"])
        else:
            h.f16_gemm(state["y"], state["x"], state["image"], None, m, k, n, n, 0, workspace=state["ws"])
        return state["y"].t
    if op == "aux":
        h.model_aux(state["y"], state["x"], state["w"], state["b"], workspace=state["ws"], **state["args"])
        return state["y"].t
    if h.lib().htp_ops_execute_message(state["address"], len(state["msg"])) != 0:
        raise h.HtpOpsError("htp_ops_execute_message: invalid message")
    for i in range(state["count"]):
        rc = h.request_state(state["msg"], state["offsets"], i)
        if rc != 0:
            raise h.HtpOpsError("request %d returned %d: %s" % (i, rc, h.last_error()))
    return {name: state["buf"][name].t for name in ("q", "k", "v", "x1", "out")}


# ---- what a pass cannot do without ----------------------------------------------


def _w8a8_work(m, k, n):
    return 4 * m * k + k * n + 8 * n + 4 * k + 4 * m * n, 2 * m * k * n


def _f16_work(m, k, n, weight_bytes=None):
    return 4 * m * k + (2 * k * n if weight_bytes is None else weight_bytes) + 4 * n + 4 * m * n, 2 * m * k * n


def work(case):
    op = case["op"]
    if op == "w8a8":
        b, f = _w8a8_work(case["m"], case["k"], case["n"])
    elif op == "mlp":
        (b1, f1), (b2, f2) = _f16_work(case["m"], case["d"], case["f"]), _f16_work(case["m"], case["f"], case["d"])
        b, f = b1 + b2, f1 + f2
    elif op == "conv":
        b, f = _f16_work(case["m"], case["k"], case["c"])
    elif op == "qk0":
        k, n = case["k"], case["n"]
        bits = 272 if case["type"] == h.GGML_Q8_0 else 144
        b, f = _f16_work(case["m"], k, n, k * n // 256 * bits if case["m"] <= 16 else None)
    elif op == "aux":
        n, extra = case["rows"] * case["width"], {"swiglu": 2, "rope": 1}.get(case["what"], 1)
        b, f = 4 * n * (1 + extra) + (512 * case["rows"] if case["what"] == "rope" else 0), 10 * n
    else:
        t, d = case["image"] + case["text"], case["heads"] * 64
        parts = [_w8a8_work(t, d, d), _w8a8_work(t, d, 4 * d), _w8a8_work(t, 4 * d, d)]
        # two norms (read, write), the gates (two reads, one write), GELU, and Q/K/V with its fp16 outputs and rotations
        b = sum(p[0] for p in parts) + 4 * t * d * (4 + 6 + 8) + 4 * t * d + 12 * d * d + 6 * t * d + 512 * t
        f = sum(p[1] for p in parts) + 6 * t * d * d
    return {"bytes": b, "flops": f}


def tolerance(case):
    op = case["op"]
    if op == "w8a8":
        # whole-number sums, then two 32-bit products (and one 32-bit GELU): measured 6e-8 (3e-7)
        return {"rel": 2e-6, "max": 2e-5}
    if op == "aux":
        # 32-bit element-wise steps after sums in 64 bits: measured below 2e-7
        return {"rel": 2e-6, "max": 2e-5}
    if op == "block":
        # fp16 outputs and int8 steps that a last-bit change upstream can move
        return {"rel": 1.2e-3, "max": 0.05}
    # one rounding of each product to fp16: measured 2.5e-4 (once in 2^11, spread evenly)
    return {"rel": 1.0e-3, "max": 5e-3}


# ---- the same mathematics in 64 bits --------------------------------------------


def _gelu(v):
    return 0.5 * v * (1.0 + torch.tanh(0.7978845608028654 * (v + 0.044715 * v * v * v)))


def _w8a8_exact(x, tiles, sw, inv):
    """Quantized rows (32-bit steps, as opcode 15 defines them) times the whole-number weights, exactly."""
    n, k = sw.numel(), inv.numel()
    w = tiles.permute(0, 2, 4, 1, 3, 5).reshape(n, k).double()
    t = x.float() * inv
    s = torch.clamp(t.abs().amax(dim=1, keepdim=True) / 127.0, min=1e-12)
    q = torch.round(torch.clamp(t * (1.0 / s) + 128.0, 1.0, 255.0)) - 128.0
    return (q.double() @ w.t()) * sw.double() * s.double()


def _f16_weight(t):
    """[n][k] of a permuted fp16 weight."""
    nb, kb = t.shape[:2]
    return t.permute(0, 3, 1, 2, 4).reshape(nb * 32, kb * 32).double()


def _f16_exact(x, t, bias):
    y = x.half().double() @ _f16_weight(t).t()
    return y if bias is None else y + bias.double()


def _dequant(blocks, k, n, kind):
    """The permuted fp16 weight that quantized super-blocks stand for: value times scale, rounded once."""
    scale = blocks[:, :16].contiguous().view(torch.float16).float().repeat_interleave(32, dim=1)
    codes = blocks[:, 16:]
    if kind == h.GGML_Q8_0:
        value = codes.contiguous().view(torch.int8).float()
    else:
        even, odd = codes[:, 0::2], codes[:, 1::2]
        nib = torch.cat([even & 15, odd & 15, even >> 4, odd >> 4], dim=1).long()
        book = list(range(-8, 8)) if kind == h.GGML_Q4_0 else [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38,
                                                               53, 69, 89, 113]
        value = torch.tensor(book, dtype=torch.float32, device="cuda")[nib]
    return (value * scale).half().reshape(n // 32, k // 32, 16, 32, 2)


def _aux_exact(case, x, w, b):
    what, x = case["what"], x.double()
    w, b = (None if v is None else v.double() for v in (w, b))
    r, width = case["rows"], case["width"]
    if what == "group norm":
        gr = x.reshape(32, -1)
        y = ((gr - gr.mean(1, keepdim=True)) / torch.sqrt(gr.var(1, unbiased=False, keepdim=True) + 1e-6)).reshape(
            r, width) * w[:, None] + b[:, None]
        return torch.nn.functional.silu(y).reshape(-1)
    if what == "layer norm":
        return _norm_modulated(x, w, b).reshape(-1)
    if what == "rms norm":
        return (x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6) * w).reshape(-1)
    if what == "swiglu":
        return (torch.nn.functional.silu(x[:, :width]) * x[:, width:]).reshape(-1)
    if what == "gelu":
        return _gelu(x).reshape(-1)
    if what == "transpose":
        return x.t().reshape(-1)
    return _rotate(x.reshape(r, width // 64, 64), w).permute(1, 0, 2).reshape(-1)


def _norm_modulated(x, w, b):
    y = (x - x.mean(1, keepdim=True)) / torch.sqrt(x.var(1, unbiased=False, keepdim=True) + 1e-6)
    return y + y * w + b


def _rotate(x, pe):
    """[token][head][width] times the 2x2 matrices of its token."""
    m = pe.double()[:, None, :, :]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * m[..., 0] + x1 * m[..., 1], x0 * m[..., 2] + x1 * m[..., 3]], -1).flatten(-2)


def _block_exact(case, p):
    t, heads, hd, a = case["image"] + case["text"], case["heads"], 64, case["image"]
    d, tiles = heads * hd, (t + 31) // 32
    x = p["x"].double()
    h1 = _norm_modulated(x, p["scale1"].double(), p["shift1"].double()).float()
    raw = {"q": [], "k": [], "v": []}
    for part, rows, pe in (("image", h1[:a], p["pe"][:a]), ("text", h1[a:], p["pe"][a:])):
        y = _f16_exact(rows, p[part + "_w"], p[part + "_b"]).reshape(-1, 3, heads, hd)
        for i, name in enumerate(("q", "k")):
            v = y[:, i]
            v = v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-6) * p["%s_%sn" % (part, name)].double()
            raw[name].append(_rotate(v, pe))
        raw["v"].append(y[:, 2])
    out = {}
    for name, parts in raw.items():  # the packed tile orders of the attention kernels that read them
        v = torch.zeros(tiles * 32, heads, hd, dtype=torch.float64, device="cuda")
        v[:t] = torch.cat(parts)
        if name == "k":
            v = v.reshape(tiles, 32, heads, hd // 64, 32, 2).permute(2, 0, 3, 4, 1, 5)
        else:
            v = v.reshape(tiles, 16, 2, heads, hd // 32, 32)
            v = v.permute(3, 0, 4, 1, 5, 2) if name == "q" else v.permute(3, 4, 0, 1, 5, 2)
        out[name] = v.reshape(-1)
    x1 = _w8a8_exact(p["attn"], *p["o"][1:]) * p["gate1"].double() + x
    h2 = _norm_modulated(x1, p["scale2"].double(), p["shift2"].double()).float()
    act = _gelu(_w8a8_exact(h2, *p["up"][1:])).float()
    out["x1"], out["out"] = x1, _w8a8_exact(act, *p["down"][1:]) * p["gate2"].double() + x1
    return out


def exact(case, seed):
    p, op = _inputs(case, seed), case["op"]
    if op == "w8a8":
        y = _w8a8_exact(p["x"], p["tiles"], p["sw"], p["inv"])
        return _gelu(y) if case["gelu"] else y
    if op == "mlp":
        v = _f16_exact(p["x"], p["w1"], p["b1"])
        v = _gelu(v) if case["mode"] == 1 else v * torch.sigmoid(1.702 * v)
        return [v, _f16_exact(v.float(), p["w2"], p["b2"])]
    if op == "conv":
        return _f16_exact(p["x"], p["w"], p["b"]).t().contiguous()
    if op == "qk0":
        return _f16_exact(p["x"], _dequant(p["blocks"], case["k"], case["n"], case["type"]), None)
    if op == "aux":
        return _aux_exact(case, p["x"], p["w"], p["b"])
    return _block_exact(case, p)
