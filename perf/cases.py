"""What the framework is timed on: the image encoder's blocks and whole
trunk, the text path's attention, the point-prompt decoder, its mask
postprocessing and the linear layer under them all, each through the entry
point that a program calls (the ctypes mirror of include/sam3_hip.h).

One pass is one call on device buffers that the program already holds, as the
C API is used: weights uploaded once, work buffers and graphs made once,
activations resident. Weights are random (Xavier-uniform matrices, PyTorch's
default biases, LayerNorm affine near (1, 0)), activations N(0, 1), images
(u - 0.5) / 0.5 of U(0, 1), prompts uniform points of the image.

The three precisions are the library's options: fp32 (the default), fp16
(weight matrices stored as half, float arithmetic) and bf16 (bf16 MFMA).
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _load_hip():
    if "sam3_hip" in sys.modules:
        return sys.modules["sam3_hip"]
    spec = importlib.util.spec_from_file_location(
        "sam3_hip", os.path.join(_ROOT, "i.sam3.opencl_amd", "sam3_hip.py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules["sam3_hip"] = mod
    spec.loader.exec_module(mod)
    mod.lib()
    return mod


hip = _load_hip()
DEV = "cuda:0"
PATCH = 14   # image pixels per token side
HD = 64      # ViT head width
_backends = {}


def backend(precision):
    """The program's one backend of this precision (hipb_init)."""
    if precision not in _backends:
        _backends[precision] = hip.Backend(precision=precision)
    return _backends[precision]


class _Device:
    """Device memory of a library buffer for torch (CUDA array interface).
    A tensor made of it holds `owner`, the state that frees the buffer."""

    def __init__(self, owner, mem, shape, typestr):
        if math.prod(shape) * int(typestr[2:]) > mem.contents.bytes:
            raise ValueError("the buffer is smaller than %s" % (shape,))
        self.owner = owner
        self.__cuda_array_interface__ = {
            "shape": tuple(shape), "typestr": typestr, "strides": None,
            "data": (mem.contents.ptr, False), "version": 2}


_TORCH = {hip.F32: ("<f4", None), hip.F16: ("<f2", None),
          hip.BF16: ("<i2", torch.bfloat16)}


def view(owner, mem, *shape):
    """The buffer as a torch tensor of its element type (no copy)."""
    typestr, dt = _TORCH[mem.contents.dtype]
    t = torch.as_tensor(_Device(owner, mem, shape, typestr), device=DEV)
    return t if dt is None else t.view(dt)


def bytes_view(owner, mem, *shape):
    return torch.as_tensor(_Device(owner, mem, shape, "|u1"), device=DEV)


class State:
    """The buffers and handles of one case; released with it."""

    def __init__(self, precision):
        self.be = backend(precision)
        self.mems = []
        self.model = self.dec = None
        self.blocks = []

    def dev(self, t):
        """A float buffer holding t."""
        m = self.be.alloc(4 * t.numel())
        self.mems.append(m)
        view(self, m, *t.shape).copy_(t)
        return m

    def weight(self, t):
        """t as hipb_upload_weight stores it: half, bf16 or float."""
        dt = hip.F16 if self.be.fp16w else hip.BF16 if self.be.bf16 else hip.F32
        m = self.be.alloc_typed(t.numel(), dt)
        self.mems.append(m)
        view(self, m, *t.shape).copy_(t)
        return m

    def empty(self, n):
        m = self.be.alloc(4 * n)
        self.mems.append(m)
        return m

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.dec is not None:
                self.dec.free()
            if self.model is not None:
                self.model.free()
            for m in self.mems:
                self.be.release(m)
        except Exception:  # the interpreter's own end
            pass


# ------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _uniform(g, bound, *shape):
    return (2 * torch.rand(*shape, generator=g, device=DEV) - 1) * bound


def _block_weights(g, E, mlp):
    def xavier(o, i):
        return _uniform(g, math.sqrt(6.0 / (i + o)), o, i)

    def norm():
        return 1 + 0.1 * _normal(g, E), 0.1 * _normal(g, E)

    w = {}
    w["n1w"], w["n1b"] = norm()
    w["qkvw"], w["qkvb"] = xavier(3 * E, E), _uniform(g, E ** -0.5, 3 * E)
    w["projw"], w["projb"] = xavier(E, E), _uniform(g, E ** -0.5, E)
    w["n2w"], w["n2b"] = norm()
    w["l1w"], w["l1b"] = xavier(mlp, E), _uniform(g, E ** -0.5, mlp)
    w["l2w"], w["l2b"] = xavier(E, mlp), _uniform(g, mlp ** -0.5, E)
    return w


_MATRICES = ("qkvw", "projw", "l1w", "l2w")


def _rope_table(side):
    """Axial 2D RoPE, (cos, sin) per position and pair [side^2, 32, 2]."""
    f = 10000.0 ** (-4.0 * torch.arange(HD // 4, dtype=torch.float64) / HD)
    p = torch.arange(side * side)
    ang = torch.cat([(p % side).double()[:, None] * f,
                     (p // side).double()[:, None] * f], 1)
    return torch.stack([ang.cos(), ang.sin()], -1).float().to(DEV)


def _windows(c):
    """Window side of each trunk block: every eighth one global (blocks 7,
    15, 23, 31 of 32), and the last."""
    n = c["depth"]
    return [0 if (i + 1) % 8 == 0 or i == n - 1 else c["window"]
            for i in range(n)]


def _trunk_inputs(c, seed):
    g = _gen(seed)
    E, grid = 64 * c["heads"], c["grid"]
    img = (torch.rand(3, grid * PATCH, grid * PATCH, generator=g,
                      device=DEV) - 0.5) / 0.5
    pe_w = _uniform(g, math.sqrt(6.0 / (3 * PATCH ** 2 + E)), E, 3 * PATCH ** 2)
    pos = 0.02 * _normal(g, grid * grid, E)
    lnpw, lnpb = 1 + 0.1 * _normal(g, E), 0.1 * _normal(g, E)
    return img, pe_w, pos, lnpw, lnpb, g


def _attend_inputs(c, seed):
    g = _gen(seed)
    D = c["heads"] * c["hd"]
    q, k, v = (_normal(g, c["nq"], D), _normal(g, c["nk"], D),
               _normal(g, c["nk"], D))
    if not c["box"]:
        return q, k, v, None, None
    h, w = c["nk"] // c["box"], c["box"]
    return (q, k, v, 2 * _normal(g, c["nq"], h, c["heads"]),
            2 * _normal(g, c["nq"], w, c["heads"]))


def _linear_inputs(c, seed):
    g = _gen(seed)
    x = _normal(g, c["rows"], c["nin"])
    w = _uniform(g, math.sqrt(6.0 / (c["nin"] + c["nout"])), c["nout"], c["nin"])
    return x, w, _uniform(g, c["nin"] ** -0.5, c["nout"])


def _decode_inputs(c, seed):
    r = np.random.default_rng(seed)
    g = _gen(seed)
    T = c["grid"] ** 2
    pts = r.uniform(0, c["grid"] * PATCH, (c["prompts"], 2)).astype(np.float32)
    return (pts, _normal(g, T, 256), _normal(g, 16 * T, 32),
            _normal(g, 4 * T, 64), hip.random_decoder_weights(seed))


# -------------------------------------------------------------- cases

def listed():
    return [
        # One 1008 x 1008 image through the whole 32-block encoder: what
        # every image, crop or tile costs first; the captured graph, as a
        # program that encodes many images keeps it.
        {"name": "trunk_bf16", "kind": "trunk", "precision": "bf16",
         "grid": 72, "heads": 16, "window": 24, "depth": 32},
        # The encoder's common layer (28 of 32) at the same image size.
        {"name": "block_window_bf16", "kind": "block", "precision": "bf16",
         "grid": 72, "heads": 16, "window": 24},
        # The default precision, the layer with the longest sequence.
        {"name": "block_global_fp32", "kind": "block", "precision": "fp32",
         "grid": 72, "heads": 16, "window": 0},
        # Half weights, a smaller image (700 pixels) whose grid the windows
        # do not divide (padded windows).
        {"name": "block_window_fp16_50", "kind": "block", "precision": "fp16",
         "grid": 50, "heads": 16, "window": 24},
        # Fusion encoder self-attention over the image tokens.
        {"name": "attend_fusion_bf16", "kind": "attend", "precision": "bf16",
         "nq": 5184, "nk": 5184, "heads": 8, "hd": 32, "causal": False, "box": 0},
        # Detection decoder: presence + 200 queries over the image, with
        # the box relative position bias, at the default precision.
        {"name": "attend_box_fp32", "kind": "attend", "precision": "fp32",
         "nq": 201, "nk": 5184, "heads": 8, "hd": 32, "causal": False, "box": 72},
        # Text encoder attention of one prompt: the smallest call.
        {"name": "attend_text_fp32", "kind": "attend", "precision": "fp32",
         "nq": 32, "nk": 32, "heads": 16, "hd": 64, "causal": True, "box": 0},
        # The text encoder's MLP layer around it.
        {"name": "linear_text_fp32", "kind": "linear", "precision": "fp32",
         "rows": 32, "nin": 1024, "nout": 4096, "act": 1, "residual": False},
        # Automatic mask generation: a batch of 64 point prompts.
        {"name": "decode_64_bf16", "kind": "decode", "precision": "bf16",
         "grid": 72, "prompts": 64, "graph": True},
        # One click on an image, interactive: latency.
        {"name": "decode_1_fp32", "kind": "decode", "precision": "fp32",
         "grid": 72, "prompts": 1, "graph": False},
        # The batch at the default precision.
        {"name": "decode_32_fp32", "kind": "decode", "precision": "fp32",
         "grid": 72, "prompts": 32, "graph": False},
        # The batch's best masks at the size of a photograph, with their
        # statistics.
        {"name": "masks_64", "kind": "masks", "precision": "bf16",
         "grid": 72, "planes": 64, "out_h": 1080, "out_w": 1440},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block"] * 5 + ["attend"] * 4 + ["decode"] * 4 +
                      ["linear"] * 3 + ["trunk", "masks"])
    prec = rng.choice(["fp32", "fp16", "bf16"])
    c = {"kind": kind, "precision": prec}
    if kind == "trunk":
        c.update(grid=rng.randint(24, 72), heads=rng.choice([12, 16]),
                 window=rng.choice([14, 16, 24]),
                 depth=rng.randint(2, 6) if prec == "bf16" else rng.randint(1, 2))
    elif kind == "block":
        c.update(grid=rng.randint(20, 72), heads=rng.choice([8, 12, 16, 16]),
                 window=rng.choice([0, 0, 14, 16, 24, 24]))
        if c["window"] > c["grid"]:
            c["window"] = 0
    elif kind == "attend":
        hd = rng.choice([32, 64])
        form = rng.choice(["self", "cross", "box", "causal"])
        heads = rng.choice([8, 12, 16]) if hd == 64 else 8
        nk = _log(rng, 32, 5184)
        nq = nk if form in ("self", "causal") else _log(rng, 8, 600)
        box = 0
        if form == "causal":
            nq = nk = _log(rng, 8, 600)
        if form == "box":
            box = rng.randint(24, 80)
            nk = box * rng.randint(24, 64)
        c.update(nq=nq, nk=nk, heads=heads, hd=hd, causal=form == "causal", box=box)
    elif kind == "decode":
        c.update(grid=rng.randint(24, 72), prompts=_log(rng, 1, 64),
                 graph=rng.random() < 0.5)
    elif kind == "linear":
        c.update(rows=_log(rng, 1, 6000), nin=64 * _log(rng, 2, 64),
                 nout=rng.choice([64 * _log(rng, 2, 64), _log(rng, 50, 4100)]),
                 act=rng.choice([0, 1, 2]), residual=rng.random() < 0.3)
    else:
        c.update(grid=rng.randint(24, 72), planes=_log(rng, 1, 96),
                 out_h=rng.randint(300, 1200), out_w=rng.randint(300, 1500))
    return c


# ------------------------------------------------------------ prepare

def _make_blocks(s, c, g, windows):
    E = HD * c["heads"]
    for ws in windows:
        w = _block_weights(g, E, 4 * E)
        blk = hip.VitBlock()
        for k, t in w.items():
            setattr(blk, k, s.weight(t) if k in _MATRICES else s.dev(t))
        blk.window = ws
        s.blocks.append(blk)
    s.model = hip.Model(s.be, grid=c["grid"], embed=E, heads=c["heads"],
                        blocks=s.blocks, mlp=4 * E)
    if any(windows):
        s.model.m.rope_win = s.dev(_rope_table(max(windows)))
    s.model.m.rope_glob = s.dev(_rope_table(c["grid"]))


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = State(c["precision"])
    s.case = c
    if kind == "trunk":
        img, pe_w, pos, lnpw, lnpb, g = _trunk_inputs(c, seed)
        _make_blocks(s, c, g, _windows(c))
        m = s.model.m
        m.patch = PATCH
        m.pe_w = s.weight(pe_w)
        m.pos, m.lnpw, m.lnpb = s.dev(pos), s.dev(lnpw), s.dev(lnpb)
        s.img = img.cpu().numpy()
        torch.cuda.synchronize()
        hip.sam_encode_trunk(s.model, s.img)
        hip.sam_trunk_graph(s.model, True)
    elif kind == "block":
        g = _gen(seed)
        x = _normal(g, c["grid"] ** 2, HD * c["heads"])
        _make_blocks(s, c, g, [c["window"]])
        s.x = s.dev(x)
    elif kind == "attend":
        q, k, v, dy, dx = _attend_inputs(c, seed)
        s.model = hip.Model(s.be, embed=c["heads"] * c["hd"], heads=c["heads"],
                            hd=c["hd"])
        s.q, s.k, s.v = s.dev(q), s.dev(k), s.dev(v)
        s.o = s.empty(q.numel())
        s.dy = s.dev(dy) if dy is not None else None
        s.dx = s.dev(dx) if dx is not None else None
    elif kind == "linear":
        x, w, b = _linear_inputs(c, seed)
        s.model = hip.Model(s.be, embed=1024, heads=16)
        s.x, s.w, s.b = s.dev(x), s.weight(w), s.dev(b)
        s.y = s.empty(c["rows"] * c["nout"])
        if c["residual"]:
            s.r = s.dev(_normal(_gen(seed + 1), c["rows"], c["nout"]))
    elif kind == "decode":
        pts, emb, s0, s1, w = _decode_inputs(c, seed)
        s.model = hip.Model(s.be, embed=1024, heads=16)
        s.model.m.grid = c["grid"]
        s.dec = hip.Decoder(s.model, w, c["prompts"], img=c["grid"] * PATCH)
        s.dec.set_image(emb.cpu().numpy(), s0.cpu().numpy(), s1.cpu().numpy())
        s.pts = pts
        if c["graph"]:
            s.dec.graph(c["prompts"])
    else:
        g = _gen(seed)
        n, L = c["planes"], 4 * c["grid"]
        s.model = hip.Model(s.be, embed=1024, heads=16)
        s.model.m.grid = c["grid"]
        s.dec = hip.Decoder(s.model, hip.random_decoder_weights(seed),
                            -(-n // 3), img=c["grid"] * PATCH)
        # Logits of a blob per mask: positive inside, negative outside,
        # smooth, with a little texture.
        low = _normal(g, 1, n, 9, 9)
        low = torch.nn.functional.interpolate(low, size=(L, L), mode="bicubic")
        low = 8 * low[0] + 0.5 * _normal(g, n, L, L) - 2
        view(s, s.dec.buf("lowres"), -(-n // 3) * 3, L, L)[:n].copy_(low)
        s.sel = np.arange(n, dtype=np.int32)
    torch.cuda.synchronize()
    return s


def run(s):
    c, kind = s.case, s.case["kind"]
    if kind == "trunk":
        hip.sam_encode_trunk(s.model, s.img)
        return view(s, s.model.m.x, c["grid"] ** 2, HD * c["heads"])
    if kind == "block":
        # The tokens of the block before, then the block in place.
        n = c["grid"] ** 2 * HD * c["heads"]
        s.be.copy(s.x, s.model.m.x, 0, 0, 4 * n)
        hip.vit_block(s.model, s.blocks[0])
        return view(s, s.model.m.x, c["grid"] ** 2, HD * c["heads"])
    if kind == "attend":
        D = c["heads"] * c["hd"]
        hip.attend(s.model, c["nq"], c["nk"], c["heads"], c["hd"], s.q, D, s.k,
                   D, s.v, D, s.o, D, causal=c["causal"], dy=s.dy, dx=s.dx,
                   W=c["box"])
        return view(s, s.o, c["nq"], D)
    if kind == "linear":
        if c["residual"]:
            s.be.copy(s.r, s.y, 0, 0, 4 * c["rows"] * c["nout"])
        hip.linear(s.model, c["rows"], c["nin"], c["nout"], s.x, 0, s.w, s.b,
                   s.y, 0, c["act"], int(c["residual"]))
        return view(s, s.y, c["rows"], c["nout"])
    if kind == "decode":
        iou = s.dec.decode(s.pts)
        return {"iou": iou, "lowres": view(s, s.dec.buf("lowres"), c["prompts"], 3,
                                           4 * c["grid"], 4 * c["grid"])}
    stats = s.dec.postprocess(s.sel, c["out_h"], c["out_w"], 1.0, False)
    return {"stats": stats, "masks": bytes_view(s, s.dec.buf("mask"), c["planes"],
                                                c["out_h"], c["out_w"])}


# --------------------------------------------------------------- work

def _wbytes(c):
    return 4 if c["precision"] == "fp32" else 2


def _block_work(c, window):
    E, T = HD * c["heads"], c["grid"] ** 2
    side = window or c["grid"]
    n = (-(-c["grid"] // side)) ** 2
    rows, N = n * side * side, side * side
    flops = (2.0 * rows * E * 4 * E + 16.0 * T * E * E +
             4.0 * n * c["heads"] * N * N * HD)
    return {"bytes": 2 * 4.0 * T * E + _wbytes(c) * 12.0 * E * E + 4.0 * 13 * E,
            "flops": flops}


def work(case):
    c, kind = case, case["kind"]
    if kind == "block":
        return _block_work(c, c["window"])
    if kind == "trunk":
        E, T = HD * c["heads"], c["grid"] ** 2
        K = 3 * PATCH ** 2
        b = [_block_work(c, w) for w in _windows(c)]
        weights = sum(w["bytes"] - 8.0 * T * E for w in b)
        return {"bytes": 4.0 * T * (K + 2 * E) + _wbytes(c) * K * E + weights,
                "flops": 2.0 * T * K * E + sum(w["flops"] for w in b)}
    if kind == "attend":
        D = c["heads"] * c["hd"]
        pairs = c["nq"] * c["nk"]
        if c["causal"]:
            pairs = c["nq"] * (c["nk"] + 1) / 2.0
        bias = c["nq"] * c["heads"] * (c["box"] + c["nk"] // c["box"]) if c["box"] else 0
        return {"bytes": 4.0 * (2 * c["nq"] * D + 2 * c["nk"] * D + bias),
                "flops": 4.0 * pairs * D}
    if kind == "linear":
        r, i, o = c["rows"], c["nin"], c["nout"]
        return {"bytes": 4.0 * (r * i + r * o * (2 if c["residual"] else 1) + o) +
                _wbytes(c) * i * o, "flops": 2.0 * r * i * o}
    if kind == "decode":
        P, T = c["prompts"], c["grid"] ** 2
        # Per prompt and image token: the five 256 <-> 128 projections of the
        # per-prompt keys, the output projection of layer 0, the upscaling's
        # two products and the logits; the tokens' own layers beside them.
        per_token = (2.0 * 256 * 128 * 7 + 4.0 * 8 * 128 * 5 +
                     2.0 * 256 * 256 + 2.0 * 4 * 64 * 128 + 2.0 * 16 * 96)
        tokens = 8 * 2.0 * (8 * 256 * 256 + 9 * 256 * 128 + 4 * 256 * 2048)
        return {"bytes": 4.0 * T * (2 * 256 + 16 * 32 + 4 * 64 + 3 * 128) +
                4.0 * P * 48 * T + _wbytes(c) * 4.1e6,
                "flops": P * (T * per_token + tokens)}
    n, L = c["planes"], 4 * c["grid"]
    return {"bytes": 4.0 * n * L * L + n * c["out_h"] * c["out_w"],
            "flops": 10.0 * n * c["out_h"] * c["out_w"]}


def tolerance(case):
    """About four times the distance of a pass from exact() as measured:
    on the bf16 path, whose operands carry 8 bits, 1.1e-3 through a block and
    2.8e-3 to 3.5e-3 through an attention, a decode or the trunk; on the
    float paths, which sum in 32 bits, 2e-7 to 7e-7 (1.5e-6 at the longest
    sums)."""
    if case["kind"] == "masks":
        return "exact"
    if case["precision"] == "bf16":
        return {"rel": 0.005 if case["kind"] == "block" else 0.014}
    return {"rel": 6e-6}


# -------------------------------------------------------------- exact

def _stored(t, c):
    """A weight matrix as the backend stores it, in 64 bits."""
    if c["precision"] == "fp16":
        t = t.half()
    elif c["precision"] == "bf16":
        t = t.bfloat16()
    return t.double()


def _ln(x, w, b, eps=1e-5):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + eps) * w.double() + b.double()


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


def _rope(x, table):
    """Rotate the pairs (2 k, 2 k + 1) of x [..., N, 64]."""
    a, b = x[..., 0::2], x[..., 1::2]
    cos, sin = table[..., 0].double(), table[..., 1].double()
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _sdpa(q, k, v, scale, mask=None):
    """One unit at a time: softmax(q k^T scale + mask) v in 64 bits."""
    out = []
    for u in range(q.shape[0]):
        sc = (q[u] * scale) @ k[u].t().contiguous()
        if mask is not None:
            sc = sc + mask(u)
        out.append(torch.softmax(sc, -1) @ v[u])
    return torch.stack(out)


def _exact_block(x, c, w, window):
    E, G, H = HD * c["heads"], c["grid"], c["heads"]
    y = _ln(x, w["n1w"], w["n1b"])
    side = window or G
    nw = -(-G // side)
    pad = torch.zeros(nw * side, nw * side, E, dtype=torch.float64, device=DEV)
    pad[:G, :G] = y.view(G, G, E)
    y = pad.view(nw, side, nw, side, E).transpose(1, 2).reshape(-1, side * side, E)
    qkv = y @ _stored(w["qkvw"], c).t().contiguous() + w["qkvb"].double()
    qkv = qkv.view(nw * nw, side * side, 3, H, HD).permute(2, 0, 3, 1, 4)
    table = _rope_table(side)
    q, k, v = (t.reshape(-1, side * side, HD).contiguous() for t in qkv)
    o = _sdpa(_rope(q, table), _rope(k, table), v, HD ** -0.5)
    o = o.view(nw, nw, H, side, side, HD).permute(0, 3, 1, 4, 2, 5)
    o = o.reshape(nw * side, nw * side, E)[:G, :G].reshape(G * G, E)
    x = x + o @ _stored(w["projw"], c).t().contiguous() + w["projb"].double()
    h = _ln(x, w["n2w"], w["n2b"]) @ _stored(w["l1w"], c).t().contiguous()
    h = _gelu(h + w["l1b"].double())
    return x + h @ _stored(w["l2w"], c).t().contiguous() + w["l2b"].double()


def _exact_decode(c, seed):
    pts, emb, s0, s1, w = _decode_inputs(c, seed)
    f = {}
    for k, a in w.items():
        t = torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
        matrix = k.endswith("w") and a.ndim == 2
        f[k] = _stored(t, c) if matrix else t.double()
    G, T = c["grid"], c["grid"] ** 2
    side = float(c["grid"] * PATCH)

    def pe(xy):
        a = 2 * math.pi * ((2 * xy - 1) @ f["gauss"])
        return torch.cat([a.sin(), a.cos()], -1)

    ax = (torch.arange(G, dtype=torch.float64, device=DEV) + 0.5) / G
    grid_xy = torch.stack([ax.repeat(G), ax.repeat_interleave(G)], -1)
    kpe = pe(grid_xy)
    src = emb.double() + f["no_mask"]

    def lin(x, p):
        return x @ f[p + "w"].t().contiguous() + f[p + "b"]

    def att(p, q, k, v):
        q, k, v = lin(q, p + "q"), lin(k, p + "k"), lin(v, p + "v")
        B, D = q.shape[0], q.shape[-1]

        def split(t):
            return t.reshape(B, -1, 8, D // 8).transpose(1, 2).contiguous()

        sc = split(q) @ split(k).transpose(-1, -2).contiguous() / math.sqrt(D // 8)
        o = torch.softmax(sc, -1) @ split(v)
        return lin(o.transpose(1, 2).reshape(B, -1, D), p + "o")

    def ln(x, p, eps=1e-5):
        return _ln(x, f[p + "w"], f[p + "b"], eps)

    def mlp(x, p, n=3):
        for j in range(n):
            x = lin(x, "%s%d" % (p, j))
            if j < n - 1:
                x = x.clamp(min=0)
        return x

    def convt(x, wt, b, n, co):
        t = (x @ wt).view(-1, n, n, co, 2, 2).permute(0, 1, 4, 2, 5, 3)
        return t.reshape(-1, 2 * n, 2 * n, co) + b

    ious, lows = [], []
    for p0 in range(0, c["prompts"], 8):
        xy = torch.from_numpy(pts[p0:p0 + 8]).double().to(DEV)
        P = xy.shape[0]
        tok = torch.zeros(P, 8, 256, dtype=torch.float64, device=DEV)
        tok[:, 0], tok[:, 1] = f["obj_token"], f["iou_token"]
        tok[:, 2:6] = f["mask_tokens"]
        tok[:, 6] = pe((xy + 0.5) / side) + f["point_emb"][1]
        tok[:, 7] = f["not_a_point"]
        qs, keys = tok.clone(), src.expand(P, T, 256).contiguous()
        for layer in range(2):
            p = "layers.%d." % layer
            if layer == 0:
                qs = att(p + "self.", qs, qs, qs)
            else:
                qs = qs + att(p + "self.", qs + tok, qs + tok, qs)
            qs = ln(qs, p + "n1")
            qs = ln(qs + att(p + "t2i.", qs + tok, keys + kpe, keys), p + "n2")
            h = lin(qs, p + "m1").clamp(min=0)
            qs = ln(qs + lin(h, p + "m2"), p + "n3")
            keys = ln(keys + att(p + "i2t.", keys + kpe, qs + tok, qs), p + "n4")
        qs = ln(qs + att("final_t2i.", qs + tok, keys + kpe, keys), "nf")
        u = convt(keys, f["up0w"], f["up0b"], G, 64)
        u = _gelu(ln(u + s1.double().view(2 * G, 2 * G, 64), "up1", 1e-6))
        u = convt(u.reshape(P, -1, 64), f["up3w"], f["up3b"], 2 * G, 32)
        u = _gelu(u + s0.double().view(4 * G, 4 * G, 32)).reshape(P, -1, 32)
        hyper = torch.stack([mlp(qs[:, 2 + i], "hyper.%d." % i) for i in (1, 2, 3)], 1)
        lows.append((hyper @ u.transpose(1, 2).contiguous()).reshape(P, 3, 4 * G, 4 * G))
        ious.append(torch.sigmoid(mlp(qs[:, 1], "iou.")[:, 1:]))
    return {"iou": torch.cat(ious), "lowres": torch.cat(lows)}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "masks":
        return None  # bits and whole numbers
    if kind == "trunk":
        img, pe_w, pos, lnpw, lnpb, g = _trunk_inputs(c, seed)
        G = c["grid"]
        cols = img.double().view(3, G, PATCH, G, PATCH).permute(1, 3, 0, 2, 4)
        x = cols.reshape(G * G, -1) @ _stored(pe_w, c).t().contiguous()
        x = _ln(x + pos.double(), lnpw, lnpb)
        for ws in _windows(c):
            E = HD * c["heads"]
            x = _exact_block(x, c, _block_weights(g, E, 4 * E), ws)
        return x
    if kind == "block":
        g = _gen(seed)
        x = _normal(g, c["grid"] ** 2, HD * c["heads"]).double()
        E = HD * c["heads"]
        return _exact_block(x, c, _block_weights(g, E, 4 * E), c["window"])
    if kind == "attend":
        q, k, v, dy, dx = _attend_inputs(c, seed)
        H, hd = c["heads"], c["hd"]

        def heads(t):
            return t.double().view(-1, H, hd).transpose(0, 1).contiguous()

        mask = None
        if c["causal"]:
            ninf = torch.full((c["nq"], c["nk"]), -math.inf, dtype=torch.float64,
                              device=DEV).triu(1)
            mask = lambda u: ninf  # noqa: E731
        elif dy is not None:
            def mask(u):
                b = dy[:, :, u].double()[:, :, None] + dx[:, :, u].double()[:, None]
                return b.reshape(c["nq"], c["nk"])
        o = _sdpa(heads(q), heads(k), heads(v), hd ** -0.5, mask)
        return o.transpose(0, 1).reshape(c["nq"], H * hd)
    if kind == "linear":
        x, w, b = _linear_inputs(c, seed)
        y = x.double() @ _stored(w, c).t().contiguous() + b.double()
        y = _gelu(y) if c["act"] == 1 else y.clamp(min=0) if c["act"] == 2 else y
        if c["residual"]:
            y = y + _normal(_gen(seed + 1), c["rows"], c["nout"]).double()
        return y
    return _exact_decode(c, seed)
