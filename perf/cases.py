"""Workloads of the Depth-Anything-3 token path, for timing and comparison.

Each case is one pass of work that a depth program hands to the library:
single layers (attention, the MLP, the QKV projection, the patch embedding,
the per-token operations), one whole block, and one whole frame.  Sizes are
the ViT-B / ViT-L shapes of the benchmark (a 504x336 image: a 24 x 36 patch
grid, 866 tokens; twelve such views: 10,392 rows; 1008x672: 3,458 tokens);
`draw` spreads over the grids, view counts, widths and parameter types
around them.

One runtime serves every state, as in a program; inputs are torch tensors on
the GPU, wrapped without a copy.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "vestra-engine_amd"))
import vestra_hip as vh  # noqa: E402

HD = 64
PATCH = 14
MEAN, STD = (0.485, 0.456, 0.406), (0.229, 0.224, 0.225)
LN_EPS, QK_EPS, HEAD_EPS, FREQ = 1e-6, 1e-5, 1e-5, 100.0
N_SPECIAL = 2  # class token and one register
DEPTH, ALT_START, OUT_LAYERS = 12, 4, (2, 5, 8, 11)
# widths: embedding, heads, MLP
WIDTH = {"B": (768, 12, 3072), "L": (1024, 16, 4096)}

# Largest relative difference (2-norm) of another correct float32
# implementation: about four times what the library's float32 sums are off
# the 64-bit values (attention 0.8-1.4e-6, the MLP 6e-7, the QKV projection
# and the patch embedding 3-4e-7, the per-token operations 4e-8-1.1e-7; a
# block and a frame carry the residual stream, which dilutes their layers').
REL = {"head": 5e-7, "ops": 5e-7, "patch": 1.5e-6, "qkv": 1.5e-6, "mlp": 2.5e-6,
       "attention": 6e-6, "block": 5e-7, "frame": 2.5e-6}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a camera frame resized to the model's input (once per frame; bytes out)
        dict(name="preprocess_frame", kind="preprocess", h=427, w=640, size=504),
        # one image to tokens: the first launch of every single-frame pass
        dict(name="patch_image", kind="patch", gh=24, gw=36, views=1, width="B"),
        # the views of a multi-view batch to tokens in one call
        dict(name="patch_views", kind="patch", gh=24, gw=36, views=12, width="B"),
        # a captured feature map handed to the depth head: LayerNorm, then channel-major
        dict(name="head_image", kind="head", tokens=864, channels=1536),
        # one block's per-token operations for one image: launches count
        dict(name="ops_image", kind="ops", gh=24, gw=36, views=1, width="B", f16=False, glob=False,
             sequential=False),
        # the same over a twelve-view global layer: the benchmark's own step
        dict(name="ops_views", kind="ops", gh=24, gw=36, views=12, width="B", f16=False, glob=True,
             sequential=False),
        # the QKV projection with Q/K-norm and RoPE for one image (few rows)
        dict(name="qkv_image", kind="qkv", gh=24, gw=36, views=1, width="B", f16=False, glob=False),
        # FC1 + GELU, FC2 + LayerScale + residual over twelve views (many rows)
        dict(name="mlp_views", kind="mlp", rows=10392, width="B", f16=False),
        # attention of one image (few query tiles)
        dict(name="attention_image", kind="attention", seqs=12, n=866),
        # a global layer's attention: every view's tokens attend to all others
        dict(name="attention_views", kind="attention", seqs=12, n=10392),
        # one ViT-L block of a 1008x672 image, weights stored as F16
        dict(name="block_large", kind="block", gh=48, gw=72, views=1, width="L", f16=True,
             glob=False),
        # a whole frame: image to tokens, twelve blocks, four captures
        dict(name="frame_image", kind="frame", gh=24, gw=36, views=1, width="B"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["preprocess", "patch", "patch", "head", "ops", "ops", "qkv", "qkv", "mlp",
                       "mlp", "attention", "attention", "attention", "block", "block", "frame"])
    width = rng.choice("BBL")
    f16 = rng.random() < 0.4
    gh, gw = _log_int(rng, 6, 48), _log_int(rng, 6, 72)
    views = 1 if rng.random() < 0.4 else _log_int(rng, 2, 12)
    glob = views > 1 and rng.random() < 0.5
    if kind == "preprocess":
        return dict(kind=kind, h=_log_int(rng, 120, 1080), w=_log_int(rng, 160, 1920),
                    size=rng.choice([252, 504, 518, 700, 1008]))
    if kind == "patch":
        # a view of a batch starts on 8 bytes
        if views > 1 and (gh * gw) % 2:
            gw += 1
        return dict(kind=kind, gh=gh, gw=gw, views=views, width=width)
    if kind == "head":
        return dict(kind=kind, tokens=gh * gw, channels=rng.choice([768, 1024, 1536, 2048]))
    if kind == "ops":
        return dict(kind=kind, gh=gh, gw=gw, views=views, width=width, f16=f16, glob=glob,
                    sequential=rng.random() < 0.2)
    if kind == "qkv":
        return dict(kind=kind, gh=gh, gw=gw, views=views, width=width, f16=f16, glob=glob)
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 38, 10392), width=width, f16=f16)
    if kind == "attention":
        heads = WIDTH[width][1]
        n = N_SPECIAL + gh * gw
        return dict(kind=kind, seqs=heads if glob else heads * views, n=n * views if glob else n)
    if kind == "block":
        return dict(kind=kind, gh=gh, gw=gw, views=views, width=width, f16=f16, glob=glob)
    gh, gw = _log_int(rng, 8, 24), _log_int(rng, 8, 36)
    views = rng.choice([1, 1, 2, 3])
    if views > 1 and (gh * gw) % 2:
        gw += 1
    return dict(kind="frame", gh=gh, gw=gw, views=views, width="B")


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most and all({k: v for k, v in x.items() if k != "name"} != c
                                    for x in listed()):
            return c


# ------------------------------------------------------------------ work
def _rows(c):
    return c["views"] * (N_SPECIAL + c["gh"] * c["gw"])


def _block_work(rows, n, seqs, D, M, wbytes):
    flops = 2 * rows * (4 * D * D + 2 * D * M) + 4 * HD * seqs * n * n
    return 2 * 4 * rows * D + wbytes * (4 * D * D + 2 * D * M), flops


def work(case):
    k = case["kind"]
    if k == "preprocess":
        oh, ow = _rt().preprocess_shape(case["h"], case["w"], case["size"], PATCH)
        return {"bytes": 3 * (case["h"] * case["w"] + oh * ow), "flops": 0}
    if k == "patch":
        D, np_ = WIDTH[case["width"]][0], case["gh"] * case["gw"]
        px = 3 * PATCH * PATCH
        return {"bytes": case["views"] * (np_ * px + 4 * (np_ + N_SPECIAL) * D) + 4 * px * D
                + 4 * (np_ + 1) * D, "flops": 2 * case["views"] * np_ * px * D}
    if k == "head":
        return {"bytes": 8 * case["tokens"] * case["channels"], "flops": 0}
    if k == "attention":
        s, n = case["seqs"], case["n"]
        return {"bytes": 4 * 4 * s * n * HD, "flops": 4 * HD * s * n * n}
    D, H, M = WIDTH[case["width"]]
    w = 2 if case.get("f16") else 4
    if k == "mlp":
        r = case["rows"]
        return {"bytes": 4 * r * 3 * D + w * 2 * D * M, "flops": 4 * r * D * M}
    rows = _rows(case)
    if k == "qkv":
        return {"bytes": 4 * rows * 4 * D + w * 3 * D * D, "flops": 6 * rows * D * D}
    if k == "ops":
        # tokens in and out and LN1; Q and K in and out; attention, MLP and
        # hidden in, hidden and LN2 out
        return {"bytes": 4 * rows * (3 * D + 4 * D + 2 * D + 2 * M + D), "flops": 0}
    n = rows if case.get("glob") else rows // case["views"]
    seqs = H if case.get("glob") else H * case["views"]
    if k == "block":
        b, f = _block_work(rows, n, seqs, D, M, w)
        return {"bytes": b, "flops": f}
    p = work(dict(kind="patch", gh=case["gh"], gw=case["gw"], views=case["views"], width="B"))
    total_b, total_f = p["bytes"], p["flops"]
    for layer in range(DEPTH):
        g = _is_global(layer)
        b, f = _block_work(rows, rows if g else n, H if g else H * case["views"], D, M, 4)
        total_b += b - 8 * rows * D  # the stream between blocks is not an output
        total_f += f
    total_b += 4 * rows * D + len(OUT_LAYERS) * 4 * 2 * D * (rows - case["views"])
    return {"bytes": total_b, "flops": total_f}


def _cost(case):
    if case["kind"] == "preprocess":
        return 6 * case["h"] * case["w"]
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def tolerance(case):
    k = case["kind"]
    return "exact" if k == "preprocess" else {"rel": REL[k], "max": 50 * REL[k]}


# ------------------------------------------------------------------ inputs
_RT = None


def _rt():
    global _RT
    if _RT is None:
        _RT = vh.Runtime(0)
    return _RT


def _wrap(t):
    """A library tensor over a torch tensor's memory, which it keeps alive."""
    kind = {torch.float32: vh.VK_F32, torch.float16: vh.VK_F16, torch.uint8: vh.VK_U8}[t.dtype]
    h = ctypes.c_void_p()
    status = vh.lib.vk_tensor_wrap(_rt().handle, kind, t.data_ptr(), t.numel(), ctypes.byref(h))
    if status != vh.VK_OK:
        raise vh.VestraError(status, vh.lib.vk_last_error().decode())
    w = vh.Tensor(_rt(), h)
    w.torch = t
    return w


class _Draws:
    """Seeded inputs: activations ~ N(0, 1), weights and biases of the
    benchmark's initialisation."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, scale=1.0, shift=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * scale + shift

    def gamma(self, n, f16=False):
        return self.stored(self.normal(n, scale=0.02, shift=1.0), f16)

    def small(self, *shape, f16=False):
        return self.stored(self.normal(*shape, scale=0.02), f16)

    def ls(self, n, f16=False):
        return self.stored(torch.rand(n, generator=self.g, device="cuda") * 0.1, f16)

    def image(self, views, h, w):
        return torch.randint(0, 256, (views, h, w, 3), generator=self.g, device="cuda",
                             dtype=torch.uint8)

    @staticmethod
    def stored(t, f16):
        return t.half() if f16 else t


def _linear(w, b, ls=None):
    host = [None if t is None else t.float().cpu().numpy() for t in (b, ls)]
    make = _rt().prepare_linear_w16 if w.dtype == torch.float16 else _rt().prepare_linear_f32
    return make(w.shape[0], w.shape[1], w.cpu().numpy(), host[0], host[1])


def _block_params(d, width, f16):
    D, _, M = WIDTH[width]
    return {"norm1_gamma": d.gamma(D, f16), "norm1_beta": d.small(D, f16=f16),
            "qkv_w": d.small(D, 3 * D, f16=f16), "qkv_b": d.small(3 * D),
            "qnorm_gamma": d.gamma(HD, f16), "qnorm_beta": d.small(HD, f16=f16),
            "knorm_gamma": d.gamma(HD, f16), "knorm_beta": d.small(HD, f16=f16),
            "proj_w": d.small(D, D, f16=f16), "proj_b": d.small(D), "ls1": d.ls(D),
            "norm2_gamma": d.gamma(D, f16), "norm2_beta": d.small(D, f16=f16),
            "fc1_w": d.small(D, M, f16=f16), "fc1_b": d.small(M),
            "fc2_w": d.small(M, D, f16=f16), "fc2_b": d.small(D), "ls2": d.ls(D)}


VECTORS = ("norm1_gamma", "norm1_beta", "qnorm_gamma", "qnorm_beta", "knorm_gamma", "knorm_beta",
           "norm2_gamma", "norm2_beta")


def _block_weights(p):
    keep = {k: _wrap(p[k]) for k in VECTORS}
    keep.update(qkv=_linear(p["qkv_w"], p["qkv_b"]), proj=_linear(p["proj_w"], p["proj_b"], p["ls1"]),
                fc1=_linear(p["fc1_w"], p["fc1_b"]), fc2=_linear(p["fc2_w"], p["fc2_b"], p["ls2"]))
    return vh.block_weights_struct(**keep), keep


def _config(width):
    D, H, M = WIDTH[width]
    return vh.VitConfig(embed_dim=D, num_heads=H, head_dim=HD, mlp_hidden=M,
                        num_register=N_SPECIAL - 1, ln_eps=LN_EPS, qk_norm_eps=QK_EPS,
                        rope_freq=FREQ, rope_start=0, qknorm_start=0, alt_start=ALT_START,
                        rope_mode=0)


def _is_global(layer):
    return layer >= ALT_START and layer % 2 == 1


def _layer(case):
    return ALT_START + 1 if case["glob"] else 0


def _tensors(case, seed):
    """The inputs and parameters of a case as torch tensors."""
    d, k = _Draws(seed), case["kind"]
    if k == "preprocess":
        return {"frame": d.image(1, case["h"], case["w"])[0]}
    if k == "attention":
        s, n = case["seqs"], case["n"]
        return {"q": d.normal(s, n, HD, scale=1.5), "k": d.normal(s, n, HD, scale=1.5),
                "v": d.normal(s, n, HD)}
    if k == "head":
        c = case["channels"]
        return {"tok": d.normal(case["tokens"], c), "gamma": d.gamma(c), "beta": d.small(c)}
    D, H, M = WIDTH[case["width"]]
    if k == "mlp":
        p = _block_params(d, case["width"], case["f16"])
        t = {n: p[n] for n in ("fc1_w", "fc1_b", "fc2_w", "fc2_b", "ls2")}
        return dict(t, x=d.normal(case["rows"], D), residual=d.normal(case["rows"], D))
    rows = _rows(case)
    if k in ("patch", "frame"):
        n = case["gh"] * case["gw"]
        t = {"image": d.image(case["views"], PATCH * case["gh"], PATCH * case["gw"]),
             "w": d.small(D, 3, PATCH, PATCH), "b": d.small(D), "cls": d.small(D),
             "reg": d.small((N_SPECIAL - 1) * D), "pos": d.small(1 + n, D)}
        if k == "frame":
            t.update(camera=d.normal(2 * D), norm_gamma=d.gamma(D), norm_beta=d.small(D),
                     blocks=[_block_params(d, "B", False) for _ in range(DEPTH)])
        return t
    p = _block_params(d, case["width"], case["f16"])
    if k == "qkv":
        names = ("qkv_w", "qkv_b", "qnorm_gamma", "qnorm_beta", "knorm_gamma", "knorm_beta")
        return dict({n: p[n] for n in names}, x=d.normal(rows, D))
    if k == "block":
        return dict(p, tokens=d.normal(rows, D))
    names = VECTORS + ("ls1", "ls2")
    return dict({n: p[n] for n in names}, tokens=d.normal(rows, D), q=d.normal(rows * D),
                k=d.normal(rows * D), attn_proj=d.normal(rows, D), hidden=d.normal(rows, M),
                mlp_out=d.normal(rows, D))


def prepare(case, seed):
    rt, t, k = _rt(), _tensors(case, seed), case["kind"]
    s = {"case": case, "rt": rt, "t": t}

    def empty(*shape, dtype=torch.float32):
        return torch.empty(*shape, device="cuda", dtype=dtype)

    if k == "preprocess":
        h, w, size = case["h"], case["w"], case["size"]
        oh, ow = rt.preprocess_shape(h, w, size, PATCH)
        need = int(vh.lib.vk_preprocess_workspace_bytes(h, w, size, PATCH, 1))
        s["out"] = empty(oh, ow, 3, dtype=torch.uint8)
        s["ws"] = empty(max(need, 1), dtype=torch.uint8)
        s.update(src=_wrap(t["frame"]), dst=_wrap(s["out"]), work=_wrap(s["ws"]))
    elif k == "attention":
        s["out"] = torch.empty_like(t["q"])
        s["a"] = [_wrap(t[n]) for n in "qkv"] + [_wrap(s["out"])]
    elif k == "head":
        s["out"] = empty(case["channels"], case["tokens"])
        s["a"] = [_wrap(t[n]) for n in ("tok", "gamma", "beta")] + [_wrap(s["out"])]
    elif k == "mlp":
        s["fc1"], s["fc2"] = _linear(t["fc1_w"], t["fc1_b"]), _linear(t["fc2_w"], t["fc2_b"], t["ls2"])
        s["hidden"] = empty(case["rows"], WIDTH[case["width"]][2])
        s.update(x=_wrap(t["x"]), h=_wrap(s["hidden"]), r=_wrap(t["residual"]))
    elif k == "qkv":
        s["lin"] = _linear(t["qkv_w"], t["qkv_b"])
        D, H, _ = WIDTH[case["width"]]
        s["out"] = [empty(H, _rows(case), HD) for _ in range(3)]
        s["x"], s["o"] = _wrap(t["x"]), [_wrap(o) for o in s["out"]]
        s["n"] = [_wrap(t[n]) for n in ("qnorm_gamma", "qnorm_beta", "knorm_gamma", "knorm_beta")]
    elif k == "ops":
        D = WIDTH[case["width"]][0]
        s["ln1"], s["ln2"] = empty(_rows(case), D), empty(_rows(case), D)
        s["keep"] = {n: _wrap(t[n]) for n in t}
        s["act_t"] = dict({n: s["keep"][n] for n in ("tokens", "q", "k", "attn_proj", "hidden",
                                                     "mlp_out")}, ln1=_wrap(s["ln1"]),
                          ln2=_wrap(s["ln2"]))
        s["layer"] = vh.layer_struct(**{n: s["keep"][n] for n in VECTORS + ("ls1", "ls2")})
        s["act"] = vh.activations_struct(**s["act_t"])
        s["cfg"] = _config(case["width"])
    elif k == "block":
        D, _, M = WIDTH[case["width"]]
        s["w"], s["keep"] = _block_weights(t)
        s["tokens"], s["cfg"] = _wrap(t["tokens"]), _config(case["width"])
        s["ws"] = rt.block_workspace(_rows(case), D, M)
    if k in ("patch", "frame"):
        D, _, M = WIDTH[case["width"]]
        s["proj"] = rt.prepare_linear_oihw_f32(3 * PATCH * PATCH, D, t["w"].cpu().numpy(),
                                               t["b"].cpu().numpy())
        s["tokens_t"] = empty(_rows(case), D)
        s["a"] = {n: _wrap(t[n]) for n in ("image", "cls", "reg", "pos")}
        s["tokens"] = _wrap(s["tokens_t"])
    if k == "frame":
        made = [_block_weights(p) for p in t["blocks"]]
        s["blocks"], s["keep"] = [m[0] for m in made], [m[1] for m in made]
        s["camera"], s["ng"], s["nb"] = (_wrap(t[n]) for n in ("camera", "norm_gamma", "norm_beta"))
        n = case["gh"] * case["gw"]
        s["feats_t"] = [empty(case["views"], n, 2 * D) for _ in OUT_LAYERS]
        s["cams_t"] = [empty(case["views"], 2 * D) for _ in OUT_LAYERS]
        s["feats"], s["cams"] = [_wrap(x) for x in s["feats_t"]], [_wrap(x) for x in s["cams_t"]]
        s["local"], s["cfg"] = rt.alloc_f32(_rows(case) * D), _config("B")
        s["ws"] = rt.block_workspace(_rows(case), D, M)
    torch.cuda.synchronize()  # the runtime's stream is its own
    return s


# ------------------------------------------------------------------ one pass
def _patch(s):
    c, rt, a = s["case"], s["rt"], s["a"]
    h, w = PATCH * c["gh"], PATCH * c["gw"]
    if c["views"] == 1:
        rt.patch_embed_u8(a["image"], h, w, PATCH, MEAN, STD, s["proj"], a["cls"], a["reg"],
                          N_SPECIAL - 1, a["pos"], s["tokens"])
    else:
        rt.patch_embed_views_u8(a["image"], c["views"], h, w, PATCH, MEAN, STD, s["proj"],
                                a["cls"], a["reg"], N_SPECIAL - 1, a["pos"], s["tokens"])


def run(s):
    c, rt, k = s["case"], s["rt"], s["case"]["kind"]
    if k == "preprocess":
        status = vh.lib.vk_preprocess_resize_u8(rt.handle, s["src"].handle, c["h"], c["w"],
                                                c["size"], PATCH, 1, s["work"].handle,
                                                s["dst"].handle)
        if status != vh.VK_OK:
            raise vh.VestraError(status, vh.lib.vk_last_error().decode())
        return s["out"]
    if k == "attention":
        q, key, v, out = s["a"]
        rt.attention_into_f32(q, key, v, c["seqs"], c["n"], HD, out)
        return s["out"]
    if k == "head":
        tok, g, b, out = s["a"]
        rt.token_to_chw_f32(tok, c["tokens"], c["channels"], g, b, HEAD_EPS, out)
        return s["out"]
    if k == "mlp":
        s["fc1"].run_gelu(s["x"], c["rows"], s["h"])
        s["fc2"].run_residual(s["h"], c["rows"], s["r"])
        return {"hidden": s["hidden"], "residual": s["t"]["residual"]}
    if k == "qkv":
        s["lin"].run_qkv_hnd_norm_rope(s["x"], _rows(c), WIDTH[c["width"]][1], *s["o"], *s["n"],
                                       N_SPECIAL, c["gh"], c["gw"], c["views"], c["glob"], FREQ,
                                       QK_EPS)
        return s["out"]
    if k == "ops":
        if c["sequential"]:
            rt.set_layernorm_order(vh.VK_LN_ORDER_SEQUENTIAL)
        rt.vit_block_fused_ops(s["cfg"], _layer(c), s["layer"], None, s["act"], c["gh"], c["gw"],
                               c["views"], None, vh.VK_BLOCK_FUSE_LS_LN)
        if c["sequential"]:
            rt.set_layernorm_order(vh.VK_LN_ORDER_TREE)
        t = s["t"]
        return {"ln1": s["ln1"], "q": t["q"], "k": t["k"], "ln2": s["ln2"], "hidden": t["hidden"],
                "tokens": t["tokens"]}
    if k == "block":
        rt.vit_block_forward_f32(s["cfg"], _layer(c), s["w"], s["tokens"], c["gh"], c["gw"],
                                 c["views"], None, s["ws"].struct)
        return s["t"]["tokens"]
    _patch(s)
    if k == "patch":
        return s["tokens_t"]
    rt.backbone_forward_f32(s["cfg"], s["blocks"], s["tokens"], c["gh"], c["gw"], c["views"],
                            s["camera"], s["ng"], s["nb"], True, OUT_LAYERS, s["feats"], s["cams"],
                            s["ws"], s["local"])
    return {"feats": s["feats_t"], "cams": s["cams_t"], "tokens": s["tokens_t"]}


# ------------------------------------------------------------------ in 64 bits
def _ln(x, g, b, eps):
    m = x.mean(-1, keepdim=True)
    var = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(var + eps) * g.double() + b.double()


def _gelu(x):
    """GELU with the library's stated erf (Abramowitz-Stegun 7.1.26)."""
    a = x.abs() / math.sqrt(2.0)
    t = 1.0 / (1.0 + 0.3275911 * a)
    poly = ((((1.0614054 * t - 1.4531520) * t + 1.4214137) * t - 0.28449674) * t
            + 0.25482959) * t
    return 0.5 * x * (1.0 + torch.sign(x) * (1.0 - poly * torch.exp(-a * a)))


def _rope(x, case, views_outer=False):
    """2D RoPE of head-major rows [..., view * token, 64] (or one view's)."""
    gh, gw = case["gh"], case["gw"]
    p = torch.arange(gh * gw)
    yx = torch.stack([p // gw + 1, p % gw + 1], 1)
    if case["glob"]:
        yx = torch.ones_like(yx)
    pos = torch.cat([torch.zeros(N_SPECIAL, 2, dtype=yx.dtype), yx])
    if not views_outer:
        pos = pos.repeat(case["views"], 1)
    inv = torch.tensor([1.0 / FREQ ** (2.0 * j / 32) for j in range(16)],
                       dtype=torch.float64).float()
    out = x.clone()
    for base, coord in ((0, 0), (32, 1)):
        ang = (pos[:, coord].float()[:, None] * inv[None, :]).double().to(x.device)
        c, s = torch.cos(ang), torch.sin(ang)
        a, b = x[..., base:base + 16], x[..., base + 16:base + 32]
        out[..., base:base + 16] = a * c - b * s
        out[..., base + 16:base + 32] = b * c + a * s
    return out


def _attention(q, k, v):
    out = torch.empty_like(q)
    step = max(1, int(2e8 // k.shape[1]))
    for h in range(q.shape[0]):
        for i in range(0, q.shape[1], step):
            p = torch.softmax(q[h, i:i + step] @ k[h].T.contiguous() / 8.0, -1)
            out[h, i:i + step] = p @ v[h]
    return out


def _qkv(x, p, case):
    rows, D = x.shape
    y = x @ p["qkv_w"].double() + p["qkv_b"].double()
    q, k, v = (y[:, i * D:(i + 1) * D].reshape(rows, -1, HD).transpose(0, 1).contiguous()
               for i in range(3))
    q = _rope(_ln(q, p["qnorm_gamma"], p["qnorm_beta"], QK_EPS), case)
    k = _rope(_ln(k, p["knorm_gamma"], p["knorm_beta"], QK_EPS), case)
    return q, k, v


def _block(x, p, case):
    rows, D = x.shape
    q, k, v = _qkv(_ln(x, p["norm1_gamma"], p["norm1_beta"], LN_EPS), p, case)
    shape = q.shape
    if not case["glob"]:
        q, k, v = (t.reshape(-1, rows // case["views"], HD) for t in (q, k, v))
    a = _attention(q, k, v).reshape(shape).transpose(0, 1).reshape(rows, D)
    x = x + (a @ p["proj_w"].double() + p["proj_b"].double()) * p["ls1"].double()
    h = _ln(x, p["norm2_gamma"], p["norm2_beta"], LN_EPS)
    h = _gelu(h @ p["fc1_w"].double() + p["fc1_b"].double())
    return x + (h @ p["fc2_w"].double() + p["fc2_b"].double()) * p["ls2"].double()


def _tokens(t, case):
    gh, gw, n = case["gh"], case["gw"], case["gh"] * case["gw"]
    mean, std = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in (MEAN, STD))
    x = (t["image"].double() / 255.0 - mean) / std
    x = x.reshape(case["views"], gh, PATCH, gw, PATCH, 3).permute(0, 1, 3, 5, 2, 4)
    w = t["w"].double().reshape(t["w"].shape[0], -1).T.contiguous()
    y = x.reshape(case["views"] * n, -1) @ w + t["b"].double()
    y = y.reshape(case["views"], n, -1) + t["pos"][1:].double()
    first = torch.cat([(t["cls"].double() + t["pos"][0].double())[None],
                       t["reg"].double().reshape(N_SPECIAL - 1, -1)])
    return torch.cat([first.expand(case["views"], -1, -1), y], 1).reshape(-1, w.shape[1])


def exact(case, seed):
    k = case["kind"]
    if k == "preprocess":
        return None
    t = _tensors(case, seed)
    if k == "attention":
        return _attention(*(t[n].double() for n in "qkv"))
    if k == "head":
        return _ln(t["tok"].double(), t["gamma"], t["beta"], HEAD_EPS).T.contiguous()
    if k == "mlp":
        h = _gelu(t["x"].double() @ t["fc1_w"].double() + t["fc1_b"].double())
        y = (h @ t["fc2_w"].double() + t["fc2_b"].double()) * t["ls2"].double()
        return {"hidden": h, "residual": t["residual"].double() + y}
    if k == "qkv":
        return list(_qkv(t["x"].double(), t, case))
    if k == "ops":
        x, D = t["tokens"].double(), t["tokens"].shape[1]
        H, n = WIDTH[case["width"]][1], x.shape[0] // case["views"]
        shape = (H, x.shape[0], HD) if case["glob"] else (case["views"], H, n, HD)
        out = {"ln1": _ln(x, t["norm1_gamma"], t["norm1_beta"], LN_EPS)}
        for m in "qk":
            y = _ln(t[m].double().reshape(shape), t[m + "norm_gamma"], t[m + "norm_beta"], QK_EPS)
            out[m] = _rope(y, case, views_outer=not case["glob"]).reshape(-1)
        x = x + t["attn_proj"].double() * t["ls1"].double()
        out["ln2"] = _ln(x, t["norm2_gamma"], t["norm2_beta"], LN_EPS)
        out["hidden"] = _gelu(t["hidden"].double())
        out["tokens"] = x + t["mlp_out"].double() * t["ls2"].double()
        return out
    if k == "block":
        return _block(t["tokens"].double(), t, case)
    x = _tokens(t, case)
    if k == "patch":
        return x
    n, views, D = case["gh"] * case["gw"] + N_SPECIAL, case["views"], x.shape[1]
    feats, cams, local = [], [], x
    for layer, p in enumerate(t["blocks"]):
        g = _is_global(layer)
        if layer == ALT_START:
            x = x.clone().reshape(views, n, D)
            x[0, 0], x[1:, 0] = t["camera"][:D].double(), t["camera"][D:].double()
            x = x.reshape(-1, D)
        x = _block(x, p, dict(case, glob=g))
        if layer in OUT_LAYERS:
            lv, xv = (local if g else x).reshape(views, n, D), x.reshape(views, n, D)
            normed = _ln(xv[:, N_SPECIAL:], t["norm_gamma"], t["norm_beta"], LN_EPS)
            feats.append(torch.cat([lv[:, N_SPECIAL:], normed], 2))
            cams.append(torch.cat([lv[:, 0], xv[:, 0]], 1))
        if not g:
            local = x
    return {"feats": feats, "cams": cams, "tokens": x}
