"""The workloads this framework is measured on: Depth-Anything-3 BASE inference
through the public entry points of ``vestra_hip``, from one encoder block of a
thumbnail to the twelve-layer encoder of a batch, with the projections,
attention, Q8_0 products, DPT head and unfused row operations that a program
also calls one by one.

A case is a dict of plain values; ``kind`` selects the path.  ``prepare`` holds
what a program keeps between calls (uploaded weights, uploaded inputs, the
runtime), ``run`` is one pass, ``exact`` the same pass in float64 torch.
"""
import math
import os
import sys

import numpy as np
import torch

for _p in (os.path.join(os.getcwd(), "vestra-kernels_amd"),
           os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                        "vestra-kernels_amd")):
    if os.path.isdir(_p) and _p not in sys.path:
        sys.path.append(_p)

import vestra_hip as vh  # noqa: E402
from vestra_hip import da3  # noqa: E402

DIM, HEADS, MLP, PATCH = da3.DIM, da3.HEADS, da3.MLP, da3.PATCH
DEV = "cuda"


def listed():
    return [
        # A 168 x 112 thumbnail (8 x 12 patches and the CLS token): one block,
        # where launches and latency are everything.
        {"name": "block_97", "kind": "block", "images": 1, "rows": 8, "cols": 12, "late": False,
         "q8": False},
        # DA3-BASE at its 504 x 336 input: the block the framework is built around.
        {"name": "block_865", "kind": "block", "images": 1, "rows": 24, "cols": 36, "late": False,
         "q8": False},
        # The same block with Q8_0 weights (GGUF checkpoints).
        {"name": "block_865_q8", "kind": "block", "images": 1, "rows": 24, "cols": 36,
         "late": False, "q8": True},
        # A late block (Q/K LayerNorm) over one 1008 x 672 image: the longest sequence.
        {"name": "block_3457_late", "kind": "block", "images": 1, "rows": 48, "cols": 72,
         "late": True, "q8": False},
        # The whole encoder of a batch of four images, from pixels: patch
        # embedding, token assembly, twelve layers of which the last four are late.
        {"name": "encoder_4x865", "kind": "encoder", "images": 4, "rows": 24, "cols": 36,
         "layers": 12, "late_from": 8},
        # Attention alone at the encoder's shape, token-major as the
        # out-projection reads it.
        {"name": "attention_865", "kind": "attention", "heads": 12, "tokens": 865, "head_dim": 64,
         "token_major": True},
        # The generic attention of a narrow-headed model at a ragged length.
        {"name": "attention_online_500x40", "kind": "attention", "heads": 8, "tokens": 500,
         "head_dim": 40, "token_major": False},
        # One fused projection, fc1 with bias and GELU.
        {"name": "fc1_gelu_865", "kind": "projection", "mode": "gelu", "m": 865, "k": 768,
         "n": 3072},
        # A plain product of two activations with no friendly dimension.
        {"name": "gemm_1153x1003x771", "kind": "gemm", "m": 1153, "k": 1003, "n": 771},
        # A Q8_0 projection alone: quantise the rows, block-dot product, bias.
        {"name": "q8_linear_865", "kind": "q8_linear", "m": 865, "k": 768, "n": 3072},
        # One level of the DPT head: projection to CHW, 4x transposed
        # convolution, layer_rn, a residual convolution, upsampling fusion.
        {"name": "dpt_24x36", "kind": "dpt", "rows": 24, "cols": 36, "features": 128},
        # The unfused row operations over a batch's tokens: LayerNorm, residual
        # add, GELU.
        {"name": "rows_3460", "kind": "rows", "rows": 3460, "cols": 768},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "encoder", "attention", "attention", "projection",
                       "projection", "gemm", "q8_linear", "dpt", "rows"])
    if kind in ("block", "encoder"):
        images = rng.choice([1, 1, 1, 2, 3, 4])
        tokens = _log_int(rng, 20, 3456 // images)
        rows = max(2, _log_int(rng, max(2, math.sqrt(tokens) / 1.6), math.sqrt(tokens) * 1.2))
        cols = max(2, tokens // rows)
        if kind == "block":
            return {"kind": "block", "images": images, "rows": rows, "cols": cols,
                    "late": rng.random() < 0.3, "q8": rng.random() < 0.25}
        layers = rng.randint(2, 6)
        return {"kind": "encoder", "images": images, "rows": rows, "cols": cols, "layers": layers,
                "late_from": rng.randint(1, layers)}
    if kind == "attention":
        hd = rng.choice([64, 64, 64, 32, 16, rng.randint(5, 63)])
        return {"kind": "attention", "heads": rng.choice([1, 6, 12, 12, 24]),
                "tokens": _log_int(rng, 16, 3500), "head_dim": hd, "token_major": rng.random() < 0.5}
    if kind == "projection":
        mode = rng.choice(["run", "gelu", "residual", "chw", "qkv"])
        k = rng.choice([768, 768, 3072, 588, 32 * rng.randint(2, 64), rng.randint(40, 1500)])
        n = 192 * rng.choice([4, 6, 12]) if mode == "qkv" else rng.choice(
            [768, 3072, 96, 192, 384, rng.randint(40, 3000)])
        return {"kind": "projection", "mode": mode, "m": _log_int(rng, 16, 4000), "k": k, "n": n}
    if kind == "gemm":
        return {"kind": "gemm", "m": _log_int(rng, 16, 3500), "k": _log_int(rng, 16, 3100),
                "n": _log_int(rng, 16, 3100)}
    if kind == "q8_linear":
        return {"kind": "q8_linear", "m": _log_int(rng, 16, 3500), "k": 32 * rng.randint(4, 96),
                "n": rng.choice([768, 2304, 3072, rng.randint(40, 3000)])}
    if kind == "dpt":
        return {"kind": "dpt", "rows": rng.randint(6, 26), "cols": rng.randint(6, 38),
                "features": rng.choice([64, 96, 128])}
    return {"kind": "rows", "rows": _log_int(rng, 16, 8000), "cols": rng.choice([768, 768, 64, 1024,
                                                                              rng.randint(40, 1500)])}


# ---- inputs --------------------------------------------------------------------
# Every input is a function of (case, seed): prepare uploads it, exact computes on it.


def _normal(rng, n, std=1.0, mean=0.0):
    return rng.standard_normal(n, dtype=np.float32) * np.float32(std) + np.float32(mean)


def _block_weights(rng, late):
    """A trained block's scales: weights of std 0.02, LayerNorm gamma about 1, LayerScale
    per channel, so that each branch moves the residual stream."""
    def vec(n):
        return (0.1 + 0.9 * rng.random(n)).astype(np.float32)

    w = {"ln1_gamma": 0.5 + vec(DIM), "ln1_beta": _normal(rng, DIM, 0.1),
         "w_qkv": _normal(rng, DIM * 3 * DIM, 0.02), "b_qkv": _normal(rng, 3 * DIM, 0.02),
         "w_proj": _normal(rng, DIM * DIM, 0.02), "b_proj": _normal(rng, DIM, 0.02),
         "ls1": vec(DIM),
         "ln2_gamma": 0.5 + vec(DIM), "ln2_beta": _normal(rng, DIM, 0.1),
         "w_fc1": _normal(rng, DIM * MLP, 0.02), "b_fc1": _normal(rng, MLP, 0.02),
         "w_fc2": _normal(rng, MLP * DIM, 0.02), "b_fc2": _normal(rng, DIM, 0.02),
         "ls2": vec(DIM)}
    if late:
        for n in ("q_norm", "k_norm"):
            w[n + "_gamma"] = _normal(rng, 64, 0.1, 1.0)
            w[n + "_beta"] = _normal(rng, 64, 0.02)
    return w


def _tokens_in(rng, rows):
    """Residual-stream rows: unit spread, a row offset and a few large channels, as a ViT's are."""
    x = _normal(rng, rows * DIM).reshape(rows, DIM)
    x += _normal(rng, rows, 0.5)[:, None]
    x[:, [5, 130, 577]] += np.float32([12.0, -8.0, 20.0])
    return x.reshape(-1)


def _rng(case, seed):
    return np.random.default_rng([int(seed), len(case["kind"]), 77])


def _inputs(case, seed):
    rng = _rng(case, seed)
    kind = case["kind"]
    if kind == "block":
        t = case["rows"] * case["cols"] + 1
        return {"w": [_block_weights(rng, case["late"])], "x": _tokens_in(rng, case["images"] * t)}
    if kind == "encoder":
        pk = 3 * PATCH * PATCH
        return {"w": [_block_weights(rng, i >= case["late_from"]) for i in range(case["layers"])],
                "pixels": [_normal(rng, 3 * case["rows"] * case["cols"] * PATCH * PATCH)
                           for _ in range(case["images"])],
                "embed_w": _normal(rng, pk * DIM, 0.03), "embed_b": _normal(rng, DIM, 0.02),
                "cls": _normal(rng, DIM), "pos": _normal(rng, (case["rows"] * case["cols"] + 1) * DIM, 0.5)}
    if kind == "attention":
        n = case["heads"] * case["tokens"] * case["head_dim"]
        return {c: _normal(rng, n) for c in "qkv"}
    if kind == "projection":
        m, k, n = case["m"], case["k"], case["n"]
        d = {"x": _normal(rng, m * k), "w": _normal(rng, k * n, 0.02), "b": _normal(rng, n, 0.02)}
        if case["mode"] in ("run", "residual"):
            d["g"] = (0.1 + 0.9 * rng.random(n)).astype(np.float32)
        if case["mode"] == "residual":
            d["r"] = _normal(rng, m * n)
        return d
    if kind == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return {"a": _normal(rng, m * k), "b": _normal(rng, k * n, 1.0 / math.sqrt(k))}
    if kind == "q8_linear":
        m, k, n = case["m"], case["k"], case["n"]
        blocks = np.zeros(n * k // 32, vh.BLOCK_Q8_0)
        blocks["qs"] = rng.integers(-127, 128, (n * k // 32, 32), dtype=np.int8)
        blocks["d"] = (1e-4 + 4e-4 * rng.random(n * k // 32)).astype(np.float16).view(np.uint16)
        return {"x": _normal(rng, m * k), "blocks": blocks, "b": _normal(rng, n, 0.02)}
    if kind == "dpt":
        r, c, f = case["rows"], case["cols"], case["features"]
        return {"x": _normal(rng, r * c * DIM), "proj_w": _normal(rng, DIM * 96, 0.03),
                "proj_b": _normal(rng, 96, 0.02), "up_w": _normal(rng, 96 * 96 * 16, 0.1),
                "up_b": _normal(rng, 96, 0.02), "rn_w": _normal(rng, f * 96 * 9, 0.03),
                "res_w": _normal(rng, f * f * 9, 0.03), "res_b": _normal(rng, f, 0.02),
                "out_w": _normal(rng, 32 * f * 9, 0.03), "out_b": _normal(rng, 32, 0.02)}
    rows, cols = case["rows"], case["cols"]
    return {"x": _normal(rng, rows * cols), "y": _normal(rng, rows * cols),
            "g": _normal(rng, cols, 0.1, 1.0), "b": _normal(rng, cols, 0.1)}


# ---- the path --------------------------------------------------------------------

_RT = None


def _runtime():
    global _RT
    if _RT is None:
        _RT = vh.Runtime(torch.cuda.current_device())
    return _RT


class _Shared:
    """A device tensor of the framework as torch sees it (no copy); keeps it alive."""

    def __init__(self, t, shape):
        self.t = t
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "version": 2,
                                         "data": (t.device_ptr, False)}


def _view(t, *shape):
    return torch.as_tensor(_Shared(t, shape), device=DEV)


def prepare(case, seed):
    rt = _runtime()
    d = _inputs(case, seed)
    kind = case["kind"]
    s = {"case": case, "rt": rt}
    if kind == "block":
        s["tokens"] = case["rows"] * case["cols"] + 1
        s["block"] = rt.prepare_block(d["w"][0], q8_0=case["q8"])
        s["in"] = rt.upload_f32(d["x"])
        s["x"] = rt.alloc_f32(d["x"].size)
        s["pos"] = da3.positions_yx(case["rows"], case["cols"])
        s["out"] = _view(s["x"], case["images"] * s["tokens"], DIM)
    elif kind == "encoder":
        s["tokens"] = case["rows"] * case["cols"] + 1
        s["blocks"] = [rt.prepare_block(w) for w in d["w"]]
        s["embed"] = rt.prepare_linear_f32(3 * PATCH * PATCH, DIM, d["embed_w"], d["embed_b"])
        s["pixels"] = [rt.upload_f32(p) for p in d["pixels"]]
        s["cls"], s["posemb"] = rt.upload_f32(d["cls"]), rt.upload_f32(d["pos"])
        s["pos"] = da3.positions_yx(case["rows"], case["cols"])
        s["x"] = rt.alloc_f32(case["images"] * s["tokens"] * DIM)
        s["out"] = _view(s["x"], case["images"] * s["tokens"], DIM)
    elif kind == "attention":
        s.update({c: rt.upload_f32(d[c]) for c in "qkv"})
    elif kind == "projection":
        s["lin"] = rt.prepare_linear_f32(case["k"], case["n"], d["w"], d["b"], d.get("g"))
        s["x"] = rt.upload_f32(d["x"])
        if case["mode"] == "residual":
            s["in"], s["r"] = rt.upload_f32(d["r"]), rt.alloc_f32(d["r"].size)
            s["out"] = _view(s["r"], case["m"], case["n"])
    elif kind == "gemm":
        s["a"], s["b"] = rt.upload_f32(d["a"]), rt.upload_f32(d["b"])
    elif kind == "q8_linear":
        s["lin"] = rt.prepare_linear_q8_0(case["k"], case["n"], d["blocks"], d["b"])
        s["x"] = rt.upload_f32(d["x"])
    elif kind == "dpt":
        f = case["features"]
        s["x"] = rt.upload_f32(d["x"])
        s["proj"] = rt.prepare_linear_f32(DIM, 96, d["proj_w"], d["proj_b"])
        s["up"] = rt.prepare_conv_transpose2d_f32(96, 96, 4, 4, 4, d["up_w"], d["up_b"])
        s["rn"] = rt.prepare_conv2d_f32(96, f, 3, 3, 1, 1, d["rn_w"])
        s["res"] = rt.prepare_conv2d_f32(f, f, 3, 3, 1, 1, d["res_w"], d["res_b"])
        s["head"] = rt.prepare_conv2d_f32(f, 32, 3, 3, 1, 1, d["out_w"], d["out_b"])
    else:
        s.update({c: rt.upload_f32(d[c]) for c in "xygb"})
    return s


def run(s):
    rt, case = s["rt"], s["case"]
    kind = case["kind"]
    if kind == "block":
        rt.overwrite_prefix_f32(s["x"], s["in"], len(s["in"]))
        rt.vit_block_run(s["block"], s["x"], case["images"], s["tokens"], s["pos"])
        return s["out"]
    if kind == "encoder":
        n, t = case["rows"] * case["cols"], s["tokens"]
        for i, px in enumerate(s["pixels"]):
            p = rt.patchify_nchw_f32(px, case["rows"] * PATCH, case["cols"] * PATCH, PATCH, 3)
            e = s["embed"].run(p, n)
            x = rt.prepend_cls_add_pos_f32(e, s["cls"], s["posemb"], n, DIM)
            rt.copy_segment_into_f32(s["x"], i * t * DIM, x, 0, t * DIM)
        rt.encoder_run(s["blocks"], s["x"], case["images"], t, s["pos"])
        return s["out"]
    if kind == "attention":
        h, t, hd = case["heads"], case["tokens"], case["head_dim"]
        if hd == 64:
            o = rt.flash_attention_f32_da3_base(s["q"], s["k"], s["v"], h, t, case["token_major"])
        else:
            o = rt.attention_online_f32(s["q"], s["k"], s["v"], h, t, hd)
        return _view(o, h * t * hd)
    if kind == "projection":
        m, n, mode, lin = case["m"], case["n"], case["mode"], s["lin"]
        if mode == "residual":
            rt.overwrite_prefix_f32(s["r"], s["in"], m * n)
            lin.run_residual(s["x"], m, s["r"])
            return s["out"]
        if mode == "qkv":
            q, k, v = lin.run_qkv_hnd(s["x"], 1, m, n // 192)
            return [_view(t, m * n // 3) for t in (q, k, v)]
        o = (lin.run_gelu if mode == "gelu" else lin.run_chw if mode == "chw" else lin.run)(s["x"], m)
        return _view(o, m * n)
    if kind == "gemm":
        return _view(rt.gemm_row_major_f32(s["a"], s["b"], case["m"], case["k"], case["n"]),
                     case["m"], case["n"])
    if kind == "q8_linear":
        return _view(s["lin"].run(s["x"], case["m"]), case["m"], case["n"])
    if kind == "dpt":
        r, c, f = case["rows"], case["cols"], case["features"]
        p = s["proj"].run_chw(s["x"], r * c)
        u = s["up"].run(p, r, c)
        a = s["rn"].run(u, 4 * r, 4 * c)
        b = s["res"].run_relu_input(a, 4 * r, 4 * c)
        rt.add_f32_in_place(b, a)
        o = s["head"].run_resize_align_corners(b, 4 * r, 4 * c, 7 * r, 7 * c)
        return [_view(b, f, 4 * r, 4 * c), _view(o, 32, 7 * r, 7 * c)]
    y = rt.layernorm_f32(s["x"], s["g"], s["b"], case["rows"], case["cols"], da3.LN_EPS)
    rt.add_f32_in_place(y, s["y"])
    rt.gelu_f32_in_place(y)
    return _view(y, case["rows"], case["cols"])


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("block", "encoder"):
        t = case["rows"] * case["cols"] + 1
        m = case["images"] * t
        layers = case.get("layers", 1)
        params = 3 * DIM * DIM + DIM * DIM + 2 * DIM * MLP
        flops = layers * (2.0 * m * params + 4.0 * m * t * DIM)
        wbytes = params * (34.0 / 32.0 if case.get("q8") else 4.0)
        if kind == "encoder":
            pk = 3 * PATCH * PATCH
            flops += 2.0 * m * pk * DIM
            return {"bytes": layers * wbytes + 4.0 * (m * (pk + DIM) + pk * DIM), "flops": flops}
        return {"bytes": wbytes + 8.0 * m * DIM, "flops": flops}
    if kind == "attention":
        n = case["heads"] * case["tokens"] * case["head_dim"]
        return {"bytes": 16.0 * n, "flops": 4.0 * n * case["tokens"]}
    if kind in ("projection", "gemm"):
        m, k, n = case["m"], case["k"], case["n"]
        io = m * k + k * n + m * n * (2 if case.get("mode") == "residual" else 1)
        return {"bytes": 4.0 * io, "flops": 2.0 * m * k * n}
    if kind == "q8_linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4.0 * m * k + n * k * 34.0 / 32.0 + 4.0 * m * n, "flops": 2.0 * m * k * n}
    if kind == "dpt":
        hw, f = case["rows"] * case["cols"], case["features"]
        flops = 2.0 * hw * (DIM * 96 + 96 * 96 * 16 + 16 * (96 * f * 9 + f * f * 9) + 49 * f * 32 * 9)
        weights = DIM * 96 + 96 * 96 * 16 + 96 * f * 9 + f * f * 9 + f * 32 * 9
        return {"bytes": 4.0 * (weights + hw * DIM + hw * 16 * f + hw * 49 * 32), "flops": flops}
    n = case["rows"] * case["cols"]
    return {"bytes": 12.0 * n, "flops": 20.0 * n}


def tolerance(case):
    # About four times what the path is off from `exact` (2-norm), largest over its sizes:
    # block 2.1e-7, encoder 9.5e-7 (twelve layers), attention 4.2e-7, projections and
    # products 5.9e-7 at K = 1000 and with its square root beyond, rows 1.0e-7, dpt 4.0e-6
    # (the resize's float32 coordinates).
    kind = case["kind"]
    if kind == "q8_linear":
        return "exact"  # integer block sums folded in a fixed order
    if kind == "block" and case["q8"]:
        # A last-bit change of the attention moves a rounded int8 here and there.
        return {"rel": 3e-4, "max": 2e-2}
    return {"rel": {"block": 1e-6, "encoder": 4e-6, "attention": 2e-6, "projection": 4e-6,
                    "gemm": 4e-6, "dpt": 1.6e-5, "rows": 5e-7}[kind]}


# ---- the same in float64 -----------------------------------------------------------


def _d(a, *shape):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV).double().reshape(shape)


def _ln(x, g, b, eps=da3.LN_EPS):
    mu = x.mean(-1, keepdim=True)
    return (x - mu) / torch.sqrt(((x - mu) ** 2).mean(-1, keepdim=True) + eps) * g + b


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _rope(z, pos, freq=da3.ROPE_FREQ):
    """z [heads, tokens, 64]; the rotation angles as the float32 path defines them."""
    inv = np.float32(freq) ** (-2.0 * np.arange(16, dtype=np.float32) / np.float32(32.0))
    z = z.clone()
    for ax in range(2):
        ang = _d(np.float32(pos.reshape(-1, 2)[:, ax:ax + 1]) * inv.astype(np.float32), -1, 16)
        sn, cs = torch.sin(ang), torch.cos(ang)
        a, b = z[..., 32 * ax:32 * ax + 16].clone(), z[..., 32 * ax + 16:32 * ax + 32].clone()
        z[..., 32 * ax:32 * ax + 16] = a * cs - b * sn
        z[..., 32 * ax + 16:32 * ax + 32] = b * cs + a * sn
    return z


def _attend(q, k, v, scale):
    out = []
    for h in range(q.shape[0]):  # a head at a time: the scores of all would be large
        out.append(torch.softmax((q[h] @ k[h].t()) * scale, -1) @ v[h])
    return torch.stack(out)


def _block_exact(x, w, images, t, pos):
    f = {n: _d(a, -1) for n, a in w.items()}
    qkv = _ln(x, f["ln1_gamma"], f["ln1_beta"]) @ f["w_qkv"].reshape(DIM, 3 * DIM) + f["b_qkv"]
    att = []
    for i in range(images):
        q, k, v = qkv[i * t:(i + 1) * t].reshape(t, 3, HEADS, 64).permute(1, 2, 0, 3)
        if "q_norm_gamma" in f:
            q = _ln(q, f["q_norm_gamma"], f["q_norm_beta"])
            k = _ln(k, f["k_norm_gamma"], f["k_norm_beta"])
        o = _attend(_rope(q, pos), _rope(k, pos), v, 0.125)
        att.append(o.permute(1, 0, 2).reshape(t, DIM))
    x = x + (torch.cat(att) @ f["w_proj"].reshape(DIM, DIM) + f["b_proj"]) * f["ls1"]
    h = _gelu(_ln(x, f["ln2_gamma"], f["ln2_beta"]) @ f["w_fc1"].reshape(DIM, MLP) + f["b_fc1"])
    return x + (h @ f["w_fc2"].reshape(MLP, DIM) + f["b_fc2"]) * f["ls2"]


def exact(case, seed):
    kind = case["kind"]
    if kind == "q8_linear" or (kind == "block" and case["q8"]):
        return None  # rounded to int8 on the way: the path's own arithmetic defines the result
    d = _inputs(case, seed)
    if kind == "block":
        t = case["rows"] * case["cols"] + 1
        return _block_exact(_d(d["x"], -1, DIM), d["w"][0], case["images"], t,
                            da3.positions_yx(case["rows"], case["cols"]))
    if kind == "encoder":
        r, c = case["rows"], case["cols"]
        t, pk = r * c + 1, 3 * PATCH * PATCH
        xs = []
        for p in d["pixels"]:
            img = _d(p, 3, r, PATCH, c, PATCH).permute(1, 3, 0, 2, 4).reshape(r * c, pk)
            e = img @ _d(d["embed_w"], pk, DIM) + _d(d["embed_b"], -1)
            xs.append(torch.cat([_d(d["cls"], 1, DIM), e]) + _d(d["pos"], t, DIM))
        x = torch.cat(xs)
        pos = da3.positions_yx(r, c)
        for w in d["w"]:
            x = _block_exact(x, w, case["images"], t, pos)
        return x
    if kind == "attention":
        h, t, hd = case["heads"], case["tokens"], case["head_dim"]
        o = _attend(*(_d(d[c], h, t, hd) for c in "qkv"), 1.0 / math.sqrt(hd))
        if hd == 64 and case["token_major"]:
            o = o.permute(1, 0, 2)
        return o.reshape(-1)
    if kind == "projection":
        m, k, n, mode = case["m"], case["k"], case["n"], case["mode"]
        y = _d(d["x"], m, k) @ _d(d["w"], k, n) + _d(d["b"], -1)
        if "g" in d:
            y = y * _d(d["g"], -1)
        if mode == "gelu":
            y = _gelu(y)
        if mode == "residual":
            return y + _d(d["r"], m, n)
        if mode == "qkv":
            return [z.reshape(-1) for z in y.reshape(m, 3, n // 192, 64).permute(1, 2, 0, 3)]
        return (y.t() if mode == "chw" else y).reshape(-1)
    if kind == "gemm":
        return _d(d["a"], case["m"], case["k"]) @ _d(d["b"], case["k"], case["n"])
    if kind == "dpt":
        F = torch.nn.functional
        r, c, f = case["rows"], case["cols"], case["features"]
        p = (_d(d["x"], r * c, DIM) @ _d(d["proj_w"], DIM, 96) + _d(d["proj_b"], -1)).t()
        # kernel == stride: one product per tap
        u = torch.einsum("iyx,iokl->oykxl", p.reshape(96, r, c), _d(d["up_w"], 96, 96, 4, 4))
        u = u.reshape(96, 4 * r, 4 * c) + _d(d["up_b"], 96, 1, 1)

        def conv(z, w, b, out_c):
            cols = F.unfold(z[None], 3, padding=1)[0]
            y = _d(w, out_c, -1) @ cols
            return (y if b is None else y + _d(b, out_c, 1)).reshape(out_c, *z.shape[1:])

        a = conv(u, d["rn_w"], None, f)
        b = conv(torch.relu(a), d["res_w"], d["res_b"], f) + a
        up = F.interpolate(b[None], size=(7 * r, 7 * c), mode="bilinear", align_corners=True)[0]
        return [b, conv(up, d["out_w"], d["out_b"], 32)]
    x = _ln(_d(d["x"], case["rows"], case["cols"]), _d(d["g"], -1), _d(d["b"], -1))
    return _gelu(x + _d(d["y"], case["rows"], case["cols"]))
