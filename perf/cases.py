"""What this framework is used for, as timed cases over the C ABI (include/ns2.h through ns2.py).

Each case is a dict of plain values whose "kind" names the work:

  pass       one whole DiT pass on resident latent tokens (the order of js/nanosaur2.js)
  block      one image block of the pass: normMod, q|k|v, attention, projection, GLU MLP
  text       one text-refine block and what the pass takes from the text (keys/values, pooling)
  attention  the joint attention of fp32 q, k, v views with 2-D RoPE and text-key biases
  linear     one int8 ConvRot linear on fp32 activations (tiled or file-layout weight)
  adaln      the one-row bf16 projections that make the modulation vectors
  encode     the Gemma3 text encoder's 17 layers on embedded tokens

Sizes: latent grids of 832x1216, 768x768 and 512x512 images (1/16 of the image side), prompts of
up to 300 tokens, and whatever lies between; widths are those of the two models. Weights are
int8 in {-127..127} with row scales that keep activations near unit size, bf16 weights and norm
vectors as the checkpoints have them in magnitude; all drawn from the seed on the device.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "nanosaur2-web_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ns2  # noqa: E402

DEV = "cuda:0"
D, HEADS, HD, MLP, BLOCKS, JOINT, CH = 1536, 16, 96, 4096, 18, 9, 64
E, EH, EHD, EMLP, ELAYERS = 640, 4, 256, 2048, 17  # Gemma3: width, heads, head dim, MLP, layers run
EPS = 1e-6
RANK = 32


# ---- the cases ------------------------------------------------------------------------------

def listed():
    return [
        # the framework's headline: one denoising pass of an 832x1216 image, 256 prompt tokens
        {"name": "pass_832x1216", "kind": "pass", "h": 76, "w": 52, "T": 256},
        # the pass's joint block at that size: 9 of its 18 blocks
        {"name": "block_832x1216", "kind": "block", "h": 76, "w": 52, "T": 256, "lora": 0},
        # a preview-sized image (512x512) with a short prompt: few rows for 256 CUs
        {"name": "block_512x512", "kind": "block", "h": 32, "w": 32, "T": 77, "lora": 0},
        # an odd latent grid (no multiple of 16 rows) with a rank-32 LoRA on every linear
        {"name": "block_lora_752x976", "kind": "block", "h": 61, "w": 47, "T": 131, "lora": RANK},
        # the text side of a pass, once per step: an ordinary prompt
        {"name": "text_120", "kind": "text", "T": 120},
        # classifier-free guidance: both batch elements' joint attention in one call
        {"name": "attention_832x1216_pair", "kind": "attention", "batch": 2, "h": 76, "w": 52, "T": 256},
        # joint attention of a 768x768 image
        {"name": "attention_768x768", "kind": "attention", "batch": 1, "h": 48, "w": 48, "T": 128},
        # the MLP's second linear on 2304 image + 128 text rows, weight re-tiled at load
        {"name": "linear_down_2432", "kind": "linear", "M": 2432, "N": 1536, "K": 6144, "tiled": True},
        # the q|k|v linear on a file-layout weight (the reference's op sequence)
        {"name": "linear_qkv_rows_2432", "kind": "linear", "M": 2432, "N": 4608, "K": 1536, "tiled": False},
        # the smallest call of a pass: the shared and final adaLN projections, one row
        {"name": "adaln_12288", "kind": "adaln", "N": 12288},
        # a full prompt through the text encoder
        {"name": "encode_256", "kind": "encode", "L": 256},
        # a short prompt: launches and latency
        {"name": "encode_37", "kind": "encode", "L": 37},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "block", "text", "attention", "attention", "linear", "adaln", "encode"])
    if kind == "block":
        while True:
            h, w = _log_int(rng, 12, 84), _log_int(rng, 12, 84)
            if h * w <= 3952:
                return {"kind": kind, "h": h, "w": w, "T": rng.choice([0, _log_int(rng, 4, 300)]),
                        "lora": rng.choice([0, 0, RANK])}
    if kind == "text":
        return {"kind": kind, "T": _log_int(rng, 9, 300)}
    if kind == "attention":
        while True:
            h, w = _log_int(rng, 12, 84), _log_int(rng, 12, 84)
            if h * w <= 3952:
                return {"kind": kind, "batch": rng.choice([1, 2]), "h": h, "w": w, "T": _log_int(rng, 4, 256)}
    if kind == "linear":
        N, K = rng.choice([(4608, 1536), (1536, 1536), (6144, 1536), (8192, 1536), (1536, 4096), (1536, 6144)])
        return {"kind": kind, "M": _log_int(rng, 33, 4096), "N": N, "K": K, "tiled": rng.random() < 0.7}
    if kind == "adaln":
        return {"kind": kind, "N": rng.choice([1536, 3072, 9216, 12288, 18432])}
    return {"kind": kind, "L": _log_int(rng, 9, 300)}


# ---- inputs ---------------------------------------------------------------------------------

class _Rand:
    """Seeded tensors on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device=DEV) * std + mean

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def bf16(self, *shape, std):
        return self.normal(*shape, std=std).to(torch.bfloat16)

    def i8(self, N, K):
        """int8 rows and the scales that give outputs of about unit size for unit inputs."""
        q = torch.randint(-127, 128, (N, K), generator=self.g, device=DEV, dtype=torch.int8)
        return q, self.uniform(0.5, 1.5, N) / (73.3 * math.sqrt(K))


def _lib():
    lib = ns2.load(0)
    lib.set_stream(torch.cuda.current_stream().cuda_stream)
    return lib


def _f32(*shape):
    return torch.empty(*shape, device=DEV)


def _tiled(rows, cols):
    return torch.empty((rows + 63) // 64 * 64 * cols, dtype=torch.int16, device=DEV)


def _rope2d(h, w):
    """cos block then sin block, [h*w][HD/2] each: x on the first half of the pairs, y on the rest."""
    quarter = HD // 4
    f = 1.0 / 10000.0 ** (torch.arange(quarter, dtype=torch.float64) * 2 / (HD // 2))
    y, x = torch.meshgrid(torch.arange(h, dtype=torch.float64) - (h - 1) / 2,
                          torch.arange(w, dtype=torch.float64) - (w - 1) / 2, indexing="ij")
    a = torch.cat([x.reshape(-1, 1) * f, y.reshape(-1, 1) * f], 1)
    return torch.cat([a.cos().reshape(-1), a.sin().reshape(-1)]).float().to(DEV)


def _rope1d(L, theta):
    a = torch.arange(L, dtype=torch.float64).reshape(-1, 1) / theta ** (torch.arange(EHD // 2, dtype=torch.float64) * 2 / EHD)
    return torch.cat([a.cos().reshape(-1), a.sin().reshape(-1)]).float().to(DEV)


def _i8_weight(lib, r, N, K, glu=False, lora=0):
    """An int8 linear as the host keeps it: the re-tiled weight, its scales and its LoRA pair."""
    q, s = r.i8(N, K)
    wt = torch.empty_like(q)
    (lib.tile_i8_weight_glu if glu else lib.tile_i8_weight)(q, wt, N, K)
    pair = None
    if lora:
        pair = (r.normal(lora, K, std=1 / math.sqrt(K)).half(), r.normal(N, lora, std=0.3 / math.sqrt(lora)).half(), lora)
    return {"q": q, "s": s, "wt": wt, "N": N, "K": K, "lora": pair}


def _block_weights(lib, r, lora=0, glu=True):
    return {"n1": r.normal(D, std=0.1, mean=1.0), "n2": r.normal(D, std=0.1, mean=1.0),
            "qn": r.normal(HD, std=0.1, mean=1.0), "kn": r.normal(HD, std=0.1, mean=1.0),
            "qkv": _i8_weight(lib, r, 3 * D, D, lora=lora), "proj": _i8_weight(lib, r, D, D, lora=lora),
            "w12": _i8_weight(lib, r, 2 * MLP, D, glu=glu, lora=lora), "w3": _i8_weight(lib, r, D, MLP, lora=lora)}


def _drop_row_major(*weights):
    for W in weights:
        del W["q"]


def _bf16_tiled(lib, r, N, K, std):
    w = r.bf16(N, K, std=std)
    wt = torch.empty_like(w)
    lib.tile_bf16_weight(w, wt, N, K)
    return {"w": w, "wt": wt, "N": N, "K": K}


def _block_buffers(lib, L, T):
    vpk = None
    if L % 16 == 0:
        vpk = torch.empty(lib.attention_vpack_bytes(L + T, HEADS, HD) // 2, dtype=torch.int16, device=DEV)
    return {"nr": _tiled(L, D), "qkv": _f32(L, 3 * D), "a": _f32(L, D), "gr": _tiled(L, MLP), "vpk": vpk}


def _prompt(r, T):
    """Log prompt weights of T tokens."""
    return r.uniform(0.5, 1.5, T).log()


def _prepare_block(c, r):
    lib, L, T = _lib(), c["h"] * c["w"], c["T"]
    return {"lib": lib, "L": L, "T": T, "x0": r.normal(L, D), "x": _f32(L, D), "b": _block_weights(lib, r, c["lora"]),
            "mod": r.normal(6 * D, std=0.3), "kv_text": r.normal(T, JOINT * 2 * D) if T else None,
            "bias": _prompt(r, T) if T else None, "cs": _rope2d(c["h"], c["w"]), "slot": 2 * D * (JOINT // 2),
            "buf": _block_buffers(lib, L, T)}


def _prepare_text(c, r):
    lib, T = _lib(), c["T"]
    return {"lib": lib, "T": T, "x0": r.normal(T, D), "x": _f32(T, D), "b": _block_weights(lib, r, glu=False),
            "kv": _i8_weight(lib, r, JOINT * 2 * D, D), "mod": r.normal(6 * D, std=0.3), "pool": r.uniform(0.5, 1.5, T),
            "buf": _text_buffers(T)}


def _text_buffers(T):
    return {"nr": _tiled(T, D), "qkv": _f32(T, 3 * D), "a": _f32(T, D), "h": _f32(T, 2 * MLP), "gr": _tiled(T, MLP),
            "kv_text": _f32(T, JOINT * 2 * D), "pooled": _f32(D)}


def _prepare_attention(c, r):
    L, Lk, B = c["h"] * c["w"], c["h"] * c["w"] + c["T"], c["batch"]
    return {"lib": _lib(), "c": c, "L": L, "Lk": Lk, "q": r.normal(B, L, D), "k": r.normal(B, Lk, D),
            "v": r.normal(B, Lk, D), "bias": _prompt(r, B * c["T"]).reshape(B, -1), "cs": _rope2d(c["h"], c["w"]),
            "o": _f32(B, L, D)}


def _prepare_linear(c, r):
    lib, M, N, K = _lib(), c["M"], c["N"], c["K"]
    s = {"lib": lib, "c": c, "x": r.normal(M, K), "y": _f32(M, N)}
    if c["tiled"]:
        s["W"] = _i8_weight(lib, r, N, K)
        s["xr"] = _tiled(M, K)
    else:
        q, sc = r.i8(N, K)
        s["W"] = {"q": q, "s": sc}
    return s


def _prepare_adaln(c, r):
    return {"lib": _lib(), "N": c["N"], "x": r.normal(1, D, std=0.6), "W": r.bf16(c["N"], D, std=0.02), "y": _f32(1, c["N"])}


def _prepare_encode(c, r):
    lib, L = _lib(), c["L"]
    layers = []
    for i in range(ELAYERS):
        W = {n: r.normal(E, std=0.1, mean=1.0) for n in ("in", "post_attn", "pre_mlp", "post_mlp")}
        W.update({n: r.normal(EHD, std=0.1, mean=1.0) for n in ("qn", "kn")})
        W["qkv"] = _bf16_tiled(lib, r, (EH + 2) * EHD, E, 0.03)
        W["o"] = _bf16_tiled(lib, r, E, EH * EHD, 0.03)
        W["gate_up"] = _bf16_tiled(lib, r, 2 * EMLP, E, 0.03)
        W["down"] = _bf16_tiled(lib, r, E, EMLP, 0.03)
        W["global"] = (i + 1) % 6 == 0
        layers.append(W)
    return {"lib": lib, "L": L, "x0": r.normal(L, E), "x": _f32(L, E), "layers": layers, "norm": r.normal(E, std=0.1, mean=1.0),
            "cs": (_rope1d(L, 1e4), _rope1d(L, 1e6)), "h": _f32(L, E), "ht": _tiled(L, E), "qkv": _f32(L, (EH + 2) * EHD),
            "part_o": _f32(EH, L, E), "part_d": _f32(EMLP // 128, L, E), "out": _f32(L, E)}


def _prepare_pass(c, r):
    lib, L, T = _lib(), c["h"] * c["w"], c["T"]
    s = {"lib": lib, "L": L, "T": T, "tokens": r.normal(L, CH), "y": r.normal(T, D), "temb": r.uniform(-1, 1, 1, 256),
         "bias": _prompt(r, T), "pool": r.uniform(0.5, 1.5, T), "cs": _rope2d(c["h"], c["w"]),
         "embed": _bf16_tiled(lib, r, D, CH, 0.125), "sprint": _bf16_tiled(lib, r, D, D, 0.01),
         "final": _bf16_tiled(lib, r, CH, D, 0.025), "t1": r.bf16(D, 256, std=0.06), "t2": r.bf16(D, D, std=0.025),
         "pool_w": r.bf16(D, D, std=0.02), "text_ada": r.bf16(2 * 6 * D, D, std=0.01), "cond_ada": r.bf16(8 * D, D, std=0.01),
         "offsets": r.normal(BLOCKS, 6 * D, std=0.1), "text": [_block_weights(lib, r, glu=False) for _ in range(2)],
         "blocks": [_block_weights(lib, r) for _ in range(BLOCKS)], "kv": _i8_weight(lib, r, JOINT * 2 * D, D)}
    for b in s["text"] + s["blocks"]:
        _drop_row_major(b["qkv"], b["proj"], b["w12"], b["w3"])
    _drop_row_major(s["kv"])
    s["buf"] = _block_buffers(lib, L, T)
    s["tbuf"] = _text_buffers(T)
    s["tt"], s["x"], s["g"], s["d"], s["n"], s["out"] = (_tiled(L, CH), _f32(L, D), _f32(L, D), _tiled(L, D), _tiled(L, D),
                                                        _f32(L, CH))
    s["th"], s["t"], s["tc"], s["tmods"], s["txt"] = _f32(D), _f32(D), _f32(D), _f32(2 * 6 * D), _f32(T, D)
    s["ada"], s["mods"] = _f32(8 * D), _f32(BLOCKS, 6 * D)
    return s


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, _Rand(seed))
    state["kind"] = case["kind"]
    return state


# ---- one pass of each kind --------------------------------------------------------------------

def _attend(lib, buf, L, T, b, cs, kv_text, slot, bias, vpk):
    """Joint (or, without text, image-only) attention over the q|k|v rows, the text keys and
    values read from the stacked projection."""
    view = dict(Lq=L, Lk=L + T, H=HEADS, D=HD, ldq=3 * D, ldk=3 * D, ldv=3 * D, ldo=D, kOff=D, vOff=2 * D,
                key_bias=bias, biasStart=L, q_norm=b["qn"], k_norm=b["kn"], eps=EPS, rope_cs=cs,
                sin_off=L * HD // 2 if cs is not None else 0, rope_rows=L if cs is not None else 0)
    if T:
        at = kv_text.data_ptr() + 4 * slot
        view.update(k_text=at, v_text=at + 4 * D, ld_text=kv_text.shape[1], text_start=L)
    qkv, a = buf["qkv"], buf["a"]
    if vpk is not None:
        lib.attention_vpacked(qkv, qkv, qkv, a, vpk, L, **view)
    elif T:
        lib.attention_text(qkv, qkv, qkv, a, **view)
    else:
        lib.attention(qkv, qkv, qkv, a, **view)


def _block(lib, x, L, T, b, mod, cs, kv_text, slot, bias, buf):
    nr, qkv, a, gr, vpk = buf["nr"], buf["qkv"], buf["a"], buf["gr"], buf["vpk"]
    W = b["qkv"]
    lib.norm_mod_rotate_f16(x, mod, 0, D, L, D, b["n1"], nr, EPS, tiled=True)
    if vpk is not None:
        lib.linear_i8_tiled_vpack(nr, W["wt"], W["s"], qkv, L, 3 * D, D, vpk, vcol0=2 * D, H=HEADS, D=HD, Lk=L + T,
                                  lora=W["lora"])
    else:
        lib.linear_i8_tiled(nr, W["wt"], W["s"], qkv, L, 3 * D, D, lora=W["lora"])
    _attend(lib, buf, L, T, b, cs, kv_text, slot, bias, vpk)
    W = b["proj"]
    lib.rotate_f16(a, D, nr, D, L, D, tiled=True)
    lib.linear_i8_tiled(nr, W["wt"], W["s"], x, L, D, D, resid=True, gate=mod, gOff=2 * D, lora=W["lora"])
    W = b["w12"]
    lib.norm_mod_rotate_f16(x, mod, 3 * D, 4 * D, L, D, b["n2"], nr, EPS, tiled=True)
    lib.linear_i8_glu_rot_tiled(nr, W["wt"], W["s"], gr, L, 2 * MLP, D, act="silu", lora=W["lora"])
    W = b["w3"]
    lib.linear_i8_tiled(gr, W["wt"], W["s"], x, L, D, MLP, resid=True, gate=mod, gOff=5 * D, lora=W["lora"])


def _text_block(lib, x, T, b, mod, buf):
    nr, qkv, a, h, gr = buf["nr"], buf["qkv"], buf["a"], buf["h"], buf["gr"]
    lib.norm_mod_rotate_f16(x, mod, 0, D, T, D, b["n1"], nr, EPS, tiled=True)
    lib.linear_i8_tiled(nr, b["qkv"]["wt"], b["qkv"]["s"], qkv, T, 3 * D, D)
    _attend(lib, buf, T, 0, b, None, None, 0, None, None)
    lib.rotate_f16(a, D, nr, D, T, D, tiled=True)
    lib.linear_i8_tiled(nr, b["proj"]["wt"], b["proj"]["s"], x, T, D, D, resid=True, gate=mod, gOff=2 * D)
    lib.norm_mod_rotate_f16(x, mod, 3 * D, 4 * D, T, D, b["n2"], nr, EPS, tiled=True)
    lib.linear_i8_tiled(nr, b["w12"]["wt"], b["w12"]["s"], h, T, 2 * MLP, D)
    lib.glu_rotate_f16(h, gr, T, MLP, "silu", tiled=True)
    lib.linear_i8_tiled(gr, b["w3"]["wt"], b["w3"]["s"], x, T, D, MLP, resid=True, gate=mod, gOff=5 * D)


def _text_outputs(lib, x, T, kv, pool, buf):
    """What the pass takes from the refined text: every joint block's keys and values, the pooled row."""
    lib.rotate_f16(x, D, buf["nr"], D, T, D, tiled=True)
    lib.linear_i8_tiled(buf["nr"], kv["wt"], kv["s"], buf["kv_text"], T, kv["N"], D)
    lib.row_sum(x, pool, buf["pooled"], T, D, 1.0 / T)


def _run_block(s):
    lib = s["lib"]
    lib.elementwise("copy", s["x0"], None, s["x"], s["L"] * D)
    _block(lib, s["x"], s["L"], s["T"], s["b"], s["mod"], s["cs"], s["kv_text"], s["slot"], s["bias"], s["buf"])
    return s["x"]


def _run_text(s):
    lib, T = s["lib"], s["T"]
    lib.elementwise("copy", s["x0"], None, s["x"], T * D)
    _text_block(lib, s["x"], T, s["b"], s["mod"], s["buf"])
    _text_outputs(lib, s["x"], T, s["kv"], s["pool"], s["buf"])
    return [s["x"], s["buf"]["kv_text"], s["buf"]["pooled"]]


def _run_attention(s):
    c, L, Lk = s["c"], s["L"], s["Lk"]
    s["lib"].attention(s["q"], s["k"], s["v"], s["o"], Lq=L, Lk=Lk, H=HEADS, D=HD, ldq=D, ldk=D, ldv=D, ldo=D,
                       batch=c["batch"], qBatch=L * D, kBatch=Lk * D, vBatch=Lk * D, oBatch=L * D, key_bias=s["bias"],
                       biasStart=L, biasBatch=c["T"], rope_cs=s["cs"], sin_off=L * HD // 2, rope_rows=L)
    return s["o"]


def _run_linear(s):
    lib, c, W = s["lib"], s["c"], s["W"]
    M, N, K = c["M"], c["N"], c["K"]
    if c["tiled"]:
        lib.rotate_f16(s["x"], K, s["xr"], K, M, K, tiled=True)
        lib.linear_i8_tiled(s["xr"], W["wt"], W["s"], s["y"], M, N, K)
    else:
        lib.linear_i8(s["x"], 0, K, W["q"], W["s"], s["y"], M, N, K)
    return s["y"]


def _run_adaln(s):
    s["lib"].linear_bf16(s["x"], D, s["W"], s["y"], 1, s["N"], D)
    return s["y"]


def _run_encode(s):
    lib, L, x, ht, qkv = s["lib"], s["L"], s["x"], s["ht"], s["qkv"]
    layers, width = s["layers"], (EH + 2) * EHD
    kv16 = qkv.data_ptr() + 4 * EH * EHD  # k and v as fp16 in the front of their fp32 columns
    lib.elementwise("copy", s["x0"], None, x, L * E)
    lib.rmsnorm(x, layers[0]["in"], s["h"], L, E, EPS)
    lib.to_tiled_f16(s["h"], E, ht, L, E)
    for i, W in enumerate(layers):
        cs = s["cs"][1 if W["global"] else 0]
        lib.linear_f16w_tiled_head_norm_f16kv(ht, W["qkv"]["wt"], None, qkv, L, width, E, W["qn"], EH, W["kn"], 1, EHD,
                                              kv16, 2 * width, cs, L * EHD // 2, L, EPS)
        lib.attention_rows_f16kv_oproj(qkv, qkv, qkv, W["o"]["wt"], s["part_o"], Lq=L, Lk=L, H=EH, D=EHD, ldq=width,
                                       ldk=2 * width, ldv=2 * width, N=E, kOff=2 * EH * EHD, vOff=2 * EH * EHD + EHD,
                                       group=EH, causal=True)
        lib.parts_add_rmsnorm_tiled(s["part_o"], EH, None, x, W["post_attn"], W["pre_mlp"], ht, L, E, EPS)
        lib.linear_f16w_tiled_glu_down(ht, W["gate_up"]["wt"], None, L, 2 * EMLP, E, W["down"]["wt"], E, s["part_d"])
        if i + 1 < len(layers):
            lib.parts_add_rmsnorm_tiled(s["part_d"], EMLP // 128, None, x, W["post_mlp"], layers[i + 1]["in"], ht, L, E, EPS)
        else:
            lib.parts_add_rmsnorm(s["part_d"], EMLP // 128, None, x, W["post_mlp"], s["norm"], s["out"], L, E, EPS)
    return s["out"]


def _run_pass(s):
    lib, L, T, x, g = s["lib"], s["L"], s["T"], s["x"], s["g"]
    W = s["embed"]
    lib.to_tiled_f16(s["tokens"], CH, s["tt"], L, CH)
    lib.linear_f16w_tiled(s["tt"], W["wt"], x, L, D, CH)
    # conditioning: timestep embedding, refined text, pooled text, modulations of every block
    lib.linear_bf16(s["temb"], 256, s["t1"], s["th"], 1, D, 256, act="silu")
    lib.linear_bf16(s["th"], D, s["t2"], s["t"], 1, D, D)
    lib.elementwise("silu", s["t"], None, s["tc"], D)
    lib.elementwise("copy", s["y"], None, s["txt"], T * D)
    lib.linear_bf16(s["tc"], D, s["text_ada"], s["tmods"], 1, 2 * 6 * D, D)
    for i, b in enumerate(s["text"]):
        _text_block(lib, s["txt"], T, b, s["tmods"][i * 6 * D:], s["tbuf"])
    _text_outputs(lib, s["txt"], T, s["kv"], s["pool"], s["tbuf"])
    lib.linear_bf16(s["tbuf"]["pooled"], D, s["pool_w"], s["t"], 1, D, D, resid=True)
    lib.elementwise("silu", s["t"], None, s["tc"], D)
    lib.linear_bf16(s["tc"], D, s["cond_ada"], s["ada"], 1, 8 * D, D)
    lib.add_rows(s["ada"], s["offsets"], s["mods"], BLOCKS, 6 * D)

    def block(i, stream):
        joint = i % 2 == 0
        _block(lib, stream, L, T if joint else 0, s["blocks"][i], s["mods"][i], s["cs"], s["tbuf"]["kv_text"],
               2 * D * (i // 2), s["bias"] if joint else None, s["buf"])

    for i in range(2):
        block(i, x)
    lib.elementwise("copy", x, None, g, L * D)
    for i in range(2, BLOCKS - 2):
        block(i, g)
    W = s["sprint"]
    lib.to_tiled_f16(g, D, s["d"], L, D, sub=x, ldsub=D)
    lib.linear_f16w_tiled(s["d"], W["wt"], x, L, D, D, resid=True)
    for i in range(BLOCKS - 2, BLOCKS):
        block(i, x)
    W = s["final"]
    lib.norm_mod_f16(x, s["ada"][6 * D:], 0, D, L, D, None, s["n"], EPS)
    lib.linear_f16w_tiled(s["n"], W["wt"], s["out"], L, CH, D)
    return s["out"]


def run(state):
    state["lib"].set_stream(torch.cuda.current_stream().cuda_stream)
    return _RUN[state["kind"]](state)


# ---- the work a pass cannot do without ----------------------------------------------------------

def _block_work(L, T):
    weights = D * 3 * D + D * D + D * 2 * MLP + MLP * D
    return 2 * L * weights + 4 * L * (L + T) * D, weights


def work(case):
    c, kind = case, case["kind"]
    if kind in ("block", "pass"):
        L, T = c["h"] * c["w"], c["T"]
        flops, weights = _block_work(L, T)
        if kind == "block":
            lora = 2 * L * c["lora"] * (4 * D + D + MLP + 4 * D + 2 * MLP + D)
            return {"bytes": 8 * L * D + weights + 4 * T * 2 * D, "flops": flops + lora}
        image_only, _ = _block_work(L, 0)
        tflops, tweights = _block_work(T, 0)
        flops = JOINT * flops + (BLOCKS - JOINT) * image_only + 2 * tflops + 2 * T * D * JOINT * 2 * D
        flops += 2 * L * (CH * D + D * D + D * CH) + 2 * D * (256 + D + D + 20 * D)
        nbytes = (BLOCKS * weights + 2 * tweights + JOINT * 2 * D * D + 2 * (2 * CH * D + D * D) + 2 * D * (256 + 2 * D + 20 * D)
                  + 8 * L * CH + 4 * T * D)
        return {"bytes": nbytes, "flops": flops}
    if kind == "text":
        flops, weights = _block_work(c["T"], 0)
        kv = JOINT * 2 * D
        return {"bytes": 8 * c["T"] * D + weights + kv * D + 4 * c["T"] * kv, "flops": flops + 2 * c["T"] * D * kv}
    if kind == "attention":
        L, Lk, B = c["h"] * c["w"], c["h"] * c["w"] + c["T"], c["batch"]
        return {"bytes": 4 * B * D * (2 * L + 2 * Lk), "flops": 4 * B * L * Lk * D}
    if kind == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": 4 * M * K + N * K + 4 * M * N, "flops": 2 * M * N * K}
    if kind == "adaln":
        return {"bytes": 2 * c["N"] * D + 4 * c["N"], "flops": 2 * c["N"] * D}
    L = c["L"]
    weights = E * (EH + 2) * EHD + EH * EHD * E + E * 2 * EMLP + EMLP * E
    return {"bytes": ELAYERS * 2 * weights + 8 * L * E, "flops": ELAYERS * (2 * L * weights + 2 * L * L * EH * EHD)}


# ---- results ------------------------------------------------------------------------------------

def tolerance(case):
    # fp16 operands with fp32 sums (2^-11 per product input), fp32 elsewhere; about four times the
    # error against exact() (relative: linear 2.1e-4, attention 4.2e-4, block 1.1e-4, encode 1e-3)
    return {"pass": {"rel": 4e-3, "max": 0.03}, "block": {"rel": 4.5e-4, "max": 0.006}, "text": {"rel": 1e-3, "max": 0.006},
            "attention": {"rel": 1.7e-3, "max": 0.015}, "linear": {"rel": 8.5e-4, "max": 0.006},
            "adaln": {"rel": 1e-5, "max": 5e-5}, "encode": {"rel": 4e-3, "max": 0.02}}[case["kind"]]


def _had256():
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device=DEV)
    h = h4
    for _ in range(3):
        h = torch.kron(h, h4)
    return h / 16


def _x_i8(x, W, had):
    """The int8 linear in float64: rotate x per 256 columns, multiply, scale, add the LoRA term."""
    xr = (x.reshape(x.shape[0], -1, 256) @ had).reshape(x.shape)
    y = (xr @ W["q"].double().T) * W["s"].double()
    if W["lora"] is not None:
        y += xr @ W["lora"][0].double().T @ W["lora"][1].double().T
    return y


def _x_rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _x_norm_mod(x, w, mod, shift, scale):
    m = mod.double()
    return _x_rms(x, w) * (1 + m[scale:scale + D]) + m[shift:shift + D]


def _x_rope(x, cs, rows):
    """Split-half RoPE on the first `rows` rows of x [rows.., heads, dim]."""
    half = x.shape[-1] // 2
    n = rows * half
    c, s = cs[:n].double().reshape(rows, 1, half), cs[n:].double().reshape(rows, 1, half)
    a, b = x[:rows, :, :half], x[:rows, :, half:]
    return torch.cat([torch.cat([a * c - b * s, b * c + a * s], -1), x[rows:]], 0)


def _x_attention(q, k, v, bias=None, causal=False):
    """q [L, H, d], k and v [Lk, H, d] -> [L, H*d], one head at a time."""
    out = []
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h].T / math.sqrt(q.shape[-1])
        if bias is not None:
            s = s + bias
        if causal:
            s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
        out.append(torch.softmax(s, -1) @ v[:, h])
    return torch.cat(out, -1)


def _x_block(x, b, mod, cs, k_text, v_text, bias, had):
    L = x.shape[0]
    qkv = _x_i8(_x_norm_mod(x, b["n1"], mod, 0, D), b["qkv"], had).reshape(L, 3, HEADS, HD)
    q, k, v = _x_rms(qkv[:, 0], b["qn"]), _x_rms(qkv[:, 1], b["kn"]), qkv[:, 2]
    if cs is not None:
        q, k = _x_rope(q, cs, L), _x_rope(k, cs, L)
    if k_text is not None:
        T = k_text.shape[0]
        k = torch.cat([k, _x_rms(k_text.double().reshape(T, HEADS, HD), b["kn"])])
        v = torch.cat([v, v_text.double().reshape(T, HEADS, HD)])
        bias = torch.cat([torch.zeros(L, dtype=torch.float64, device=DEV), bias.double()])
    gate = mod.double()
    x = x + gate[2 * D:3 * D] * _x_i8(_x_attention(q, k, v, bias), b["proj"], had)
    h = _x_i8(_x_norm_mod(x, b["n2"], mod, 3 * D, 4 * D), b["w12"], had)
    act = torch.nn.functional.silu(h[:, :MLP]) * h[:, MLP:]
    return x + gate[5 * D:6 * D] * _x_i8(act, b["w3"], had)


def _x_encode(s):
    x, L = s["x0"].double(), s["L"]
    for W in s["layers"]:
        qkv = (_x_rms(x, W["in"]) @ W["qkv"]["w"].double().T).reshape(L, EH + 2, EHD)
        cs = s["cs"][1 if W["global"] else 0]
        q, k = _x_rope(_x_rms(qkv[:, :EH], W["qn"]), cs, L), _x_rope(_x_rms(qkv[:, EH:EH + 1], W["kn"]), cs, L)
        a = _x_attention(q, k.expand(-1, EH, -1), qkv[:, EH + 1:].expand(-1, EH, -1), causal=True)
        x = x + _x_rms(a @ W["o"]["w"].double().T, W["post_attn"])
        t = _x_rms(x, W["pre_mlp"]) @ W["gate_up"]["w"].double().T
        y = torch.nn.functional.gelu(t[:, :EMLP], approximate="tanh") * t[:, EMLP:]
        x = x + _x_rms(y @ W["down"]["w"].double().T, W["post_mlp"])
    return _x_rms(x, s["norm"])


def exact(case, seed):
    kind = case["kind"]
    if kind == "pass":
        return None  # 18 blocks in float64 take too long; its block is a case of its own
    s = prepare(case, seed)
    if kind == "block":
        k = v = None
        if s["T"]:
            k, v = s["kv_text"][:, s["slot"]:s["slot"] + D], s["kv_text"][:, s["slot"] + D:s["slot"] + 2 * D]
        return _x_block(s["x0"].double(), s["b"], s["mod"], s["cs"], k, v, s["bias"], _had256())
    if kind == "text":
        had = _had256()
        x = _x_block(s["x0"].double(), s["b"], s["mod"], None, None, None, None, had)
        return [x, _x_i8(x, s["kv"], had), s["pool"].double() @ x / s["T"]]
    if kind == "attention":
        out = []
        for b in range(case["batch"]):
            q, k, v = (t[b].double().reshape(-1, HEADS, HD) for t in (s["q"], s["k"], s["v"]))
            bias = torch.cat([torch.zeros(s["L"], dtype=torch.float64, device=DEV), s["bias"][b].double()])
            out.append(_x_attention(_x_rope(q, s["cs"], s["L"]), _x_rope(k, s["cs"], s["L"]), v, bias))
        return torch.stack(out)
    if kind == "linear":
        W = {"q": s["W"]["q"], "s": s["W"]["s"], "lora": None}
        return _x_i8(s["x"].double(), W, _had256())
    if kind == "adaln":
        return s["x"].double() @ s["W"].double().T
    return _x_encode(s)


_PREPARE = {"pass": _prepare_pass, "block": _prepare_block, "text": _prepare_text, "attention": _prepare_attention,
            "linear": _prepare_linear, "adaln": _prepare_adaln, "encode": _prepare_encode}
_RUN = {"pass": _run_pass, "block": _run_block, "text": _run_text, "attention": _run_attention, "linear": _run_linear,
        "adaln": _run_adaln, "encode": _run_encode}
