"""The one-launch linears of a short sequence (q|k|v with head norms, gate/up with GLU and down shares) at
their edges: row tiles with and without rows, two row tiles per block, chunks of one and five k-tiles, both
sides of the rules that choose between one launch and two (which of them ran is read back), the largest weight
slice of one launch, outputs that overlap the rows or the weights.

The operands are fp16 and given, the reference is float64: fp32 sums of K products are off by at most
sqrt(K) 2^-24 of the result's size (a random walk), values rounded to fp16 by 2^-11 of theirs.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-6


def tiled(x):
    """fp16 [M, K] -> the tiled operand [ceil(M/64)][K/64][8][64][8]; padding rows are NaN (never used)."""
    M, K = x.shape
    p = torch.full(((M + 63) // 64 * 64, K), math.nan, dtype=torch.float16, device=x.device)
    p[:M] = x
    return p.reshape(-1, 64, K // 64, 8, 8).permute(0, 2, 3, 1, 4).contiguous()


def weight(lib, N, K, g):
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    t = torch.empty_like(w)
    lib.tile_bf16_weight(w, t, N, K)
    return w.half().double(), t


def close(got, ref, tol, what):
    rel = ((got.double() - ref).norm() / ref.norm()).item()
    print(f"[parity] {what}: rel-L2 {rel:.2e} (tol {tol:.1e})", flush=True)
    assert torch.isfinite(got).all() and rel <= tol, what


SHAPES = [(1, 640), (16, 64), (17, 1920), (37, 640), (65, 1984), (128, 704), (256, 640), (257, 640), (300, 960), (272, 1024),
          (511, 320), (1024, 128), (1025, 640)]


@pytest.mark.parametrize("M,K", SHAPES)
@pytest.mark.parametrize("D,heads,H1,H2,bias", [(256, 6, 4, 1, False), (128, 5, 2, 2, True), (64, 3, 0, 1, False)])
def test_head_norm(ns2lib, M, K, D, heads, H1, H2, bias):
    print(f"[case] head norm {M}x{heads * D}x{K}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + K + D)
    N, rope = heads * D, M - M // 3
    x = torch.randn(M, K, generator=g, device=DEV).half()
    w, wt = weight(ns2lib, N, K, g)
    w1, w2 = (torch.randn(D, generator=g, device=DEV) for _ in range(2))
    b = torch.randn(N, generator=g, device=DEV) if bias else None
    ang = torch.rand(rope, D // 2, generator=g, device=DEV, dtype=torch.float64) * 6
    cs = torch.cat([ang.cos().reshape(-1), ang.sin().reshape(-1)]).float()
    c = torch.full((M + 2, N), 5.0, device=DEV)
    ldkv = (heads - H1) * D + 8
    kv = torch.full((M + 2, ldkv), 5.0, dtype=torch.float16, device=DEV)
    ns2lib.linear_f16w_tiled_head_norm_f16kv(tiled(x), wt, b, c, M, N, K, w1, H1, w2, H2, D, kv, ldkv, cs, rope * D // 2, rope, EPS)
    torch.cuda.synchronize()
    y = x.double() @ w.T
    if bias:
        y = y + b.double()
    y = y.reshape(M, heads, D)
    for h in range(H1 + H2):
        v = y[:, h]
        v = v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + EPS) * (w1 if h < H1 else w2).double()
        lo, hi = v[:rope, :D // 2], v[:rope, D // 2:]
        co, si = cs[:rope * D // 2].double().reshape(rope, -1), cs[rope * D // 2:].double().reshape(rope, -1)
        y[:, h] = torch.cat([torch.cat([lo * co - hi * si, hi * co + lo * si], 1), v[rope:]])
    if H1:
        close(c[:M, :H1 * D], y[:, :H1].reshape(M, -1), 2 * math.sqrt(max(K, 256)) * 2.0**-24, "q")
    close(kv[:M, :ldkv - 8].float(), y[:, H1:].reshape(M, -1), 2.0**-11, "k and v")
    assert (c[M:] == 5.0).all() and (c[:, H1 * D:] == 5.0).all() and (kv[M:] == 5.0).all() and (kv[:, ldkv - 8:] == 5.0).all()


@pytest.mark.parametrize("M,K", SHAPES)
@pytest.mark.parametrize("inner,Nd,act,bias", [(2048, 640, "gelu_tanh", False), (128, 64, "silu", True), (384, 1088, "none", False)])
def test_glu_down(ns2lib, M, K, inner, Nd, act, bias):
    print(f"[case] glu down {M}x{inner}x{K} -> {Nd}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + K + Nd)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    w, wt = weight(ns2lib, 2 * inner, K, g)
    wd, wdt = weight(ns2lib, Nd, inner, g)
    b = torch.randn(2 * inner, generator=g, device=DEV) if bias else None
    shares = inner // 128
    part = torch.full((shares * M + 1, Nd), 7.0, device=DEV)
    ns2lib.linear_f16w_tiled_glu_down(tiled(x), wt, b, M, 2 * inner, K, wdt, Nd, part, act=act)
    torch.cuda.synchronize()
    t = x.double() @ w.T
    if bias:
        t = t + b.double()
    f = {"gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh"), "silu": torch.nn.functional.silu, "none": lambda v: v}[act]
    y = f(t[:, :inner]) * t[:, inner:]
    assert (part[shares * M:] == 7.0).all()
    for s in range(shares):
        ref = y[:, 128 * s:128 * s + 128] @ wd[:, 128 * s:128 * s + 128].T
        close(part[s * M:s * M + M], ref, 2.0**-11, f"share {s}")


# M, D, heads, K of the q|k|v linear, or M, GLU columns, Nd, K: both sides of the rules that choose between one launch
# and two, with the largest weight slices that one launch takes
@pytest.mark.parametrize("one,M,D,heads,K", [(True, 16, 256, 6, 896), (False, 16, 256, 6, 1024), (True, 37, 64, 2, 960),
                                             (False, 37, 64, 2, 1024), (True, 256, 128, 8, 1472), (False, 256, 128, 8, 1536),
                                             (True, 257, 256, 6, 896), (False, 257, 256, 6, 960), (False, 300, 256, 1, 256)])
def test_head_norm_route(ns2lib, one, M, D, heads, K):
    ns2lib.profile_reset()
    ns2lib.profile(True)
    try:
        test_head_norm(ns2lib, M, K, D, heads, heads - 1, 0, True)
        names = ns2lib.profile_report()
    finally:
        ns2lib.profile(False)
    assert ("linear_head_norm_f16kv" in names) == one and ("head_norm_f16kv" in names) != one


@pytest.mark.parametrize("one,M,inner,Nd,K", [(True, 16, 2048, 640, 448), (False, 16, 2048, 640, 512), (True, 17, 8192, 64, 1024),
                                              (False, 17, 8192, 64, 1088), (False, 64, 256, 640, 576), (True, 65, 1024, 64, 1152),
                                              (False, 65, 1024, 64, 1216), (True, 65, 512, 64, 768), (False, 257, 256, 64, 384),
                                              (True, 257, 384, 64, 960), (True, 10, 6144, 64, 512)])
def test_glu_down_route(ns2lib, one, M, inner, Nd, K):
    ns2lib.profile_reset()
    ns2lib.profile(True)
    try:
        test_glu_down(ns2lib, M, K, inner, Nd, "silu", True)
        names = ns2lib.profile_report()
    finally:
        ns2lib.profile(False)
    assert ("linear_glu_down" in names) == one and ("glu_down" in names) != one


def test_outputs_over_the_rows(ns2lib):
    """An output that overlaps the tiled rows (only the last launch of a call may store)."""
    M, K, N, D = 100, 640, 1536, 256
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    _, wt = weight(ns2lib, N, K, g)
    w = torch.randn(D, generator=g, device=DEV)
    outs = []
    for shared in (False, True):
        a = tiled(x)
        c = torch.zeros(M, N, device=DEV)
        kv = torch.zeros(M, 2 * D, dtype=torch.float16, device=DEV)
        if shared:  # the rows start inside C
            c.view(-1).view(torch.float16)[4096:4096 + a.numel()] = a.reshape(-1)
            a = c.view(-1).view(torch.float16)[4096:4096 + a.numel()]
        ns2lib.linear_f16w_tiled_head_norm_f16kv(a, wt, None, c, M, N, K, w, 4, w, 1, D, kv, 2 * D)
        torch.cuda.synchronize()
        outs.append((c[:, :4 * D].clone(), kv))
    close(outs[1][0], outs[0][0].double(), 2.0**-19, "q over the rows")
    close(outs[1][1].float(), outs[0][1].double(), 2.0**-11, "k and v")


def test_outputs_over_the_weights(ns2lib):
    """An output that overlaps the weights, which only the first of two launches reads."""
    M, K, inner, Nd = 200, 640, 1024, 640
    g = torch.Generator(device=DEV).manual_seed(4)
    x = tiled(torch.randn(M, K, generator=g, device=DEV).half())
    _, wt = weight(ns2lib, 2 * inner, K, g)
    _, wdt = weight(ns2lib, Nd, inner, g)
    alone = torch.empty(inner // 128 * M, Nd, device=DEV)
    ns2lib.linear_f16w_tiled_glu_down(x, wt, None, M, 2 * inner, K, wdt, Nd, alone)
    part = torch.empty_like(alone)
    part.view(-1)[:wt.numel() // 2] = wt.reshape(-1).view(torch.float32)
    ns2lib.linear_f16w_tiled_glu_down(x, part, None, M, 2 * inner, K, wdt, Nd, part)
    torch.cuda.synchronize()
    close(part, alone.double(), 2.0**-11, "shares over the weights")
    w, c = torch.randn(256, generator=g, device=DEV), torch.empty(M, 2 * inner, device=DEV)
    kv, over = (torch.empty(M, 1024, dtype=torch.float16, device=DEV) for _ in range(2))
    ns2lib.linear_f16w_tiled_head_norm_f16kv(x, wt, None, c, M, 2 * inner, K, w, 4, w, 1, 256, kv, 1024)
    buf = wt.reshape(-1).view(torch.float16).clone()
    ns2lib.linear_f16w_tiled_head_norm_f16kv(x, buf, None, c, M, 2 * inner, K, w, 4, w, 1, 256, buf, 1024)
    torch.cuda.synchronize()
    over.copy_(buf[:M * 1024].reshape(M, 1024))
    close(over.float(), kv.double(), 2.0**-10, "k and v over the weights")
