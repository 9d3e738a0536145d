"""The flash kernels' softmax state: two key parts per block (small grids) against one, at the edges of
tiles, parts and query blocks, and references that must agree between the two lanes of a query.

The reference is the same attention in float64 on the fp32 inputs. q, k, v and P are rounded to fp16
(2^-11 each): a score is off by about |q||k| 2^-11 / sqrt(D), which stays below 2^-9 for unit inputs,
and the output by that plus P's and v's rounding, under 2^-8 of its size in all.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(q, k, v, bias, start):
    """q [B, Lq, H, D], k and v [B, Lk, H, D] -> [B, Lq, H, D] in float64."""
    s = (q.double().transpose(1, 2).unsqueeze(3) * k.double().transpose(1, 2).unsqueeze(2)).sum(-1) / math.sqrt(q.shape[-1])
    if bias is not None:
        s[..., start:] += bias.double()[:, None, None, :]
    return (torch.softmax(s, -1).unsqueeze(-1) * v.double().transpose(1, 2).unsqueeze(2)).sum(3).transpose(1, 2)


def run(lib, q, k, v, bias=None, start=0):
    B, Lq, H, D = q.shape
    Lk = k.shape[1]
    o = torch.full((B, Lq + 3, H, D), 9.0, device=DEV)
    W = H * D
    lib.attention(q, k, v, o, Lq=Lq, Lk=Lk, H=H, D=D, ldq=W, ldk=W, ldv=W, ldo=W, batch=B, qBatch=Lq * W, kBatch=Lk * W,
                  vBatch=Lk * W, oBatch=(Lq + 3) * W, key_bias=bias, biasStart=start, biasBatch=Lk - start if bias is not None else 0)
    torch.cuda.synchronize()
    assert (o[:, Lq:] == 9.0).all(), "rows past Lq were written"
    return o[:, :Lq]


def check(got, ref, what):
    rel = ((got.double() - ref).norm() / ref.norm()).item()
    print(f"[parity] {what}: rel-L2 {rel:.2e}", flush=True)
    assert torch.isfinite(got).all() and rel <= 2.0**-8, what


# (batch, heads, queries): 64-query blocks in two parts, 128-query blocks in two parts, one part, wide
ROUTES = {"parts, 64 queries": (1, 4, 65), "parts, 128 queries": (2, 64, 129), "one part": (2, 120, 129), "wide": (2, 128, 65)}


@pytest.mark.parametrize("route", ROUTES)
@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_half_of_a_tile_vanishes(ns2lib, route, D):
    """The keys one lane of a query holds all underflow in the first tile, and no later score reaches the
    first tile's maximum: the lanes' references have to stay together all the same."""
    B, H, Lq = ROUTES[route]
    Lk = 256
    g = torch.Generator(device=DEV).manual_seed(D)
    v = torch.randn(B, Lk, H, D, generator=g, device=DEV)
    q = torch.ones(B, Lq, H, D, device=DEV)
    key = torch.arange(Lk, device=DEV)
    for lane in (0, 4):
        score = torch.where(key < 64, torch.where((key & 4) == lane, 0.0, -40.0), -3.0)  # of sqrt(D)-scaled q k
        k = (score / math.sqrt(D))[None, :, None, None].expand(B, Lk, H, D).contiguous()
        check(run(ns2lib, q, k, v), reference(q, k, v, None, 0), f"{route} D={D} lane bit {lane}")


@pytest.mark.parametrize("D", [32, 64, 96])
@pytest.mark.parametrize("Lq,Lk,start", [(1, 65, None), (63, 128, None), (64, 129, 65), (65, 129, 64), (33, 192, 100),
                                         (200, 193, 128), (17, 256, 255), (129, 257, 70), (64, 64, 10), (5, 449, 66)])
def test_key_parts(ns2lib, Lq, Lk, start, D):
    """Tiles that split evenly or not between the parts, and biases from the first key of a part on:
    text weights, keys masked by -inf and by the lowest fp32 value."""
    B, H = 2, 3
    g = torch.Generator(device=DEV).manual_seed(Lq + Lk + D)
    q, k, v = (torch.randn(B, L, H, D, generator=g, device=DEV) for L in (Lq, Lk, Lk))
    bias = None
    if start is not None:
        bias = torch.rand(B, Lk - start, generator=g, device=DEV).log()
        bias[0, ::2] = -math.inf
        bias[1, 1::3] = torch.finfo(torch.float32).min
    check(run(ns2lib, q, k, v, bias, start or 0), reference(q, k, v, bias, start or 0), f"{Lq}x{Lk} from {start} D={D}")


def test_key_parts_large_scores(ns2lib):
    """Scores far from 0 in both directions and different in each part (the merge weighs the parts)."""
    B, H, D, Lq, Lk = 1, 2, 96, 70, 330
    g = torch.Generator(device=DEV).manual_seed(1)
    v = torch.randn(B, Lk, H, D, generator=g, device=DEV)
    q = torch.ones(B, Lq, H, D, device=DEV)
    tile = torch.arange(Lk, device=DEV) // 64
    for even, odd in ((-300.0, -299.0), (250.0, 248.5), (-300.0, 200.0), (90.0, -90.0)):
        score = torch.where(tile % 2 == 0, even, odd) + (torch.arange(Lk, device=DEV) % 5) * 0.25
        k = (score / math.sqrt(D)).half().float()[None, :, None, None].expand(B, Lk, H, D).contiguous()
        check(run(ns2lib, q, k, v), reference(q, k, v, None, 0), f"scores {even} / {odd}")


@pytest.mark.parametrize("route", ROUTES)
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("low", [-3000.0, -1e9, -1e30])
def test_first_tiles_masked(ns2lib, route, D, low):
    """A finite low mask over whole key tiles in front of the others: the reference taken from them must not
    swallow the scores of the tiles behind (fp32 spacing at 1.4e9: 128)."""
    B, H, Lq = ROUTES[route]
    Lk = 300
    g = torch.Generator(device=DEV).manual_seed(D)
    q, k, v = (torch.randn(B, L, H, D, generator=g, device=DEV) for L in (Lq, Lk, Lk))
    key = torch.arange(Lk, device=DEV)
    for what, masked in (("first tile", key < 64), ("first two tiles", key < 128), ("even tiles", key // 64 % 2 == 0)):
        bias = torch.where(masked, low, 0.0).expand(B, Lk).contiguous()
        check(run(ns2lib, q, k, v, bias, 0), reference(q, k, v, bias, 0), f"{route} D={D} {what} masked by {low}")
