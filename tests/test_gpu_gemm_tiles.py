"""The block tiles of the tiled int8 / fp16 linears at their edges: ragged last rows and columns, the
shortest K, split K, old outputs, the LoRA term, the activations and the packed values, each at a size whose
launch takes the named tile (asked of the library, which chooses it by a time model).

The operands are given (fp16 activations, int8 weights), so the reference is the same product in
float64 and the only error is that of fp32 sums: the K products of an output are added in fp32, a
random walk of at most sqrt(K) 2^-24 of the result's size (4.7e-6 at K = 6144).
"""

import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def tiled(x):
    """fp16 [M, K] -> the tiled operand [ceil(M/64)][K/64][8][64][8], padding rows zero."""
    M, K = x.shape
    p = torch.zeros((M + 63) // 64 * 64, K, dtype=torch.float16, device=x.device)
    p[:M] = x
    return p.reshape(-1, 64, K // 64, 8, 8).permute(0, 2, 3, 1, 4).contiguous()


def tile_of(lib, ops, M, N, K, act="none", resid=False, rank=0, packed=False):
    """The block tile and K splits of a linear; ops: 0 int8 tiles, 1 fp16 tiles, 2 row-major operands."""
    fn, splits = lib.dll.ns2_internal_tile, ctypes.c_int()
    fn.restype = ctypes.c_char_p
    name = fn(ops, M, N, K, {"none": 0, "silu": 1, "gelu_tanh": 2}[act], int(resid), rank, int(packed), ctypes.byref(splits))
    return name.decode(), splits.value


def close(got, ref, K, what):
    rel = ((got.double() - ref).norm() / ref.norm()).item()
    print(f"[parity] {what}: rel-L2 {rel:.2e}", flush=True)
    assert torch.isfinite(got).all() and rel <= math.sqrt(K) * 2.0**-24, what


def assert_tile(lib, tile, ops, M, N, K, **form):
    name, splits = tile_of(lib, ops, M, N, K, **form)
    assert name == tile.split()[0] and (splits > 1) == ("split" in tile), (name, splits)


CASES = [
    # tile, M, N, K, resid, LoRA rank; K2: two k groups, S3: three stages
    ("64x64", 33, 1536, 256, False, 0),
    ("64x64 split K", 65, 1536, 4096, True, 0),
    ("64x64", 120, 1536, 6144, False, 32),
    ("64x64 split K", 120, 1536, 6144, False, 0),
    ("64x64", 64, 64, 1536, True, 32),
    ("64x128K2", 1501, 1536, 1536, True, 0),
    ("64x128K2", 1460, 1536, 1536, False, 32),
    ("64x128K2S3", 1025, 1536, 1536, True, 0),
    ("64x128K2S3", 999, 1536, 1536, False, 32),
    ("64x128K2S3", 1000, 1472, 1536, False, 0),
    ("64x128K2", 511, 4672, 1536, False, 0),
    ("64x128K2", 513, 4672, 1536, True, 32),
    ("64x128", 257, 4608, 256, False, 0),
    ("64x128", 257, 4608, 256, True, 32),
    ("128x128", 1537, 4672, 1536, False, 0),
    ("128x128", 1800, 4608, 256, False, 32),
    ("128x192", 2305, 4672, 1536, False, 0),
    ("128x192", 2433, 4608, 1536, True, 32),
    ("128x192K2", 3951, 1536, 4096, True, 0),
    ("128x192K2", 2867, 1600, 6144, False, 32),
    ("128x128", 3951, 4672, 1536, False, 0),
    ("64x128", 3800, 4608, 256, False, 0),
    ("192x384", 3329, 4672, 1536, False, 0),
    ("256x256", 1501, 8256, 512, False, 0),
]


@pytest.mark.parametrize("tile,M,N,K,resid,rank", CASES)
def test_i8_tiles(ns2lib, tile, M, N, K, resid, rank):
    print(f"[case] {tile} {M}x{N}x{K} resid {resid} rank {rank}", flush=True)
    assert_tile(ns2lib, tile, 0, M, N, K, resid=resid, rank=rank)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
    bias = torch.randn(N, generator=g, device=DEV)
    gate = torch.randn(N, generator=g, device=DEV)
    wt = torch.empty_like(q)
    ns2lib.tile_i8_weight(q, wt, N, K)
    ref = (x.double() @ q.double().T) * s.double() + bias.double()
    lora = None
    if rank:
        a = (torch.randn(rank, K, generator=g, device=DEV) / math.sqrt(K)).half()
        b = (torch.randn(N, rank, generator=g, device=DEV) / math.sqrt(rank)).half()
        lora = (a, b, rank)
        # the term's own rounding: t = x a^T is rounded to fp16 for the second product
        ref = ref + (x.double() @ a.double().T).half().double() @ b.double().T
    buf = torch.randn(M + 300, N, generator=g, device=DEV)
    before = buf.clone()
    ns2lib.linear_i8_tiled(tiled(x), wt, s, buf, M, N, K, bias=bias, resid=resid, gate=gate if resid else None, lora=lora)
    torch.cuda.synchronize()
    assert torch.equal(buf[M:], before[M:]), "rows past M were written"
    if resid:
        ref = before[:M].double() + gate.double() * ref
    if rank:
        # t computed in fp32 may round to the other fp16 neighbour: 2^-11 of the term in few places
        rel = ((buf[:M].double() - ref).norm() / ref.norm()).item()
        assert rel <= 2.0**-12, f"{tile}: {rel:.2e}"
    else:
        close(buf[:M], ref, K, f"{tile} {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [(40, 64, 256), (40, 128, 4096), (70, 12288, 512)])
def test_rows_far_apart(ns2lib, M, N, K):
    """Old outputs and stores where 31 output rows span more than 2^31 (70 rows) or 2^32 (40 rows) elements, in
    20 GB that are never filled."""
    ldc = (1 << (32 if M == 40 else 31)) // 31 + 64
    buf = torch.empty(M * ldc, device=DEV)
    c = buf.as_strided((M, N), (ldc, 1))
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
    wt = torch.empty_like(q)
    ns2lib.tile_i8_weight(q, wt, N, K)
    old = torch.randn(M, N, generator=g, device=DEV)
    c.copy_(old)
    ns2lib.linear_i8_tiled(tiled(x), wt, s, buf, M, N, K, ldc=ldc, resid=True)
    torch.cuda.synchronize()
    close(c.contiguous(), old.double() + (x.double() @ q.double().T) * s.double(), K, f"{M}x{N}x{K} ldc {ldc}")
    del buf, c
    torch.cuda.empty_cache()


@pytest.mark.parametrize("tile,M,N,K,resid", [("64x64", 70, 64, 64, False), ("64x64 split K", 65, 1536, 1600, True),
                                              ("64x128", 1000, 1536, 64, False), ("128x128", 3951, 1600, 1536, True)])
def test_f16w_tiles(ns2lib, tile, M, N, K, resid):
    print(f"[case] {tile} {M}x{N}x{K} resid {resid}", flush=True)
    assert_tile(ns2lib, tile, 1, M, N, K, resid=resid)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
    wt = torch.empty_like(w)
    ns2lib.tile_bf16_weight(w, wt, N, K)
    buf = torch.randn(M + 200, N, generator=g, device=DEV)
    before = buf.clone()
    ns2lib.linear_f16w_tiled(tiled(x), wt, buf, M, N, K, resid=resid)
    torch.cuda.synchronize()
    assert torch.equal(buf[M:], before[M:]), "rows past M were written"
    ref = x.double() @ w.half().double().T
    close(buf[:M], before[:M].double() + ref if resid else ref, max(K, 1024), f"{tile} {M}x{N}x{K}")


# both sides of the rule that takes file-layout operands to the block tiles: rows, work, 64-row weight blocks,
# the number of tiles
@pytest.mark.parametrize("route,M,N,K,resid,rank,act", [
    ("tiled", 400, 2560, 1024, True, 0, "none"), ("rows", 399, 2560, 1024, True, 0, "none"),
    ("tiled", 1001, 1600, 768, False, 32, "none"), ("rows", 1001, 1616, 768, False, 32, "none"),
    ("rows", 3953, 64, 4096, True, 0, "silu"), ("rows", 3953, 64, 3840, True, 0, "silu"),
    ("tiled", 8193, 64, 4096, True, 0, "silu"), ("tiled", 2500, 4608, 1536, False, 0, "none"),
    ("tiled", 3953, 1536, 1536, False, 0, "none"), ("tiled", 1025, 1536, 1536, True, 0, "none"),
])
def test_i8_file_layout(ns2lib, route, M, N, K, resid, rank, act):
    """The int8 linear on a file-layout weight (every int8 value, strided rows, a column window of C) for
    its three input formats; fp16-exact inputs, so the error is that of fp32 sums."""
    print(f"[case] file layout {route} {M}x{N}x{K} resid {resid} rank {rank} {act}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    lda, ldc = K + 64, N + 32
    x = torch.randn(M, lda, generator=g, device=DEV).half()
    q = torch.randint(-128, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
    bias, gate = torch.randn(N, generator=g, device=DEV), torch.randn(N, generator=g, device=DEV)
    xk = x[:, :K].double()
    ref = (xk @ q.double().T) * s.double() + bias.double()
    lora = None
    if rank:
        a = (torch.randn(rank, K, generator=g, device=DEV) / math.sqrt(K)).half()
        b = (torch.randn(N, rank, generator=g, device=DEV) / math.sqrt(rank)).half()
        lora = (a, b, rank)
        ref = ref + (xk @ a.double().T).half().double() @ b.double().T
    if act == "silu":
        ref = torch.nn.functional.silu(ref)
    base = torch.randn(M, ldc, generator=g, device=DEV)
    if resid:
        ref = base[:, 32:].double() + gate.double() * ref
    kw = dict(bias=bias, resid=resid, gate=gate if resid else None, lora=lora, ldc=ldc, cOff=32, act=act)
    outs = {}
    for fmt, src in ((1, x), (2, x.float())):
        y = base.clone()
        ns2lib.linear_i8(src, fmt, lda, q, s, y, M, N, K, **kw)
        torch.cuda.synchronize()
        assert torch.equal(y[:, :32], base[:, :32]), "columns left of the window were written"
        outs[fmt] = y
    assert torch.equal(outs[1], outs[2])
    got = outs[1][:, 32:]
    if rank:  # t = x a^T may round to the other fp16 neighbour
        assert ((got.double() - ref).norm() / ref.norm()).item() <= 2.0**-12
    else:
        close(got, ref, K, f"file layout {route} {M}x{N}x{K}")
    # unrotated fp32 input: the same as the rotated rows given as fp16
    xr = torch.empty(M, K, dtype=torch.float16, device=DEV)
    ns2lib.rotate_f16(x.float(), lda, xr, K, M, K)
    y0, y1 = base.clone(), base.clone()
    ns2lib.linear_i8(x.float(), 0, lda, q, s, y0, M, N, K, **kw)
    ns2lib.linear_i8(xr, 1, K, q, s, y1, M, N, K, **kw)
    torch.cuda.synchronize()
    assert torch.equal(y0, y1)


def test_i8_file_layout_rotated_rows_keep_to_themselves(ns2lib):
    """The linear on rotated fp16 rows and a file-layout weight uses no memory but its operands: none is
    allocated, and calls that overlap on two streams do not meet."""
    M, N, K = 512, 8192, 8192
    g = torch.Generator(device=DEV).manual_seed(7)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    q = [torch.randint(-128, 128, (N, K), generator=g, device=DEV, dtype=torch.int8) for _ in range(2)]
    s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
    y, alone = ([torch.empty(M, N, device=DEV) for _ in range(2)] for _ in range(2))
    main, streams = torch.cuda.current_stream(), [torch.cuda.Stream() for _ in range(2)]
    ns2lib.linear_i8(x, 1, K, q[0], s, alone[0], 64, N, K)  # the kernels' code is loaded
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for i in range(2):
        ns2lib.linear_i8(x, 1, K, q[i], s, alone[i], M, N, K)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < N * K // 2, "device memory was allocated"
    close(alone[0], (x.double() @ q[0].double().T) * s.double(), K, "file layout 512x8192x8192")
    try:
        for _ in range(8):
            for i in range(2):
                ns2lib.set_stream(streams[i].cuda_stream)
                ns2lib.linear_i8(x, 1, K, q[i], s, y[i], M, N, K)
    finally:
        ns2lib.set_stream(main.cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(y[0], alone[0]) and torch.equal(y[1], alone[1])


@pytest.mark.parametrize("M,N,K", [(1001, 1616, 768), (65, 4120, 256)])
def test_lora_ragged_columns(ns2lib, M, N, K):
    """Row-major kernel, LoRA, N no multiple of 32: the last columns' low-rank term takes every lane's
    rows (t's fp16 rounding: 2^-12 of the result)."""
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
    a = (torch.randn(32, K, generator=g, device=DEV) / math.sqrt(K)).half()
    b = (torch.randn(N, 32, generator=g, device=DEV) / math.sqrt(32)).half()
    y = torch.empty(M, N, device=DEV)
    ns2lib.linear_i8(x, 1, K, q, s, y, M, N, K, lora=(a, b, 32))
    ref = (x.double() @ q.double().T) * s.double() + (x.double() @ a.double().T).half().double() @ b.double().T
    for cols in (slice(0, N), slice(N // 32 * 32, N)):
        rel = ((y[:, cols].double() - ref[:, cols]).norm() / ref[:, cols].norm()).item()
        assert rel <= 2.0**-12, f"columns {cols}: {rel:.2e}"


@pytest.mark.parametrize("M,act", [(96, "silu"), (1000, "gelu_tanh")])
def test_i8_activation(ns2lib, M, act):
    N, K = 1536, 512
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
    wt, y = torch.empty_like(q), torch.empty(M, N, device=DEV)
    ns2lib.tile_i8_weight(q, wt, N, K)
    ns2lib.linear_i8_tiled(tiled(x), wt, s, y, M, N, K, act=act)
    torch.cuda.synchronize()
    z = (x.double() @ q.double().T) * s.double()
    ref = torch.nn.functional.silu(z) if act == "silu" else torch.nn.functional.gelu(z, approximate="tanh")
    close(y, ref, 1024, act)


# a size per operand kind at which every form a tile is built for takes it
SIZES = {
    0: {"64x64": (65, 192, 768), "64x128K2": (777, 2624, 1536), "64x128K2S3": (65, 8256, 512), "64x128": (257, 4608, 256),
        "128x128": (1801, 4608, 256), "128x192": (2867, 1536, 256), "128x192K2": (1537, 2624, 1536), "192x384": (3329, 4672, 1536),
        "256x256": (1501, 8256, 512)},
    1: {"64x64": (65, 192, 768), "64x128K2S3": (65, 8256, 512), "64x128": (999, 4160, 256), "128x128": (1460, 1536, 256),
        "128x192": (2305, 4608, 256), "256x256": (2867, 4608, 256)},
    2: {"64x64": (511, 1536, 1536), "64x128K2": (777, 2560, 1024), "64x128K2S3": (401, 2560, 1024), "64x128": (511, 4672, 512),
        "128x128": (999, 8256, 512), "128x192": (511, 8256, 512), "128x192K2": (1801, 2560, 1024), "192x384": (3329, 4672, 1536),
        "256x256": (1501, 8256, 512)},
}
FORMS = [("none", False, 0), ("none", True, 0), ("none", False, 64), ("none", True, 32), ("silu", False, 0), ("gelu_tanh", True, 0),
         ("gelu_tanh", False, 32), ("silu", True, 32)]


@pytest.mark.parametrize("ops,tile", [(o, t) for o in SIZES for t in SIZES[o]])
@pytest.mark.parametrize("act,resid,rank", FORMS)
def test_tile_forms(ns2lib, ops, tile, act, resid, rank):
    """Every kernel of every block tile: old outputs, the LoRA term, the activations and what combines them,
    a column window of a wider output, with fp16-exact operands. Beside the fp32 sums the activation is off
    by a few ulp (__expf and the quotient: 2^-21 of a value), and t of the LoRA may round to the other fp16
    neighbour in few places (2^-12 of the result)."""
    M, N, K = SIZES[ops][tile]
    if tile == "192x384" and (act, resid, rank) != ("none", False, 0) or tile == "128x128" and resid and rank:
        assert tile_of(ns2lib, ops, M, N, K, act, resid, rank)[0] != tile
        return
    print(f"[case] ops {ops} {tile} {M}x{N}x{K} {act} resid {resid} rank {rank}", flush=True)
    assert_tile(ns2lib, tile, ops, M, N, K, act=act, resid=resid, rank=rank)
    g = torch.Generator(device=DEV).manual_seed(M + N + K + rank)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    bias, gate = torch.randn(N, generator=g, device=DEV), torch.randn(N, generator=g, device=DEV)
    if ops == 1:
        w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).to(torch.bfloat16)
        ref = x.double() @ w.half().double().T
    else:
        w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
        s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
        ref = (x.double() @ w.double().T) * s.double()
    ref = ref + bias.double()
    lora = None
    if rank:
        a = (torch.randn(rank, K, generator=g, device=DEV) / math.sqrt(K)).half()
        b = (torch.randn(N, rank, generator=g, device=DEV) / math.sqrt(rank)).half()
        lora = (a, b, rank)
        ref = ref + (x.double() @ a.double().T).half().double() @ b.double().T
    if act != "none":
        ref = torch.nn.functional.silu(ref) if act == "silu" else torch.nn.functional.gelu(ref, approximate="tanh")
    ldc = N + 32
    buf = torch.randn(M + 300, ldc, generator=g, device=DEV)
    before = buf.clone()
    if resid:
        ref = before[:M, 32:].double() + gate.double() * ref
    kw = dict(bias=bias, act=act, resid=resid, gate=gate if resid else None, lora=lora, ldc=ldc, cOff=32)
    if ops == 2:
        ns2lib.linear_i8(x, 1, K, w, s, buf, M, N, K, **kw)
    else:
        wt = torch.empty_like(w)
        if ops == 1:
            ns2lib.tile_bf16_weight(w, wt, N, K)
            ns2lib.linear_f16w_tiled(tiled(x), wt, buf, M, N, K, **kw)
        else:
            ns2lib.tile_i8_weight(w, wt, N, K)
            ns2lib.linear_i8_tiled(tiled(x), wt, s, buf, M, N, K, **kw)
    torch.cuda.synchronize()
    assert torch.equal(buf[M:], before[M:]) and torch.equal(buf[:, :32], before[:, :32]), "values outside the window were written"
    got = buf[:M, 32:]
    rel = ((got.double() - ref).norm() / ref.norm()).item()
    tol = math.sqrt(max(K, 1024)) * 2.0**-24 + (2.0**-21 if act != "none" else 0) + (2.0**-12 if rank else 0)
    print(f"[parity] ops {ops} {tile}: rel-L2 {rel:.2e} (tol {tol:.1e})", flush=True)
    assert torch.isfinite(got).all() and rel <= tol


# 1030: 17 row blocks of 64, so the last 128-row tile holds one real block; 1090: a ragged second one
@pytest.mark.parametrize("tile,M,N,K,rank", [("128x512", 1030, 8192, 256, 0), ("128x512", 1090, 8192, 1536, 32),
                                             ("64x512", 1024, 8192, 256, 0), ("64x512", 2100, 8192, 256, 32),
                                             ("64x512S3", 70, 1024, 2304, 0), ("64x512S3", 401, 2048, 4096, 32)])
def test_glu_tiles(ns2lib, tile, M, N, K, rank):
    """The GLU + rotation epilogue's block tiles: one fp16 rounding of the result (2^-11 of a value at
    most), with a LoRA the rounding of its down-projection too; rows past the last row block stay."""
    print(f"[case] glu {tile} {M}x{N}x{K} rank {rank}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
    h = (x.double() @ q.double().T) * s.double()
    lora = None
    if rank:
        a = (torch.randn(rank, K, generator=g, device=DEV) / math.sqrt(K)).half()
        b = (torch.randn(N, rank, generator=g, device=DEV) / math.sqrt(rank)).half()
        lora = (a, b, rank)
        h = h + (x.double() @ a.double().T).half().double() @ b.double().T
    I, rows = N // 2, (M + 63) // 64 * 64
    y = (torch.nn.functional.silu(h[:, :I]) * h[:, I:]).reshape(M, I // 256, 256)
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device=DEV)
    had = torch.kron(torch.kron(h4, h4), torch.kron(h4, h4)) / 16
    ref = (y @ had).reshape(M, I)
    wt = torch.empty_like(q)
    ns2lib.tile_i8_weight_glu(q, wt, N, K)
    out = torch.full((rows + 64, I), -7.0, dtype=torch.float16, device=DEV)
    ns2lib.linear_i8_glu_rot_tiled(tiled(x), wt, s, out, M, N, K, act="silu", lora=lora)
    torch.cuda.synchronize()
    assert (out[rows:] == -7.0).all(), "rows past the last row block were written"
    got = out[:rows].reshape(rows // 64, I // 64, 8, 64, 8).permute(0, 3, 1, 2, 4).reshape(rows, I)[:M]
    rel = ((got.double() - ref).norm() / ref.norm()).item()
    print(f"[parity] glu {tile}: rel-L2 {rel:.2e}", flush=True)
    assert torch.isfinite(got).all() and rel <= (2.0**-10 if rank else 2.0**-11)


@pytest.mark.parametrize("M", [100, 1100])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "none"])
def test_glu_activation(ns2lib, M, act):
    """The fused GLU launch computes the activation of the plain epilogue, bit for bit: small integers make
    the products' fp32 sums exact in any order, act(h1) comes from the plain linear, and the modulation
    producer (scale -1, the row as its shift) rotates act(h1) * h2 as the GLU epilogue does."""
    print(f"[case] glu activation {M} {act}", flush=True)
    I, K = 4096, 256
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randint(-8, 9, (M, K), generator=g, device=DEV).half()
    q = torch.randint(-127, 128, (2 * I, K), generator=g, device=DEV, dtype=torch.int8)
    s = torch.full((2 * I,), 2.0**-12, device=DEV)
    wt, wg = torch.empty_like(q), torch.empty_like(q)
    ns2lib.tile_i8_weight(q, wt, 2 * I, K)
    ns2lib.tile_i8_weight_glu(q, wg, 2 * I, K)
    a, h = torch.empty(M, I, device=DEV), torch.empty(M, 2 * I, device=DEV)
    ns2lib.linear_i8_tiled(tiled(x), wt, s, a, M, I, K, act=act)  # the first I weight rows are the first tiles
    ns2lib.linear_i8_tiled(tiled(x), wt, s, h, M, 2 * I, K)
    out = torch.empty((M + 63) // 64, I // 64, 8, 64, 8, dtype=torch.float16, device=DEV)
    ns2lib.linear_i8_glu_rot_tiled(tiled(x), wg, s, out, M, 2 * I, K, act=act)
    got = out.permute(0, 3, 1, 2, 4).reshape(-1, I)[:M]
    one, minus = torch.ones(I, device=DEV), torch.full((I,), -1.0, device=DEV)
    ref = torch.empty(M, I, dtype=torch.float16, device=DEV)
    for m in range(0, M, 7):
        ns2lib.norm_mod_rotate_f16(one, torch.cat([a[m] * h[m, I:], minus]), 0, I, 1, I, one, ref[m])
    torch.cuda.synchronize()
    differ = (got[::7] != ref[::7]).sum().item()
    assert differ == 0, f"{differ} values differ"


# head dims and counts whose value columns start inside a wave's columns (3200 is no multiple of 96)
@pytest.mark.parametrize("M,N,K,H,HD", [(3952, 4608, 512, 22, 64), (3328, 4608, 512, 16, 96), (2304, 4608, 512, 22, 64),
                                        (1536, 4608, 512, 16, 96), (48, 4608, 512, 22, 64)])
def test_vpack_tiles(ns2lib, M, N, K, H, HD):
    """The packed values equal the fp16 roundings of the plain store's columns, key by key, and the
    other columns equal the plain store's."""
    print(f"[case] vpack {M}x{N}x{K} heads {H}x{HD}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M)
    x = tiled(torch.randn(M, K, generator=g, device=DEV).half())
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) + 0.5) / (73 * math.sqrt(K))
    wt = torch.empty_like(q)
    ns2lib.tile_i8_weight(q, wt, N, K)
    Lk, vcol0 = M + 20, N - H * HD
    tiles = (Lk + 63) // 64
    plain, y = torch.empty(M, N, device=DEV), torch.zeros(M, N, device=DEV)
    vpk = torch.zeros(H * tiles * 64 * HD, dtype=torch.float16, device=DEV)
    ns2lib.linear_i8_tiled(x, wt, s, plain, M, N, K)
    ns2lib.linear_i8_tiled_vpack(x, wt, s, y, M, N, K, vpk, vcol0=vcol0, H=H, D=HD, Lk=Lk)
    torch.cuda.synchronize()
    assert torch.equal(y[:, :vcol0], plain[:, :vcol0])
    # [head][tile][chunk][dim][8]: chunk 2g + hi holds keys 16g + 4hi + {0..3}, 16g + 8 + 4hi + {0..3}
    v = vpk.reshape(H, tiles, 4, 2, HD, 2, 4).permute(1, 2, 5, 3, 6, 0, 4).reshape(tiles * 64, H * HD)
    # both launches take the same tile, and neither splits K
    assert tile_of(ns2lib, 0, M, N, K) == tile_of(ns2lib, 0, M, N, K, packed=True)
    assert torch.equal(v[:M], plain[:, vcol0:].half())
