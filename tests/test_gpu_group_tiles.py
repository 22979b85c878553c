"""The K-group tiles (the K steps split over wave groups, the groups' sums added in LDS) on an MI355X: every tile at
its edges — one row, a row and a column past the tile, a K with fewer steps than groups, one that does not divide
among them and one that does —, each epilogue, output type, output layout and weight layout, bit for bit against the
128 × 256 kernel on the same operands (W8A8 sums are exact integers: any split of K gives the same bits)."""
import pytest
import torch

from test_gpu_parity import DEV, dev

pytestmark = pytest.mark.gpu

W8A8_TILES = ["g32x32k8", "g32x64k8", "g64x64k4", "g64x96k4", "g64x128k4", "g96x96k4", "g96x128k4", "g128x96k4",
              "g128x128k2", "g96x192k2", "g128x192k2"]


def _w8a8_operands(m, k, n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    codes = torch.randint(-128, 128, (m, k), dtype=torch.int8, device=DEV, generator=g)
    w = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=DEV, generator=g)
    sx, s = (torch.rand(size, device=DEV, generator=g) * 1e-2 + 1e-3 for size in (m, n))
    return codes, sx, w, s, torch.randn(n, device=DEV, generator=g)


@pytest.mark.parametrize("tile", W8A8_TILES)
def test_w8a8_group_tile_same_bits(tile_gemm, tile):
    bm, bn = (int(v) for v in tile[1:].split("k")[0].split("x"))
    got, want = tile_gemm(tile), tile_gemm("128")
    cases = [(1, 128, bn, None, torch.float32, False), (bm + 1, 640, bn + 32, "gelu_tanh", torch.bfloat16, False),
             (bm, 1024, bn + 4, None, torch.bfloat16, True), (2 * bm - 1, 1152, 2 * bn + 1, None, torch.float32, False),
             (bm - 1, 200, bn - 3, "gelu_tanh", torch.float32, False)]
    if bn % 64 == 0:
        cases += [(bm + 3, 640, 2 * (bn // 2 + 5), "silu_glu", torch.bfloat16, False),
                  (bm, 1024, 2 * bn, "situ_glu", torch.float32, False)]
    for m, k, n, epi, out, nk in cases:
        print(f"{tile}: {m} x {k} x {n} {epi} {out} {'nk' if nk else 'packed'}", flush=True)
        codes, sx, w, s, b = _w8a8_operands(m, k, n, m + k + n)
        if not nk:
            w = want.pack(w, layout="nk", glu=epi in ("silu_glu", "situ_glu"))
        ys = [g.product_w8a8(codes, sx, w, s, bias=b, epilogue=epi, out_dtype=out) for g in (got, want)]
        torch.cuda.synchronize()
        assert torch.equal(*ys)
    # Three outputs (row-major, head-major), and the residual stream in place.
    m, k, d = bm + 2, 1024, 128
    codes, sx, w, s, b = _w8a8_operands(m, k, 3 * d, 7)
    w = want.pack(w, layout="nk")
    for head_dim in (0, 32):
        parts = [g.product_w8a8_qkv(codes, sx, w, s, bias=b, head_dim=head_dim) for g in (got, want)]
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(*parts))
    gate = torch.linspace(-1.0, 1.0, 3 * d, device=DEV)
    streams = [torch.ones((m, 3 * d), device=DEV) for _ in range(2)]
    for g, x in zip((got, want), streams):
        g.product_w8a8_residual(x, codes, sx, w, s, bias=b, gate=gate)
    torch.cuda.synchronize()
    assert torch.equal(*streams)


Q8_TILES = {"16": (16, 64), "32": (32, 64), "48": (48, 64), "64": (64, 64), "80": (80, 64), "128x128": (128, 128),
            "128x256": (128, 256), "64x256": (64, 256)}


@pytest.fixture(scope="module")
def q8_gemm(gemm):
    """Block-scale contexts on a forced tile (SQ8_Q8_TILE)."""
    import os
    import siliconed_amd as sq
    made = {}
    for name in Q8_TILES:
        os.environ["SQ8_Q8_TILE"] = name
        try:
            made[name] = sq.TensorGEMM.make(0)
        finally:
            del os.environ["SQ8_Q8_TILE"]
    return made


@pytest.mark.parametrize("tile", Q8_TILES)
def test_q8_tile_sums_in_k_order(gemm, q8_gemm, tile):
    """Block scales at every tile's edges (one row, a row and a column past the tile; one K step, counts that leave each
    remainder of the kernels' unrolled steps; a K of 32·odd), plain and GLU, bf16 and fp32 out, the rounded and the fp32
    route. Integer activations make each block's sum exact, so acc = fl(P·d + acc) per block in K order, then the bias,
    is the whole arithmetic: restated in float64 (which holds P·d + acc exactly), bit for bit on fp32 outputs; the
    activations' outputs bit for bit against the 16-row tile's."""
    bm, bn = Q8_TILES[tile]
    ctx = q8_gemm[tile]
    for m, k, n, epi, out, exact in [
            (1, 64, 8, None, torch.float32, False), (bm + 1, 320, bn + 4, None, torch.float32, False),
            (bm, 96, bn + 1, None, torch.float32, False), (2 * bm - 1, 704, bn, None, torch.float32, False),
            (bm - 1, 576, 130, None, torch.float32, True), (bm + 3, 448, 2 * (bn // 2 + 5), "silu_glu", torch.bfloat16, False),
            (bm + 2, 1024, 2 * bn, "situ_glu", torch.float32, False), (bm + 5, 832, bn + 2, "gelu_tanh", torch.bfloat16, False)]:
        print(f"q8 tile {tile}: {m} x {k} x {n} {epi} {out} {'fp32 route' if exact else ''}", flush=True)
        g = torch.Generator(device=DEV).manual_seed(m + k + n)
        x = torch.randint(-5, 6, (m, k), device=DEV, generator=g).float()
        q = torch.randint(-127, 128, (n, k), device=DEV, generator=g, dtype=torch.int8)
        d = (torch.rand((n, k // 32), device=DEV, generator=g) * 0.02 + 1e-3).half()
        b = torch.randn(n, device=DEV, generator=g)
        w = ctx.pack_blocks(q, d, 32, layout="nk", glu=epi in ("silu_glu", "situ_glu"))
        a = x if exact else x.bfloat16()
        y = ctx.product_blocks(a, w, bias=b, epilogue=epi, out_dtype=out, rounding=not exact)
        torch.cuda.synchronize()
        if epi is None:
            acc = torch.zeros((m, n), device=DEV)
            for i in range(k // 32):
                part = x[:, 32 * i:32 * i + 32].double() @ q[:, 32 * i:32 * i + 32].double().t()
                acc = (part * d[:, i].double() + acc.double()).float()
            assert torch.equal(y, acc + b)
        else:
            z = q8_gemm["16"].product_blocks(a, w, bias=b, epilogue=epi, out_dtype=out, rounding=not exact)
            torch.cuda.synchronize()
            assert torch.equal(y, z)


BF16_TILES = ["g32x32k4", "g32x64k4", "g64x64k4", "g64x96k4", "g64x128k4", "g64x128k2", "g64x192k2", "g96x96k4", "g96x128k4",
              "g128x96k4", "g128x128k2", "g96x192k2", "g128x192k2"]
F32_TILES = [t for t in BF16_TILES if t not in ("g96x128k4", "g128x96k4")]


@pytest.mark.parametrize("route,tile", [("bf16", t) for t in BF16_TILES] + [("fp32", t) for t in F32_TILES])
def test_group_tile_exact_sums_same_bits(tile_gemm, route, tile):
    """The bf16 and fp32 routes on operands whose every partial sum is exact in fp32 (so any split and order of K gives
    the same bits), against the 128-row tiles: int8 and fp8 codes, both layouts, every epilogue, output type and output
    layout. fp32 route: values of two and of three non-zero bf16 parts (12 and 18 significant bits)."""
    bm, bn = (int(v) for v in tile[1:].split("k")[0].split("x"))
    got, want = tile_gemm(tile), tile_gemm("128")
    cases = [(1, 64, bn, None, torch.float32, False, True), (bm + 1, 320, bn + 32, "gelu_tanh", torch.bfloat16, False, False),
             (bm, 512, bn + 4, None, torch.bfloat16, True, False), (2 * bm - 1, 448, 2 * bn + 1, None, torch.float32, False, True),
             (bm - 1, 200, bn - 3, "gelu_tanh", torch.float32, False, False)]
    if bn % 64 == 0:
        cases += [(bm + 3, 320, 2 * (bn // 2 + 5), "silu_glu", torch.bfloat16, False, False),
                  (bm, 512, 2 * bn, "situ_glu", torch.float32, True, True)]

    def operands(m, k, n, seed, fp8):
        g = torch.Generator(device=DEV).manual_seed(seed)
        q = torch.randint(-3, 4, (n, k), device=DEV, generator=g)
        s = torch.rand(n, device=DEV, generator=g) * 1e-2 + 1e-3
        if route == "bf16":
            x = torch.randint(-5, 6, (m, k), device=DEV, generator=g).bfloat16()
        elif k > 64:
            x = torch.randint(-2047, 2048, (m, k), device=DEV, generator=g).float() / 1024     # |sum| < 2^24 / 1024
        else:
            x = torch.randint(-(2 ** 16), 2 ** 16 + 1, (m, k), device=DEV, generator=g).float() / 65536 * 1.0
            x = x + torch.randint(-1, 2, (m, k), device=DEV, generator=g) / 65536 / 2           # 18 bits; |q| ≤ 1 below
            q = q.clamp(-1, 1)
        return x, q.to(torch.float8_e4m3fn if fp8 else torch.int8), s, torch.randn(n, device=DEV, generator=g)

    for m, k, n, epi, out, nk, fp8 in cases:
        print(f"{route} {tile}: {m} x {k} x {n} {epi} {out} {'nk' if nk else 'packed'} {'fp8' if fp8 else 'int8'}", flush=True)
        x, q, s, b = operands(m, k, n, m + k + n, fp8)
        w = q if nk else want.pack(q, layout="nk", glu=epi in ("silu_glu", "situ_glu"))
        ys = [g.product(x, w, s, bias=b, epilogue=epi, out_dtype=out, rounding=route == "bf16") for g in (got, want)]
        torch.cuda.synchronize()
        assert torch.equal(*ys)
    if route == "bf16":
        m, k, d = bm + 2, 320, 128
        x, q, s, b = operands(m, k, 3 * d, 7, False)
        w = want.pack(q, layout="nk")
        for head_dim in (0, 32):
            parts = [g.product_qkv(x, w, s, bias=b, head_dim=head_dim) for g in (got, want)]
            torch.cuda.synchronize()
            assert all(torch.equal(u, v) for u, v in zip(*parts))
        gate = torch.linspace(-1.0, 1.0, 3 * d, device=DEV)
        streams = [torch.ones((m, 3 * d), device=DEV) for _ in range(2)]
        for g, y in zip((got, want), streams):
            g.product_residual(y, x, w, s, bias=b, gate=gate)
        torch.cuda.synchronize()
        assert torch.equal(*streams)


def _same(x, y):
    """The same values, NaN in the same places."""
    return torch.equal(x.isnan(), y.isnan()) and torch.equal(x.nan_to_num(), y.nan_to_num())


@pytest.mark.parametrize("route,tile", [("bf16", "g32x64k4"), ("bf16", "g128x192k2"), ("fp32", "g64x96k4"), ("fp32", "g96x192k2")])
def test_group_tile_infinities_and_nan(tile_gemm, route, tile):
    """NaN and infinite activations reach their own rows only, NaN fp8 codes their own columns, through the split of K
    (a K of 200 padded to whole steps; 7 steps over the groups), as in the 128-row tiles."""
    got, want = tile_gemm(tile), tile_gemm("128")
    for m, k, n, fp8, epi in [(40, 448, 200, False, None), (131, 200, 96, True, "gelu_tanh"), (33, 512, 128, True, "silu_glu")]:
        g = torch.Generator(device=DEV).manual_seed(m)
        q = torch.randint(-3, 4, (n, k), device=DEV, generator=g).to(torch.float8_e4m3fn if fp8 else torch.int8)
        if fp8:
            q.view(torch.uint8)[17, k - 1] = 0x7F
        x = torch.randint(-5, 6, (m, k), device=DEV, generator=g).float()
        x[5, 7], x[9, 3], x[12, k - 1], x[31, 64] = float("nan"), float("inf"), float("-inf"), float("inf")
        x = x if route == "fp32" else x.bfloat16()
        s, b = torch.rand(n, device=DEV, generator=g) * 1e-2 + 1e-3, torch.randn(n, device=DEV, generator=g)
        s[3] = float("inf")
        w = want.pack(q, layout="nk", glu=epi == "silu_glu")
        ys = [c.product(x, w, s, bias=b, epilogue=epi, out_dtype=torch.float32, rounding=route == "bf16") for c in (got, want)]
        torch.cuda.synchronize()
        assert _same(*ys)
        assert ys[0][5].isnan().all() and (ys[0].isnan().sum(1) < n // 4).sum() >= m - 5


@pytest.mark.parametrize("tile", Q8_TILES)
def test_q8_tile_infinities_and_nan(q8_gemm, tile):
    """The same through the block scales: an infinite scale meets one block of one column; the padded half step's zero
    codes and scales (a K of 32·odd) stay out of every sum."""
    m, k, n = 37, 352, 136
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randint(-5, 6, (m, k), device=DEV, generator=g).float()
    x[5, 7], x[9, 3], x[12, k - 1] = float("nan"), float("inf"), float("-inf")
    q = torch.randint(-127, 128, (n, k), device=DEV, generator=g, dtype=torch.int8)
    d = (torch.rand((n, k // 32), device=DEV, generator=g) * 0.02 + 1e-3).half()
    d[20, 4] = float("inf")
    ctx = q8_gemm[tile]
    y = ctx.product_blocks(x.bfloat16(), ctx.pack_blocks(q, d, 32, layout="nk"), out_dtype=torch.float32)
    torch.cuda.synchronize()
    acc = torch.zeros((m, n), dtype=torch.float64)
    xs, qs, ds = x.double().cpu(), q.double().cpu(), d.double().cpu()
    for i in range(k // 32):
        part = (xs[:, None, 32 * i:32 * i + 32] * qs[None, :, 32 * i:32 * i + 32]).sum(-1)
        acc = (part * ds[:, i] + acc).float().double()
    assert _same(y.cpu(), acc.float())
    assert torch.isfinite(y).sum() == (m - 3) * (n - 1)


@pytest.mark.parametrize("kind,tile", [("bf16", "g64x96k4"), ("bf16", "g96x192k2"), ("w8a8", "g32x64k8"), ("w8a8", "g128x96k4")])
def test_group_tile_outputs_off_the_four_column_grid(tile_gemm, kind, tile):
    """Stores one column at a time: three outputs off the 16-byte grid, rows and heads that end inside a wave's columns; a
    residual stream of an odd width, off the grid, with and without a gate; a plain output one element in. Bit for bit the
    128-row tiles'."""
    got, want = tile_gemm(tile), tile_gemm("128")
    m, k = 75, 384
    off = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)

    def operands(n, seed):
        g = torch.Generator(device=DEV).manual_seed(seed)
        q = torch.randint(-3, 4, (n, k), device=DEV, generator=g).to(torch.int8)
        x = torch.randint(-5, 6, (m, k), device=DEV, generator=g)
        s, b = torch.rand(n, device=DEV, generator=g) * 1e-2 + 1e-3, torch.randn(n, device=DEV, generator=g)
        sx = torch.rand(m, device=DEV, generator=g) + 0.5
        return ((x.bfloat16(),) if kind == "bf16" else (x.to(torch.int8), sx)), want.pack(q, layout="nk"), s, b

    for d, head_dim in ((100, 0), (100, 20), (96, 12), (36, 4)):
        x, w, s, b = operands(3 * d, d + head_dim)
        shape = (m, d) if head_dim == 0 else (d // head_dim, m, head_dim)
        for dtype in (torch.bfloat16, torch.float32):
            outs = [tuple(f(torch.zeros(shape, device=DEV, dtype=dtype)) for f in (off, off, torch.clone)) for _ in range(2)]
            for ctx, out in zip((got, want), outs):
                (ctx.product_qkv if kind == "bf16" else ctx.product_w8a8_qkv)(*x, w, s, bias=b, head_dim=head_dim, out=out,
                                                                             out_dtype=dtype)
            torch.cuda.synchronize()
            assert all(torch.equal(u, v) for u, v in zip(*outs)) and all(u.any() for u in outs[0])
    for n in (385, 384):
        x, w, s, b = operands(n, n)
        for gate in (None, off(torch.linspace(-1.0, 1.0, n, device=DEV))):
            streams = [off(torch.ones((m, n), device=DEV)) for _ in range(2)]
            for ctx, y in zip((got, want), streams):
                (ctx.product_residual if kind == "bf16" else ctx.product_w8a8_residual)(y, *x, w, s, bias=b, gate=gate)
            torch.cuda.synchronize()
            assert torch.equal(*streams) and not torch.equal(streams[0], torch.ones_like(streams[0]))
        outs = [off(torch.zeros((m, n), device=DEV, dtype=torch.bfloat16)) for _ in range(2)]
        for ctx, y in zip((got, want), outs):
            (ctx.product if kind == "bf16" else ctx.product_w8a8)(*x, w, s, bias=b, out=y)
        torch.cuda.synchronize()
        assert torch.equal(*outs)
