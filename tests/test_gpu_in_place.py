"""Products on codes as they lie ([K, N] of a map, [N, K] of a published weight) that the kernels do not read in place — a
ragged K or N, a row stride or base at any byte, an activation not aligned for 16-byte loads — on an MI355X: staged per
product, bit for bit the product of the packed weight; and under stream capture before any product of that size, where the
context's buffers may not grow, on the kernels that read the codes as they lie."""
import pytest
import torch

from siliconed_amd import _abi as abi
from test_gpu_parity import DEV

pytestmark = pytest.mark.gpu


def _operands(m, k, n, seed, fp8=False):
    """Operands whose every partial sum is exact in fp32: any kernel's sums have the same bits."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = torch.randint(-7, 8, (n, k), device=DEV, generator=g)
    x = torch.randint(-5, 6, (m, k), device=DEV, generator=g).bfloat16()
    s = torch.rand(n, device=DEV, generator=g) * 1e-2 + 1e-3
    return x, q.to(torch.float8_e4m3fn if fp8 else torch.int8), s, torch.randn(n, device=DEV, generator=g)


def _at(t, offset, pad):
    """`t` in a buffer of rows `pad` elements longer, starting `offset` elements in (other values around it)."""
    rows, cols = t.shape
    buf = torch.full((offset + rows * (cols + pad),), 3, device=DEV).to(t.dtype)
    view = buf[offset:].view(rows, cols + pad)[:, :cols]
    view.copy_(t)
    return view


@pytest.mark.parametrize("layout", ["kn", "nk"])
@pytest.mark.parametrize("m,k,n,offset,pad", [
    (1, 64, 64, 0, 0), (33, 200, 100, 0, 0), (130, 320, 264, 3, 5), (5, 256, 128, 1, 0), (70, 512, 320, 0, 16),
    (300, 1000, 77, 2, 1), (17, 8, 8, 0, 0), (64, 1, 3, 0, 0)])
def test_in_place_same_bits_as_packed(gemm, layout, m, k, n, offset, pad):
    for epi, fp8, out in (("gelu_tanh", False, torch.bfloat16), (None, True, torch.float32), ("silu_glu", False, torch.float32)):
        if epi == "silu_glu" and n % 2:
            continue
        print(f"{layout} {m} x {k} x {n} offset {offset} pad {pad} {epi} fp8 {fp8}", flush=True)
        x, q, s, b = _operands(m, k, n, m + k + n, fp8)
        want = gemm.product(x, gemm.pack(q, layout="nk", glu=epi == "silu_glu"), s, bias=b, epilogue=epi, out_dtype=out)
        w = _at(q if layout == "nk" else q.t().contiguous(), offset, pad)
        for a in (x, _at(x, offset, pad)):
            got = gemm.product(a, w, s, layout=layout, bias=b, epilogue=epi, out_dtype=out)
            torch.cuda.synchronize()
            assert torch.equal(got, want)
    x, q, s, b = _operands(m, k, n, 5)
    want = gemm.product(x.float(), gemm.pack(q, layout="nk"), s, rounding=False, out_dtype=torch.float32)
    w = _at(q if layout == "nk" else q.t().contiguous(), offset, pad)
    run = lambda: gemm.product(_at(x.float(), offset, pad), w, s, layout=layout, rounding=False, out_dtype=torch.float32)
    if layout == "nk" and k % 64 == 0 and (offset % 16 or (k + pad) % 16):
        with pytest.raises(abi.Unsupported):  # the fp32 route has no kernel for such codes
            run()
    else:
        got = run()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("layout,m,k,n,before", [("kn", 40, 512, 192, False), ("kn", 40, 200, 100, False),
                                                 ("nk", 40, 200, 100, False), ("kn", 40, 200, 100, True),
                                                 ("nk", 40, 200, 100, True)])
def test_in_place_under_capture(layout, m, k, n, before):
    """In a graph, with and without room in the context's buffers; a larger product afterwards grows (and so frees) them."""
    import siliconed_amd as sq
    x, q, s, b = _operands(m, k, n, 9)
    w = q if layout == "nk" else q.t().contiguous()
    want = (x.double() @ q.double().t() * s.double()).float() + b
    stream = torch.cuda.Stream()
    ctx = sq.TensorGEMM.make(0, stream)
    y = torch.zeros((m, n), device=DEV)
    torch.cuda.synchronize()
    if before:
        with torch.cuda.stream(stream):
            ctx.product(x, w, s, layout=layout, bias=b, out=y)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.product(x, w, s, layout=layout, bias=b, out=y)
    for i in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(y, want, rtol=2e-6, atol=1e-6)
        if k % 256:
            with torch.cuda.stream(stream):  # eager, larger each time
                big = [t.repeat(i + 2, 1) for t in (x, w)]
                got = ctx.product(big[0], big[1] if layout == "nk" else w, s if layout == "kn" else s.repeat(i + 2),
                                  layout=layout, bias=b if layout == "kn" else b.repeat(i + 2), out_dtype=torch.float32)
            torch.cuda.synchronize()
            assert torch.allclose(got[:m, :n], want, rtol=2e-6, atol=1e-6)


@pytest.mark.parametrize("kind", ["kn_slabs", "fp32_rounded", "fp32_route", "rotated", "padded_k", "w8a8", "w8a8_kn", "q8_kn"])
def test_graph_buffers_outlive_growth(kind):
    """A captured product that uses the context's buffers, replayed after larger products have outgrown them: the same bits as
    before the capture, and the larger products' own as on another context."""
    import siliconed_amd as sq
    k = 200 if kind == "padded_k" else 512
    x, q, s, b = _operands(40, k, 192, 11)
    a = x.float() if kind in ("fp32_rounded", "fp32_route", "w8a8", "w8a8_kn") else x
    d = torch.rand((k // 32, 192), device=DEV) * 0.02 + 1e-3

    def product(ctx, a, y):
        if kind in ("w8a8", "w8a8_kn"):
            return ctx.product_quantized(a, w, s, group=64, bias=b, out=y, layout="kn" if kind == "w8a8_kn" else "nk")
        if kind == "q8_kn":
            return ctx.product_blocks(a, w, d, 32, layout="kn", bias=b, out=y)
        return ctx.product(a, w, s, bias=b, out=y, layout="kn" if kind == "kn_slabs" else "nk", rounding=kind != "fp32_route",
                           rotation=64 if kind == "rotated" else 0)

    stream = torch.cuda.Stream()
    ctx, other = sq.TensorGEMM.make(0, stream), sq.TensorGEMM.make(0, stream)
    w = q.t().contiguous() if kind in ("kn_slabs", "w8a8_kn", "q8_kn") else ctx.pack(q, layout="nk") if kind == "padded_k" else q
    big = [a.repeat(8 << i, 1) for i in range(3)]  # each needs a larger scratch
    wide = [_operands(40, 512, 256 << i, i) for i in range(3)]  # and each a larger packing buffer
    y, want = torch.zeros((40, 192), device=DEV), torch.zeros((40, 192), device=DEV)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        product(ctx, a, want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        product(ctx, a, y)
    for rows, (xw, qw, sw, bw) in zip(big, wide):
        y.zero_()
        with torch.cuda.stream(stream):
            outs = [product(c, rows, torch.zeros((rows.shape[0], 192), device=DEV)) for c in (ctx, other)]
            outs += [c.product(xw, qw.t().contiguous(), sw, layout="kn", bias=bw) for c in (ctx, other)]
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[2], outs[3])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
    torch.cuda.synchronize()
