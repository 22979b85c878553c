"""The product's own tile choice, on a seeded sweep of shapes around the rule's boundaries, on an MI355X.

Every tile of the weight-direct main kernels (256- and 224-row tiles, 128/64/32-row tiles of 64-column
waves, 64 × 128 and 64 × 192 tiles of one-block waves) runs one MFMA sequence over K, so whatever the
rule picks among them gives the bits of the 128-row tiles; the skinny kernel splits K over its waves and
gives the bits of its own 32-row tiles, the short-M kernel (up to 16 rows) its own, and the K-group tiles
(the K steps split over four or two wave groups) one set of bits per group count. So the default product
equals one of those five bit for bit, and
is judged against the oracle's fp64 truth on sampled rows at the reference's bars (Diagnostic.swift:105-107,
DiagnosticProbes.swift:75-82).
"""
import random

import numpy as np
import pytest
import torch

from refgen import bitwise_equal
from test_gpu_parity import bf16_dev, dev, judge, problem, weight_tensor

pytestmark = pytest.mark.gpu

_NAMES = {"none": None, "gelu": "gelu_tanh", "silu": "silu_glu"}


def _case(i):
    rng = random.Random(4100 + i)
    k = 64 * rng.choice([1, 3, 8, 16, 48])
    # Rows and columns on both sides of the rule's boundaries (tile counts 128, 144, 256 at the heights).
    m = rng.choice([1, 17, 64, 100, 129, 256, 353, 400, 512, 704, 705, 1024, 1280, 1408, 1500, 2048, 4100])
    n = rng.choice([64, 192, 320, 1024, 1344, 2880, 3000, 3072, 4608, 6144, 9216, 12288])
    epi = rng.choice(["none", "gelu", "gelu", "silu"])
    if epi == "silu" and n % 64:
        n += 64 - n % 64
    out = rng.choice([torch.bfloat16, torch.float32])
    fp8 = rng.random() < 0.25
    layout = rng.choice(["packed", "nk"])
    return m, k, n, epi, out, fp8, layout


@pytest.mark.parametrize("i", range(80))
def test_default_tile_matches_a_fixed_tile(gemm, orc, tile_gemm, i):
    m, k, n, epi, out, fp8, layout = _case(i)
    print(f"tile rule case {i}: m {m} k {k} n {n} {epi} {out} fp8 {fp8} {layout}", flush=True)
    x, q, s, b = problem(orc, m, k, n, fp8, 4200 + i)
    w = weight_tensor(q, fp8, "nk")
    if layout == "packed":
        w = gemm.pack(w, layout="nk", glu=epi == "silu")
    ys = {}
    for name, g in (("default", gemm), ("128", tile_gemm("128")), ("s32", tile_gemm("s32")), ("gemv", tile_gemm("gemv")),
                    ("k32x32", tile_gemm("k32x32")), ("k64x128", tile_gemm("k64x128"))):
        y = g.product(bf16_dev(x), w, dev(s), layout="nk", bias=dev(b), epilogue=_NAMES[epi], out_dtype=out)
        torch.cuda.synchronize()
        ys[name] = y.float().cpu().numpy()
    assert any(bitwise_equal(ys["default"], ys[t]) == 0 for t in ("128", "s32", "gemv", "k32x32", "k64x128"))
    if m >= 31:
        judge(orc, ys["default"], x, q, fp8, s, b, epi, out, rows=orc.sample_rows(m, 32))


def _random_operands(m, k, n, f32, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((m, k), device="cuda", generator=g)
    q = torch.randint(-127, 128, (n, k), device="cuda", generator=g, dtype=torch.int8)
    s = torch.rand(n, device="cuda", generator=g) * 1e-2 + 1e-3
    return x if f32 else x.bfloat16(), q, s, torch.randn(n, device="cuda", generator=g)


@pytest.mark.parametrize("route,k,n,chunks", [
    ("bf16", 1024, 3840, (4608, 4608)), ("bf16", 3072, 3072, (5760, 4096)), ("bf16", 320, 1088, (4100, 5377)),
    ("fp32", 1024, 3072, (4096, 7168))])
def test_chunks_of_4096_rows_have_one_calls_bits(gemm, route, k, n, chunks):
    """A host's row chunks of 4096 or more give the bits of the one call over all rows (past 1024 columns)."""
    x, q, s, b = _random_operands(sum(chunks), k, n, route == "fp32", n + k)
    w = gemm.pack(q, layout="nk")
    run = lambda rows: gemm.product(rows, w, s, bias=b, out_dtype=torch.float32, rounding=route == "bf16")
    whole = run(x)
    parts = torch.cat([run(rows) for rows in x.split(chunks)])
    torch.cuda.synchronize()
    assert torch.equal(whole, parts)


@pytest.mark.parametrize("route,m,k,n", [("bf16", 2737, 3072, 3072), ("bf16", 1088, 3072, 9216), ("bf16", 333, 1024, 3072),
                                         ("fp32", 1282, 3072, 9216)])
def test_bits_do_not_depend_on_alignment_or_output_type(gemm, route, m, k, n):
    """The order of sums is the shape's alone: outputs, scales and biases off the 16-byte grid, and a bf16 output, round
    the same sums."""
    x, q, s, b = _random_operands(m, k, n, route == "fp32", n + k)
    w = gemm.pack(q, layout="nk")
    off = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)
    run = lambda s, b, out: gemm.product(x, w, s, bias=b, out=out, rounding=route == "bf16")
    want = run(s, b, torch.empty((m, n), device="cuda"))
    plain = run(s, b, torch.empty((m, n), device="cuda", dtype=torch.bfloat16))
    for dtype in (torch.float32, torch.bfloat16):
        for ss, bb in ((s, b), (off(s), off(b))):
            y = run(ss, bb, off(torch.zeros((m, n), device="cuda", dtype=dtype)))
            torch.cuda.synchronize()
            assert torch.equal(y, want if dtype == torch.float32 else plain)
    assert torch.equal(want.bfloat16(), plain)
