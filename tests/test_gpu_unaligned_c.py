"""Outputs whose rows start off the vector boundaries: the tile epilogues store
whole runs at any alignment, single elements only where a run straddles N.
Against the same call into an aligned output (bit for bit) and, around C, the
bytes it must leave alone."""
import pytest
import torch

import hxm.ops as ops

pytestmark = pytest.mark.gpu

TILES = [(64, 64, 128, 2, 2, 4), (128, 128, 128, 2, 2, 3), (256, 256, 128, 2, 2, 2)]


def _window(M, N, dtype, pad, off):
    """An [M, N] view with odd rows inside a guard buffer."""
    buf = torch.full((M + 2, N + pad), 7, dtype=dtype, device="cuda")
    return buf, buf[1:M + 1, off:off + N]


def _check(buf, view, want, off):
    M, N = want.shape
    assert torch.equal(view, want)
    guard = buf.clone()
    guard[1:M + 1, off:off + N] = 7
    assert torch.equal(guard, torch.full_like(buf, 7))


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N", [(1, 1), (257, 255), (130, 67), (300, 515)])
@pytest.mark.parametrize("kind", ["f16", "bf16", "f16_f32", "i8", "dequant"])
@pytest.mark.parametrize("accumulate", [False, True])
def test_matmul_rows_off_the_vector_boundary(tile, M, N, kind, accumulate):
    if kind == "dequant" and accumulate:
        pytest.skip("the dequant epilogue overwrites")
    K, g = 160, torch.Generator(device="cuda").manual_seed(3)
    eb = 1 if kind in ("i8", "dequant") else 2
    cfg = (tile[0], tile[1], tile[2] // eb, tile[3], tile[4], tile[5], 1)
    # The aligned reference: rows of a multiple of 16 elements, N + its remainder.
    pad_n = (N + 15) // 16 * 16
    if eb == 1:
        A = torch.randint(-127, 128, (M, K), generator=g, device="cuda", dtype=torch.int8)
        B = torch.randint(-127, 128, (pad_n, K), generator=g, device="cuda", dtype=torch.int8)
    else:
        dt = torch.bfloat16 if kind == "bf16" else torch.float16
        A = torch.randn(M, K, generator=g, device="cuda").to(dt)
        B = torch.randn(pad_n, K, generator=g, device="cuda").to(dt)
    out_dt = {"f16": torch.float16, "bf16": torch.bfloat16, "f16_f32": torch.float32,
              "i8": torch.int32, "dequant": torch.float16}[kind]
    rs = torch.rand(M, generator=g, device="cuda") * 0.01
    cs = torch.rand(pad_n, generator=g, device="cuda") * 0.01

    def call(n, out):
        if kind == "dequant":
            return ops.gemm_i8_dequant(A, B[:n], rs, cs[:n], out=out, b_layout="nk", config=cfg)
        f = ops.gemm_i8 if kind == "i8" else ops.matmul
        return f(A, B[:n], out=out, b_layout="nk", accumulate=accumulate, config=cfg)

    start = 7 if accumulate else 0
    want = call(pad_n, torch.full((M, pad_n), start, dtype=out_dt, device="cuda"))[:, :N]
    for pad, off in ((3, 1), (4, 3)):
        buf, view = _window(M, N, out_dt, pad, off)
        call(N, view)
        _check(buf, view, want, off)


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("M,N", [(257, 255), (130, 67)])
def test_w8a16_rows_off_the_vector_boundary(M, N, residual):
    K, g = 160, torch.Generator(device="cuda").manual_seed(5)
    pad_n = (N + 15) // 16 * 16
    cfg = (128, 128, 64, 2, 2, 3, 1)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    W = torch.randint(-127, 128, (pad_n, K), generator=g, device="cuda", dtype=torch.int8)
    s = torch.rand(pad_n, generator=g, device="cuda") * 0.01
    r = torch.randn(M, pad_n, generator=g, device="cuda").half()
    want = ops.gemm_w8a16(x, W, s, residual=r if residual else None, config=cfg)[:, :N]
    buf, view = _window(M, N, torch.float16, 4, 1)
    ops.gemm_w8a16(x, W[:N], s[:N], out=view, config=cfg,
                   residual=r[:, :N].contiguous() if residual else None)
    _check(buf, view, want, 1)


# The default tile where N is off the vector boundary: two-stage 128x128 from
# 257 tiles to 16 stages of K, not at 256 tiles nor beyond 16 stages.
@pytest.mark.parametrize("M,N,kb,two_stage", [(2050, 2011, 336, True), (1990, 2010, 400, False),
                                              (2050, 2011, 2048, True), (2050, 2011, 2064, False)])
@pytest.mark.parametrize("i8", [False, True])
def test_default_tile_at_ragged_n(M, N, kb, two_stage, i8):
    g = torch.Generator(device="cuda").manual_seed(7)
    if i8:
        A, B = (torch.randint(-127, 128, (r, kb), generator=g, device="cuda", dtype=torch.int8)
                for r in (M, N))
    else:
        A, B = (torch.randn(r, kb // 2, generator=g, device="cuda").half() for r in (M, N))
    f = ops.gemm_i8 if i8 else ops.matmul
    C = f(A, B, b_layout="nk")
    c = ops.last_plan()["config"]
    assert ((c[0], c[1], c[5]) == (128, 128, 2)) == two_stage
    assert torch.equal(C, f(A, B, b_layout="nk", config=(256, 256, 128 if i8 else 64,
                                                         2, 2, 2, 1)))
