"""The skinny matmul (csrc/skinny_kernel.h), the default of the matmuls of few
rows, against the CPU oracle: at the edges of its row blocks (4, 16, 32,
64, several of 64), with channels and K that end inside a group, a slab and a 64-byte piece
of one.  Operands are views of wider buffers whose padding holds NaN (x) or
127 (W), so a chunk read past K or M would show, and the output's padding
must keep its fill."""
import numpy as np
import pytest
import torch

import hxm
import hxm.ops as ops
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# fp32 sums of f16 x int8 products in any order, one f16 rounding: the
# tolerance the W8A16 entries state.
TOL = dict(rtol=1e-2, atol=1e-3)
SKINNY = (16, 16, 64, 1, 8, 0, 1)


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def padded(t, fill, dev, rows=3, cols=16):
    """t as a view of a wider buffer on the GPU filled with `fill`."""
    buf = torch.full((t.shape[0] + rows, t.shape[1] + cols), fill, dtype=t.dtype, device=dev)
    v = buf[:t.shape[0], :t.shape[1]]
    v.copy_(t)
    return buf, v


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 32, 33, 64, 65, 256])
@pytest.mark.parametrize("N,K", [(8, 16), (100, 112), (333, 656), (272, 2064)])
def test_w8a16_and_residual(dev, M, N, K):
    print(f"skinny w8a16 M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    x = torch.randn(M, K, generator=g).half()
    W = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    s = (torch.rand(N, generator=g) * 0.019 + 0.001).half().float()
    r = (4 * torch.randn(M, N, generator=g)).half()
    _, xd = padded(x, float("nan"), dev)
    _, Wd = padded(W, 127, dev)
    ybuf, y = padded(torch.zeros(M, N).half(), 7.0, dev)
    ops.gemm_w8a16(xd, Wd, s.to(dev), out=y)
    assert ops.last_plan()["config"] == SKINNY
    ref = orc.f16_bits_to_f32(orc.gemm_w8a16(bits(x), W.numpy(), s.numpy()))
    np.testing.assert_allclose(y.float().cpu().numpy(), ref, **TOL)
    assert (ybuf[:, N:] == 7).all() and (ybuf[M:] == 7).all()
    _, z = padded(r, 7.0, dev)                       # in place: out is the residual
    ops.gemm_w8a16(xd, Wd, s.to(dev), out=z, residual=z)
    ref = orc.f16_bits_to_f32(orc.gemm_w8a16_residual(bits(x), W.numpy(), s.numpy(), bits(r)))
    np.testing.assert_allclose(z.float().cpu().numpy(), ref, **TOL)


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 32, 33, 64, 150])
@pytest.mark.parametrize("I,K", [(16, 16), (100, 656), (200, 1040)])
def test_swiglu(dev, M, I, K):
    print(f"skinny swiglu M={M} I={I} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + I + K)
    x = torch.randn(M, K, generator=g).half()
    Wg, Wu = (torch.randint(-127, 128, (I, K), generator=g, dtype=torch.int8) for _ in range(2))
    sg, su = (torch.rand(I, generator=g) * 0.004 + 0.001 for _ in range(2))
    Wgu, sgu = ops.swiglu_pack(Wg.to(dev), Wu.to(dev), sg.to(dev), su.to(dev))
    _, xd = padded(x, float("nan"), dev)
    hbuf, h = padded(torch.zeros(M, I).half(), 7.0, dev)
    ops.gemm_w8a16_swiglu(xd, Wgu, sgu, I, out=h)
    assert ops.last_plan()["config"] == SKINNY
    ref = orc.f16_bits_to_f32(orc.swiglu_gateup(bits(x), Wg.numpy(), Wu.numpy(), sg.numpy(),
                                                su.numpy()))
    np.testing.assert_allclose(h.float().cpu().numpy(), ref, **TOL)
    assert (hbuf[:, I:] == 7).all() and (hbuf[M:] == 7).all()


@pytest.mark.parametrize("M", [1, 16, 40, 64])
def test_exact_sums_match_the_tiles_bit_for_bit(dev, M):
    """Small integers: every summation order gives the same fp32 sum, so the
    skinny kernel and a staged tile must agree to the bit.  SwiGLU's last
    product is not pinned in fp32 (the compiler may round it once, to f16, or
    twice), so there the two may differ by one f16 ulp, 2^-10 of the value
    (2^-24 below the normal range)."""
    g = torch.Generator().manual_seed(M)
    N, K = 200, 512
    x = torch.randint(-4, 5, (M, K), generator=g).half().to(dev)
    W = torch.randint(-8, 9, (N, K), generator=g, dtype=torch.int8).to(dev)
    s = (torch.rand(N, generator=g) + 0.5).to(dev)
    r = torch.randn(M, N, generator=g).half().to(dev)
    tile = ops.w8a16_configs(swiglu=True)[0]
    for res in (None, r):
        assert torch.equal(ops.gemm_w8a16(x, W, s, residual=res),
                           ops.gemm_w8a16(x, W, s, residual=res, config=tile))
    Wgu, sgu = ops.swiglu_pack(W, W, s * 0.01, s * 0.01)
    np.testing.assert_allclose(ops.gemm_w8a16_swiglu(x, Wgu, sgu, N).float().cpu().numpy(),
                               ops.gemm_w8a16_swiglu(x, Wgu, sgu, N,
                                                     config=tile).float().cpu().numpy(),
                               rtol=2.0 ** -10, atol=2.0 ** -24)


def test_named_config_and_tuner(dev):
    x = torch.randn(257, 64, device=dev).half()
    W = torch.ones(32, 64, dtype=torch.int8, device=dev)
    s = torch.ones(32, device=dev)
    with pytest.raises(hxm.HxmError, match="no-kernel"):
        ops.gemm_w8a16(x, W, s, config=SKINNY)           # 257 rows
    y = ops.gemm_w8a16(x[:64], W, s, config=SKINNY)
    assert ops.last_plan()["source"] == "caller"
    hxm.lib.hxm_tune_cache_clear()
    _, rep = ops.tune_w8a16(x[:64], W, s, y, reps=3)     # the control is the default
    ctl = rep["configs"][rep["control"]]
    assert ctl["tiles"] == [16, 16, 64] and ctl["stages"] == 0
    assert all(c["verified"] for c in rep["configs"] if c["q50"] is not None)
    hxm.lib.hxm_tune_cache_clear()


@pytest.mark.parametrize("M", [1, 5, 17, 32, 33, 64, 100])
@pytest.mark.parametrize("N,K", [(8, 2048), (333, 2064), (40, 272)])
def test_int8(dev, M, N, K):
    """int32 (plain and accumulated) and dequant outputs, bit for bit."""
    print(f"skinny int8 M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    B = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    _, Ad = padded(A, 111, dev)
    _, Bd = padded(B, 111, dev)
    ref = orc.gemm_i8(A.numpy(), B.numpy(), b_nk=True)
    C0 = torch.randint(-1000, 1000, (M, N), generator=g, dtype=torch.int32)
    cbuf, c = padded(C0, 7, dev)
    ops.gemm_i8(Ad, Bd, out=c, b_layout="nk", config=SKINNY)
    assert np.array_equal(c.cpu().numpy(), ref)
    c.copy_(C0)
    ops.gemm_i8(Ad, Bd, out=c, b_layout="nk", accumulate=True, config=SKINNY)
    assert np.array_equal(c.cpu().numpy(), ref + C0.numpy())
    assert (cbuf[:, N:] == 7).all() and (cbuf[M:] == 7).all()
    rs, cs = (torch.rand(n, generator=g) * 0.019 + 0.001 for n in (M, N))
    D = ops.gemm_i8_dequant(Ad, Bd, rs.to(dev), cs.to(dev), b_layout="nk", config=SKINNY)
    assert np.array_equal(bits(D), orc.dequant_f16(ref, rs.numpy(), cs.numpy()))


@pytest.mark.parametrize("M", [1, 5, 17, 32, 33, 64, 100])
@pytest.mark.parametrize("N,K", [(8, 1024), (333, 1032), (40, 136)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_float(dev, dt, M, N, K):
    """f16 / bf16 operands into f32 (accumulated too) and their own dtype; the
    padding of A and B is NaN."""
    print(f"skinny {dt} M={M} N={N} K={K}", flush=True)
    name = "f16" if dt == torch.float16 else "bf16"
    g = torch.Generator().manual_seed(M + N + K)
    A = (torch.rand(M, K, generator=g) * 2 - 1).to(dt)
    B = (torch.rand(N, K, generator=g) * 2 - 1).to(dt)
    _, Ad = padded(A, float("nan"), dev)
    _, Bd = padded(B, float("nan"), dev)
    C0 = torch.randn(M, N, generator=g)
    ref = orc.matmul(bits(A), bits(B), ab_dtype=name, c_dtype="f32", b_nk=True)
    cbuf, c = padded(C0, 7.0, dev)
    ops.matmul(Ad, Bd, out=c, b_layout="nk", config=SKINNY)
    np.testing.assert_allclose(c.cpu().numpy(), ref, rtol=1e-4, atol=1e-4)
    c.copy_(C0)
    ops.matmul(Ad, Bd, out=c, b_layout="nk", accumulate=True, config=SKINNY)
    np.testing.assert_allclose(c.cpu().numpy(), ref + C0.numpy(), rtol=1e-4, atol=1e-4)
    assert (cbuf[:, N:] == 7).all() and (cbuf[M:] == 7).all()
    h = ops.matmul(Ad, Bd, b_layout="nk", config=SKINNY)
    np.testing.assert_allclose(h.float().cpu().numpy(), ref, rtol=1e-2, atol=1e-3)


# The GEMV takes any number of rows, 16 at a time: 261 and 300 end in partial blocks
# past the row limit of the GEMMs.
@pytest.mark.parametrize("M", [2, 4, 5, 16, 17, 40, 261, 300])
@pytest.mark.parametrize("N,K", [(40, 16), (333, 656), (100, 2064)])
def test_gemv_plain_weights(dev, M, N, K):
    print(f"skinny gemv M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).half()
    W = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    s = (torch.rand(N, generator=g) * 0.019 + 0.001).half()
    _, xd = padded(x, float("nan"), dev)
    _, Wd = padded(W, 127, dev)
    ybuf, y = padded(torch.zeros(M, N).half(), 7.0, dev)
    ops.gemv_w8a16(xd, Wd, s.to(dev), out=y)
    ref = orc.f16_bits_to_f32(orc.gemv_w8a16(bits(x), W.numpy(), bits(s)))
    np.testing.assert_allclose(y.float().cpu().numpy(), ref, **TOL)
    assert (ybuf[:, N:] == 7).all() and (ybuf[M:] == 7).all()


@pytest.mark.parametrize("M", [1, 5, 32, 33, 100])
@pytest.mark.parametrize("N,K", [(16, 16), (33, 272), (100, 2064), (333, 144)])
def test_int8_reads_kn_operands_as_they_are(dev, M, N, K):
    """A [K, N] B without a transposed copy, from rows off any alignment."""
    print(f"skinny int8 kn M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    B = torch.randint(-127, 128, (K, N), generator=g, dtype=torch.int8)
    _, Ad = padded(A, 111, dev)
    ref = orc.gemm_i8(A.numpy(), B.numpy())
    for cols in (0, 3):
        _, Bd = padded(B, 111, dev, rows=0, cols=cols)
        C = ops.gemm_i8(Ad, Bd, config=SKINNY)
        assert ops.last_plan()["workspace_bytes"] == 0
        assert np.array_equal(C.cpu().numpy(), ref)


@pytest.mark.parametrize("M", [1, 5, 32, 33, 100])
@pytest.mark.parametrize("N,K", [(8, 8), (9, 136), (33, 1032), (333, 72)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_float_reads_kn_operands_as_they_are(dev, dt, M, N, K):
    print(f"skinny kn {dt} M={M} N={N} K={K}", flush=True)
    name = "f16" if dt == torch.float16 else "bf16"
    g = torch.Generator().manual_seed(M + N + K)
    A = (torch.rand(M, K, generator=g) * 2 - 1).to(dt)
    B = (torch.rand(K, N, generator=g) * 2 - 1).to(dt)
    _, Ad = padded(A, float("nan"), dev)
    ref = orc.matmul(bits(A), bits(B), ab_dtype=name, c_dtype="f32")
    for cols in (0, 3):
        _, Bd = padded(B, float("nan"), dev, rows=0, cols=cols)
        c = ops.matmul(Ad, Bd, out_dtype=torch.float32, config=SKINNY)
        np.testing.assert_allclose(c.cpu().numpy(), ref, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("M,N,K", [(16, 8, 8), (17, 9, 40), (33, 31, 72), (100, 70, 200),
                                   (256, 256, 256), (1, 500, 128)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_small_output_kernel_reads_kn_operands_as_they_are(dev, dt, M, N, K):
    """The small-output kernel on a plain [K, N] B off any alignment gives the
    bits it gives on the [N, K] image."""
    print(f"small kn {dt} M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    A = (torch.rand(M, K, generator=g) * 2 - 1).to(dt).to(dev)
    B = (torch.rand(K, N, generator=g) * 2 - 1).to(dt)
    want = ops.matmul(A, B.t().contiguous().to(dev), b_layout="nk")
    for cols in (0, 3):
        _, Bd = padded(B, float("nan"), dev, rows=0, cols=cols)
        got = ops.matmul(A, Bd)
        assert ops.last_plan()["config"] == (16, 16, 32, 1, 1, 0, 1)
        assert torch.equal(got, want)
