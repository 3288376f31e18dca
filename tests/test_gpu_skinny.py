"""The skinny matmul (csrc/skinny_kernel.h), the default of the W8A16 GEMMs at 1 to 64
rows, against the CPU oracle: at the edges of its row blocks (4, 16, 32,
64), with channels and K that end inside a group, a slab and a 64-byte piece
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


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 32, 33, 64])
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


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 32, 33, 64])
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
    x = torch.randn(65, 64, device=dev).half()
    W = torch.ones(32, 64, dtype=torch.int8, device=dev)
    s = torch.ones(32, device=dev)
    with pytest.raises(hxm.HxmError, match="no-kernel"):
        ops.gemm_w8a16(x, W, s, config=SKINNY)           # 65 rows
    y = ops.gemm_w8a16(x[:64], W, s, config=SKINNY)
    assert ops.last_plan()["source"] == "caller"
    hxm.lib.hxm_tune_cache_clear()
    _, rep = ops.tune_w8a16(x[:64], W, s, y, reps=3)     # the control is the default
    ctl = rep["configs"][rep["control"]]
    assert ctl["tiles"] == [16, 16, 64] and ctl["stages"] == 0
    assert all(c["verified"] for c in rep["configs"] if c["q50"] is not None)
    hxm.lib.hxm_tune_cache_clear()
