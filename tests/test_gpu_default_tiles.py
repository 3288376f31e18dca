"""The default tile of a matmul at shapes that take each tile of the rule, with
remainders on every edge, against the oracle: int8 bit for bit, f16 within
the contract's tolerance and bit-identical to the 256x256 tile (every tile
groups K into the same k-steps)."""
import numpy as np
import pytest
import torch

import hxm
import hxm.ops as ops
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


# (M, N, K bytes, tile): K ends inside a stage; M and N inside a tile.
SHAPES = [(260, 333, 2576, (64, 64)), (300, 4001, 1040, (64, 64)), (1001, 1500, 2576, (128, 64)),
          (1990, 2010, 400, (128, 128)), (2041, 4072, 272, (256, 128))]


@pytest.mark.parametrize("M,N,kb,tile", SHAPES)
def test_default_tile_int8(dev, M, N, kb, tile):
    g = torch.Generator().manual_seed(M)
    A = torch.randint(-127, 128, (M, kb), generator=g, dtype=torch.int8)
    B = torch.randint(-127, 128, (N, kb), generator=g, dtype=torch.int8)
    print(f"int8 {M}x{N}x{kb}", flush=True)
    C = ops.gemm_i8(A.to(dev), B.to(dev), b_layout="nk")
    assert ops.last_plan()["config"][:2] == tile
    assert np.array_equal(C.cpu().numpy(), orc.gemm_i8(A.numpy(), B.numpy(), b_nk=True))


@pytest.mark.parametrize("M,N,kb,tile", SHAPES)
def test_default_tile_f16(dev, M, N, kb, tile):
    g = torch.Generator().manual_seed(N)
    K = kb // 2
    A = (torch.rand(M, K, generator=g) * 2 - 1).half()
    B = (torch.rand(N, K, generator=g) * 2 - 1).half()
    print(f"f16 {M}x{N}x{K}", flush=True)
    Ad, Bd = A.to(dev), B.to(dev)
    C = ops.matmul(Ad, Bd, b_layout="nk")
    assert ops.last_plan()["config"][:2] == tile
    assert torch.equal(C, ops.matmul(Ad, Bd, b_layout="nk", config=S0))
    rows = np.unique(np.linspace(0, M - 1, 16).astype(int))
    ref = orc.f16_bits_to_f32(orc.matmul(bits(A)[rows], bits(B), b_nk=True))
    np.testing.assert_allclose(C.float().cpu().numpy()[rows], ref, rtol=1e-2, atol=1e-3)


S0 = (256, 256, 64, 2, 2, 2, 1)


# Accumulating calls: (M, N, K bytes, tile, stages).
ACC = [(1500, 2047, 528, (64, 64), 2), (700, 3001, 144, (64, 64), 2), (3500, 2004, 3984, (128, 128), 2),
       (260, 333, 2576, (64, 64), 4), (1001, 1500, 2576, (128, 64), 4)]


@pytest.mark.parametrize("M,N,kb,tile,stages", ACC)
def test_default_tile_accumulating(dev, M, N, kb, tile, stages):
    g = torch.Generator().manual_seed(M + N)
    for dt, K in ((torch.int8, kb), (torch.bfloat16, kb // 2)):
        print(f"accumulate {dt} {M}x{N}x{K}", flush=True)
        if dt == torch.int8:
            A, B = (torch.randint(-127, 128, s, generator=g, dtype=dt) for s in ((M, K), (N, K)))
            C0 = torch.randint(-2**31, 2**31 - 1, (M, N), generator=g, dtype=torch.int32)
        else:
            A, B = ((torch.rand(*s, generator=g) * 2 - 1).to(dt) for s in ((M, K), (N, K)))
            C0 = torch.randn(M, N, generator=g).to(dt)
        fn = ops.gemm_i8 if dt == torch.int8 else ops.matmul
        Ad, Bd = A.to(dev), B.to(dev)
        C, D = C0.to(dev), C0.to(dev)
        fn(Ad, Bd, out=C, b_layout="nk", accumulate=True)
        plan = ops.last_plan()
        assert plan["source"] == "default"
        assert plan["config"][:2] == tile and plan["config"][5] == stages
        fn(Ad, Bd, out=D, b_layout="nk", accumulate=True,
           config=(256, 256, 128 // Ad.element_size(), 2, 2, 2, 1))
        assert torch.equal(C, D)
        if dt == torch.int8:
            ref = orc.gemm_i8(A.numpy(), B.numpy(), b_nk=True)
            ref = (ref.astype(np.int64) + C0.numpy()).astype(np.int32)   # wraps
            assert np.array_equal(C.cpu().numpy(), ref)
        else:
            rows = np.unique(np.linspace(0, M - 1, 16).astype(int))
            ref = orc.to_f32(orc.matmul(bits(A)[rows], bits(B), ab_dtype="bf16", c_dtype="f32",
                                        b_nk=True), "f32") + C0.float().numpy()[rows]
            # fp32 sums, one rounding to bf16 (2^-9 of the value)
            np.testing.assert_allclose(C.float().cpu().numpy()[rows], ref, rtol=1e-2, atol=1e-3)
