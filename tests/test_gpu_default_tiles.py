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
