"""Operand packs (csrc/pack.hip) at the edges of their 128-byte tiles: the [K, N] ->
[N, K] image is the transpose bit for bit, from sources that start and stride
off any boundary into images of any row stride (whose padding keeps its
fill), and the f32 operands of a matmul reach the fp16 MFMA as
float16(x + 0.0), zero past K."""
import numpy as np
import pytest
import torch

import hxm.ops as ops

pytestmark = pytest.mark.gpu

EDGES = [(1, 1), (16, 3), (63, 65), (64, 64), (65, 63), (127, 129), (128, 128), (129, 200),
         (300, 131)]


@pytest.mark.parametrize("K,N", EDGES)
@pytest.mark.parametrize("dt", [torch.int8, torch.float16, torch.bfloat16])
def test_prepack_is_the_transpose_at_tile_edges(dev, dt, K, N):
    print(f"prepack {dt} {K}x{N}", flush=True)
    g = torch.Generator().manual_seed(K + N)
    B = torch.randint(-127, 128, (K, N), generator=g).to(dt)
    for off, pad, opad in ((0, 0, 0), (1, 3, 5)):
        buf = torch.full((K * (N + pad) + off,), 77, dtype=torch.int32).to(dt).to(dev)
        src = buf[off:].view(K, N + pad)[:, :N]
        src.copy_(B)
        obuf = torch.full((N * (K + opad) + off,), 55, dtype=torch.int32).to(dt).to(dev)
        out = obuf[off:].view(N, K + opad)[:, :K]
        ops.prepack_weight(src, out)
        assert torch.equal(out.cpu(), B.t())
        rest = obuf[off:].view(N, K + opad)[:, K:]
        assert (rest == 55).all() and (obuf[:off] == 55).all(), "wrote outside the image"


@pytest.mark.parametrize("K", [1, 7, 8, 9, 63, 64, 65, 130])
@pytest.mark.parametrize("layout", ["kn", "nk"])
def test_f32_operands_are_quantised_exactly(dev, layout, K):
    """One operand the identity: each output is one fp16 value of the other."""
    g = torch.Generator().manual_seed(K)
    X = (4 * torch.randn(70, K + 3, generator=g)).to(dev)[:, 1:1 + K]   # off the 16-byte grid
    eye = torch.eye(K, device=dev)
    want = (X.cpu() + 0.0).half()
    assert torch.equal(ops.matmul(X, eye, b_layout=layout, out_dtype=torch.float16).cpu(), want)
    Xt = X if layout == "nk" else X.t().contiguous()                    # X as B
    got = ops.matmul(eye, Xt, b_layout=layout, out_dtype=torch.float16).cpu()
    assert torch.equal(got, want.t())


def test_resident_f32_image_at_tile_edges(dev):
    for K, N in ((64, 64), (72, 130), (200, 65)):
        B = torch.randn(K, N, generator=torch.Generator().manual_seed(K)).to(dev)
        img = ops.resident_weight(B)
        assert torch.equal(img.cpu(), (B.cpu() + 0.0).half().t())
