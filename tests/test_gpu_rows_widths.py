"""Row kernels at the widths where the launch changes (waves per row, vectors
per lane, four rows to a wave, the streamed rows), one element either side of
each, against the oracle: rows that start off the 16-byte boundary, with a
leading dimension that is no multiple of a vector, into an output whose
padding must keep its fill."""
import numpy as np
import pytest
import torch

import hxm.ops as ops
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

TDT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
# rtol 1e-2 / atol 1e-3 is the 16-bit contract.  f32: sums of up to 131073 terms
# in another order than the oracle's, the mean's rounding scaled by rstd.
TOL = {"f16": dict(rtol=1e-2, atol=1e-3), "bf16": dict(rtol=1e-2, atol=1e-3),
       "f32": dict(rtol=1e-4, atol=1e-5)}
EDGES = (64, 128, 192, 256, 384, 512, 768, 1024, 1536, 2048, 3072, 4096, 8192, 16384)


def bits(t, name):
    t = t.contiguous().cpu()
    return t.numpy() if name == "f32" else t.view(torch.int16).numpy().view(np.uint16)


def check(dev, name, rows, cols):
    print(f"{name} {rows}x{cols}", flush=True)
    g = torch.Generator().manual_seed(rows + cols)
    x = (2 * torch.randn(rows, cols, generator=g) + 0.5).to(TDT[name])
    if cols > 2:
        x[0, cols // 2:] = torch.finfo(TDT[name]).min    # a mask of the lowest value
    w = (1 + 0.1 * torch.randn(cols, generator=g)).to(TDT[name])
    b = (0.1 * torch.randn(cols, generator=g)).to(TDT[name])
    xbuf = torch.full((rows * (cols + 3) + 1,), float("nan"), dtype=TDT[name], device=dev)
    xd = xbuf[1:].view(rows, cols + 3)[:, :cols]         # off by one element, ld = cols + 3
    xd.copy_(x)
    ybuf = torch.full((rows, cols + 5), 7.0, dtype=TDT[name], device=dev)
    y = ybuf[:, :cols]
    wd, bd = w.to(dev), b.to(dev)
    ops.softmax(xd, out=y)
    ref = orc.to_f32(orc.softmax_rows(bits(x, name), name), name)
    np.testing.assert_allclose(y.float().cpu().numpy(), ref, **TOL[name], err_msg="softmax")
    x[0] = x[-1]                                         # the norms on ordinary values
    xd.copy_(x)
    ops.rms_norm(xd, (cols,), wd, eps=1e-6, out=y)
    ref = orc.to_f32(orc.rmsnorm_rows(bits(x, name), bits(w, name), 1e-6, name), name)
    np.testing.assert_allclose(y.float().cpu().numpy(), ref, **TOL[name], err_msg="rms_norm")
    _, mean, rstd = ops.layer_norm(xd, (cols,), wd, bd, eps=1e-5, out=y, return_stats=True)
    ry, rmean, rrstd = orc.layernorm_rows(bits(x, name), bits(w, name), bits(b, name), 1e-5, name)
    np.testing.assert_allclose(y.float().cpu().numpy(), orc.to_f32(ry, name), **TOL[name],
                               err_msg="layer_norm")
    np.testing.assert_allclose(mean.cpu().numpy(), rmean, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(rstd.cpu().numpy(), rrstd, rtol=1e-4)
    assert (ybuf[:, cols:] == 7).all(), "wrote past the row"


@pytest.mark.parametrize("nv", EDGES)
@pytest.mark.parametrize("name", ["f16", "bf16", "f32"])
def test_widths(dev, name, nv):
    cols = nv * (4 if name == "f32" else 8)
    for c in (cols - 1, cols, cols + 1):
        check(dev, name, 3, c)


@pytest.mark.parametrize("nv", [1, 16, 32, 48, 63])
@pytest.mark.parametrize("name", ["f16", "bf16", "f32"])
def test_many_short_rows(dev, name, nv):
    cols = nv * (4 if name == "f32" else 8)
    for c in (max(1, cols - 1), cols, cols + 1):
        check(dev, name, 2051, c)


def extreme_rows(name, cols, g):
    """Softmax rows whose maximum is large: wholly masked ones (the lowest value,
    -1e10), one peak near the largest value, and steps of one unit or less at
    growing offsets, where a scaled maximum rounds by more than the steps."""
    big = torch.finfo(TDT[name]).max
    ten = 1e10 if name != "f16" else 6e4
    x = [torch.full((cols,), v) for v in (-big, -ten, ten, big)]
    x.append(2 * torch.randn(cols, generator=g))
    x[-1][cols // 3] = big * 0.88
    x.append(torch.where(torch.arange(cols) % 3 == 0, big, -big))
    steps = -torch.randint(0, 40, (cols,), generator=g) * 0.5
    x += [steps + off for off in (1e3, -1e3, 4e4, -4e4)]
    if name != "f16":
        x += [steps + off for off in (4194300.0, -4194300.0, 4194400.0, -4194400.0)]
        x += [v * (1 + steps / 3e7) for v in (3.5e9, -3.5e9, 2e38, -2e38)]
    return torch.stack(x).to(TDT[name])


@pytest.mark.parametrize("nv", [1, 16, 48, 63] + list(EDGES))
@pytest.mark.parametrize("name", ["f16", "bf16", "f32"])
def test_softmax_of_large_maxima(dev, name, nv):
    for c in (-1, 0, 1):
        cols = nv * (4 if name == "f32" else 8) + c
        x = extreme_rows(name, cols, torch.Generator().manual_seed(cols))
        if nv < 64:
            x = x.repeat(2048 // len(x) + 1, 1)          # four short rows to a wave
        print(f"{name} {tuple(x.shape)}", flush=True)
        y = ops.softmax(x.to(dev)).float().cpu().numpy()
        ref = orc.to_f32(orc.softmax_rows(bits(x, name), name), name)
        np.testing.assert_allclose(y, ref, **TOL[name])
        np.testing.assert_allclose(y.sum(1, dtype=np.float64), 1, rtol=1e-2)
