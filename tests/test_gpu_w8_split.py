"""The K split of the W8A16 GEMMs (csrc/gemm_w8part.hip) against the CPU oracle:
one slice to more slices than stages fill, rows and channels that end inside a
tile and a four-column run, output rows off every alignment; the untuned choice
of it; and its planes under graph capture."""
import threading

import numpy as np
import pytest
import torch

import hxm
import hxm.ops as ops
from hxm import search as S
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# fp32 sums of f16 x int8 products in any order, one f16 rounding: the
# tolerance the W8A16 entries state.
TOL = dict(rtol=1e-2, atol=1e-3)


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def operands(M, N, K, n_weights=1):
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    x = torch.randn(M, K, generator=g).half()
    W = [torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8) for _ in range(n_weights)]
    s = [torch.rand(N, generator=g) * 0.004 + 0.001 for _ in range(n_weights)]
    return g, x, W, s


def padded(M, N, dev, pad):
    buf = torch.full((M + 1, N + pad), 7.0, dtype=torch.float16, device=dev)
    return buf, buf[:M, :N]


def untouched(buf, M, N):
    return bool((buf[:, N:] == 7).all() and (buf[M:] == 7).all())


@pytest.mark.parametrize("M,N,K,S", [(1, 1, 16, 2), (57, 333, 656, 2), (128, 128, 1024, 16),
                                     (129, 130, 2064, 5), (57, 258, 1040, 16), (300, 515, 720, 3)])
@pytest.mark.parametrize("tile,pad", [((128, 128, 64, 2, 2, 3), 0), ((128, 128, 64, 2, 2, 3), 3),
                                      ((64, 128, 64, 1, 2, 4), 1)])
def test_against_oracle(dev, M, N, K, S, tile, pad):
    print(f"w8 split M={M} N={N} K={K} S={S} tile={tile} pad={pad}", flush=True)
    cfg = tile + (S,)
    g, x, (W,), (s,) = operands(M, N, K)
    r = (4 * torch.randn(M, N, generator=g)).half()
    buf, y = padded(M, N, dev, pad)
    ops.gemm_w8a16(x.to(dev), W.to(dev), s.to(dev), out=y, config=cfg)
    assert ops.last_plan()["config"] == cfg
    ref = orc.f16_bits_to_f32(orc.gemm_w8a16(bits(x), W.numpy(), s.numpy()))
    np.testing.assert_allclose(y.float().cpu().numpy(), ref, **TOL)
    assert untouched(buf, M, N)
    buf, z = padded(M, N, dev, pad)                  # in place: out is the residual
    z.copy_(r)
    ops.gemm_w8a16(x.to(dev), W.to(dev), s.to(dev), out=z, residual=z, config=cfg)
    ref = orc.f16_bits_to_f32(orc.gemm_w8a16_residual(bits(x), W.numpy(), s.numpy(), bits(r)))
    np.testing.assert_allclose(z.float().cpu().numpy(), ref, **TOL)
    assert untouched(buf, M, N)

    _, x, (Wg, Wu), (sg, su) = operands(M, N, K, 2)
    Wgu, sgu = ops.swiglu_pack(Wg.to(dev), Wu.to(dev), sg.to(dev), su.to(dev))
    buf, h = padded(M, N, dev, pad)
    ops.gemm_w8a16_swiglu(x.to(dev), Wgu, sgu, N, out=h, config=cfg)
    ref = orc.f16_bits_to_f32(orc.swiglu_gateup(bits(x), Wg.numpy(), Wu.numpy(), sg.numpy(),
                                                su.numpy()))
    np.testing.assert_allclose(h.float().cpu().numpy(), ref, **TOL)
    assert untouched(buf, M, N)


def test_untuned_choice_and_capture(dev, tmp_path):
    """57 rows of a long K are split when untuned, and by a tuned winner that is
    a split.  A capture of either runs unsplit, also on a stream that has the
    planes: its graph holds no workspace, so graphs captured on one stream
    replay at once, beside an eager split call of that stream."""
    g, x, (W,), (s,) = operands(57, 1024, 8192)
    xs = [x.to(dev), torch.randn(57, 8192, generator=g).half().to(dev)]
    W, s = W.to(dev), s.to(dev)
    ys = [torch.empty(57, 1024, dtype=torch.float16, device=dev) for _ in xs]
    eager = torch.empty_like(ys[0])
    hxm.lib.hxm_tune_cache_clear()
    cache = tmp_path / "tune.txt"
    S.tune_cache_save(str(cache))                    # this build's header
    with open(cache, "a") as f:
        f.write("16 57 1024 8192 128 128 64 2 2 3 4 3\n")
    others = [torch.cuda.Stream(), torch.cuda.Stream()]
    try:
        for tuned in (False, True):
            print(f"capture tuned={tuned}", flush=True)
            if tuned:
                assert S.tune_cache_load(str(cache)) == 1
            warm = torch.cuda.Stream()
            with torch.cuda.stream(warm):
                ops.gemm_w8a16(xs[1], W, s, out=eager)
            plan = ops.last_plan()
            assert plan["source"] == ("tuned" if tuned else "default")
            assert plan["config"][6] > 1 and plan["workspace_bytes"] > 0
            torch.cuda.synchronize()
            split = eager.clone()
            graphs = []
            for xi, yi in zip(xs, ys):
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=warm):
                    ops.gemm_w8a16(xi, W, s, out=yi)
                plan = ops.last_plan()
                assert plan["config"][6] <= 1 and plan["workspace_bytes"] == 0
                graph.replay()
                torch.cuda.synchronize()
                graphs.append(graph)
            want = [y.clone() for y in ys]
            for xi, w in zip(xs, want):
                ref = orc.f16_bits_to_f32(orc.gemm_w8a16(bits(xi), W.cpu().numpy(),
                                                         s.cpu().numpy()))
                np.testing.assert_allclose(w.float().cpu().numpy(), ref, **TOL)
            for rep in range(20):
                for y in ys + [eager]:
                    y.fill_(-7.0)
                torch.cuda.synchronize()
                for graph, st in zip(graphs, others):
                    with torch.cuda.stream(st):
                        graph.replay()
                with torch.cuda.stream(warm):
                    ops.gemm_w8a16(xs[1], W, s, out=eager)
                torch.cuda.synchronize()
                for y, w in zip(ys, want):
                    assert torch.equal(y, w), rep
                assert torch.equal(eager, split), rep
    finally:
        hxm.lib.hxm_tune_cache_clear()


def test_requested_split_in_a_graph(dev):
    """A split asked for by config is captured with the stream's planes: its
    replays give the eager call's bits, also after the planes have grown."""
    cfg = (128, 128, 64, 2, 2, 3, 4)
    _, x, (W,), (s,) = operands(57, 1024, 8192)
    x, W, s = x.to(dev), W.to(dev), s.to(dev)
    y = torch.empty(57, 1024, dtype=torch.float16, device=dev)
    warm = torch.cuda.Stream()
    with torch.cuda.stream(warm):
        ops.gemm_w8a16(x, W, s, out=y, config=cfg)
    torch.cuda.synchronize()
    want = y.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=warm):
        ops.gemm_w8a16(x, W, s, out=y, config=cfg)
    assert ops.last_plan()["config"] == cfg
    big = torch.randn(512, 8192, device=dev).half()
    with torch.cuda.stream(warm):                    # grows that stream's planes
        ops.gemm_w8a16(big, W, s, config=cfg[:6] + (16,))
    for rep in range(3):
        y.fill_(-7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), rep


def test_planes_grow_beside_a_capture(dev):
    """An untuned call that takes its planes for the first time, then one that
    has to grow them, on another thread and stream while a graph is captured:
    the capture stays valid."""
    g, x, (W,), (s,) = operands(57, 1024, 8192)
    xs = [x.to(dev), torch.randn(200, 8192, generator=g).half().to(dev)]
    W, s = W.to(dev), s.to(dev)
    ys = [torch.empty(xi.shape[0], 1024, dtype=torch.float16, device=dev) for xi in xs]
    a = torch.randn(64, 4096, generator=g).half().to(dev)
    o = torch.empty_like(a)
    ops.softmax(a, out=o)
    torch.cuda.synchronize()
    want = o.clone()
    other, stream, plans, errors = torch.cuda.Stream(), torch.cuda.Stream(), [], []
    hxm.lib.hxm_release_cache()                      # no planes on any stream

    def work():
        try:
            for xi, yi in zip(xs, ys):
                ops.gemm_w8a16(xi, W, s, out=yi, stream=other)
                plans.append(ops.last_plan())
        except Exception as e:                       # reported by the main thread
            errors.append(e)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        t = threading.Thread(target=work)
        t.start()
        t.join()
        ops.softmax(a, out=o)
    assert not errors
    assert all(p["config"][6] > 1 for p in plans)
    assert plans[1]["workspace_bytes"] > max(plans[0]["workspace_bytes"], 1 << 20)
    for xi, yi in zip(xs, ys):
        ref = orc.f16_bits_to_f32(orc.gemm_w8a16(bits(xi), W.cpu().numpy(), s.cpu().numpy()))
        np.testing.assert_allclose(yi.float().cpu().numpy(), ref, **TOL)
    for rep in range(3):
        o.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want), rep
