"""GPU: the prompt GEMM (the engine's projections of 17 to 768 tokens)."""
import pytest
import torch

import my_cuda_engine_cpp as ops
from mycustomcudaengine_amd import _lib
from mycustomcudaengine_amd.engine.projections import (linear, linear_add, linear_add_norm,
                                                       linear_swiglu)

pytestmark = pytest.mark.gpu


def rnd(dev, *shape, dtype=torch.float16, std=1.0, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed + sum(shape))
    return torch.empty(*shape, dtype=dtype, device=dev).normal_(0, std, generator=g)


def close(out, ref, dtype, k):
    """Half an ulp of the output plus fp32 sums of k products."""
    tol = (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) + k * 2.0 ** -24
    err = (out.double() - ref).abs()
    assert (err <= tol * ref.abs() + 4 * k ** 0.5 * 2.0 ** -24 + 1e-3 * 2.0 ** -11).all(), err.max().item()


# every tile (64, 128 and 256 tokens) at its smallest and largest, one token
# past it, and token counts that leave a tile's last rows empty; K cut into
# slices (few columns) and whole (many), K not a multiple of the slices.  (n
# from 2048 up: SwiGLU's n / 2 columns below 1024 go to the library, which
# rounds gate and up to 16 bits first and is outside the bound.)
@pytest.mark.parametrize("m", [17, 64, 65, 128, 129, 256, 257, 384, 385, 512])
@pytest.mark.parametrize("n,k", [(2048, 2048), (3072, 8192), (9216, 2112)])
def test_projections_match_fp64(dev, m, n, k):
    dtype = torch.float16 if (m + n) % 2 else torch.bfloat16
    x, w = rnd(dev, m, k + 8, dtype=dtype)[:, 8:], rnd(dev, n, k, dtype=dtype, std=k ** -0.5)
    acc = x.double() @ w.double().T
    close(linear(x, w), acc, dtype, k)
    g, u = acc.chunk(2, 1)
    # SwiGLU: an fp32 sum of k products of unit-variance sums is off by about
    # d = sqrt(k) 2^-24 (4 d at most here), and |d(silu(g) u)| <= 1.1 (|u| dg + |g| du)
    out, ref = linear_swiglu(x, w).double(), torch.nn.functional.silu(g) * u
    tol = 2.0 ** (-10 if dtype == torch.float16 else -7)
    d = 4 * k ** 0.5 * 2.0 ** -24
    assert ((out - ref).abs() <= tol * ref.abs() + 1.1 * d * (g.abs() + u.abs()) + 2.0 ** -24).all()
    res = rnd(dev, m, n, dtype=dtype, seed=1)
    want = res.double() + acc
    a = res.clone()
    linear_add(x, w, a)
    close(a, want, dtype, k)


# the residual add's own sizes: short K on the 128-token tile to 448, long K on
# the 256-token tile past 512; the store's multiples of 32
@pytest.mark.parametrize("m,n,k,add", [(385, 3072, 3072, True), (448, 3072, 3072, True),
                                       (513, 3072, 8192, True), (768, 3072, 8192, True),
                                       (160, 5120, 3072, False), (224, 5120, 3072, False)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_sizes_of_one_epilogue(dev, m, n, k, add, dtype):
    assert _lib.load().mce_prompt_gemm_takes(m, n, k, 1 if add else 0)
    x, w = rnd(dev, m, k, dtype=dtype), rnd(dev, n, k, dtype=dtype, std=k ** -0.5)
    acc = x.double() @ w.double().T
    if not add:
        close(linear(x, w), acc, dtype, k)
        return
    a, nw = rnd(dev, m, n, dtype=dtype, seed=1), rnd(dev, n, dtype=dtype)
    want = a.double() + acc
    y = linear_add_norm(x, w, a, nw, 1e-5)
    close(a, want, dtype, k)
    assert torch.equal(y, ops.rmsnorm(a, nw, 1e-5))


@pytest.mark.parametrize("m,n,k", [(17, 2048, 2048), (100, 3072, 8192), (256, 3072, 3072),
                                   (500, 3072, 8192), (300, 4096, 6144), (40, 5120, 2048)])
def test_add_norm_equals_add_then_rmsnorm(dev, m, n, k):
    """The norm that comes with the residual add has rmsnorm()'s bits for the
    updated rows, and the residual those of the add alone."""
    x, w, nw = rnd(dev, m, k), rnd(dev, n, k, std=k ** -0.5), rnd(dev, n)
    a = rnd(dev, m, n, seed=2)
    b = a.clone()
    y = linear_add_norm(x, w, a, nw, 1e-5)
    linear_add(x, w, b)
    assert torch.equal(a, b) and torch.equal(y, ops.rmsnorm(a, nw, 1e-5))


def test_first_call_binds_the_library(dev, monkeypatch):
    """A process whose first op is a projection takes the same path as a later one."""
    calls = []
    load = _lib.load
    monkeypatch.setattr(_lib, "load", lambda: calls.append(1) or load())
    linear(rnd(dev, 64, 2048), rnd(dev, 1024, 2048, std=0.02))
    assert calls


def test_takes_and_leaves(dev):
    """Sizes outside its rule, autograd and odd layouts go to the library."""
    lib = _lib.load()
    takes = lib.mce_prompt_gemm_takes
    assert takes(160, 5120, 3072, 0) and takes(448, 3072, 3072, 1) and takes(768, 3072, 8192, 1)
    assert takes(17, 3072, 3072, 0) and takes(512, 3072, 8192, 1) and takes(512, 8192, 3072, 2)
    for m, n, k, e in ((16, 3072, 3072, 0), (129, 5120, 3072, 0), (288, 5120, 3072, 0),
                       (449, 3072, 3072, 1), (769, 3072, 8192, 1), (513, 8192, 3072, 2), (64, 3072, 3080, 0),
                       (64, 3080, 3072, 0), (64, 512, 3072, 0)):
        assert not takes(m, n, k, e)
        assert lib.mce_prompt_gemm(0, None, None, None, m, n, k, k, n, e, None, 0.0, None, None, 0,
                                   None) == _lib.MCE_ERR_UNSUPPORTED
    x, w = rnd(dev, 64, 2048), rnd(dev, 1024, 2048, std=0.02).requires_grad_()
    y = linear(x, w)
    assert y.requires_grad and torch.equal(y, torch.matmul(x, w.T))
    xt = rnd(dev, 2048, 64).t()
    assert torch.equal(linear(xt, w.detach()), torch.matmul(xt, w.detach().T))


def test_graph_replays(dev):
    """K slices (partials in a torch-allocated workspace) captured and replayed
    with eager calls of another shape in between."""
    x, w, nw = rnd(dev, 40, 8192), rnd(dev, 3072, 8192, std=0.01), rnd(dev, 3072)
    x2, w2 = rnd(dev, 90, 8192), rnd(dev, 3072, 8192, std=0.01, seed=3)
    res = rnd(dev, 40, 3072)

    def run():
        a = res.clone()
        return linear_add_norm(x, w, a, nw, 1e-5), a
    want = run()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        run()
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = run()
    other = linear(x2, w2)
    for _ in range(3):
        g.replay()
        assert torch.equal(linear(x2, w2), other)
        torch.cuda.synchronize()
        assert all(torch.equal(p, q) for p, q in zip(got, want))
