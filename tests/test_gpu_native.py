"""GPU: every op's native call against the Python path behind it, over the
layouts each of them takes -- the same bits, the same refusals."""
import pytest
import torch

from mycustomcudaengine_amd import ops

pytestmark = pytest.mark.gpu
F16, BF16 = torch.float16, torch.bfloat16


class Declines:
    """Stands in for the native module: every call goes to the Python path."""

    def __getattr__(self, name):
        return lambda *args: NotImplemented


def both(monkeypatch, fn, expect_native=True):
    """fn() through the native module and through Python; fn returns tensors.
    expect_native: whether the native module is meant to take the call."""
    took = []
    native = ops._native

    class Spy:
        def __getattr__(self, name):
            def run(*args):
                r = getattr(native, name)(*args)
                took.append(r is not NotImplemented)
                return r
            return run

    with monkeypatch.context() as m:
        m.setattr(ops, "_native", Spy())
        a = fn()
    with monkeypatch.context() as m:
        m.setattr(ops, "_native", Declines())
        b = fn()
    assert took and all(t == expect_native for t in took), took
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype
        assert torch.equal(x.contiguous().view(torch.int16), y.contiguous().view(torch.int16))


def rnd(dev, *shape, dtype=F16, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g).to(dtype).to(dev)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("shape,view", [((5, 3072), None), ((2, 3, 1000), None), ((0, 64), None),
                                        ((7, 13), None), ((6, 128), "transposed")])
def test_norm_and_swiglu(dev, monkeypatch, shape, view, dtype):
    x, w = rnd(dev, *shape, dtype=dtype), rnd(dev, shape[-1], dtype=dtype)
    if view:
        x = x.t().contiguous().t()
    both(monkeypatch, lambda: [ops.rmsnorm(x, w, 1e-5)], view is None)
    if shape[-1] % 2 == 0:
        both(monkeypatch, lambda: [ops.swiglu(x)], view is None)


def pool(dev, b, width, hkv, dtype, bs=16):
    kc, vc = (rnd(dev, b * width + 3, bs, hkv, 128, dtype=dtype, seed=s) for s in (1, 2))
    tables = torch.randperm(b * width, generator=torch.Generator().manual_seed(b)).view(b, width)
    return kc, vc, tables.to(torch.int32).to(dev)


@pytest.mark.parametrize("dtype,hq,hkv,width,view", [(F16, 24, 8, 8, False), (BF16, 8, 8, 100, False),
                                                     (F16, 24, 8, 70, True)])
def test_decode_and_paged_prefill(dev, monkeypatch, dtype, hq, hkv, width, view):
    b = 3
    kc, vc, tables = pool(dev, b, width, hkv, dtype)
    ctx = torch.tensor([width * 16, 50, 120], dtype=torch.int32, device=dev)
    q = rnd(dev, b, hq, 128, dtype=dtype)
    qs = rnd(dev, b, 50, hq, 128, dtype=dtype)
    if view:
        q, qs = rnd(dev, b, hq + 1, 128, dtype=dtype)[:, 1:], qs.transpose(1, 2).contiguous().transpose(1, 2)
    both(monkeypatch, lambda: [ops.paged_attention_decode(q, kc, vc, tables, ctx, width, 16, 0.09)],
         not view)
    for split in (True, False):
        both(monkeypatch, lambda: [ops.prefill_attention_paged(qs, kc, vc, tables, ctx, 0.09, split)],
             not view)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("layout,native", [("plain", True), ("fused", True), ("heads", False),
                                           ("kv differ", False)])
def test_prefill(dev, monkeypatch, layout, native, dtype):
    b, s = 2, 65
    qkv = rnd(dev, b, s, 40, 128, dtype=dtype)
    q, k, v = qkv[:, :, :24], qkv[:, :, 24:32], qkv[:, :, 32:]
    if layout == "plain":
        q, k, v = (t.contiguous() for t in (q, k, v))
    elif layout == "heads":
        q = q.transpose(1, 2).contiguous().transpose(1, 2)
    elif layout == "kv differ":
        v = v.contiguous()
    both(monkeypatch, lambda: [ops.prefill_attention(q, k, v, 0.09)], native)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("hd,fused,native", [(128, True, True), (128, False, True), (64, True, True),
                                             (20, True, False)])
def test_rope_and_stores(dev, monkeypatch, hd, fused, native, dtype):
    n, hq, hkv = 9, 6, 2
    cos, sin = rnd(dev, 40, hd // 2).float(), rnd(dev, 40, hd // 2, seed=1).float()
    pos = torch.tensor([0, 5, 39, 40, -1, 7, 8, 9, 10], dtype=torch.int32, device=dev)
    slots = torch.tensor([3, -1, 5, 6, 7, 100000, 0, 1, 2], dtype=torch.int32, device=dev)

    def tensors():
        qkv = rnd(dev, n, (hq + 2 * hkv), hd, dtype=dtype)
        q, k, v = qkv[:, :hq], qkv[:, hq:hq + hkv], qkv[:, hq + hkv:]
        if not fused:
            q, k, v = (t.contiguous() for t in (q, k, v))
        kc, vc = (torch.zeros(2, 16, hkv, hd, dtype=dtype, device=dev) for _ in range(2))
        return q, k, v, kc, vc

    def kv_store():
        q, k, v, kc, vc = tensors()
        ops.paged_kv_store(k, v, kc, vc, slots)
        return kc, vc

    def rope(with_key):
        q, k, v, kc, vc = tensors()
        ops.rope_inplace(q.unsqueeze(0), k.unsqueeze(0) if with_key else None, cos, sin, pos)
        return q, k

    def rope_store(with_out):
        q, k, v, kc, vc = tensors()
        qo = torch.zeros(n, hq, hd, dtype=dtype, device=dev) if with_out else None
        ops.rope_kv_store(q, k, v, kc, vc, cos, sin, pos, slots, query_out=qo)
        return (q, k, kc, vc) + ((qo,) if with_out else ())

    both(monkeypatch, kv_store)
    for flag in (True, False):
        both(monkeypatch, lambda: rope(flag))
        both(monkeypatch, lambda: rope_store(flag), native)


@pytest.mark.parametrize("b", [1, 4])
def test_decode_rope_attention(dev, monkeypatch, b):
    kc0, vc0, tables = pool(dev, b, 20, 8, F16)
    qkv = rnd(dev, b, 40 * 128)
    q, k, v = (t.unflatten(1, (-1, 128)) for t in qkv.split([3072, 1024, 1024], 1))
    cos, sin = rnd(dev, 400, 64).float(), rnd(dev, 400, 64, seed=1).float()
    ctx = torch.arange(100, 100 + 37 * b, 37, dtype=torch.int32, device=dev)
    slots = torch.stack([tables[i, (int(ctx[i]) - 1) // 16] * 16 + (ctx[i] - 1) % 16
                         for i in range(b)]).to(torch.int32)

    def run():
        kc, vc = kc0.clone(), vc0.clone()
        out = ops.decode_rope_attention(q, k, v, kc, vc, cos, sin, ctx - 1, slots, tables, ctx, 20, 0.09)
        return out, kc, vc

    both(monkeypatch, run)


@pytest.mark.parametrize("m", [1, 8, 13])
def test_projections(dev, monkeypatch, m):
    x, w, nw = rnd(dev, m, 2048), rnd(dev, 320, 2048) * 0.02, rnd(dev, 2048)
    out = rnd(dev, m, 400)[:, :320]
    for epi in ("store", "swiglu", "add"):
        def plain():
            o = out.clone(memory_format=torch.preserve_format) if epi == "add" else None
            return [ops.decode_gemm(x, w, out=o, epilogue=epi)]

        def normed():
            o = out.clone() if epi == "add" else None
            return [ops.rmsnorm_decode_gemm(x, nw, 1e-5, w, out=o, epilogue=epi)]

        both(monkeypatch, plain)
        both(monkeypatch, normed)
    o = torch.zeros(m, 320, dtype=F16, device=dev)
    assert ops.decode_gemm(x, w, out=o) is o


def test_other_streams_devices_and_refusals(dev, monkeypatch):
    """The current stream is the one launched on, and wrong arguments raise the
    Python path's errors."""
    x, w = rnd(dev, 64, 3072), rnd(dev, 3072)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        a = ops.rmsnorm(x, w, 1e-5)
        ev = s.record_event()
    ev.synchronize()
    assert torch.equal(a, ops.rmsnorm(x, w, 1e-5))
    for bad in (lambda: ops.rmsnorm(x, w[:-1], 1e-5), lambda: ops.rmsnorm(x.float(), w, 1e-5),
                lambda: ops.rmsnorm(x.cpu(), w, 1e-5), lambda: ops.swiglu(x[:, :3071]),
                lambda: ops.prefill_attention(x.view(1, 64, 24, 128), x.view(1, 64, 24, 128),
                                              x[:, :1024].reshape(1, 64, 8, 128), 0.1)):
        with pytest.raises(RuntimeError) as native:
            bad()
        with monkeypatch.context() as m:
            m.setattr(ops, "_native", Declines())
            with pytest.raises(RuntimeError) as python:
                bad()
        assert str(native.value) == str(python.value)
    sub = torch.nn.Parameter(w)  # a Parameter is as good as its tensor
    assert torch.equal(ops.rmsnorm(x, sub, 1e-5), a)
