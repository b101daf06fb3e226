"""GPU: layouts and sizes at which a kernel takes another path."""
import pytest
import torch

import my_cuda_engine_cpp as ops

pytestmark = pytest.mark.gpu


def gen(seed):
    return torch.Generator().manual_seed(seed)


# one shape per launch of the prefill kernel: 64-row items, 128-row items on two
# key streams (with items left over for a second pick), one key stream
@pytest.mark.parametrize("b,s,dtype", [(1, 1, torch.float16), (2, 77, torch.bfloat16),
                                       (1, 1800, torch.float16), (1, 2048, torch.bfloat16),
                                       (5, 700, torch.float16)])
def test_prefill_reads_projection_views_in_place(dev, b, s, dtype):
    """q, k and v as views into one fused projection [B, S, (24 + 8 + 8) 128]
    give the bits of their contiguous copies, with NaN rows behind every
    sequence (keys past the end read as zeros, not as the next sequence)."""
    buf = torch.full((b, s + 3, 40 * 128), float("nan"), dtype=dtype)
    buf[:, :s] = torch.randn(b, s, 40 * 128, generator=gen(b + s)).to(dtype)
    buf = buf.to(dev)[:, :s]
    q = buf[:, :, :3072].unflatten(2, (24, 128))
    k = buf[:, :, 3072:4096].unflatten(2, (8, 128))
    v = buf[:, :, 4096:].unflatten(2, (8, 128))
    got = ops.prefill_attention(q, k, v, 128 ** -0.5)
    want = ops.prefill_attention(q.contiguous(), k.contiguous(), v.contiguous(), 128 ** -0.5)
    assert got.is_contiguous() and not torch.isnan(got).any()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_prefill_copies_the_layouts_it_cannot_read(dev):
    """Transposed heads, k and v of different strides, a misaligned view."""
    g = gen(7)
    q, k, v = (torch.randn(2, 90, h, 128, generator=g).half().to(dev) for h in (24, 8, 8))
    want = ops.prefill_attention(q, k, v, 0.1)
    qt = q.transpose(1, 2).contiguous().transpose(1, 2)
    kw = torch.zeros(2, 90, 10, 128, dtype=torch.float16, device=dev)
    kw[:, :, :8] = k
    vm = torch.zeros(2 * 90 * 8 * 128 + 1, dtype=torch.float16, device=dev)[1:].view(2, 90, 8, 128)
    vm.copy_(v)
    assert torch.equal(ops.prefill_attention(qt, kw[:, :, :8], v, 0.1), want)
    with pytest.raises(RuntimeError, match="aligned"):  # contiguous but misaligned: refused
        ops.prefill_attention(q, k, vm, 0.1)
    qm = torch.zeros(2, 90, 3072 + 4, dtype=torch.float16, device=dev)[:, :, 4:].unflatten(2, (24, 128))
    qm.copy_(q)
    assert torch.equal(ops.prefill_attention(qm, k, v, 0.1), want)


@pytest.mark.parametrize("n,k", [(33360, 2048), (40976, 3072)])
def test_decode_gemm_walks_uneven_tile_ranges(dev, n, k):
    """9-16 tokens on a wide weight: one workgroup per CU walks a contiguous
    range of 16-column tiles, here of unequal counts; |err| <= 2e-3 + 4e-3 |ref|
    against fp32 (fp16 rounding of the output and fp32 sums)."""
    from mycustomcudaengine_amd.ops import decode_gemm
    g = gen(n)
    x = torch.randn(13, k, generator=g).half()
    w = (torch.randn(n, k, generator=g) * 0.02).half()
    out = decode_gemm(x.to(dev), w.to(dev)).float().cpu()
    ref = x.float() @ w.float().T
    assert ((out - ref).abs() <= 2e-3 + 4e-3 * ref.abs()).all()


# rows of fewer than 64 groups of 8 (flat kernel), 64 and more (row kernel: a
# partial last workgroup, more rows than grid.y holds), and a call of over 192 MB
# (non-temporal loads)
@pytest.mark.parametrize("rows,inter,dtype", [(3, 504, torch.float16), (5, 512, torch.bfloat16),
                                              (7, 2056, torch.float16), (65540, 512, torch.float16),
                                              (4100, 8192, torch.bfloat16)])
def test_swiglu_row_kernels(dev, rows, inter, dtype):
    """silu(g) u against fp64: half an ulp of the output type plus the fp32
    exponential's error (2^-11 and 2^-8 of the value, doubled for the sum)."""
    g = torch.Generator(device=dev).manual_seed(rows)
    x = torch.empty(rows, 2 * inter, dtype=dtype, device=dev).normal_(generator=g)
    out = ops.swiglu(x)
    gate, up = (t.double() for t in x.chunk(2, 1))
    ref = gate * torch.sigmoid(gate) * up
    tol = 2.0 ** (-10 if dtype == torch.float16 else -7)
    assert ((out.double() - ref).abs() <= tol * ref.abs() + 1e-7).all()


# up to 4 sequences over tables past 1024 tokens take one kv head per workgroup
# (ranges of whole sequences): contexts at a range's and a tile's edges, an empty
# sequence, lengths so uneven that the range length has to be searched; the
# last three stay with the whole-page split (5 sequences, long tables, kv heads)
@pytest.mark.parametrize("ctx,width,hq,hkv,dtype", [
    ([1100], 70, 24, 8, torch.float16), ([1], 65, 24, 8, torch.float16),
    ([128, 129], 66, 24, 8, torch.bfloat16), ([0, 3000], 190, 8, 8, torch.float16),
    ([17, 5000, 1], 320, 6, 2, torch.float16), ([2048, 33, 0, 1999], 128, 32, 8, torch.bfloat16),
    ([4000, 100, 4000, 16], 256, 14, 7, torch.float16), ([1500, 7, 900, 16, 2000], 128, 24, 8, torch.float16),
    ([1, 20000, 5, 300], 1250, 24, 8, torch.float16), ([1100, 3000], 200, 32, 32, torch.float16)])
def test_decode_of_few_sequences(dev, ctx, width, hq, hkv, dtype):
    """Against fp64 on the gathered K/V; the unused pool is NaN."""
    g = gen(sum(ctx) + hq)
    b, nb = len(ctx), sum(-(-c // 16) for c in ctx) + 3
    kc, vc = (torch.full((nb, 16, hkv, 128), float("nan"), dtype=dtype) for _ in range(2))
    tables, perm, off = torch.zeros(b, width, dtype=torch.int32), torch.randperm(nb, generator=g), 0
    q = torch.randn(b, hq, 128, generator=g).to(dtype)
    ref = torch.zeros(b, hq, 128, dtype=torch.float64)
    for i, c in enumerate(ctx):
        n = -(-c // 16)
        blocks = perm[off:off + n]
        off += n
        tables[i, :n] = blocks.to(torch.int32)
        k, v = (torch.randn(n * 16, hkv, 128, generator=g).to(dtype) for _ in range(2))
        k[c:], v[c:] = float("nan"), float("nan")
        kc[blocks], vc[blocks] = k.view(n, 16, hkv, 128), v.view(n, 16, hkv, 128)
        if c:
            kk, vv = (t[:c].double().repeat_interleave(hq // hkv, 1) for t in (k, v))
            p = torch.softmax(torch.einsum("hd,thd->ht", q[i].double(), kk) * 128 ** -0.5, -1)
            ref[i] = torch.einsum("ht,thd->hd", p, vv)
    out = ops.paged_attention_decode(q.to(dev), kc.to(dev), vc.to(dev), tables.to(dev),
                                     torch.tensor(ctx, dtype=torch.int32, device=dev), width, 16,
                                     128 ** -0.5).cpu()
    # P rounds to the element type (2^-11 / 2^-8 relative), |v| <= 5, and so does the output
    tol = 5 * (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7)
    assert (out.double() - ref).abs().max().item() <= tol
