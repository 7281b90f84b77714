"""The kernels that stage tiles in LDS (pipelined, short-K direct,
register-staged), at more outputs than the small-tile kernel takes: the calls
of the parity tests again on larger batches, each checked to run the kernel it
is here for. Integer results: equal bytes."""
import numpy as np
import pytest

import nnr_amd as H
from nnr_amd import _lib
from oracle import pyoracle as O
from test_gpu_small_tiles import host, on, rand, variants

pytestmark = pytest.mark.gpu


def ran(names, kernel):
    """kernel: 'small', 'dma', 'direct' or 'reg', the one GEMM kernel that a run launched."""
    want = {"small": "variant:small<", "dma": "variant:dma<", "direct": "variant:direct", "reg": "variant:qgemm_reg"}[kernel]
    return bool(names) and all(n.startswith(want) for n in names)


@pytest.mark.parametrize("m,n,k,adt,bdt,azp,bzp,batch,kernel", [
    # a zero point of B: column and row sums. K at the edges of the column sums'
    # 8 rows a wave, N of their 64 columns
    (1000, 65, 128, np.uint8, np.uint8, 7, 131, 52, "reg"), (1000, 65, 129, np.uint8, np.uint8, 0, 3, 52, "reg"),
    (13200, 255, 16, np.int8, np.uint8, -4, 200, 1, "reg"), (3400, 1000, 77, np.uint8, np.int8, 9, -5, 1, "reg"),
    (1840, 1840, 1, np.uint8, np.int8, 3, 2, 1, "reg"),
    (400, 77, 512, np.uint8, np.int8, 127, 0, 55, "dma"), (1100, 64, 1040, np.int8, np.int8, 5, 0, 24, "dma"),
    (27000, 64, 16, np.uint8, np.int8, 1, 0, 1, "dma")])
@pytest.mark.parametrize("shared_b", [False, True])
def test_matmul_integer(dev, m, n, k, adt, bdt, azp, bzp, batch, kernel, shared_b):
    rng = np.random.default_rng(m + k)
    a, b = rand(rng, adt, (batch, m, k)), rand(rng, bdt, (1 if shared_b else batch, k, n))
    ref = np.matmul(a.astype(np.float32) - azp, b.astype(np.float32) - bzp)   # |sums| < 2^24 for K <= 257
    if k > 257:
        ref = O.matmul_integer(a, np.broadcast_to(b, (batch, k, n)).copy(), azp, bzp)
    op = H.MatMulInteger(m, n, k, adt, bdt, max_batch=batch)
    ad, bd = on(dev, a), on(dev, b)
    y, names = variants(lambda: op(ad, bd, azp, bzp, batch=batch, b_bstride=0 if shared_b else k * n))
    assert ran(names, kernel), names
    assert np.array_equal(y.reshape(ref.shape), ref.astype(np.int32))


@pytest.mark.parametrize("N,C,hw,OC,k,group,kernel", [
    (7, 32, 28, 192, 1, 1, "small"), (8, 32, 28, 192, 1, 1, "direct"),        # K = 64: 1.2 M
    (41, 128, 14, 200, 3, 1, "small"), (43, 128, 14, 200, 3, 1, "dma"), (4, 256, 28, 512, 1, 1, "small"),
    (5, 256, 28, 512, 1, 1, "dma"), (29, 64, 28, 72, 3, 1, "small"), (30, 64, 28, 72, 3, 1, "dma"),   # 1.65 M
    (57, 512, 7, 512, 3, 1, "small"), (58, 512, 7, 512, 3, 1, "dma"),         # K = 4608: 1.45 M
    (48, 128, 14, 128, 3, 2, "small"), (49, 128, 14, 128, 3, 2, "dma"),       # groups: 1.22 M
    (25, 256, 14, 256, 3, 8, "small"), (26, 256, 14, 256, 3, 8, "dma"),       # of 32 channels: 1.3 M
    (27, 256, 14, 128, 1, 2, "small"), (28, 256, 14, 128, 1, 2, "dma")])      # of K = 128: 0.7 M
def test_conv_limits(dev, N, C, hw, OC, k, group, kernel):
    """Both sides of the output counts at which the kernels change over."""
    rng = np.random.default_rng(N + OC)
    x, w = rand(rng, np.uint8, (N, hw, hw, C)), rand(rng, np.int8, (OC, C // group, k, k))
    kw = dict(pads=(k // 2,) * 4, x_nhwc=1, y_nhwc=1, x_scale=0.02, x_zp=128, y_scale=0.5, y_zp=3, group=group,
              w_scale=rng.uniform(0.001, 0.01, OC).astype(np.float32), bias=rng.integers(-4096, 4097, OC).astype(np.int32))
    ref, _ = O.Conv(N, C, hw, hw, OC, k, k, **kw).run(x, w)
    op = H.QLinearConv(N, C, hw, hw, w, **kw)
    y, names = variants(lambda: op(on(dev, x)))
    assert ran(names, kernel), names
    assert np.array_equal(y, ref)


@pytest.mark.parametrize("N,C,hw,OC,k,kernel", [
    (4, 64, 56, 64, 1, "small"), (5, 64, 56, 64, 1, "dma"),       # K = 64: 1.0 M
    (5, 64, 28, 320, 1, "dma"), (6, 64, 28, 320, 1, "small"),     # but 1.65 M from 32 row tiles
    (7, 64, 28, 320, 1, "dma"),                                   # (weights in registers)
    (3, 128, 28, 512, 1, "small"), (4, 128, 28, 512, 1, "dma"),   # K = 128: 1.25 M
    (7, 256, 14, 1024, 1, "small"), (8, 256, 14, 1024, 1, "dma"),   # K = 256: 1.5 M
    (16, 512, 7, 2048, 1, "small"), (17, 512, 7, 2048, 1, "dma"), (6, 64, 56, 80, 3, "small"), (7, 64, 56, 80, 3, "dma")])
@pytest.mark.parametrize("conv_is_a", [0, 1])
def test_fused_add_limits(dev, N, C, hw, OC, k, kernel, conv_is_a):
    rng = np.random.default_rng(C + OC)
    x, w = rand(rng, np.uint8, (N, hw, hw, C)), rand(rng, np.int8, (OC, C, k, k))
    kw = dict(pads=(k // 2,) * 4, x_nhwc=1, y_nhwc=1, x_scale=0.02, x_zp=128, y_scale=0.5, y_zp=3,
              w_scale=rng.uniform(0.001, 0.01, OC).astype(np.float32), bias=rng.integers(-4096, 4097, OC).astype(np.int32))
    conv, _ = O.Conv(N, C, hw, hw, OC, k, k, **kw).run(x, w)
    other = rand(rng, np.uint8, conv.shape)
    q = (0.041, 7, 0.023, 131, 0.06, 2)
    ref = O.qlinear_add(0, *((conv, other) if conv_is_a else (other, conv)), *q)
    op = H.QLinearConv(N, C, hw, hw, w, **kw)
    assert op.fuse_add(conv_is_a, *q)
    xd, od = on(dev, x), on(dev, other)
    y, names = variants(lambda: op.run_add(xd, od))
    assert ran(names, kernel), names
    assert np.array_equal(y, ref)


@pytest.mark.parametrize("m,n,k,gelu,pairs,kernel", [
    (100, 768, 128, 1, 1, "dma"), (100, 768, 192, 1, 1, "small"), (100, 768, 256, 0, 1, "dma"),
    (100, 768, 320, 0, 1, "small"), (320, 3072, 768, 0, 1, "small"), (321, 3072, 768, 0, 1, "dma"),   # 240, 288 tiles
    (537, 3072, 768, 1, 1, "small"), (538, 3072, 768, 1, 1, "dma"), (537, 3072, 64, 0, 0, "small"),
    (538, 3072, 64, 0, 0, "dma")])
@pytest.mark.parametrize("codes", [0, 1])
def test_chain_limits(dev, m, n, k, gelu, pairs, kernel, codes):
    """Fused QLinearMatMul -> DequantizeLinear -> + bias (-> Gelu): the values
    against the oracle's bytes, with Gelu against the kernel of its own; the
    bytes; the pairs."""
    import torch
    rng = np.random.default_rng(m + k)
    a, b = rand(rng, np.uint8, (m, k)), rand(rng, np.int8, (k, n))
    ys, yz, bias = float(0.02 * 0.004 * 74 * k ** 0.5), 121, rng.standard_normal(n).astype(np.float32)
    q = O.qlinear_matmul(a, np.float32(0.02), 120, b, 0.004, 0, ys, yz)
    ref = (O.dequantize_linear(q, ys, yz) + bias).astype(np.float32)
    if gelu:
        r = on(dev, ref)
        _lib.check(_lib.lib().nnrh_gelu_f32(r.data_ptr(), r.data_ptr(), r.numel(), _lib.cur_stream()))
        ref = host(r)
    op = H.QLinearMatMul(b, 0.02, 120, 0.004, 0, ys, yz, m=m)
    op.fuse_dq_bias(ys, yz, bias)
    if gelu:
        op.fuse_gelu()
    if pairs:
        parts = torch.full((2 * op.minmax_count(1),), float("nan"), dtype=torch.float32, device=dev)
        op.set_minmax_out(parts)
    if codes:
        op.set_codes_out()
    ad = on(dev, a)
    y, names = variants(lambda: op(ad))
    assert ran(names, kernel), names
    assert np.array_equal(y, q) if codes else np.array_equal(y.view(np.uint32), ref.view(np.uint32))
    if pairs:
        p = host(parts).reshape(-1, 2)
        assert not np.isnan(p).any()
        assert p[:, 0].min() == min(0.0, ref.min()) and p[:, 1].max() == max(0.0, ref.max())
