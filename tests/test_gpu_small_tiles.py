"""The small-tile GEMM kernel against the oracle: edges of its 16 x 16 .. 32 x
64 tiles and of the 128-byte K units split over a block's waves, every operand
alignment and epilogue, and both sides of the output count where the pipelined
and register-staged kernels take over. Integer results: equal bytes."""
import numpy as np
import pytest

import nnr_amd as H
from nnr_amd import _lib
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def on(dev, a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy()


def rand(rng, dt, shape):
    return rng.integers(np.iinfo(dt).min, np.iinfo(dt).max + 1, shape, dtype=dt)


def variants(run):
    """run()'s result and the GEMM variants it launched."""
    _lib.profile_reset()
    _lib.profile_enable(True)
    try:
        y = host(run())
    finally:
        _lib.profile_enable(False)
    names = sorted(_lib.profile_read(variants=True))
    _lib.profile_reset()
    return y, names


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (15, 17, 16), (16, 16, 64), (17, 33, 65), (1, 3072, 768), (31, 4, 128),
                                   (33, 130, 192), (49, 512, 4608), (96, 96, 72), (61, 8, 24), (3, 1000, 2041),
                                   (634, 1024, 48), (635, 1024, 48), (1318, 1024, 512), (1319, 1024, 512),
                                   (1611, 1024, 48), (1612, 1024, 48), (3222, 1024, 20), (3223, 1024, 20)])
@pytest.mark.parametrize("dt", [np.uint8, np.int8])
def test_matmul(dev, m, n, k, dt):
    rng = np.random.default_rng(m + n + k)
    a, b = rand(rng, dt, (m, k)), rand(rng, np.int8, (k, n))
    args = (0.021, 121 if dt == np.uint8 else -9, b, 0.0047, 0, 0.0021 * k ** 0.5, 128 if dt == np.uint8 else 3)
    ref = O.qlinear_matmul(a, args[0], args[1], b, args[3], 0, args[5], args[6], dt)
    op = H.QLinearMatMul(b, *args[:2], *args[3:], m=m, a_dtype=dt, y_dtype=dt)
    y, names = variants(lambda: op(on(dev, a)))
    assert np.array_equal(y.reshape(ref.shape), ref)
    # the pipelined kernel takes K % 16 == 0, the register-staged one the rest.
    # (One limit of 1650000 for every K had the small-tile kernel run K = 64 at
    # 800000 outputs and more, 1.1 to 1.27 times the pipelined kernel's time)
    limit = 3300000 if k % 16 else 650000 if k <= 64 else 1350000
    assert any("small" in v for v in names) == (m * n <= limit), names


@pytest.mark.parametrize("m,n,k,adt,bdt,azp,bzp,batch", [
    (77, 77, 64, np.uint8, np.uint8, 127, 131, 5), (1, 16, 16, np.uint8, np.int8, 3, 0, 1),
    (33, 65, 200, np.int8, np.uint8, -4, 255, 2), (50, 31, 37, np.uint8, np.uint8, 0, 1, 3),
    (128, 512, 1024, np.int8, np.int8, 5, -7, 1), (1300, 1300, 64, np.uint8, np.int8, 9, 0, 1)])
@pytest.mark.parametrize("shared_b", [False, True])
def test_matmul_integer(dev, m, n, k, adt, bdt, azp, bzp, batch, shared_b):
    """The zero-point sums formed from the operands; B repacked per call."""
    rng = np.random.default_rng(m + k)
    a = rand(rng, adt, (batch, m, k))
    b = rand(rng, bdt, (1 if shared_b else batch, k, n))
    ref = O.matmul_integer(a, np.broadcast_to(b, (batch, k, n)).copy(), azp, bzp)
    op = H.MatMulInteger(m, n, k, adt, bdt, max_batch=batch)
    y = op(on(dev, a), on(dev, b), azp, bzp, batch=batch, b_bstride=0 if shared_b else k * n)
    assert np.array_equal(host(y).reshape(ref.shape), ref)


CONVS = [
    # N, C, H, W, OC, k, options
    (1, 64, 7, 7, 64, 3, dict(x_nhwc=1, y_nhwc=1, pads=(1, 1, 1, 1))),
    (1, 16, 9, 5, 40, 3, dict(x_nhwc=1, y_nhwc=1, stride=(2, 2), pads=(1, 1, 1, 1))),        # RQ-B' columns
    (2, 48, 11, 13, 88, 1, dict(x_nhwc=1, y_nhwc=1, stride=(2, 2))),
    (1, 32, 10, 10, 24, 5, dict(x_nhwc=1, y_nhwc=1, pads=(2, 2, 2, 2), dil=(2, 2))),
    (2, 24, 6, 6, 96, 1, dict(x_nhwc=1, y_nhwc=1)),                                          # 8-byte rows
    (1, 36, 23, 23, 50, 3, dict(pads=(1, 1, 1, 1), act_dtype=np.int8)),                       # scalar tails, NCHW
    (2, 20, 17, 9, 33, 3, dict(pads=(1, 1, 1, 1), stride=(2, 1))),
    (1, 32, 12, 12, 48, 3, dict(group=4, x_nhwc=1, y_nhwc=1, pads=(1, 1, 1, 1))),             # 8 channels a group
    (2, 24, 9, 9, 12, 3, dict(group=2, pads=(1, 1, 1, 1), stride=(2, 2))),                    # 12: 4-byte pieces
    (1, 15, 9, 9, 10, 3, dict(group=5, x_nhwc=1, y_nhwc=1, pads=(1, 1, 1, 1))),               # 3: single bytes
    (1, 32, 9, 9, 24, 3, dict(x_nhwc=1, y_nhwc=1, pads=(1, 1, 1, 1), w_zp=(5,))),             # row sums
    (2, 32, 9, 9, 8, 1, dict(group=2, w_zp=tuple(range(8)))),                                 # per-channel w_zp
    (8, 64, 56, 56, 64, 3, dict(x_nhwc=1, y_nhwc=1, pads=(1, 1, 1, 1))),                      # 1.6 M outputs
    (17, 64, 28, 28, 128, 3, dict(pads=(1, 1, 1, 1))),                                        # 1.7 M, NCHW
]


@pytest.mark.parametrize("case", range(len(CONVS)))
def test_conv(dev, case):
    N, C, Hh, W, OC, k, kw = CONVS[case]
    rng = np.random.default_rng(case)
    kw = dict(kw)
    act = kw.get("act_dtype", np.uint8)
    xn = kw.pop("x_nhwc", 0)
    w = rand(rng, np.int8, (OC, C // kw.get("group", 1), k, k))
    kw.update(w_scale=rng.uniform(0.001, 0.01, OC).astype(np.float32), x_scale=0.02,
              x_zp=128 if act == np.uint8 else -5, y_scale=0.6, y_zp=7, bias=rng.integers(-4096, 4097, OC).astype(np.int32))
    x = rand(rng, act, (N, Hh, W, C) if xn else (N, C, Hh, W))
    ref, _ = O.Conv(N, C, Hh, W, OC, k, k, x_nhwc=xn, **kw).run(x, w)
    op = H.QLinearConv(N, C, Hh, W, w, x_nhwc=xn, **kw)
    y, names = variants(lambda: op(on(dev, x)))
    assert np.array_equal(y, ref)
    assert any("small" in v for v in names), names


@pytest.mark.parametrize("N,C,hw,OC,k", [(1, 64, 7, 80, 1), (2, 128, 9, 64, 3), (1, 512, 7, 2048, 1),
                                         # above the small-tile kernel's outputs: weights in registers
                                         # (K = 64), one residual buffer (K = 128), uniform taps
                                         (10, 64, 31, 192, 1), (5, 128, 28, 512, 1), (9, 64, 56, 64, 3)])
@pytest.mark.parametrize("conv_is_a", [0, 1])
def test_fused_add(dev, N, C, hw, OC, k, conv_is_a):
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
    assert np.array_equal(host(op.run_add(on(dev, x), on(dev, other))), ref)


@pytest.mark.parametrize("m,n,k", [(37, 768, 768), (1, 64, 3072), (70, 3072, 96), (128, 200, 256), (600, 3072, 96)])
def test_fused_chain_pairs(dev, m, n, k):
    """Fused dequantize + bias + Gelu with the (min, max) pairs: every pair is
    written, however few blocks the launch has, and they cover the output."""
    import torch
    rng = np.random.default_rng(m + n)
    a, b = rand(rng, np.uint8, (m, k)), rand(rng, np.int8, (k, n))
    ys, yz = float(0.02 * 0.004 * 74 * k ** 0.5), 121
    op = H.QLinearMatMul(b, 0.02, 120, 0.004, 0, ys, yz, m=m)
    op.fuse_dq_bias(ys, yz, rng.standard_normal(n).astype(np.float32))
    op.fuse_gelu()
    parts = torch.full((2 * op.minmax_count(1),), float("nan"), dtype=torch.float32, device=dev)
    op.set_minmax_out(parts)
    y = host(op(on(dev, a)))
    p = host(parts).reshape(-1, 2)
    assert not np.isnan(p).any()
    assert p[:, 0].min() == min(0.0, y.min()) and p[:, 1].max() == max(0.0, y.max())
