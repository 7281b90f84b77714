"""The kernels that stage tiles in LDS (pipelined, short-K direct,
register-staged), at more outputs than the small-tile kernel takes: the calls
of the parity tests again on larger batches, each checked to run the kernel it
is here for. Integer results: equal bytes."""
import numpy as np
import pytest

import nnr_amd as H
import test_gpu_parity as P
from nnr_amd import _lib
from oracle import pyoracle as O
from test_gpu_small_tiles import host, on, rand, variants

pytestmark = pytest.mark.gpu
LARGE = 3350000   # outputs past every limit of the small-tile kernel


def ran(names, kernel):
    """kernel: 'small', 'dma', 'direct' or 'reg', the one GEMM kernel that a run launched."""
    want = {"small": "variant:small<", "dma": "variant:dma<", "direct": "variant:direct", "reg": "variant:qgemm_reg"}[kernel]
    return bool(names) and all(n.startswith(want) for n in names)


def launched(test):
    """The GEMM variants that a test launches."""
    _lib.profile_reset()
    _lib.profile_enable(True)
    try:
        test()
    finally:
        _lib.profile_enable(False)
    names = sorted(_lib.profile_read(variants=True))
    _lib.profile_reset()
    return names


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


# the parity tests' convolutions that the short-K direct and the register-staged
# kernel run (scalar tails, RQ-B', a weight zero point, NCHW output, channels in
# 8-, 4- and 1-byte pieces); the other GEMMs are the pipelined kernel's
DIRECT = {"nchw16_c64", "packed_c24", "direct_c24", "direct_c16_oc96", "direct_c64_oc16", "direct_c32_oc32",
          "dma_persistent_1x1", "tall2_1x1_k64"}
REG = {"packed_bprime", "packed_wzp", "packed_wzp_neg", "packed_nchw_out", "direct_c40_oc72", "direct_c24_oc8", "direct",
       "direct_tail", "grouped_s1", "grouped_s2", "float_int8act", "float_pcz", "dma_grouped_c16", "cpad_c8_3x3",
       "cpad_c24_wzp"}


@pytest.mark.parametrize("case", [c for c in P.CONV_CASES if c[0][:2] not in ("dw", "fi")], ids=lambda c: c[0])
def test_conv(dev, case):
    name, N, C, Hh, W, OC, k, kw = case
    kw = dict(kw)
    oh, ow = ((d + p - kw.get("dil", (1, 1))[0] * (k - 1) - 1) // s + 1 for d, p, s in zip(
        (Hh, W), (sum(kw.get("pads", (0,) * 4)[i::2]) for i in (0, 1)), kw.get("stride", (1, 1))))
    N = max(N, -(-LARGE // (oh * ow * OC)))
    names = launched(lambda: P.run_conv_case(dev, N, C, Hh, W, OC, k, seed=sum(name.encode()), **kw))
    assert ran(names, "direct" if name in DIRECT else "reg" if name in REG else "dma"), names
    assert all(n.endswith(",128,0,2>") for n in names) == ("ksplit" in name or name == "dma_s2_3x3"), names   # K split


@pytest.mark.parametrize("m,n,k,batch,adt,bdt,ydt,bzp,sdt", P.MM_CASES)
def test_matmul(dev, m, n, k, batch, adt, bdt, ydt, bzp, sdt):
    m = -(-LARGE // (n * batch))
    names = launched(lambda: P.test_qmatmul_shapes(dev, m, n, k, batch, adt, bdt, ydt, bzp, sdt))
    assert ran(names, "dma" if k % 16 == 0 and bzp in (0, 128 if bdt == np.uint8 else 0) else "reg"), names


@pytest.mark.parametrize("m,n,k,dt", [(1400, 1000, 512, np.uint8), (11000, 129, 256, np.int8), (400, 3500, 1024, np.uint8),
                                      (1400, 1001, 192, np.int8), (28000, 63, 48, np.uint8), (1361, 1300, 64, np.int8)])
def test_matmul_ragged(dev, m, n, k, dt):
    """Ragged last rows and columns: K split over two waves (K % 128 == 0), 64-
    and 128-byte stages, 256 x 64 tiles."""
    names = launched(lambda: P.test_qmatmul_shapes(dev, m, n, k, 1, dt, np.int8, dt, 0, np.float32))
    assert ran(names, "dma"), names
    assert all(n.endswith(",128,0,2>") for n in names) == (k % 128 == 0), names   # K split


@pytest.mark.parametrize("case", P.FUSED_ADD_CASES, ids=lambda c: c[0])
def test_fused_add(dev, case):
    name, N, C, Hh, W, OC, k, pads, conv_is_a = case
    N = max(N, -(-LARGE // (Hh * W * OC)))
    names = launched(lambda: P.test_qconv_fused_add(dev, (name, N, C, Hh, W, OC, k, pads, conv_is_a)))
    assert ran(names, "dma"), names


@pytest.mark.parametrize("rows,n,k", [(800, 768, 96), (9100, 64, 96), (601, 1000, 256)])
@pytest.mark.parametrize("mode", ["values", "bytes", "scaled"])
def test_group(dev, rows, n, k, mode):
    """Three projections of one A in a launch: each member's values, bytes, or
    MatMulInteger -> Cast -> Mul -> Add against the oracle."""
    import torch
    rng = np.random.default_rng(rows + n)
    a, bs = rand(rng, np.uint8, (rows, k)), [rand(rng, np.int8, (k, n)) for _ in range(3)]
    bias = [rng.standard_normal(n).astype(np.float32) for _ in range(3)]
    a_s, a_z, members, refs = np.float32(0.0173), 119, [], []
    for b, bi, b_s, ys, yz in zip(bs, bias, (0.004, 0.0031, 0.0057), (0.031, 0.047, 0.022), (121, 90, 140)):
        if mode == "scaled":
            ws = rng.uniform(1e-4, 2e-3, n).astype(np.float32)
            members.append(H.MatMulIntegerScaled(b, ws, bi, m=rows))
            acc = np.matmul(a.astype(np.float32) - a_z, b.astype(np.float32))   # exact: K * 255 * 128 < 2^24
            refs.append(((acc * (a_s * ws).astype(np.float32)).astype(np.float32) + bi).astype(np.float32))
        else:
            members.append(H.QLinearMatMul(b, 1.0, 0, b_s, 0, ys, yz, m=rows))
            members[-1].fuse_dq_bias(ys, yz, bi)
            q = O.qlinear_matmul(a, a_s, a_z, b, b_s, 0, ys, yz)
            refs.append(q if mode == "bytes" else (O.dequantize_linear(q, ys, yz) + bi).astype(np.float32))
    grp = H.QLinearMatMulGroup(members)
    if mode == "bytes":
        grp.set_codes_out()
    ad, sd, zd = on(dev, a), on(dev, np.array([a_s])), on(dev, np.array([a_z], np.uint8))
    outs = [torch.zeros((rows, n), dtype=torch.uint8 if mode == "bytes" else torch.float32, device=dev) for _ in refs]
    names = launched(lambda: grp(ad, outs, a_scale_dev=sd, a_zp_dev=zd))
    assert ran(names, "dma"), names
    for y, ref in zip(outs, refs):
        assert np.array_equal(host(y).view(np.uint8), ref.view(np.uint8))


@pytest.mark.parametrize("m,n,k,batch,a_dt,b_dt,bias", [
    (1300, 1300, 96, 1, np.uint8, np.int8, True), (520, 1100, 256, 3, np.int8, np.int8, False),
    (26500, 64, 48, 1, np.uint8, np.uint8, True)])
def test_matmul_integer_scaled(dev, m, n, k, batch, a_dt, b_dt, bias):
    names = launched(lambda: P.test_matmul_integer_scaled(dev, m, n, k, batch, a_dt, b_dt, bias))
    assert ran(names, "dma"), names


def test_matmul_unaligned(dev):
    """An A no multiple of 16 bytes into its buffer: the register-staged kernel's
    other load widths (K = 72 in 8s, 76 in 4s, 77 in bytes)."""
    rng = np.random.default_rng(9)
    for k, off in ((80, 8), (72, 8), (80, 4), (76, 4), (80, 1), (77, 3)):
        m, n = 3400, 1000
        a, b = rand(rng, np.uint8, (m, k)), rand(rng, np.int8, (k, n))
        args = (0.021, 121, b, 0.0047, 0, 0.31, 128)
        ref = O.qlinear_matmul(a, args[0], args[1], b, args[3], 0, args[5], args[6], np.uint8)
        op = H.QLinearMatMul(b, *args[:2], *args[3:], m=m)
        buf = on(dev, np.concatenate([np.zeros(off, np.uint8), a.reshape(-1)]))
        y, names = variants(lambda: op(buf[off:].reshape(m, k)))
        assert ran(names, "reg"), (k, off, names)
        assert np.array_equal(y, ref), (k, off)
