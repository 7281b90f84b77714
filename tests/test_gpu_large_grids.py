"""The kernels that stage tiles in LDS (pipelined, short-K direct,
register-staged), at more outputs than the small-tile kernel takes: the calls
of the parity tests again on larger batches, each checked to run the kernel it
is here for. Integer results: equal bytes."""
import numpy as np
import pytest

import nnr_amd as H
import test_gpu_parity as P
from oracle import pyoracle as O
from test_gpu_small_tiles import host, on, rand, variants

pytestmark = pytest.mark.gpu


def ran(names, kernel):
    """kernel: 'dma', 'direct' or 'reg', the one GEMM kernel that a run launched."""
    want = {"dma": "variant:dma<", "direct": "variant:direct", "reg": "variant:qgemm_reg"}[kernel]
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
