"""The attention kernel that walks the keys in steps, against float64: every
head size it takes, lengths at the edges of its 64-key steps and 64-query
blocks, infinite scores, and an output that lies over an input."""
import ctypes as C

import numpy as np
import pytest

from nnr_amd import _lib

pytestmark = pytest.mark.gpu


def attention(dev, q, k, v, heads, scale, y_over=None):
    import torch
    B, S, hidden = q.shape
    t = {n: torch.from_numpy(np.ascontiguousarray(a)).to(dev) for n, a in (("q", q), ("k", k), ("v", v))}
    n = C.c_size_t()
    _lib.check(_lib.lib().nnrh_multihead_attention_workspace(B, S, hidden, heads, C.byref(n)))
    ws = torch.empty(n.value + 256, dtype=torch.uint8, device=dev)
    y = t[y_over] if y_over else torch.full((B, S, hidden), float("nan"), dtype=torch.float32, device=dev)
    _lib.check(_lib.lib().nnrh_multihead_attention_f32(
        t["q"].data_ptr(), t["k"].data_ptr(), t["v"].data_ptr(), y.data_ptr(), B, S, hidden, heads, scale, None,
        (ws.data_ptr() + 255) & ~255, _lib.cur_stream()))
    torch.cuda.synchronize()
    return y.cpu().numpy()


def exact(q, k, v, heads, scale):
    B, S, hidden = q.shape
    sp = lambda t: t.astype(np.float64).reshape(B, S, heads, -1).transpose(0, 2, 1, 3)
    sc = np.matmul(sp(q), sp(k).transpose(0, 1, 3, 2)) * np.float32(scale)
    e = np.exp(sc - sc.max(-1, keepdims=True))
    return np.matmul(e / e.sum(-1, keepdims=True), sp(v)).transpose(0, 2, 1, 3).reshape(B, S, hidden)


def data(seed, B, S, hidden):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((B, S, hidden)).astype(np.float32) for _ in range(3)]


@pytest.mark.parametrize("hd", [32, 64, 80, 96, 128, 48])   # 48: the general path
@pytest.mark.parametrize("B,S,heads", [(2, 1, 3), (1, 63, 2), (2, 64, 1), (1, 65, 2), (1, 129, 3), (2, 200, 2),
                                       (1, 512, 2)])
def test_against_float64(dev, hd, B, S, heads):
    q, k, v = data(S + hd, B, S, heads * hd)
    y, ref = attention(dev, q, k, v, heads, hd ** -0.5), exact(q, k, v, heads, hd ** -0.5)
    # fp32: hd products a score, S terms a sum, each within an ulp (6e-8) of
    # its magnitude; random signs keep the sum of them under 20 ulps
    assert np.linalg.norm(y - ref) <= 1.2e-6 * np.linalg.norm(ref)


def test_large_scores(dev):
    """Scores of several hundred: only differences to the maximum enter exp()."""
    q, k, v = data(3, 1, 300, 128)
    y, ref = attention(dev, 40 * q, 40 * k, v, 2, 0.125), exact(40 * q, 40 * k, v, 2, 0.125)
    # a score of 4e3 carries 2e-4 of rounding, which exp() turns into a relative error
    assert np.linalg.norm(y - ref) <= 1e-3 * np.linalg.norm(ref)


@pytest.mark.parametrize("hd,S", [(64, 129), (64, 512), (32, 300), (128, 1000)])
def test_large_values(dev, hd, S):
    """Values whose sum over the keys is no float, whose weighted mean is one."""
    q, k, v = data(6 + S, 1, S, hd)
    v = np.sign(v) * np.random.default_rng(S).uniform(2e38, 3e38, v.shape).astype(np.float32)
    v[..., 0] = 3e38   # a column of equal values: nothing cancels
    q *= np.float32(0.1)
    y, ref = attention(dev, q, k, v, 1, 0.125), exact(q, k, v, 1, 0.125)
    assert np.isfinite(y).all()
    # (scaled: the squares of the norm are no floats; the bound of ordinary values)
    assert np.linalg.norm(y / 1e38 - ref / 1e38) <= 1.2e-6 * np.linalg.norm(ref / 1e38)


def test_infinite_scores(dev):
    """Keys whose scores are -inf weigh nothing, a whole step of them too (the
    first 64 keys); a row with only such keys, or with +inf, is NaN."""
    q, k, v = data(4, 1, 192, 64)
    q[0, :, 0] = 1.0
    k[0, :64, 0] = -np.inf
    y = attention(dev, q, k, v, 1, 0.125)
    sc = np.matmul(q[0].astype(np.float64), k[0, 64:].astype(np.float64).T) * 0.125
    e = np.exp(sc - sc.max(-1, keepdims=True))
    ref = np.matmul(e / e.sum(-1, keepdims=True), v[0, 64:].astype(np.float64))
    assert np.linalg.norm(y[0] - ref) <= 1.2e-6 * np.linalg.norm(ref)
    q[0, 7, 0] = -1.0   # this query's first 64 scores are +inf
    y = attention(dev, q, k, v, 1, 0.125)
    assert np.isnan(y[0, 7]).all() and not np.isnan(np.delete(y[0], 7, 0)).any()


@pytest.mark.parametrize("over,S,hd", [("q", 260, 64), ("k", 260, 64),
                                       ("v", 64, 32), ("v", 64, 48), ("v", 64, 128)])   # one block a head
def test_output_over_an_input(dev, over, S, hd):
    q, k, v = data(5, 2, S, 2 * hd)
    y, ref = attention(dev, q, k, v, 2, 0.125, over), exact(q, k, v, 2, 0.125)
    assert np.linalg.norm(y - ref) <= 1.2e-6 * np.linalg.norm(ref)
