"""Prefill attention over an int64 cache at the edges of its two routes, byte for byte against the oracle: keys or values
at the largest that the digit planes hold and one beyond it (one element decides for the whole call), head dims on and off
the 16-dim tile, lengths around a 64-key step, row counts on both sides of where the planes fit the score space, and the
bound refusals on either route."""
import numpy as np
import pytest

from oracle import attention as oat, fixedpoint as fx

pytestmark = pytest.mark.gpu
CAP = 2139062143


def _qkv(seed, H, Hkv, hd, M, L, mag=1 << 20):
    rng = np.random.default_rng(seed)
    q = rng.integers(-(1 << 18), 1 << 18, size=(H, M, hd), dtype=np.int64)
    k = rng.integers(-mag, mag, size=(Hkv, L, hd), dtype=np.int64)
    v = rng.integers(-mag, mag, size=(Hkv, L, hd), dtype=np.int64)
    return q, k, v


@pytest.mark.parametrize("H,Hkv,hd,M,start", [
    (8, 2, 128, 33, 0), (8, 2, 128, 64, 63), (8, 2, 128, 31, 1), (4, 4, 128, 130, 0), (8, 1, 64, 17, 47),
    (6, 2, 96, 40, 25), (4, 2, 16, 9, 0), (4, 2, 40, 33, 5), (2, 1, 128, 2, 300),
])
@pytest.mark.parametrize("edge", ["plain", "k_cap", "v_cap", "k_over", "v_over", "both_huge"])
def test_prefill_int64_routes(gpu, H, Hkv, hd, M, start, edge):
    L = start + M
    q, k, v = _qkv(H * 100 + hd + M + start, H, Hkv, hd, M, L)
    if edge == "k_cap":
        k[-1, L // 2, 3] = -CAP
    elif edge == "v_cap":
        v[0, L - 1, hd - 1] = CAP
    elif edge == "k_over":
        k[0, 0, 0] = CAP + 1
    elif edge == "v_over":
        v[-1, L - 1, 0] = -CAP - 1
    elif edge == "both_huge":
        k[0, L - 1, 1] = 1 << 33
        v[0, 0, 1] = -(1 << 36)
    isq = fx.inv_sqrt_fp(hd, 16)
    got = gpu.attention_prefill_gpu(q, k, v, start, 16, isq)
    want = oat.attention_cached(q, k, v, start, 16, isq)
    assert got is not None and np.array_equal(got, want)


@pytest.mark.parametrize("mag", [CAP, 1 << 45])
def test_prefill_int64_refusals(gpu, mag):
    """max|q| max|K| hd beyond int64, with keys inside the digit planes' range and beyond it."""
    q, k, v = _qkv(5, 4, 2, 128, 48, 48)
    q[0, 0, 0] = 1 << 40
    k[0, 47, 0] = mag
    assert gpu.attention_prefill_gpu(q, k, v, 0, 16, fx.inv_sqrt_fp(128, 16)) is None
    q[0, 0, 0] = 1
    k[0, 47, 0] = 1
    v[0, 3, 3] = 1 << 60
    assert gpu.attention_prefill_gpu(q, k, v, 0, 16, fx.inv_sqrt_fp(128, 16)) is None
