"""The Q1_0 linear of one to nine rows, bit for bit against the oracle, where its kernels' edges lie: one token with K
split over a workgroup's waves (up to 32 slabs) and beyond, two to eight tokens over odd tile counts, partial slabs
and tiles, and slabs of one limb, of the last 32-bit limb (three), of four, and of every limb beyond the staged ones."""
import numpy as np
import pytest

from oracle.q1 import q1_linear

pytestmark = pytest.mark.gpu
CAP3, CAP4 = 127 * ((256 ** 3 - 1) // 255), 127 * ((256 ** 4 - 1) // 255)


def _case(seed, T, N, nb, wide):
    rng = np.random.default_rng(seed)
    bits = rng.integers(0, 256, size=(N, nb, 16), dtype=np.uint8)
    scale = rng.integers(-(1 << 34) if wide else -4096, 1 << 34 if wide else 4097, size=(N, nb), dtype=np.int64)
    x = rng.integers(-(1 << 20), 1 << 20, size=(T, nb * 128), dtype=np.int64)
    kinds = [127, CAP3, CAP3 + 1, CAP4, CAP4 + 1, 1 << 45, (1 << 63) - 1]
    for t in range(T):                                  # a different largest value per (token, slab)
        for sl in range((nb + 3) // 4):
            k = kinds[(t + sl + seed) % len(kinds)]
            lo, hi = sl * 512, min(sl * 512 + 512, nb * 128)
            if k == 127:
                x[t, lo:hi] %= 127
            x[t, rng.integers(lo, hi)] = k if rng.random() < 0.5 else -k
    return bits, scale, x


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("T,N,nb", [
    (1, 1, 1), (1, 16, 4), (1, 333, 11), (1, 4097, 32), (1, 40, 33), (1, 70, 128), (1, 48, 130),
    (2, 17, 1), (3, 333, 5), (4, 4096, 8), (5, 100, 33), (7, 64, 96), (8, 16, 9), (8, 2000, 32), (9, 33, 8),
    (3, 32784, 4),                                      # an odd number of tiles, two per wave
    (2, 32768, 4), (2, 65552, 4), (5, 65552, 4),        # the last count of one tile per wave; the first beyond one round
])
def test_few_rows(gpu, T, N, nb, wide):
    bits, scale, x = _case(T * 1000 + nb, T, N, nb, wide)
    h = gpu.q1_register_weight(bits, scale)
    got = gpu.q1_apply_resident(h, x, N, nb, 16)
    assert np.array_equal(got, q1_linear(x, bits, scale, 16))
    gpu.q1_free_weights()


@pytest.mark.parametrize("frac", [0, 1, 31, 63])
def test_few_rows_frac(gpu, frac):
    bits, scale, x = _case(3, 4, 50, 6, False)
    for T in (1, 4):
        assert np.array_equal(gpu.q1_apply_gpu(x[:T], bits, scale, frac), q1_linear(x[:T], bits, scale, frac))
