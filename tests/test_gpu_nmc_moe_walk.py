"""The expert kernels of a batched MoE block over the edges of their walk, bit for bit against the oracle: rows of one
block, of a whole staged chunk and one past it (one group of tokens and two), output tiles of a partly filled down
workgroup, 1 to 9 tokens of one expert, five limbs (the second group holds the high ones), and block scales beyond the
32-bit factor (every block, or some of them)."""
import numpy as np
import pytest

from oracle import qk

pytestmark = pytest.mark.gpu
FW = 24


@pytest.mark.parametrize("m,n_e,k,d,ffn,mag,scale", [
    (3, 1, 1, 256, 256, 16, (5e-4, 2e-3)),            # one block, one tile of four
    (4, 2, 1, 1024, 1280, 16, (5e-4, 2e-3)),          # a chunk of two groups; one past it below
    (5, 1, 1, 1280, 1024, 16, (5e-4, 2e-3)),
    (8, 1, 1, 2048, 512, 16, (5e-4, 2e-3)),           # a chunk of one group; one past it below
    (9, 1, 1, 2304, 256, 16, (5e-4, 2e-3)),
    (3, 1, 1, 256, 2304, 16, (5e-4, 2e-3)),
    (7, 3, 2, 512, 768, 33, (2e-5, 1e-4)),            # five limbs
    (3, 1, 1, 2304, 256, 33, (2e-5, 1e-4)),
    (7, 1, 1, 512, 512, 0, (200.0, 700.0)),           # |dq| 2^24 beyond 2^31
    (6, 2, 1, 512, 512, 0, (60.0, 180.0)),            # some blocks beyond
])
def test_moe_walk(gpu, m, n_e, k, d, ffn, mag, scale):
    from integer_inference_engine_amd import qk_gpu
    rng = np.random.default_rng(d + ffn + m)
    fa, (lo, hi) = 16, scale
    experts, handles = {}, []
    for e in range(n_e):
        raws = [qk.random_blocks(11, 3 * e + i, o, n // 256, t, dlo=lo, dhi=hi, dminhi=lo)
                for i, (o, n, t) in enumerate(((ffn, d, 0), (ffn, d, 0), (d, ffn, 1)))]
        experts[e] = {n: qk.dequant(r, o, i // 256, t, FW) for n, r, (o, i, t) in
                      zip(("gate", "up", "down"), raws, ((ffn, d, 0), (ffn, d, 0), (d, ffn, 1)))}
        handles.append([qk_gpu.register_weight(r, o, i // 256, t) for r, (o, i, t) in
                        zip(raws, ((ffn, d, 0), (ffn, d, 0), (d, ffn, 1)))])
    h = rng.integers(-(1 << mag), (1 << mag) + 1, size=(m, d), dtype=np.int64)
    sel = np.stack([rng.permutation(n_e)[:k] for _ in range(m)])
    gates = rng.integers(1, 1 << fa, size=(m, k), dtype=np.int64)
    flat = sel.reshape(-1)
    got = qk_gpu.moe_ffn_batched([handles[e][0] for e in flat], [handles[e][1] for e in flat],
                                 [handles[e][2] for e in flat], m, k, h, gates, d, ffn, fa, FW)
    want = qk.moe_ffn(h, sel, gates, experts, fa, FW)
    assert got is not None and np.array_equal(got, want)
    qk_gpu.free_all()
