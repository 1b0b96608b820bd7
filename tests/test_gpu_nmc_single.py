"""One activation row against Q4_K / Q6_K weights, and the MoE block of one and two tokens, bit for bit against the
oracle: block counts around a half wave's 8 blocks and the largest the single-row kernel takes, odd output sizes,
digits at their limb edges, and rows beyond five limbs."""
import numpy as np
import pytest

from oracle import qk

pytestmark = pytest.mark.gpu
FW = 24


def _x(rng, n, kind):
    if kind == "edges":                                 # the extremes of 1..5 balanced limbs
        caps = [127 * ((256 ** l - 1) // 255) for l in range(1, 6)]
        return rng.choice(np.array(caps + [-c for c in caps] + [c - 255 for c in caps], dtype=np.int64), size=n)
    if kind.startswith("wide"):
        x = rng.integers(-(1 << 20), 1 << 20, size=n, dtype=np.int64)
        x[rng.integers(0, n)] = (1 << int(kind[4:])) + 77   # one value beyond five limbs
        return x
    return rng.integers(-(1 << int(kind)), 1 << int(kind), size=n, dtype=np.int64)


@pytest.mark.parametrize("qtype,out_f,nb,kind", [
    (0, 33, 1, "6"), (1, 17, 1, "edges"), (0, 7, 8, "20"), (1, 16, 8, "wide45"), (0, 40, 9, "edges"),
    (1, 5, 16, "30"), (0, 16, 32, "wide45"), (1, 31, 32, "20"), (0, 9, 33, "20"), (1, 3, 33, "edges"),
])
def test_single_row_linear(gpu, qtype, out_f, nb, kind):
    from integer_inference_engine_amd import qk_gpu
    rng = np.random.default_rng(nb * 10 + qtype)
    raw = qk.random_blocks(nb, qtype, out_f, nb, qtype)
    x = _x(rng, nb * 256, kind).reshape(1, -1)
    h = qk_gpu.register_weight(raw, out_f, nb, qtype)
    got = qk_gpu.apply_resident(h, x, out_f, FW)
    assert np.array_equal(got, qk.linear(x, qk.dequant(raw, out_f, nb, qtype, FW), FW))
    qk_gpu.free_all()


def test_single_row_grouped_mixed_types(gpu):
    """Q4_K and Q6_K weights of different heights in one launch, as the Q / K / V projections are."""
    from integer_inference_engine_amd import qk_gpu
    rng = np.random.default_rng(3)
    x = rng.integers(-(1 << 18), 1 << 18, size=(1, 512), dtype=np.int64)
    sizes = [(64, 0), (17, 1), (1, 0), (33, 1)]
    raws = [qk.random_blocks(5, i, o, 2, t) for i, (o, t) in enumerate(sizes)]
    hs = [qk_gpu.register_weight(r, o, 2, t) for r, (o, t) in zip(raws, sizes)]
    got = qk_gpu.apply_resident_grouped(hs, x, [o for o, _ in sizes], FW)
    for g, r, (o, t) in zip(got, raws, sizes):
        assert np.array_equal(g, qk.linear(x, qk.dequant(r, o, 2, t, FW), FW))
    qk_gpu.free_all()


@pytest.mark.parametrize("m,k,d,ffn,kind", [
    (1, 1, 256, 256, "20"), (1, 8, 512, 768, "16"), (2, 3, 256, 512, "edges"), (2, 8, 256, 256, "18"),
    (1, 2, 512, 256, "wide39"), (1, 16, 256, 512, "16"), (3, 2, 256, 256, "16"),
])
def test_moe_few_tokens(gpu, m, k, d, ffn, kind):
    from integer_inference_engine_amd import qk_gpu
    rng = np.random.default_rng(d + ffn + k)
    n_e, fa = max(k, 4), 16
    experts, handles = {}, []
    lo, hi = (0.0005, 0.002) if not kind.startswith("wide") else (5e-7, 2e-6)   # small weights for the wide row
    for e in range(n_e):
        raws = [qk.random_blocks(9, 3 * e + i, o, n // 256, t, dlo=lo, dhi=hi, dminhi=lo)
                for i, (o, n, t) in enumerate(((ffn, d, 0), (ffn, d, 0), (d, ffn, 1)))]
        experts[e] = {n: qk.dequant(r, o, i // 256, t, FW) for n, r, (o, i, t) in
                      zip(("gate", "up", "down"), raws, ((ffn, d, 0), (ffn, d, 0), (d, ffn, 1)))}
        handles.append([qk_gpu.register_weight(r, o, i // 256, t) for r, (o, i, t) in
                        zip(raws, ((ffn, d, 0), (ffn, d, 0), (d, ffn, 1)))])
    h = np.stack([_x(rng, d, kind) for _ in range(m)])
    if kind == "edges":
        h >>= 20                                        # the products stay in the int64 envelope
    sel = np.stack([rng.permutation(n_e)[:k] for _ in range(m)])
    gates = rng.integers(1, 1 << fa, size=(m, k), dtype=np.int64)
    flat = sel.reshape(-1)
    got = qk_gpu.moe_ffn_batched([handles[e][0] for e in flat], [handles[e][1] for e in flat],
                                 [handles[e][2] for e in flat], m, k, h, gates, d, ffn, fa, FW)
    want = qk.moe_ffn(h, sel, gates, experts, fa, FW)
    assert got is not None and np.array_equal(got, want)
    qk_gpu.free_all()


@pytest.mark.parametrize("k,d,ffn", [(2, 8192, 1024), (2, 8192, 1280), (16, 2048, 256), (16, 2048, 512)])
def test_moe_two_tokens_as_one_each(gpu, k, d, ffn):
    """Two tokens at and beyond the weight volume where the grouped kernels take over, against one token each (the small
    form, held to the oracle above): the same bits."""
    from integer_inference_engine_amd import qk_gpu
    rng = np.random.default_rng(d + ffn)
    handles = [[qk_gpu.register_weight(qk.random_blocks(11, 3 * e + i, o, n // 256, t), o, n // 256, t)
                for i, (o, n, t) in enumerate(((ffn, d, 0), (ffn, d, 0), (d, ffn, 1)))] for e in range(k + 1)]
    h = rng.integers(-(1 << 12), 1 << 12, size=(2, d), dtype=np.int64)
    sel = np.stack([rng.permutation(k + 1)[:k] for _ in range(2)])
    gates = rng.integers(1, 1 << 16, size=(2, k), dtype=np.int64)

    def call(tokens):
        flat = sel[tokens].reshape(-1)
        return qk_gpu.moe_ffn_batched(*([handles[e][i] for e in flat] for i in range(3)), len(tokens), k, h[tokens],
                                      gates[tokens], d, ffn, 16, FW)

    got, one = call([0, 1]), [call([t]) for t in range(2)]
    assert got is not None and np.array_equal(got, np.concatenate(one)) and got.any()
    qk_gpu.free_all()
