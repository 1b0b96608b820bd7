"""kv8 attention reads a cache's fourth digit plane only when its running maximum needs one: caches whose max|K| or
max|V| lies at the largest three-digit value, one above it and far above it, mixed over sequences and kv heads, in
decode (one new row) and prefill (33 new rows) and over the head layouts, byte for byte against the oracle layer stack;
and a row that starts behind slots written before a reset, whose maxima the reset has cleared."""
import numpy as np
import pytest

from oracle import bonsai_model as obm, c_oracle, prng, workloads
from oracle.q1 import q1_rows
from tests.bonsai_gpu_harness import register_model

pytestmark = pytest.mark.gpu

CAP = 320
CAP3 = 127 * (256 ** 3 - 1) // 255
# (H, Hkv, hd)
LAYOUTS = [(4, 4, 64), (16, 2, 96), (8, 2, 128), (8, 1, 128)]


def _net(gpu, model, B):
    from integer_inference_engine_amd.resident import ResidentNet
    cfg = model["cfg"]
    w, g = register_model(gpu, model, with_head=False)
    return ResidentNet(B=B, n_layers=cfg["n_layers"], H=cfg["H"], Hkv=cfg["Hkv"], hd=cfg["hd"], d=cfg["d"],
                       dff=cfg["dff"], cap=CAP, w=w, g=g, kv32=True)


def _cache(seed, tag, cfg, n, edges):
    """(n_layers, Hkv, n, hd) values below 2^20 with one element of kv head i of layer l set to edges[l + i]."""
    out = np.stack([prng.uniform_int(seed, tag + li, (cfg["Hkv"], n, cfg["hd"]), -(1 << 20), 1 << 20)
                    for li in range(cfg["n_layers"])])
    for li in range(cfg["n_layers"]):
        for kv in range(cfg["Hkv"]):
            out[li, kv, (7 * li + 11 * kv) % n, (5 * kv + li) % cfg["hd"]] = edges[(li + kv) % len(edges)]
    return out


def _planes(seqs):
    """seqs: per sequence the (n_layers, Hkv, n, hd) values; planes by their maxima, (n_layers, B, Hkv)."""
    return np.stack([np.where(np.abs(s).max(axis=(2, 3)) <= CAP3, 3, 4) for s in seqs], axis=1)


def _check(net, model, c, ks, vs, starts, M, seed):
    import torch
    xs = [q1_rows(*model["embed"], prng.uniform_int(seed, 20 + b, (M,), 0, 64)) for b in range(len(starts))]
    x = torch.from_numpy(np.concatenate(xs)).cuda()
    assert net.forward(x, starts, M) == 0
    got = x.cpu().numpy()
    for b, s0 in enumerate(starts):
        want = xs[b]
        for li, layer in enumerate(model["layers"]):
            want, _, _ = obm.layer_forward(want, layer, c, model["cos"], model["sin"], 16, ks[b][li], vs[b][li], s0,
                                           q1=c_oracle.q1_linear)
        bad = np.flatnonzero(got[b * M:(b + 1) * M] != want)
        assert bad.size == 0, f"sequence {b}: {bad.size} values differ"


@pytest.mark.parametrize("M", [1, 33])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_kv8_planes_by_maximum(gpu, layout, M):
    H, Hkv, hd = layout
    seed = 300 + H + 3 * Hkv + hd + M
    model = workloads.bonsai_model(seed, d=256, H=H, Hkv=Hkv, hd=hd, dff=512, n_layers=2, vocab=64, ctx=CAP)
    c = {"H": H, "Hkv": Hkv, "hd": hd}
    starts = [200, 70, 130]
    kedge = [[CAP3, CAP3 + 1], [-CAP3 - 1, -CAP3], [1 << 26, 5]]
    vedge = [[-CAP3 - 1, CAP3], [CAP3, -CAP3], [7, (1 << 27) + 3]]
    ks = [_cache(seed, 10 + 4 * b, model["cfg"], n, kedge[b]) for b, n in enumerate(starts)]
    vs = [_cache(seed, 30 + 4 * b, model["cfg"], n, vedge[b]) for b, n in enumerate(starts)]
    print(f"[kv8-planes] H={H} Hkv={Hkv} hd={hd} {starts} + {M}", flush=True)
    net = _net(gpu, model, 3)
    try:
        for b in range(3):
            net.seed(b, ks[b], vs[b])
        got = net.kv_planes()
        assert np.array_equal(got[:, 0], _planes(ks)) and np.array_equal(got[:, 1], _planes(vs))
        _check(net, model, c, ks, vs, starts, M, seed)
    finally:
        net.close()
    net = _net(gpu, model, 1)                        # one sequence: the decode path that stores its exponentials
    try:
        net.seed(0, ks[1], vs[1])
        _check(net, model, c, [ks[1]], [vs[1]], starts[1:2], M, seed)
    finally:
        net.close()


@pytest.mark.parametrize("M", [1, 33])
def test_kv8_planes_behind_a_reset(gpu, M):
    H, Hkv, hd = 8, 2, 128
    seed = 350 + M
    model = workloads.bonsai_model(seed, d=256, H=H, Hkv=Hkv, hd=hd, dff=512, n_layers=2, vocab=64, ctx=CAP)
    ks = _cache(seed, 10, model["cfg"], 100, [1 << 26, CAP3 + 1])
    vs = _cache(seed, 30, model["cfg"], 100, [CAP3 + 1, -(1 << 27)])
    net = _net(gpu, model, 1)
    try:
        net.seed(0, ks, vs)
        net.reset()
        net.reset()
        assert (net.kv_planes() == 4).all()            # some value of every cached head lay beyond three digits
        _check(net, model, {"H": H, "Hkv": Hkv, "hd": hd}, [ks], [vs], [100], M, seed)
    finally:
        net.close()
