"""Run by test_gpu_pinned_refusal.py in a process of its own: hipHostMalloc is answered by a shim that refuses every request
once armed, and the calls that read back through pinned memory are compared with the oracle. Prints one line a call."""
from __future__ import annotations

import ctypes
import sys
from pathlib import Path

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))


def prefill(gpu, shim):
    import numpy as np
    from oracle import bonsai_model as obm, fixedpoint as fx, prng, workloads
    from oracle.q1 import q1_rows
    from tests.bonsai_gpu_harness import register_model
    model = workloads.small_bonsai(seed=6)
    cfg = model["cfg"]
    w, g = register_model(gpu, model)
    for T in (9, 21):
        x0 = q1_rows(*model["embed"], prng.uniform_int(T, 99, (T,), 0, cfg["vocab"]))
        x, ks, vs = x0, [], []
        for layer in model["layers"]:
            x, k1, v1 = obm.layer_forward(x, layer, {k: cfg[k] for k in ("H", "Hkv", "hd")}, model["cos"], model["sin"], 16,
                                          None, None, 0)
            ks.append(k1), vs.append(v1)
        want = obm.head_logits(model, x[-1:], 16)[0]
        dims = (T, cfg["d"], cfg["n_layers"], cfg["H"], cfg["Hkv"], cfg["hd"], cfg["dff"])
        got = gpu.prefill_forward_gpu(x0, dims, w, g, 16, 1, fx.inv_sqrt_fp(cfg["hd"], 16), export_kv=True)
        assert got[0] is not None, "refused"
        assert np.array_equal(got[0], want) and np.array_equal(got[1], np.stack(ks)) and np.array_equal(got[2], np.stack(vs))
        print("prefill", T, "ok", flush=True)
        shim.arm(1)                                     # the second, larger call finds no pinned memory


def bank(gpu, shim):
    import numpy as np
    from integer_inference_engine_amd import qk_gpu
    from oracle import fixedpoint as fx, nmc_block as onb, qk
    from oracle.rope import apply_interleaved, build_rope_tables
    from tests import test_gpu_nmc_bank as t
    W, hs, experts, eh = t._weights(41)
    cos, sin = build_rope_tables(t.CAP, t.HD, base=50000, frac=t.FA)
    for armed in (0, 1):
        shim.arm(armed)
        cache = qk_gpu.ResidentAttentionCache(1, t.CAP, t.D, t.H, t.HKV, t.HD, t.FA, cos, sin)
        cache.configure_moe_layer(0, t.E, t.USED, t.D, t.EFF)
        for e in range(t.E):
            cache.bind_moe_expert(0, e, *eh[e])
        kc, vc = (np.zeros((t.HKV, t.CAP, t.HD), dtype=np.int64) for _ in range(2))
        x = np.random.default_rng(42).integers(-(1 << 18), 1 << 18, size=(1, t.D), dtype=np.int64)
        want, _, _, _, kc[:, 0], vc[:, 0] = onb.block_step(x, W, kc, vc, 0, None, True, cos, sin, t.CFG, experts)
        assert not cache.begin_moe_layer(0, hs["gain"], hs["router"], hs["wq"], hs["wk"], hs["wv"], hs["wo"], x, t.FW, 1,
                                         None, True)
        assert np.array_equal(cache.continue_moe_layer(0, t.FW, publish=True), want)
        got = cache.apply(0, hs["wq"], hs["wk"], hs["wv"], hs["wo"], x, t.FW, None, True)
        q, k, v = (qk.linear(x, W[n], t.FW).reshape(-1, t.HD) for n in ("wq", "wk", "wv"))
        q, k = (apply_interleaved(a[:, None, :], cos[1:2], sin[1:2], t.FA)[:, 0, :] for a in (q, k))
        kc[:, 1], vc[:, 1] = k, v
        att = onb.attention_step(q, kc, vc, 1, None, t.FA, fx.inv_sqrt_fp(t.HD, t.FA)).reshape(1, t.H * t.HD)
        assert np.array_equal(got, qk.linear(att, W["wo"], t.FW))
        cache.close()
        print("bank", armed, "ok", flush=True)


def main():
    shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)      # before the HIP runtime: its symbol comes first
    from integer_inference_engine_amd import gpu_native as gpu
    assert gpu.gpu_available()
    globals()[sys.argv[2]](gpu, shim)
    assert shim.refused() > 0, "no request reached the shim"


if __name__ == "__main__":
    main()
