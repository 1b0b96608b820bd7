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


def main():
    shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)      # before the HIP runtime: its symbol comes first
    from integer_inference_engine_amd import gpu_native as gpu
    assert gpu.gpu_available()
    globals()[sys.argv[2]](gpu, shim)
    assert shim.refused() > 0, "no request reached the shim"


if __name__ == "__main__":
    main()
