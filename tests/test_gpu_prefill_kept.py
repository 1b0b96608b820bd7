"""What whole prefills (bonsai_prefill_forward_gpu) keep between calls never shows in a result: in one process, small calls
behind large ones, another layer count and head layout, a refused call, an export on four threads whose parts are no whole
pages, a call beyond what is kept (2 GiB of workspaces, 256 MiB of export), and calls after the memory was given back.
Small calls against the oracle, large ones against the resident forward over a kv8 cache, to the bit."""
import ctypes

import numpy as np
import pytest

from oracle import bonsai_model as obm, fixedpoint as fx, prng, workloads
from tests.bonsai_gpu_harness import register_model

pytestmark = pytest.mark.gpu
A = dict(d=256, H=8, Hkv=8, hd=128, dff=256, n_layers=2, vocab=64, ctx=8400)      # 272 MB of K / V at 8320 rows
B = dict(d=256, H=4, Hkv=2, hd=96, dff=384, n_layers=3, vocab=80, ctx=1100)       # 9.2 MB at 1001


def _x(T, d):
    return prng.uniform_int(T, 5, (T, d), -(1 << 18), 1 << 18)


class _Model:
    def __init__(self, gpu, cfg, seed):
        self.gpu, self.model = gpu, workloads.bonsai_model(seed, **cfg)
        self.cfg, self.want = self.model["cfg"], {}
        self.register()

    def register(self):
        self.w, self.g = register_model(self.gpu, self.model)

    def _oracle(self, T):
        c = {k: self.cfg[k] for k in ("H", "Hkv", "hd")}
        x, ks, vs = _x(T, self.cfg["d"]), [], []
        for layer in self.model["layers"]:
            x, k, v = obm.layer_forward(x, layer, c, self.model["cos"], self.model["sin"], 16, None, None, 0)
            ks.append(k), vs.append(v)
        return obm.head_logits(self.model, x[-1:], 16)[0], np.stack(ks), np.stack(vs)

    def _resident(self, T):
        import torch
        from integer_inference_engine_amd.resident import ResidentNet
        c = self.cfg
        net = ResidentNet(B=1, n_layers=c["n_layers"], H=c["H"], Hkv=c["Hkv"], hd=c["hd"], d=c["d"], dff=c["dff"], cap=T,
                          w=self.w, g=self.g, kv32=True)
        try:
            x = torch.from_numpy(_x(T, c["d"])).cuda()
            assert net.forward(x, [0], T) == 0
            last = x[T - 1:].contiguous()
            torch.cuda.synchronize()
            logits = net.head(last, 1)[0].cpu().numpy()[0]
            kv = [net.export_kv(li, 0, T) for li in range(c["n_layers"])]
            return logits, np.stack([k for k, _ in kv]), np.stack([v for _, v in kv])
        finally:
            net.close()

    def dims(self, T):
        c = self.cfg
        return T, c["d"], c["n_layers"], c["H"], c["Hkv"], c["hd"], c["dff"]

    def call(self, T, w=None):
        inv = fx.inv_sqrt_fp(self.cfg["hd"], 16)
        return self.gpu.prefill_forward_gpu(_x(T, self.cfg["d"]), self.dims(T), w or self.w, self.g, 16, 1, inv, export_kv=True)

    def check(self, T):
        if T not in self.want:
            self.want[T] = self._oracle(T) if T <= 64 else self._resident(T)
        print(f"[kept] {self.cfg['n_layers']} layers, {T} rows", flush=True)
        for got, want, what in zip(self.call(T), self.want[T], ("logits", "K", "V")):
            assert got is not None and np.array_equal(got, want), (T, what)


def _free_bytes(so):
    free, total = ctypes.c_uint64(0), ctypes.c_uint64(0)
    assert so.bonsai_gpu_mem_info(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_kept_memory_never_shows(gpu):
    from integer_inference_engine_amd import _lib
    so = _lib.lib()
    so.imie_prefill_release()
    a, b = _Model(gpu, A, 61), _Model(gpu, B, 62)
    for m, T in ((a, 5), (b, 1001), (a, 33), (b, 7), (b, 1), (b, 1001)):
        m.check(T)

    # refused (a layer's V far beyond p V's bound): the caller's arrays are as they were, the next calls unharmed
    layer = b.model["layers"][1]
    bad = dict(b.w, wv=b.w["wv"].copy())
    bad["wv"][1] = gpu.q1_register_weight(layer["wv"][0], layer["wv"][1].astype(np.int64) << 32)
    T = 1001
    logits, k = np.full(80, 77, dtype=np.int64), np.full((2, 3, 2, T, 96), -5, dtype=np.int64)
    x, arr = _x(T, 256), {**{n: np.ascontiguousarray(bad[n]) for n in workloads.PROJ}, **b.g}
    rc = so.bonsai_prefill_forward_gpu(
        x.ctypes.data, *b.dims(T), 16, 1, fx.inv_sqrt_fp(96, 16),
        *[arr[n].ctypes.data for n in (*workloads.PROJ, "n1g", "n2g", "qng", "kng")], int(b.g["finalg"]),
        int(b.w["out_head"]), int(b.g["cos_h"]), int(b.g["sin_h"]), logits.ctypes.data, k[0].ctypes.data, k[1].ctypes.data)
    assert rc == 2 and (logits == 77).all() and (k == -5).all()
    assert b.call(7, bad)[0] is None
    b.check(7)
    b.check(1001)

    # beyond both bounds: nothing of it stays
    a.want[8320] = a._resident(8320)
    before = _free_bytes(so)
    a.check(8320)
    assert _free_bytes(so) >= before
    a.check(33)
    b.check(1001)

    # given back: by its own call, which leaves the model, and with the uploaded buffers
    before = _free_bytes(so)
    gpu.release_prefill_workspace()
    assert _free_bytes(so) > before
    b.check(7)
    a.check(33)
    so.imie_buf_free_all()
    a.register(), b.register()
    b.check(1001)
    a.check(5)
    gpu.release_prefill_workspace()
