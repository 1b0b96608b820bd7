"""kv8 pages whose byte offsets leave 32 bits: the same rows, prefilled and decoded over one huge page and over pages of 64
slots, give the same bits. 2^25 slots of 32 dims are the first block beyond the fused prefill's offsets, 286,331,200 slots
the first page beyond the decode PV's lane offsets (36 GB of K and of V)."""
import numpy as np
import pytest

from oracle import prng, workloads
from tests.bonsai_gpu_harness import register_model

pytestmark = pytest.mark.gpu
HD, FIRST = 32, 37


def _net(gpu, model, page):
    from integer_inference_engine_amd.resident import ResidentNet
    cfg = model["cfg"]
    w, g = register_model(gpu, model, with_head=False)
    return ResidentNet(B=1, n_layers=1, H=cfg["H"], Hkv=cfg["Hkv"], hd=HD, d=cfg["d"], dff=cfg["dff"], cap=64, w=w, g=g,
                       page=page, kv32=True)


def _model(H, Hkv):
    return workloads.bonsai_model(70 + H, d=256, H=H, Hkv=Hkv, hd=HD, dff=256, n_layers=1, vocab=64, ctx=64)


def _rows(gpu, model, page):
    import torch
    net = _net(gpu, model, page)
    out = []
    try:
        for start, M in ((0, FIRST), (FIRST, 1), (FIRST + 1, 1), (FIRST + 2, 9)):
            x = torch.from_numpy(prng.uniform_int(71, start, (M, 256), -(1 << 18), 1 << 18)).cuda()
            assert net.forward(x, [start], M) == 0
            out.append(x.cpu().numpy())
    finally:
        net.close()
    return out


@pytest.mark.parametrize("H,Hkv,page", [(4, 1, 1 << 25), (8, 2, 1 << 25), (4, 4, 1 << 25), (4, 1, 286331136),
                                        (4, 1, 286331200), (8, 1, 286331200)])
def test_large_pages(gpu, H, Hkv, page):
    model = _model(H, Hkv)
    print(f"[large pages] H={H} Hkv={Hkv} page={page}", flush=True)
    for got, want in zip(_rows(gpu, model, page), _rows(gpu, model, 64)):
        assert np.array_equal(got, want)


def test_large_pages_refuse_one_row_of_other_layouts(gpu):
    """One new row of three query heads per kv head goes through the fused prefill kernel: refused where the page is too
    large for it, computed where it is not."""
    import torch
    model = _model(12, 4)
    for page, ok in ((1 << 24, True), (1 << 25, False)):
        net = _net(gpu, model, page)
        try:
            x = torch.from_numpy(prng.uniform_int(72, 1, (1, 256), -(1 << 18), 1 << 18)).cuda()
            if ok:
                assert net.forward(x, [0], 1) == 0
            else:
                with pytest.raises(RuntimeError):
                    net.forward(x, [0], 1)
        finally:
            net.close()
