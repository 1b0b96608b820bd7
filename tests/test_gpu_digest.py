"""Row digests on the device against hashlib's SHA-256 at the edges of the kernel's split: rows around the 32 of a
workgroup, vocabularies whose last block is whole, one value short of or past a block, and one whose length needs a
block of its own, and odd and even block counts (two blocks of a row are expanded at a time)."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 65])
@pytest.mark.parametrize("vocab,ld", [(1, 1), (6, 6), (7, 9), (8, 8), (9, 9), (14, 14), (15, 15), (16, 17), (23, 23),
                                      (24, 24), (1000, 1003)])
def test_digest_edges(gpu, rows, vocab, ld):
    import torch
    from integer_inference_engine_amd.verify import logits_digest_dev
    rng = np.random.default_rng(rows * 10000 + vocab)
    full = rng.integers(-(1 << 63), (1 << 63) - 1, size=(rows, ld), dtype=np.int64)
    full[0, :vocab] = -1
    dev = torch.from_numpy(full).cuda()[:, :vocab]
    want = [hashlib.sha256(np.ascontiguousarray(full[r, :vocab]).tobytes()).hexdigest() for r in range(rows)]
    assert logits_digest_dev(dev) == want
