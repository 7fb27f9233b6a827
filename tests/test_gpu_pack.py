"""rta_pack at the edges of its blocks (16 rows x 8 superblocks), byte for byte against the
layout built from the GGUF blocks: partial row tiles, partial and several superblock runs,
Q6_K matrices whose rows start 2 bytes into a dword, and nothing written past the end."""
import numpy as np
import pytest

import oracle as orc
from rta import _lib, ops, synth
from test_gpu_tiled import np_pack

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,shift", [(orc.Q4_K, 0), (orc.Q6_K, 0), (orc.Q6_K, 2)])
@pytest.mark.parametrize("rows,cols", [(1, 256), (15, 7 * 256), (16, 8 * 256), (17, 9 * 256), (33, 23 * 256)])
def test_pack_edges(fmt, shift, rows, cols):
    import torch
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(rows * 7 + cols + fmt + shift)
    w = synth.random_matrix(rng, fmt, rows, cols)
    held = torch.zeros(w.size + 2, dtype=torch.uint8, device=dev)
    held[shift:shift + w.size] = torch.from_numpy(w.reshape(-1)).to(dev)
    n = ops.pack_bytes(fmt, rows, cols)
    out = torch.full((n + 64,), 0xA5, dtype=torch.uint8, device=dev)
    _lib.check(_lib.load().rta_pack(fmt, held.data_ptr() + shift, rows, cols, out.data_ptr(), ops._stream()))
    got = out.cpu().numpy()
    assert np.array_equal(got[:n], np_pack(fmt, w, rows, cols))
    assert (got[n:] == 0xA5).all()
