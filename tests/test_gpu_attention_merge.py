"""Decode attention where a few long sequences share the workgroups: the merge that gives a
quarter of a head to each workgroup (at most 64 (sequence, head) pairs, over 128 tiles), both
sides of its two lines, and tile lists whose sequences hold none, one or hundreds of the
workgroups' first tiles.  Bar as in test_gpu_attention_cases.py."""
import numpy as np
import pytest

import oracle as orc
from test_gpu_attention_cases import LAYOUTS, _sized_case, torch_dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmts", LAYOUTS)
@pytest.mark.parametrize("hq,hkv,ctx", [(16, 4, [8192]), (16, 4, [8193]), (4, 1, [40000, 1]), (8, 8, [9000] * 8),
                                        (8, 4, [9000] * 9), (16, 2, [30000, 64, 65, 1])])
def test_few_long_sequences(torch_dev, fmts, hq, hkv, ctx):  # noqa: F811
    torch, dev = torch_dev
    _sized_case(torch, dev, 71 + len(ctx), ctx, hq, hkv, fmts, gate=True)


def test_tile_list_of_70_uneven_sequences(torch_dev):  # noqa: F811
    torch, dev = torch_dev
    ctx = np.full(70, 3)
    ctx[[0, 5, 63, 64, 69]] = [6000, 64, 12000, 65, 9000]
    _sized_case(torch, dev, 72, ctx, 8, 2, (orc.Q4_K, orc.Q6_K))


@pytest.mark.parametrize("nseq", [4, 64, 66])
def test_tile_list_at_the_line_of_long_runs(torch_dev, nseq):  # noqa: F811
    """Runs of 31 to 33 workgroups and of none, side by side: up to 32 are listed by the
    sequence's own lane, longer ones by the wave."""
    torch, dev = torch_dev
    ctx = np.full(nseq, 1)
    ctx[[0, 1, 2, nseq - 1]] = [2048, 2112, 1984, 2112]
    _sized_case(torch, dev, 73 + nseq, ctx, 8, 2, (orc.Q4_K, orc.Q6_K))
