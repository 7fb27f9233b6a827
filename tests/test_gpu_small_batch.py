"""GGUF-row readouts of 2 to 4 rows below the matrix cores' line: a grid row of the batch-1
kernel per batch row, so every row is bit for bit that of a batch of 1, and (16640 columns)
the kernel of wider rows; against the fp64 oracle, max|gpu - ref| <= 1e-5 + 1e-3 max|ref|."""
import numpy as np
import pytest

import oracle as orc
from conftest import assert_close
from rta import ops
from test_gpu_wide import dev, matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [orc.Q4_K, orc.Q6_K])
@pytest.mark.parametrize("rows,cols", [(1, 256), (37, 1280), (1000, 4096), (45, 4352), (77, 8448), (61, 12544),
                                       (19, 16640)])
def test_small_batches(fmt, rows, cols):
    rng = np.random.default_rng(rows + cols + fmt)
    w, wd, f = matrix(rng, fmt, rows, cols, False, shift=2 if fmt == orc.Q6_K else 0)
    x = rng.standard_normal((4, cols)).astype(np.float32)
    x[1] *= 1e-3
    ref = orc.gemv_f64(fmt, w, rows, cols, x)
    one = np.concatenate([ops.gemv(f, wd, rows, cols, dev(x[b:b + 1])).cpu().numpy() for b in range(4)])
    for n in (2, 3, 4):
        y = ops.gemv(f, wd, rows, cols, dev(x[:n])).cpu().numpy()
        for b in range(n):
            assert_close(y[b], ref[b], f"batch {n} row {b}")
        if cols <= 16384:
            assert np.array_equal(y, one[:n]), n
        y0 = rng.standard_normal((n, rows)).astype(np.float32)
        ya = ops.gemv(f, wd, rows, cols, dev(x[:n]), y=dev(y0), accumulate=True).cpu().numpy()
        assert np.array_equal(ya, y0 + y)


@pytest.mark.parametrize("hidden,inter,batch", [(256, 256, 2), (1280, 768, 3), (4352, 512, 4)])
def test_small_batch_mlp_and_lm_head(hidden, inter, batch):
    rng = np.random.default_rng(hidden + inter + batch)
    (g, gd, _), (u, ud, _) = (matrix(rng, orc.Q4_K, inter, hidden, False) for _ in range(2))
    d, dd, _ = matrix(rng, orc.Q6_K, hidden, inter, False)
    x = rng.standard_normal((batch, hidden)).astype(np.float32)
    fm = (orc.Q4_K, orc.Q4_K, orc.Q6_K)
    act, y = ops.mlp_swiglu(fm, gd, ud, dd, hidden, inter, dev(x))
    ract, ry = orc.mlp_swiglu(fm, g, u, d, hidden, inter, x)
    assert_close(act.cpu().numpy(), ract, "activation")
    assert_close(y.cpu().numpy(), ry, "output")
    vocab = 1111
    w, wd, f = matrix(rng, orc.Q6_K, vocab, hidden, False)
    logits, ids = ops.lm_head(f, wd, vocab, hidden, dev(x))
    lg = logits.cpu().numpy()
    assert_close(lg, orc.gemv_f64(orc.Q6_K, w, vocab, hidden, x), "logits")
    for b in range(batch):
        assert int(ids.cpu().numpy().view(np.uint32)[b]) == orc.argmax_margin_f32(lg[b], 1e-4)
