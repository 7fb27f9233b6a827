"""GGUF-row readouts of 2 to 4 rows below the matrix cores' line: a grid row of the batch-1
kernel per batch row, so every row is bit for bit that of a batch of 1, or (16640 columns, some
Q6_K matrices) one reading of the weights for all rows; against the fp64 oracle, max|gpu - ref| <= 1e-5 + 1e-3 max|ref|."""
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


@pytest.mark.parametrize("rows,cols", [(15100, 1024), (15200, 1024), (16369, 1024), (15361, 1280), (15401, 1280),
                                       (3120, 6144)])
def test_q6_rows_at_the_edge_of_full_rounds(rows, cols):
    """Q6_K matrices either side of the line where 2 to 4 rows share one reading of the weights
    instead of a grid row each: 15200x1024 from 4 rows, 16369x1024 from 3, 15401x1280 from 2,
    3120x6144 (two passes a row) from 3."""
    fmt = orc.Q6_K
    rng = np.random.default_rng(rows + cols)
    w, wd, f = matrix(rng, fmt, rows, cols, False, shift=2)
    x = rng.standard_normal((4, cols)).astype(np.float32)
    x[1] *= 1e-3
    ref = orc.gemv_f64(fmt, w, rows, cols, x)
    for n in (2, 3, 4):
        y = ops.gemv(f, wd, rows, cols, dev(x[:n])).cpu().numpy()
        for b in range(n):
            assert_close(y[b], ref[b], f"batch {n} row {b}")
        y0 = rng.standard_normal((n, rows)).astype(np.float32)
        ya = ops.gemv(f, wd, rows, cols, dev(x[:n]), y=dev(y0), accumulate=True).cpu().numpy()
        assert np.array_equal(ya, y0 + y)
        logits, ids = ops.lm_head(f, wd, rows, cols, dev(x[:n]))
        lg = logits.cpu().numpy()
        assert np.array_equal(lg, y), n
        for b in range(n):
            assert int(ids.cpu().numpy().view(np.uint32)[b]) == orc.argmax_margin_f32(lg[b], 1e-4)


@pytest.mark.parametrize("inter,batch", [(7424, 4), (7680, 4), (8192, 3)])
def test_q6_swiglu_at_the_edge_of_full_rounds(inter, batch):
    hidden, q6 = 1024, orc.Q6_K
    rng = np.random.default_rng(inter + batch)
    (g, gd, _), (u, ud, _) = (matrix(rng, q6, inter, hidden, False) for _ in range(2))
    x = rng.standard_normal((batch, hidden)).astype(np.float32)
    act = ops.swiglu(q6, gd, ud, hidden, inter, dev(x)).cpu().numpy()
    gx, ux = (orc.gemv_f64(q6, m, inter, hidden, x) for m in (g, u))
    assert_close(act, gx * ux / (1 + np.exp(-gx)), "activation")


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
