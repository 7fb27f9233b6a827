"""The readouts of more than one matrix-core batch tile (over 32 rows) at the edges of the
wide kernel's blocks: 64 / 128-row batch blocks, partial row tiles and row blocks, one and
several K slabs, batches past one launch (256 rows), GGUF rows (also Q6_K rows that start 2
bytes into a dword) and packed tiles, every epilogue; and that a workspace sized for a batch
of 32 is still accepted and gives the same results to rounding.

Bar: max|gpu - ref| <= 1e-5 + 1e-3 max|ref| per tensor against the fp64 oracle; between the
two paths 1e-5 of the peak (both sum the same exact products in fp32)."""
import numpy as np
import pytest

import oracle as orc
from conftest import assert_close
from rta import _lib, ops, synth
from rta._lib import TILED

pytestmark = pytest.mark.gpu
REL, ABS = 1e-3, 1e-5


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def matrix(rng, fmt, rows, cols, packed, shift=0):
    import torch
    w = synth.random_matrix(rng, fmt, rows, cols)
    if packed:
        return w, ops.pack(fmt, dev(w), rows, cols), fmt | TILED
    held = torch.zeros(w.size + shift, dtype=torch.uint8, device="cuda:0")
    held[shift:] = dev(w.reshape(-1))
    return w, held[shift:], fmt


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("fmt", [orc.Q4_K, orc.Q6_K])
@pytest.mark.parametrize("rows,cols,batch", [(16, 256, 33), (17, 512, 64), (300, 768, 65), (1000, 2304, 128),
                                             (4096, 1024, 129), (777, 256, 256), (130, 512, 300), (8200, 2048, 200)])
def test_wide_readout(fmt, packed, rows, cols, batch):
    rng = np.random.default_rng(rows + 3 * cols + 5 * batch + fmt)
    w, wd, f = matrix(rng, fmt, rows, cols, packed, shift=2 if fmt == orc.Q6_K and not packed else 0)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x[1] *= 1e3
    x[2] *= 1e-3
    x[batch - 1] = 0
    ref = orc.gemv_f64(fmt, w, rows, cols, x)
    y = ops.gemv(f, wd, rows, cols, dev(x))
    for b in range(batch):
        assert_close(y[b].cpu().numpy(), ref[b], f"row {b}")
    y0 = rng.standard_normal((batch, rows)).astype(np.float32)
    ya = ops.gemv(f, wd, rows, cols, dev(x), y=dev(y0), accumulate=True)
    assert_close(ya.cpu().numpy(), ref + y0, "accumulated")
    # a workspace sized for 32 rows keeps the narrow tiles
    need = ops.gemv_workspace_bytes(f, rows, cols, 32)
    small = np.zeros(max(need, 1), np.uint8)
    assert ops.gemv_workspace_bytes(f, rows, cols, batch) >= need
    yn = ops.gemv(f, wd, rows, cols, dev(x), workspace=dev(small))
    peak = float(np.abs(ref).max())
    assert float((yn - y).abs().max()) <= 1e-5 * peak
    if need:
        with pytest.raises(_lib.RtaError):
            ops.gemv(f, wd, rows, cols, dev(x), workspace=dev(small[:need - 1]))


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("hidden,inter,batch", [(512, 1536, 100), (2048, 6144, 256), (768, 1024, 257)])
def test_wide_mlp(packed, hidden, inter, batch):
    rng = np.random.default_rng(hidden + inter + batch)
    (g, gd, f), (u, ud, _) = (matrix(rng, orc.Q4_K, inter, hidden, packed) for _ in range(2))
    d, dd, fd = matrix(rng, orc.Q6_K, hidden, inter, packed)
    x = rng.standard_normal((batch, hidden)).astype(np.float32)
    act, y = ops.mlp_swiglu((f, f, fd), gd, ud, dd, hidden, inter, dev(x))
    ract, ry = orc.mlp_swiglu((orc.Q4_K, orc.Q4_K, orc.Q6_K), g, u, d, hidden, inter, x)
    assert_close(act.cpu().numpy(), ract, "activation")
    assert_close(y.cpu().numpy(), ry, "output")


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("vocab,hidden,batch", [(3001, 512, 33), (20011, 1024, 65), (9000, 256, 260)])
def test_wide_lm_head(packed, vocab, hidden, batch):
    rng = np.random.default_rng(vocab + hidden + batch)
    w, wd, f = matrix(rng, orc.Q6_K, vocab, hidden, packed)
    h = (rng.standard_normal((batch, hidden)) * 2).astype(np.float32)
    logits, ids = ops.lm_head(f, wd, vocab, hidden, dev(h))
    lg, ids = logits.cpu().numpy(), ids.cpu().numpy().view(np.uint32)
    ref = orc.gemv_f64(orc.Q6_K, w, vocab, hidden, h)
    assert_close(lg, ref, "logits")
    for b in range(batch):
        assert int(ids[b]) == orc.argmax_margin_f32(lg[b], 1e-4), b


@pytest.mark.parametrize("fmt", [orc.Q4_K, orc.Q6_K])
@pytest.mark.parametrize("rows,cols", [(700, 4096), (2064, 768)])
def test_rows_of_wide_calls_do_not_depend_on_the_batch(fmt, rows, cols):
    """Bitwise: calls of 33 to 64 rows against calls of 17 to 32; within the classes
    (64, 128] and above 128 rows, across launches of 256, on packed tiles and GGUF rows."""
    rng = np.random.default_rng(rows + cols + fmt)
    x = dev(rng.standard_normal((600, cols)).astype(np.float32))
    for packed in (False, True):
        _, wd, f = matrix(rng, fmt, rows, cols, packed)
        y = {n: ops.gemv(f, wd, rows, cols, x[:n]).cpu().numpy() for n in (20, 32, 33, 64, 65, 128, 129, 257, 600)}
        for a, b in ((20, 64), (32, 33), (65, 128), (129, 600), (257, 600)):
            assert np.array_equal(y[a], y[b][:a]), (packed, a, b)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("rows,cols", [(6144, 2048), (1000, 4096)])
def test_smaller_batches_on_the_largest_batchs_workspace(rows, cols, packed):
    """Bitwise the results of a workspace of their own, where 64 rows (both shapes) and 65 to 128
    (6144x2048) are cut into more K slabs than 256."""
    rng = np.random.default_rng(rows + cols)
    _, wd, f = matrix(rng, orc.Q4_K, rows, cols, packed)
    x = dev(rng.standard_normal((256, cols)).astype(np.float32))
    largest = dev(np.zeros(ops.gemv_workspace_bytes(f, rows, cols, 256), np.uint8))
    for n in (20, 33, 64, 65, 100, 128, 129, 256):
        y = ops.gemv(f, wd, rows, cols, x[:n], workspace=largest)
        assert np.array_equal(y.cpu().numpy(), ops.gemv(f, wd, rows, cols, x[:n]).cpu().numpy()), n


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("batch", [33, 65])
def test_step_norms_in_the_wide_readouts(packed, batch):
    """A decode step whose readouts take the RMSNorm in front of them in their x preparation,
    against the fp64 composition."""
    from rta import model
    from rta._lib import Q4_K, Q6_K
    from step_reference import check_steps
    t = TILED if packed else 0
    shape = model.HybridShape(hidden=512, layers=4, full_every=2, q_heads=4, kv_heads=2, head_dim=128, rec_heads=2,
                              ff=768, vocab=3001, capacity=64, fmt_embed=Q4_K, fmt_proj=Q4_K | t, fmt_lm=Q6_K | t,
                              fmt_k=Q4_K, fmt_v=Q6_K, rope_rotary=128, eps=1e-6, margin=1e-4, rope_theta=1e6)
    m = model.DecodeModel(shape, batch, [3 + 2 * i % 90 for i in range(batch)], seed=17, keep_gguf=True)
    check_steps(m, 2)


def small_step(hidden, batch, packed):
    from rta import model
    from rta._lib import Q4_K, Q6_K
    t = TILED if packed else 0
    shape = model.HybridShape(hidden=hidden, layers=2, full_every=2, q_heads=2, kv_heads=2, head_dim=128, rec_heads=2,
                              ff=512, vocab=300, capacity=64, fmt_embed=Q4_K, fmt_proj=Q4_K | t, fmt_lm=Q6_K | t,
                              fmt_k=Q4_K, fmt_v=Q6_K, rope_rotary=128, eps=1e-6, margin=1e-4, rope_theta=1e6)
    return model.DecodeModel(shape, batch, [3 + i % 50 for i in range(batch)], seed=18, keep_gguf=True)


@pytest.mark.parametrize("batch", [256, 257])
def test_step_norms_at_one_launch_of_rows(batch):
    """The readouts take the norm up to 256 sequences; above, it is a launch of its own."""
    from step_reference import check_steps
    check_steps(small_step(512, batch, True), 1)


@pytest.mark.parametrize("batch", [33, 257])
def test_step_refuses_an_unaligned_norm_vector(batch):
    """As the norm kernel itself does, also where a readout would take the norm."""
    m = small_step(256, batch, True)
    for name in ("norm_in", "norm_post"):
        at = getattr(m.layers[1], name)
        setattr(m.layers[1], name, at + 4)
        with pytest.raises(_lib.RtaError) as e:
            m.step()
        assert e.value.status == 4, name
        setattr(m.layers[1], name, at)
    m.weights.norm_final += 4
    with pytest.raises(_lib.RtaError) as e:
        m.step()
    assert e.value.status == 4


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("fmt", [orc.Q4_K, orc.Q6_K])
@pytest.mark.parametrize("rows,cols,batch", [(130, 512, 40), (300, 768, 130), (4096, 2304, 257)])
def test_not_finite_rows_stay_apart(fmt, packed, rows, cols, batch):
    """Rows that hold a NaN or an infinity come out not finite, all others bit for bit as
    without them (the same workgroup and the same matrix-core tiles hold both)."""
    rng = np.random.default_rng(rows + batch + fmt)
    _, wd, f = matrix(rng, fmt, rows, cols, packed)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    clean = ops.gemv(f, wd, rows, cols, dev(x)).cpu().numpy()
    bad = {0: np.nan, 17: np.inf, 31: -np.inf, batch - 1: np.nan}
    for b, v in bad.items():
        x[b, (37 * b + 5) % cols] = v
    y = ops.gemv(f, wd, rows, cols, dev(x)).cpu().numpy()
    good = [b for b in range(batch) if b not in bad]
    assert np.array_equal(y[good], clean[good])
    assert not np.isfinite(y[list(bad)]).any()


@pytest.mark.parametrize("fmt", [orc.Q4_K, orc.Q6_K])
@pytest.mark.parametrize("rows,cols", [(700, 4096), (20000, 2304)])
def test_rows_of_matrix_core_calls_do_not_depend_on_the_batch(fmt, rows, cols):
    """Bitwise within 5 to 16 rows and within 17 to 64 (20000x2304: 3 K slabs of the one class,
    5 of the other), on packed tiles and GGUF rows, which give each other's results too."""
    rng = np.random.default_rng(rows + cols + fmt)
    x = dev(rng.standard_normal((64, cols)).astype(np.float32))
    both = []
    w = synth.random_matrix(rng, fmt, rows, cols)
    for wd, f in ((dev(w.reshape(-1)), fmt), (ops.pack(fmt, dev(w), rows, cols), fmt | TILED)):
        y = {n: ops.gemv(f, wd, rows, cols, x[:n]).cpu().numpy() for n in (5, 11, 16, 17, 32, 64)}
        for a, b in ((5, 16), (11, 16), (17, 32), (17, 64)):
            assert np.array_equal(y[a], y[b][:a]), (f, a, b)
        both.append(y)
    for n in both[0]:
        assert np.array_equal(both[0][n], both[1][n]), n
