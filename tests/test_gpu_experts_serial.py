"""The serial (reference-order) routed expert product at the edges of its
tiles and of the range its matrix-core form covers.

The kernel works in tiles of 128 rows and up to 64 pairs (two groups of 32, or
one group two blocks at a time), with the weights of 8 blocks in LDS; blocks
with an activation outside 0 or [2^-84, 2^80) or a scale byte outside
[87, 167] take an element-by-element path.  Every output is the oracle's
dot_mxfp4_f32_scalar sum, bit for bit (NaN where it is NaN)."""
import numpy as np
import pytest

from oracle import oracle as O
from rustyllm_amd import synth

pytestmark = pytest.mark.gpu
MX = 39


def _run(hip, w, stride, n_exp, rows, cols, x, per_pair, k, sel):
    import torch
    dev = torch.device("cuda:0")
    tw, tx, ts = (torch.from_numpy(a).to(dev) for a in (w.reshape(-1), x.reshape(-1), sel))
    ty = torch.full((sel.size * rows,), -7.0, dtype=torch.float32, device=dev)
    torch.cuda.synchronize()
    assert hip.mxfp4_experts_dev(tw.data_ptr(), stride, rows * stride, n_exp, rows, cols, tx.data_ptr(), cols,
                                 per_pair, k, ts.data_ptr(), sel.size, ty.data_ptr(), rows, False)
    return ty.cpu().numpy().reshape(sel.size, rows)


def _check(got, w, rb, rows, cols, x, per_pair, k, sel, n_exp):
    for p, e in enumerate(sel):
        if not 0 <= e < n_exp:
            assert np.all(got[p] == -7.0)
            continue
        ref = O.matvec(MX, np.ascontiguousarray(w[e, :, :rb]), x[p if per_pair else p // k], rows, cols)
        nan = np.isnan(ref)
        assert np.array_equal(np.isnan(got[p]), nan), p
        assert np.array_equal(got[p][~nan].view(np.uint32), ref[~nan].view(np.uint32)), p


@pytest.mark.parametrize("rows,cols,n_exp,k,counts", [
    (1, 32, 1, 1, [1]),
    (63, 64, 3, 1, [16, 0, 17]),
    (65, 96, 3, 1, [15, 33, 1]),
    (64, 512, 4, 1, [48, 49, 64, 65]),
    (130, 544, 2, 1, [63, 130]),
    (70, 1056, 64, 2, None),
])
@pytest.mark.parametrize("per_pair", [False, True])
def test_tile_edges(hip, rows, cols, n_exp, k, counts, per_pair):
    rng = np.random.default_rng(rows + cols)
    rb = synth.row_bytes(MX, cols)
    stride = (rb + 15) // 16 * 16
    w = np.zeros((n_exp, rows, stride), np.uint8)
    w[:, :, :rb] = synth.normal_quantized(MX, 3, n_exp * rows, cols, 0.05).reshape(n_exp, rows, rb)
    if counts is None:
        sel = np.stack([rng.choice(n_exp, size=k, replace=False) for _ in range(97)]).astype(np.int32).reshape(-1)
        sel[5], sel[40] = -1, 64  # neither names an expert
    else:
        sel = rng.permutation(np.repeat(np.arange(n_exp), counts)).astype(np.int32)
    x = synth.normal_f32(9, sel.size if per_pair else sel.size // k, cols)
    got = _run(hip, w, stride, n_exp, rows, cols, x, per_pair, k, sel)
    _check(got, w, rb, rows, cols, x, per_pair, k, sel, n_exp)


@pytest.mark.parametrize("kind", ["scales", "tiny", "huge", "zeros", "nonfinite", "mixed"])
def test_values_outside_the_matrix_core_range(hip, kind):
    rows, cols, n_exp = 66, 192, 2
    rng = np.random.default_rng(len(kind))
    rb = synth.row_bytes(MX, cols)
    stride = (rb + 15) // 16 * 16
    w = np.zeros((n_exp, rows, stride), np.uint8)
    w[:, :, :rb] = rng.integers(0, 256, (n_exp, rows, rb))  # every nibble, -0 among them
    sc = w[:, :, 16:rb:17]
    sc[:] = rng.integers(110, 140, sc.shape)
    sel = rng.integers(0, n_exp, 40).astype(np.int32)
    x = synth.normal_f32(17, sel.size, cols)
    if kind in ("scales", "mixed"):
        sc[:, ::5] = rng.choice([0, 1, 23, 60, 86, 87, 167, 168, 230, 253, 254, 255], sc[:, ::5].shape)
    if kind in ("tiny", "mixed"):
        x[::3] *= np.exp2(rng.integers(-149, -30, x[::3].shape)).astype(np.float32)
    if kind == "huge":
        x[::3] *= np.exp2(rng.integers(30, 127, x[::3].shape)).astype(np.float32)
    if kind == "zeros":
        x[::2] = 0.0
        x[1::4, ::2] = -0.0
    if kind in ("nonfinite", "mixed"):
        x[2, 40], x[5, 3], x[9, 100] = np.inf, -np.inf, np.nan
    got = _run(hip, w, stride, n_exp, rows, cols, x, True, 1, sel)
    _check(got, w, rb, rows, cols, x, True, 1, sel, n_exp)


def _weights(n_exp, rows, cols, rng, scale):
    """Random nibbles (every weight, -0 among them), one scale byte."""
    rb = synth.row_bytes(MX, cols)
    stride = (rb + 15) // 16 * 16
    w = np.zeros((n_exp, rows, stride), np.uint8)
    w[:, :, :rb] = rng.integers(0, 256, (n_exp, rows, rb))
    w[:, :, 16:rb:17] = scale
    return w, rb, stride


@pytest.mark.parametrize("rows,cols,n_pairs", [(127, 256, 3), (128, 288, 33), (129, 544, 40)])
@pytest.mark.parametrize("xe,scale", [
    (-84, 87), (-84, 167), (79, 87), (79, 167),  # every block on the matrix cores, at the edges of their range
    (-86, 87), (-84, 85), (-100, 127),           # every block outside: products below the normal range would differ
    (86, 167), (79, 174), (100, 150),            # ... and sums past the largest number
])
def test_edges_of_the_matrix_core_range(hip, rows, cols, n_pairs, xe, scale):
    rng = np.random.default_rng(rows + xe + scale)
    w, rb, stride = _weights(2, rows, cols, rng, scale)
    sel = rng.integers(0, 2, n_pairs).astype(np.int32)
    # full mantissas in [2^xe, 2^(xe + 1)), either sign
    mant = rng.integers(0, 1 << 23, (n_pairs, cols), dtype=np.uint32)
    x = (mant | np.uint32((xe + 127) << 23) | (rng.integers(0, 2, mant.shape, dtype=np.uint32) << 31)).view(np.float32)
    x[:, :32] = np.where(rng.random((n_pairs, 32)) < 0.2, np.float32(0), x[:, :32])
    _check(_run(hip, w, stride, 2, rows, cols, x, True, 1, sel), w, rb, rows, cols, x, True, 1, sel, 2)


@pytest.mark.parametrize("what", ["x below", "x above", "scale below", "scale above", "last block"])
def test_one_value_outside_the_matrix_core_range(hip, what):
    """One block of one pair or row on the element path, its neighbours not."""
    rows, cols, n_pairs = 130, 32 * 17, 37
    rng = np.random.default_rng(len(what))
    w, rb, stride = _weights(1, rows, cols, rng, 87 if "below" in what else 160)
    x = (synth.normal_f32(5, n_pairs, cols) * np.float32(2.0 ** (-82 if "below" in what else 70))).reshape(n_pairs, cols)
    x[np.abs(x) < 2.0 ** -84] = 0.0
    if what == "x below":
        x[3, 32 * 9 + 5] = np.float32(1.9 * 2.0 ** -90)
    elif what == "x above":
        x[36, 32 * 8] = np.float32(1.3 * 2.0 ** 88)
    elif what == "last block":
        x[0, cols - 1] = np.inf
    else:
        w[0, 129, 17 * 7 + 16] = 80 if what == "scale below" else 180
    sel = np.zeros(n_pairs, np.int32)
    _check(_run(hip, w, stride, 1, rows, cols, x, True, 1, sel), w, rb, rows, cols, x, True, 1, sel, 1)


@pytest.mark.parametrize("n_pairs,kind", [(800, "spread"), (1024, "spread"), (1024, "one expert"), (1000, "half unrouted"),
                                          (257, "spread"), (65, "spread"), (64, "one expert"), (1, "one expert")])
def test_pairs_found_in_the_workgroups(hip, n_pairs, kind):
    """Up to 1024 pairs the product is one launch (a list launch before it had
    made calls of few pairs slower than without)."""
    rows, n_exp, cols = 33, 64, 32
    rng = np.random.default_rng(n_pairs)
    w, rb, stride = _weights(n_exp, rows, cols, rng, 120)
    sel = rng.integers(0, n_exp, n_pairs).astype(np.int32)
    if kind == "one expert":
        sel[:] = n_exp - 1
    if kind == "half unrouted":
        sel[::2] = rng.choice([-1, -2, n_exp, 1 << 30], sel[::2].shape)
    x = synth.normal_f32(3, n_pairs, cols).reshape(n_pairs, cols)
    hip.profile_enable(True)
    try:
        got = _run(hip, w, stride, n_exp, rows, cols, x, True, 1, sel)
        launches = {name: n for name, (_, n) in hip.profile_results().items() if n}
    finally:
        hip.profile_enable(False)
    assert launches == {"mxfp4_experts": 1}
    _check(got, w, rb, rows, cols, x, True, 1, sel, n_exp)


@pytest.mark.parametrize("n_pairs", [2, 34])
def test_every_element_of_a_block_is_checked(hip, n_pairs):
    """One infinite activation at each place of a block: rows whose weight there
    is not 0 get an infinite sum, not NaN."""
    rows, cols = 40, 96
    rng = np.random.default_rng(n_pairs)
    w, rb, stride = _weights(1, rows, cols, rng, 125)
    sel = np.zeros(n_pairs, np.int32)
    base = synth.normal_f32(2, n_pairs, cols).reshape(n_pairs, cols)
    for e in range(32):
        x = base.copy()
        x[n_pairs - 1, 32 * (e % 3) + e] = np.inf
        _check(_run(hip, w, stride, 1, rows, cols, x, True, 1, sel), w, rb, rows, cols, x, True, 1, sel, 1)
