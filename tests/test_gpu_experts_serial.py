"""The serial (reference-order) routed expert product at the edges of its
tiles and of the range its matrix-core form covers.

The kernel works in tiles of 64 rows and up to 64 pairs (in groups of 16),
chunks of 2 activation and 16 weight blocks; blocks whose activations are
outside [2^-60, 2^60) or whose scale bytes are outside [87, 167] take an
element-by-element path.  Every output is the oracle's dot_mxfp4_f32_scalar
sum, bit for bit (NaN where it is NaN)."""
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
