"""The batched K-quant products' workgroup shapes (32 or 64 tokens by 128 rows,
or K split over a workgroup's waves) at their edges: rows and tokens one off a
tile, one and several blocks per row, on both sides of the dispatch lines.
Every output equals the oracle's single-token product bit for bit (a few
rows and tokens of each output, the last ones among them)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_kernels import _synth_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,rows,cols,T", [
    (12, 14336, 256, 321),   # 64-token workgroups, one block, one token in the last tile
    (12, 16385, 512, 257),   # ... one row in the last tile
    (12, 6144, 768, 127),    # 32-token workgroups, ragged
    (12, 129, 1280, 33),     # K split, five blocks over four waves
    (14, 14336, 256, 191),   # Q6_K 64-token workgroups
    (14, 8193, 512, 289),
    (14, 127, 1280, 31),     # Q6_K, K split
    (14, 6143, 512, 129),    # Q6_K 32-token workgroups, ragged
    (14, 32897, 256, 31),    # ... many of them, one token tile
    (12, 65537, 256, 17),    # Q4_K: no 64-token workgroups up to 32 tokens
])
def test_workgroup_shapes(hip, t, rows, cols, T):
    w = _synth_weight(t, rows, cols, rows + T)
    rb = w.size // rows
    xs = np.random.default_rng(T).standard_normal((T, cols)).astype(np.float32)
    out = np.full((T, rows), 7.0, np.float32)
    assert hip.kquant_matvec_batch_into(t, w, rows, cols, xs, out)
    for tok in sorted({0, 1, 31, 32, 63, 64, T // 2, T - 2, T - 1} & set(range(T))):
        ref = O.matvec(t, w, xs[tok], rows, cols, threads=8)
        assert np.array_equal(out[tok].view(np.uint32), ref.view(np.uint32)), tok
    assert rb * rows == w.size


@pytest.mark.parametrize("rows,T", [(14336, 65), (6144, 129), (64, 33)])
def test_q6k_scale_extremes(hip, rows, T):
    """Products sc (q - 32) at both ends of their range, every weight 0 or 63
    and every scale -128, -1, 0, 1 or 127, on each workgroup shape."""
    cols, rng = 512, np.random.default_rng(rows)
    w = rng.choice(np.array([0, 255], np.uint8), size=(rows * cols // 256, 210))
    w[:, 192:208] = rng.choice(np.array([-128, -1, 0, 1, 127], np.int8), size=(len(w), 16)).view(np.uint8)
    w[:, 208:] = np.array([0.01], np.float16).view(np.uint8)
    w[0, :192], w[0, 192:208] = 0, 128  # a block of the largest products, all of one sign
    w = w.reshape(-1)
    xs = rng.standard_normal((T, cols)).astype(np.float32)
    xs[0, :256] = 3.0
    out = np.full((T, rows), 7.0, np.float32)
    assert hip.kquant_matvec_batch_into(14, w, rows, cols, xs, out)
    for tok in (0, 1, T - 1):
        ref = O.matvec(14, w, xs[tok], rows, cols, threads=8)
        assert np.array_equal(out[tok].view(np.uint32), ref.view(np.uint32)), tok
