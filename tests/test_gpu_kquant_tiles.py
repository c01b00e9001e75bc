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
