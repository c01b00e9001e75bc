"""The per-op exports' pinned staging at its size limit: activations and
outputs of up to 2^20 floats cross through pinned memory, larger ones by the
runtime's copies; every output equals the oracle's bit for bit on both sides,
for one to three outputs and optional ones left out."""
import numpy as np
import pytest

from oracle import oracle as O
from rustyllm_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,rows,cols", [(8, 1048575, 32), (8, 1048576, 32), (8, 1048577, 32), (39, 40, 14336),
                                         (39, 33000, 64), (12, 3, 14336), (14, 32800, 256), (8, 1, 256)])
def test_matvec_sizes(hip, t, rows, cols):
    w = synth.normal_quantized(t, rows, rows, cols, 0.05)
    for seed in (1, 2):  # a second call finds the buffers used
        x = synth.normal_f32(seed, 1, cols)[0]
        out = np.full(rows, 9.0, np.float32)
        assert hip.matvec_into(t, w, x, rows, cols, out)
        ref = O.matvec(t, w, x, rows, cols, threads=8)
        assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("rows", [(5, 700, 64), (600000, 400000, 48576), (600000, 400000, 48577)])
def test_three_outputs(hip, rows):
    ws = [(synth.normal_quantized(t, r, r, 256, 0.05), t, r) for t, r in zip((12, 12, 14), rows)]
    x = synth.normal_f32(3, 1, 256)[0]
    outs = [np.full(r, 9.0, np.float32) for r in rows]
    assert hip.quant_matvec3_into(*ws, x, 256, outs)
    for (w, t, r), o in zip(ws, outs):
        assert np.array_equal(o.view(np.uint32), O.matvec(t, w, x, r, 256, threads=8).view(np.uint32))


@pytest.mark.parametrize("rows,cols,T", [(1024, 256, 1024), (1025, 256, 1023), (1025, 256, 1024), (16, 4096, 257)])
def test_batch(hip, rows, cols, T):
    w = synth.normal_quantized(12, T, rows, cols, 0.05)
    x, out = synth.normal_f32(5, T, cols), np.zeros((T, rows), np.float32)
    assert hip.kquant_matvec_batch_into(12, w, rows, cols, x, out)
    for t in (0, 1, T // 2, T - 1):
        assert np.array_equal(out[t].view(np.uint32), O.matvec(12, w, x[t], rows, cols, threads=8).view(np.uint32)), t


def test_weight_change_at_one_address_is_seen(hip):
    """The sampled fingerprint covers these bytes: new weights at an old
    address are uploaded again."""
    w = synth.normal_quantized(8, 1, 16, 64, 0.05)
    x, out = synth.normal_f32(4, 1, 64)[0], np.zeros(16, np.float32)
    for byte in (0, 7, 8, 15, w.size - 1):
        w[byte] ^= 0x80 if byte != w.size - 1 else 1
        assert hip.matvec_into(8, w, x, 16, 64, out)
        assert np.array_equal(out, O.matvec(8, w, x, 16, 64), equal_nan=True), byte


def test_without_pinned_memory(hip):
    """Where the pinned buffers cannot be had, the same calls go by the
    runtime's copies, and with them again afterwards."""
    cols, rows = 512, (300, 40, 7)
    ws = [(synth.normal_quantized(t, r, r, cols, 0.05), t, r) for t, r in zip((12, 12, 14), rows)]
    xs = synth.normal_f32(6, 40, cols)
    refs = [O.matvec(t, w, xs[0], r, cols) for w, t, r in ws]
    dim, hidden = 256, 512
    f = [synth.normal_quantized(t, 9 + i, r, c, 0.05) for i, (t, r, c) in
         enumerate(((12, hidden, dim), (12, hidden, dim), (14, dim, hidden)))]
    blocks = []
    try:
        for n in (1024, 0):
            assert hip.debug_alloc_limit(n)
            outs = [np.zeros(r, np.float32) for r in rows]
            assert hip.quant_matvec3_into(*ws, xs[0], cols, outs)
            batch = np.zeros((40, rows[0]), np.float32)
            assert hip.kquant_matvec_batch_into(12, ws[0][0], rows[0], cols, xs, batch)
            block = np.zeros(dim, np.float32)
            assert hip.q4k_q4k_q6k_ffn_into(*f, xs[1, :dim], dim, hidden, dim, hidden, block)
            blocks.append(block)
            for got, ref in zip(outs + [batch[0]], refs + [refs[0]]):
                assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
        assert np.array_equal(blocks[0].view(np.uint32), blocks[1].view(np.uint32)) and np.any(blocks[0])
    finally:
        hip.debug_alloc_limit(0)
