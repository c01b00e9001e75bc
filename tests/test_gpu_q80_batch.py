"""The batched Q8_0 products on the matrix cores (gemm_q8_0_f32_kernel,
gemm_q8_0_q8k_kernel) at the edges of their 64-row, 64-token, two-block tiles,
through the gpt-oss prefill that runs them: K and V of every layer and the next
logits equal the oracle's sequential forward bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from rustyllm_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,heads,n", [
    (864, 8, 301),  # f32 q/k/v over 27 blocks (an odd count)
    (608, 4, 320),  # 19 blocks, whole token tiles
    (768, 4, 257),  # int8 q/k/v below the matrix cores' line
])
def test_prefill_equals_sequential(hip, dim, heads, n):
    prev = hip.attention_mode("exact")
    try:
        cfg = dict(synth.GPTOSS_CONFIGS["tiny-gptoss-w128"], n_layers=2, dim=dim, n_heads=heads, n_kv_heads=2,
                   vocab=300, n_experts=4)
        model = synth.make_gptoss(cfg, seed=dim)
        res, orc = hip.ResidentGptOss(model, 400), O.OracleGptOss(model, 400)
        toks = synth.token_ids(n, n + 1, cfg["vocab"])
        assert res.prefill(toks[:n], 0)
        for pos in range(n):
            orc.forward(int(toks[pos]), pos)
        for layer in range(cfg["n_layers"]):
            for which, ref in ((0, orc.kc[layer]), (1, orc.vc[layer])):
                assert np.array_equal(res.kv_read(layer, which, 0, orc.storage).view(np.uint32), ref.view(np.uint32))
        emb, et = model["token_embd"]
        x = O.dequant_row(et, emb[int(toks[n]) * O.row_bytes(et, dim):], dim)
        g, r = res.decode(x, n, 0, True), orc.forward(int(toks[n]), n)
        assert np.array_equal(g.view(np.uint32), r.view(np.uint32))
    finally:
        hip.attention_mode(prev)


@pytest.mark.parametrize("dim,heads,kv,n,gemm", [
    (1536, 16, 2, 257, ("qkv", "o")),  # int8 q/k/v in one launch and wo, one token in the last tile
    (1536, 16, 2, 215, ("qkv", "o")),  # ... a ragged last token tile of 23, just above the line (4288)
    (1440, 16, 2, 195, ("qkv", "o")),  # f32 q/k/v; wo of 22.5 row tiles just above its line (4459)
    (1440, 16, 2, 193, ("qkv",)),      # ... and just below it
    (512, 8, 2, 385, ()),              # 12 tiles of 512 columns: below the line (4630)
    (608, 8, 2, 54, ("qkv",)),         # f32 just above its line (640)
    (608, 8, 2, 53, ()),               # ... and just below it
])
def test_both_sides_of_the_lines(hip, dim, heads, kv, n, gemm):
    """Which products the matrix-core kernels take, and both kernels' values."""
    prev = hip.attention_mode("exact")
    try:
        cfg = dict(synth.GPTOSS_CONFIGS["tiny-gptoss-w128"], n_layers=1, dim=dim, n_heads=heads, n_kv_heads=kv,
                   vocab=300, n_experts=4)
        model = synth.make_gptoss(cfg, seed=dim + n)
        res, orc = hip.ResidentGptOss(model, 450), O.OracleGptOss(model, 450)
        toks = synth.token_ids(n, n, cfg["vocab"])
        assert res.prefill(toks, 0)  # (allocates)
        hip.profile_enable(True)
        try:
            _, got = res.generate(toks, 0)  # n - 1 tokens in the batch, the last one decoded
            assert res.prefill(toks, 0)
            ran = {name for name, (_, c) in hip.profile_results().items() if c}
        finally:
            hip.profile_enable(False)
        for part in ("qkv", "o"):
            assert (f"pf_q80_{part}" in ran) == (part in gemm), sorted(ran)
        for pos in range(n):
            ref = orc.forward(int(toks[pos]), pos)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
        for which, want in ((0, orc.kc[0]), (1, orc.vc[0])):
            assert np.array_equal(res.kv_read(0, which, 0, orc.storage).view(np.uint32), want.view(np.uint32))
    finally:
        hip.attention_mode(prev)
