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
    (864, 8, 301),  # f32 q/k/v over 27 blocks (an odd count), wo int8 over 512 columns, 13.5 row tiles
    (608, 4, 320),  # 19 blocks, 9.5 row tiles, whole token tiles
    (768, 4, 257),  # int8 q/k/v in one launch, one token in the last tile
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
