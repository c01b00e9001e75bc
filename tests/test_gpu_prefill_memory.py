"""The batched prefill's buffers: sized by the prompt at hand, taken at 512
tokens per chunk where 1024 do not fit, given back where neither does; and a
gpt-oss prompt of more than one chunk in one call, bit-exact over the chunk
boundary."""
import numpy as np
import pytest

from oracle import oracle as O
from rustyllm_amd import synth

pytestmark = pytest.mark.gpu
CFG = dict(synth.GPTOSS_CONFIGS["tiny-gptoss-w128"], n_layers=2, vocab=300)


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@pytest.fixture
def limit(hip):
    yield hip.debug_alloc_limit
    assert hip.debug_alloc_limit(0)


def test_chunk_of_512_where_1024_does_not_fit(hip, limit):
    prev = hip.attention_mode("exact")
    try:
        model = synth.make_gptoss(CFG, seed=5)
        n = 700
        toks = synth.token_ids(3, n, CFG["vocab"])
        res = hip.ResidentGptOss(model, 2048)
        _, want = res.generate(toks, 0)  # one chunk
        kv = [res.kv_read(l, w, 0, res.slots) for l in range(2) for w in (0, 1)]
        # the largest buffer, the attention scratch, takes several MB more at 1024
        # tokens than at 512: find a limit between them
        res = hip.ResidentGptOss(model, 2048)
        refused = 1 << 10
        accepted = 1 << 34
        while accepted - refused > refused // 8:
            mid = (accepted + refused) // 2
            assert limit(mid)
            res = hip.ResidentGptOss(model, 2048)
            if res.prefill(toks[:8], 0):
                accepted = mid
            else:
                refused = mid
        assert limit(accepted)  # 512 tokens' largest buffer fits, 1024 tokens' does not
        for _ in range(2):
            _, got = res.generate(toks, 0)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        for i, ref in enumerate(kv):
            assert np.array_equal(res.kv_read(i // 2, i % 2, 0, res.slots).view(np.uint32), ref.view(np.uint32))
    finally:
        hip.attention_mode(prev)


def test_refused_prompts_keep_no_memory(hip, limit):
    model = synth.make_gptoss(CFG, seed=6)
    res = hip.ResidentGptOss(model, 2048)
    toks = synth.token_ids(4, 700, CFG["vocab"])
    assert limit(1 << 20)  # the first buffers fit, the scratch does not
    assert not res.prefill(toks, 0)
    before = _free()
    for _ in range(8):
        assert not res.prefill(toks, 0)
    assert _free() >= before
    assert limit(0)
    assert res.prefill(toks, 0)


def test_short_prompts_take_512_token_buffers(hip):
    model = synth.make_gptoss(CFG, seed=7)
    res = hip.ResidentGptOss(model, 4096)
    start = _free()
    assert res.prefill(synth.token_ids(1, 40, CFG["vocab"]), 0)
    short = start - _free()
    assert res.prefill(synth.token_ids(1, 900, CFG["vocab"]), 0)
    long = start - _free()
    assert 0 < short < 0.7 * long, (short, long)


def test_prompt_across_a_chunk_boundary(hip):
    """1100 tokens in one call: chunks of 1024 and 76 (the first with the expert
    lists' launch, the second with the pairs found in the workgroups)."""
    prev = hip.attention_mode("exact")
    try:
        n = 1100
        model = synth.make_gptoss(CFG, seed=8)
        toks = synth.token_ids(9, n, CFG["vocab"])
        res, orc = hip.ResidentGptOss(model, 1200), O.OracleGptOss(model, 1200)
        _, got = res.generate(toks, 0)
        for pos in range(n):
            ref = orc.forward(int(toks[pos]), pos)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
        for layer in range(CFG["n_layers"]):
            for which, want in ((0, orc.kc[layer]), (1, orc.vc[layer])):
                assert np.array_equal(res.kv_read(layer, which, 0, orc.storage).view(np.uint32), want.view(np.uint32))
    finally:
        hip.attention_mode(prev)
