"""Prompts of up to 64 tokens, which go through the layers once, the last token's head included, against
the same tokens decoded one by one: logits, cache rows, the greedy pick fed to the next step. The two
differ by what a decode step stores in 16 bits between its kernels (attention and SwiGLU rows: 2^-11
relative each) and by cache rows that round the other way; 3e-3 of max |logit| is the bound the chunked
prefill's 16-bit operands are held to. 65 and 66 tokens, just past the short prompts, take that prefill:
their bf16 GEMM operands round at 2^-9, eight times fp16's 2^-12, and are held to its bf16 bound of 1.5e-2."""
from __future__ import annotations

import numpy as np
import pytest

import l0llm_amd as l0
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu

# q heads, kv heads, head dim, hidden, intermediate: the group sizes and head widths of the attention
# kernels, widths that are not multiples of the 64-value steps or of the 16-column blocks
SHAPES = [(4, 2, 64, 256, 512, True), (7, 1, 128, 208, 336, False), (6, 6, 16, 96, 176, True)]


@pytest.mark.parametrize("precision,tol", [(l0.PRECISION_INT8, 3e-3), (l0.PRECISION_FLOAT16, 3e-3), (l0.PRECISION_BFLOAT16, 3e-3)])
@pytest.mark.parametrize("nh,nkv,hd,hidden,inter,bias", SHAPES)
def test_short_prompt_matches_sequential_decode(device, precision, tol, nh, nkv, hd, hidden, inter, bias):
    cfg = l0.HfConfig(hidden_size=hidden, intermediate_size=inter, num_layers=3, num_attention_heads=nh,
                      num_key_value_heads=nkv, head_dim=hd, vocab_size=515, max_position_embeddings=4096,
                      rms_norm_eps=1e-5, rope_theta=500000.0, attention_bias=bias)
    prompt = np.random.default_rng(hidden + precision).integers(0, cfg.vocab_size, 66).tolist()
    with l0.LlmModel(device, cfg, precision=precision, cache_dtype=l0.F16, max_seq_len=80) as m:
        m.init_random(77, 0.05)
        step = [m.compute_logits(t, i) for i, t in enumerate(prompt)]

        def rows(which, li, count):
            n = count * nkv * hd
            return l0.Buffer(device, n * 2, ptr=m.kv_cache(li)[which], owned=False).read(np.float16, n).astype(np.float32)

        want = [[rows(w, li, 66) for w in (0, 1)] for li in range(3)]
        for count in (1, 2, 15, 16, 17, 32, 33, 48, 49, 63, 64, 65, 66):
            got = m.prefill(prompt[:count])
            assert m.position == count
            ref = step[count - 1]
            bound = 1.5e-2 if count > 64 and precision == l0.PRECISION_BFLOAT16 else tol
            assert np.max(np.abs(got - ref)) <= bound * np.max(np.abs(ref)), count
            if count <= 64:
                for li in range(3):
                    for w in (0, 1):
                        have, exp = rows(w, li, count), want[li][w][: count * nkv * hd]
                        assert np.max(np.abs(have - exp)) <= 4e-2 * max(1.0, np.max(np.abs(exp))), (count, li, w)
            # the device's own step state: the pick of the prompt's last logits feeds the next step
            out = m.generate_greedy(prompt[:count], 3)
            assert out[0] == int(np.argmax(got))
            m.prefill(prompt[:count])
            nxt = m.decode(int(out[0]))
            if orc.top2_margin(nxt) > 1e-5 * np.max(np.abs(nxt)):
                assert out[1] == int(np.argmax(nxt))


def test_short_prompt_rejects_bad_ids(device):
    cfg = l0.HfConfig(hidden_size=64, intermediate_size=64, num_layers=1, num_attention_heads=2, num_key_value_heads=1, head_dim=32,
                      vocab_size=33, max_position_embeddings=64, rms_norm_eps=1e-5, rope_theta=1e4, attention_bias=False)
    with l0.LlmModel(device, cfg, precision=l0.PRECISION_INT8, cache_dtype=l0.F16, max_seq_len=16) as m:
        m.init_random(3, 0.05)
        for ids in ([33, 1], [1, 33], [1, -1, 2]):
            with pytest.raises(ValueError):
                m.prefill(ids)
        assert np.all(np.isfinite(m.prefill([1, 2, 3])))
