"""The dense GEMMs of a prefill (k_gemm_q8) against the per-token products (k_gemv): the logits
after a prompt prefilled in one batch and after the same prompt token by token, at column
counts that end a 64-column chunk early (by 16, 32 and 48), at rows that end a 64-row panel
early, at both group sizes and at token counts round the tiles' edges; and at rows and tokens
enough that each product form leaves the small products' tiles (32 tokens, two halves a block)
for the others, on 256 CUs: gate/up at 64 tokens a tile ("wide": 160 panels, 201 tokens), the rest
at 64 ("tall": 64 panels of attn_out, down, and q_a with kv_a, 449 tokens, 1040 or more
columns), attn_out and q_b at 32 tokens in one half ("long": 36 panels of fewer columns), and so
gate/up ("flat": 36 panels of 528 or 544 columns). The bar is the one used against
glm.c (max-abs 1e-2, rel-L2 1e-3, the same argmax): the two differ by rounding
alone, and an operand read from a wrong column by far more."""
import numpy as np
import pytest

import gmoe
from conftest import assert_close

pytestmark = pytest.mark.gpu


def config(gs, ql, nope, vh, dim, hidden=0, layers=2):
    return dict(dim=dim, hidden_dim=hidden or 3 * dim, n_layers=layers, n_heads=4, vocab_size=300, q_lora_rank=ql,
                kv_lora_rank=64, rope_dim=16, qk_nope_dim=nope, head_k_dim=nope + 16, v_head_dim=vh, group_size=gs,
                cache_cap=512, attn_layers=layers, has_l0_ffn=1, max_batch=512)


CONFIGS = {"gs16_cols48_16": config(16, 48, 16, 20, 272), "gs16_cols80_112": config(16, 112, 80, 28, 304),
           "gs32_cols32_96": config(32, 96, 32, 24, 288), "gs16_wide": config(16, 48, 16, 20, 1040, 10240, 1),
           "gs32_wide": config(32, 96, 32, 24, 1056, 10240, 1),
           "gs16_tall": config(16, 4000, 16, 260, 4096, 1040, 1), "gs32_tall": config(32, 4000, 32, 264, 4096, 1056, 1),
           "gs16_long": config(16, 112, 560, 20, 2304, 272, 1), "gs32_long": config(32, 96, 544, 24, 2304, 288, 1),
           "gs16_flat": config(16, 48, 16, 20, 528, 2304, 1), "gs32_flat": config(32, 96, 32, 24, 544, 2304, 1)}
TOKENS = {"wide": [201], "tall": [449], "long": [449], "flat": [449]}
CASES = [(name, n) for name in CONFIGS for n in TOKENS.get(name[5:], [8, 33])]


@pytest.mark.parametrize("name,n", CASES)
def test_prefill_matches_token_by_token(name, n):
    cfg = CONFIGS[name]
    g, attn = gmoe.synth_model_weights(cfg, 23)
    tokens = np.random.default_rng(9).integers(0, cfg["vocab_size"], n).astype(np.int32)
    model = gmoe.Model(cfg)
    try:
        model.upload(g)
        for l, a in enumerate(attn):
            model.upload_attn(l, a)
        print(f"[case] {name}: {n} tokens one at a time", flush=True)
        for pos, t in enumerate(tokens):
            want = model.forward_token(int(t), pos)
        want = want.copy()
        print(f"[case] {name}: {n} tokens in a batch", flush=True)
        got = model.prefill(tokens, 0)
        assert_close(got, want, f"{name} n={n}: logits")
        assert int(np.argmax(got)) == int(np.argmax(want)), f"{name} n={n}: argmax"
    finally:
        model.close()
