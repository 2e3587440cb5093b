"""The dense GEMMs of a prefill (k_gemm_q8) against the per-token products (k_gemv): the logits
after a prompt prefilled in one batch and after the same prompt token by token, at column
counts that end a 64-column chunk early (by 16, 32 and 48), at rows that end a 64-row panel
early, at both group sizes and at token counts round the tiles' edges; and with a layer 0 wide
enough that its gate/up product runs 64 tokens a tile (160 panels, 201 tokens). The bar is the one
used against glm.c (max-abs 1e-2, rel-L2 1e-3, the same argmax): the two differ by rounding
alone, and an operand read from a wrong column by far more."""
import numpy as np
import pytest

import gmoe
from conftest import assert_close

pytestmark = pytest.mark.gpu


def config(gs, ql, nope, vh, dim, hidden=0, layers=2):
    return dict(dim=dim, hidden_dim=hidden or 3 * dim, n_layers=layers, n_heads=4, vocab_size=300, q_lora_rank=ql,
                kv_lora_rank=64, rope_dim=16, qk_nope_dim=nope, head_k_dim=nope + 16, v_head_dim=vh, group_size=gs,
                cache_cap=256, attn_layers=layers, has_l0_ffn=1, max_batch=256)


CONFIGS = {"gs16_cols48_16": config(16, 48, 16, 20, 272), "gs16_cols80_112": config(16, 112, 80, 28, 304),
           "gs32_cols32_96": config(32, 96, 32, 24, 288), "gs16_wide": config(16, 48, 16, 20, 1040, 10240, 1),
           "gs32_wide": config(32, 96, 32, 24, 1056, 10240, 1)}
CASES = [(name, n) for name in CONFIGS for n in ([201] if name.endswith("wide") else [8, 33])]


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
