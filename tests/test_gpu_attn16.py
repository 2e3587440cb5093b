"""The batch attention on fp16 matrix cores with split operands (k_attn_tile16) against the
fp32 MFMA kernel it replaces (GMOE_ATTN_TILE_FP32=1), on the same model and prompt.

Both take the same tiles, chunks and partial-result slots; k_attn_tile16 forms each product
as hi.hi + hi.lo + lo.hi of fp16 halves (~22 bits of each operand) with power-of-two
exponents per query row and per cached row, so its results differ from fp32 products in
the last few bits only. The logits after a batched prefill are held to a tight bar against
the fp32 kernel's (max-abs 2e-4, rel-L2 2e-5: ~100x below the bar against glm.c, which
test_gpu_prefill.py and test_gpu_config5.py apply to the default kernel), with the same
argmax. Shapes: a small one (kv 64 + rope 16 = 80 columns: the last 32-column step is
padded with zeros) and glm.c's attention ranks (kv 512 + rope 64), 4 and 20 heads. Prompts:
300 tokens in one batch (five 64-token query tiles, several position chunks), then 200 more
at position 300 over that cache (chunks that span both batches, causal masks inside); then
a decode token with GMOE_MODEL_KEEP_CACHE at position 250 (its fp32 entries written, then
restored; the split form, which decode steps do not write, must be left as the prefill
wrote it), three tokens decoded one at a time (fp32 entries only: the next prefill converts
them with k_spl_fill before its attention) and 8 more tokens in a batch over all of them."""
import os

import numpy as np
import pytest

import gmoe
from conftest import assert_close

pytestmark = pytest.mark.gpu

KEEP_CACHE = 1  # GMOE_MODEL_KEEP_CACHE, include/gmoe_model.h


def small():
    return dict(dim=256, hidden_dim=512, n_layers=2, n_heads=4, vocab_size=300, q_lora_rank=64, kv_lora_rank=64,
                rope_dim=16, qk_nope_dim=32, head_k_dim=48, v_head_dim=32, group_size=32, cache_cap=512,
                attn_layers=2, has_l0_ffn=1, max_batch=300)


def glm_ranks(heads):
    return dict(dim=2048, hidden_dim=1024, n_layers=2, n_heads=heads, vocab_size=300, q_lora_rank=256,
                kv_lora_rank=512, rope_dim=64, qk_nope_dim=192, head_k_dim=256, v_head_dim=256, group_size=32,
                cache_cap=512, attn_layers=2, has_l0_ffn=1, max_batch=300)


CASES = {"small": small, "h4": lambda: glm_ranks(4), "h20": lambda: glm_ranks(20)}


def run(model, tokens, pos0, fp32):
    old = os.environ.get("GMOE_ATTN_TILE_FP32")
    try:
        if fp32:
            os.environ["GMOE_ATTN_TILE_FP32"] = "1"
        else:
            os.environ.pop("GMOE_ATTN_TILE_FP32", None)
        return model.prefill(tokens, pos0).copy()
    finally:
        if old is None:
            os.environ.pop("GMOE_ATTN_TILE_FP32", None)
        else:
            os.environ["GMOE_ATTN_TILE_FP32"] = old


@pytest.mark.parametrize("name", list(CASES))
def test_split_fp16_attention_matches_fp32(name):
    cfg = CASES[name]()
    g, attn = gmoe.synth_model_weights(cfg, 17)
    model = gmoe.Model(cfg)
    try:
        model.upload(g)
        for l, a in enumerate(attn):
            model.upload_attn(l, a)
        rng = np.random.default_rng(5)
        first = rng.integers(0, cfg["vocab_size"], 300).astype(np.int32)
        second = rng.integers(0, cfg["vocab_size"], 200).astype(np.int32)
        def check(what, toks, pos0):
            print(f"[case] {name}: {what}", flush=True)
            want = run(model, toks, pos0, fp32=True)
            got = run(model, toks, pos0, fp32=False)
            assert np.isfinite(got).all()
            assert_close(got, want, f"{name} {what}: logits", max_abs=2e-4, rel_l2=2e-5)
            assert int(np.argmax(got)) == int(np.argmax(want)), f"{name} {what}: argmax"

        check("300 tokens at 0", first, 0)
        check("200 tokens at 300", second, 300)
        # a kept decode token overwrites position 250's fp32 entries and restores them; tokens
        # decoded one at a time write fp32 entries only; a batch then reads both in split form
        model.forward_token(7, 250, flags=KEEP_CACHE)
        for pos in range(500, 503):
            model.forward_token(int(rng.integers(0, cfg["vocab_size"])), pos)
        check("8 tokens at 503 after kept and decoded tokens", rng.integers(0, cfg["vocab_size"], 8).astype(np.int32), 503)
    finally:
        model.close()


# The running scale and the reference score of a chunk (a16_scale; A16_SLACK): 1024 tokens of 20
# heads, whose chunks are eleven 32-position tiles. Token 0's embedding row is zero (layer 0's
# entry of it is exactly zero), those of tokens 1..3 are scaled by 2^-36, 2^-56 and 2^-76 (their
# entries, which come from x / sqrt(mean x^2 + 1e-5), lie about 2^-21, 2^-41 and 2^-61 of an ordinary
# token's); "scores" multiplies the queries by 4, which leaves the scores a standard deviation of
# 4 and 14, so that a chunk's maximum passes the slack several times.
def tall(**over):
    cfg = dict(small(), n_heads=20, cache_cap=1152, max_batch=1024)
    cfg.update(over)
    return cfg


TALL = {"kv64": tall, "kv512": lambda: tall(dim=512, kv_lora_rank=512, rope_dim=64, qk_nope_dim=192, head_k_dim=256, v_head_dim=64)}


def runs(rng, *spec):
    """Tokens run by run: (count, id), or ordinary ones where the id is None."""
    return np.concatenate([rng.integers(10, 300, n) if t is None else np.full(n, t) for n, t in spec]).astype(np.int32)


PROMPTS = {
    "zeros": lambda rng: runs(rng, (100, None), (200, 0), (200, None), (300, 0), (224, None)),
    "zeros first": lambda rng: runs(rng, (200, 0), (200, None), (624, 0)),
    "falling": lambda rng: runs(rng, (50, None), (60, 1), (90, 2), (100, 3), (52, None), (32, 1), (64, 3), (128, 2), (448, None)),
    "small then ordinary": lambda rng: runs(rng, (352, 3), (352, 2), (300, 1), (20, None)),
    "zeros after small": lambda rng: runs(rng, (40, None), (64, 3), (200, 0), (100, 2), (400, 0), (220, None)),
    "scores": lambda rng: runs(rng, (1024, None)),
}


@pytest.mark.parametrize("name", list(TALL))
@pytest.mark.parametrize("what", list(PROMPTS))
def test_running_scale_matches_fp32(name, what):
    cfg = TALL[name]()
    g, attn = gmoe.synth_model_weights(cfg, 19)
    g["tok_q"][0] = 0
    for t in (1, 2, 3):
        g["tok_s"][t] *= 2.0 ** -(16 + 20 * t)
    if what == "scores":
        for a in attn:
            a["q_b_s"] *= 4.0
    model = gmoe.Model(cfg)
    try:
        model.upload(g)
        for l, a in enumerate(attn):
            model.upload_attn(l, a)
        toks = PROMPTS[what](np.random.default_rng(7))
        assert toks.size == 1024
        print(f"[case] {name}: {what}", flush=True)
        want = run(model, toks, 0, fp32=True)
        got = run(model, toks, 0, fp32=False)
        assert np.isfinite(want).all()
        assert_close(got, want, f"{name} {what}: logits", max_abs=2e-4, rel_l2=2e-5)
        assert int(np.argmax(got)) == int(np.argmax(want)), f"{name} {what}: argmax"
    finally:
        model.close()


@pytest.mark.parametrize("name", list(TALL))
def test_entries_past_the_batch_are_not_read(name):
    """Token 4's embedding is NaN, and so are its cache entries and those that attend it. A
    prompt of 100 tokens leaves them at positions 40 and up; another of 35 over the same cache
    shares a 32-position tile with them and attends none."""
    cfg = TALL[name]()
    g, attn = gmoe.synth_model_weights(cfg, 19)
    g["tok_s"][4] = np.nan
    model = gmoe.Model(cfg)
    try:
        model.upload(g)
        for l, a in enumerate(attn):
            model.upload_attn(l, a)
        rng = np.random.default_rng(3)
        print(f"[case] {name}: stale NaN entries", flush=True)
        assert np.isnan(run(model, runs(rng, (40, None), (1, 4), (59, None)), 0, fp32=False)).all()
        toks = runs(rng, (35, None))
        got = run(model, toks, 0, fp32=False)
        want = run(model, toks, 0, fp32=True)
        assert_close(got, want, f"{name}: logits", max_abs=2e-4, rel_l2=2e-5)
    finally:
        model.close()
