"""The grouped GEMMs over glm.c's own layout (k_native_group_gu, k_native_group_down: the
native form's batches from T (K + 1) = E + 2 K on) against the oracle, at every count of
scales a 128-column chunk has (group sizes of 64 columns and more, 32, and 16 or an odd
multiple of it) and at lists of one to three tiles with remainders; and against the per-token
kernels that smaller batches take, which GMOE_GROUPED_MIN_T keeps for any T.

Bar against the oracle as elsewhere (max-abs 1e-2, rel-L2 1e-3). Between the two kernel pairs:
fp32 sums in another order and activations of 22 bits, 2^-22 of each element before random signs
average it, so rel-L2 5e-7 per product and 2e-6 through the layer's three."""
import numpy as np
import pytest

import gmoe
import oracle
from conftest import assert_close
from test_gpu_native import check

pytestmark = pytest.mark.gpu


def shape(gs, D=512, F=256):
    return gmoe.Shape(dim=D, moe_ffn_dim=F, n_routed_experts=16, n_experts_used=4, group_size=gs)


SHAPES = [pytest.param(shape(128), id="gs128"), pytest.param(shape(64), id="gs64"), pytest.param(shape(32), id="gs32"),
          pytest.param(shape(16), id="gs16"), pytest.param(shape(48, 768, 768), id="gs48"),
          pytest.param(shape(192, 768, 768), id="gs192"), pytest.param(shape(96, 768, 768), id="gs96"),
          pytest.param(gmoe.Shape(dim=256, moe_ffn_dim=256, n_routed_experts=80, n_experts_used=2, group_size=64), id="e80")]


def forward(sh, hl, x, T, flags=0):
    ctx = gmoe.Context(sh, n_layers=2, max_tokens=T, q8_form=gmoe.GMOE_Q8_NATIVE)
    try:
        ctx.upload(1, hl)
        return gmoe.forward_host(ctx, 1, x, flags=flags)
    finally:
        ctx.close()


@pytest.mark.parametrize("T", [5, 31, 70])
@pytest.mark.parametrize("sh", SHAPES)
def test_grouped_native(sh, T, monkeypatch):
    T = max(T, -(-(sh.E + 2 * sh.K) // (sh.K + 1)))  # the least T of the grouped GEMMs (28 for e80)
    hl = gmoe.HostLayer(sh, seed=61, layer=1, norm_mode=gmoe.SYNTH_NORM_RANDOM, scale_mode=gmoe.SYNTH_SCALES_FP32)
    x = gmoe.activations(61, 2, T, sh.D)
    for flags in (0, gmoe.GMOE_FLAG_NO_ROUTED):
        print(f"[case] native grouped gs={sh.gs} D={sh.D} E={sh.E} T={T} flags={flags}", flush=True)
        want = oracle.Oracle("port").layer(sh, hl, x, disable_routed=bool(flags))
        got, st = forward(sh, hl, x, T, flags)
        check(want, got, st, f"gs={sh.gs} T={T}")
        monkeypatch.setenv("GMOE_GROUPED_MIN_T", "100000")
        one, _ = forward(sh, hl, x, T, flags)
        monkeypatch.delenv("GMOE_GROUPED_MIN_T")
        assert not np.array_equal(got, one), "both runs took the same kernels"
        rel = np.linalg.norm(got.astype(np.float64) - one) / np.linalg.norm(one.astype(np.float64))
        assert rel <= 2e-6, f"gs={sh.gs} T={T}: {rel:.2e} from the per-token kernels"


@pytest.mark.parametrize("E", [16, 80])
def test_profile_counts_each_product_once(E):
    """gmoe_profile_read of a native batch: one launch a call of gate_up and of down, with the
    grouped kernels as with the per-token ones (T = 2), so that ms / launches is a layer's time."""
    sh = gmoe.Shape(dim=256, moe_ffn_dim=256, n_routed_experts=E, n_experts_used=2, group_size=64)
    ctx = gmoe.Context(sh, n_layers=2, max_tokens=64, q8_form=gmoe.GMOE_Q8_NATIVE)
    try:
        ctx.upload(1, gmoe.HostLayer(sh, seed=62, layer=1))
        for T in (2, 64):  # 64 * 3 >= E + 4: grouped
            print(f"[case] native profile E={E} T={T}", flush=True)
            ctx.profile(True)
            for _ in range(3):
                gmoe.forward_host(ctx, 1, gmoe.activations(62, 2, T, sh.D))
            ran = ctx.profile_read()
            ctx.profile(False)
            assert ran["gate_up"][0] == ran["down"][0] == 3, ran
    finally:
        ctx.close()
