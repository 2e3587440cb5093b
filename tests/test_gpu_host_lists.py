"""gmoe_forward_host's per-expert lists, which the host forms from the selections it has read
back, against k_dispatch's (gmoe_read_layer_state after the same call): one token, small and
ragged batches, and a batch with a NaN row, whose selections name no expert. The call's other
outputs, which the GPU writes into pinned host memory, against the same read-back."""
import numpy as np
import pytest

import gmoe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,nan_row", [(1, None), (1, 0), (3, 1), (37, None)])
def test_host_lists_are_the_dispatch_lists(T, nan_row):
    shape = gmoe.Shape(dim=512, moe_ffn_dim=256, n_routed_experts=16, n_experts_used=4)
    ctx = gmoe.Context(shape, n_layers=2, max_tokens=40)
    try:
        ctx.upload(1, gmoe.HostLayer(shape, seed=71, layer=1))
        x = gmoe.activations(71, 1, T, shape.D)
        if nan_row is not None:
            x[nan_row] = np.nan
        print(f"[case] host lists T={T} nan_row={nan_row}", flush=True)
        got, st = gmoe.forward_host(ctx, 1, x)
        dev = ctx.read_state(T)
        n = int(st["expert_offsets"][-1])
        assert n == T * shape.K - (0 if nan_row is None else shape.K)
        for k in ("expert_offsets", "topk_idx"):
            np.testing.assert_array_equal(st[k], dev[k], err_msg=k)
        np.testing.assert_array_equal(st["expert_tokens"][:n], dev["expert_tokens"][:n])
        for k in ("xn", "router_prob", "topk_w", "shared_out", "routed_out"):
            assert np.array_equal(st[k].view(np.uint32), dev[k].view(np.uint32)), k
    finally:
        ctx.close()
