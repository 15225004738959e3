"""The prefill layer at the group counts of the streaming products against the
CPU oracle: K / 64 of 4 .. 36 in the gate/up product, and in the down product
one superstep of two groups (ff 128), whole ones, and whole ones with two more;
up to 384 tokens (128 weight rows a block), up to 1,023 (256) and from 1,024
(64-row tiles beside them). Up to 64 tokens these shapes take the general
kernels, as one past the streaming kernels' (width 384) does at any count. 129
to 511 tokens with few experts route by the batched projection."""
import numpy as np
import pytest

from conftest import tol_ok, weights_ok
from stratacuda_amd import workload as wl
from test_gpu_moe import device_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,F,E,topk,tokens", [(256, 128, 8, 3, 7), (256, 128, 40, 3, 65), (256, 128, 8, 3, 1030), (768, 384, 12, 4, 64),
                                               (1024, 256, 64, 6, 65), (1280, 896, 10, 2, 33), (1024, 640, 9, 3, 200), (1024, 640, 40, 3, 384), (512, 640, 9, 3, 385), (256, 128, 17, 2, 511),
                                               (1792, 1024, 6, 2, 1024), (2304, 1280, 6, 2, 50), (384, 192, 8, 3, 90),
                                               (768, 384, 12, 4, 65), (768, 384, 12, 4, 385), (768, 384, 12, 4, 1024), (1280, 896, 10, 2, 66),
                                               (1280, 896, 10, 2, 390), (2304, 1280, 6, 2, 67), (2304, 1280, 6, 2, 386)])
@pytest.mark.parametrize("block", [False, True])
def test_layer_group_counts(backend, oracle, W, F, E, topk, tokens, block):
    layer = wl.DeviceLayer(backend, layer=0, width=W, ff=F, experts=E, base_seed=29)
    host = wl.host_layer(oracle, 0, width=W, ff=F, experts=E, base_seed=29)
    X = device_inputs(backend, tokens, W, 37 + tokens, False)
    Y, ids, w = backend.alloc(tokens * W), backend.alloc(tokens * topk, "i32"), backend.alloc(tokens * topk)
    x = backend.read(X)
    tail = (layer.Wr, layer.arena, layer.stride, layer.shared, layer.Wsg, W, F, E, topk, Y, ids, w)
    if block:
        ws = backend.alloc_bytes(backend.moe_block_workspace_bytes(tokens, W, F, E, topk))
        backend.moe_block(X, tokens, layer.gamma, 1e-6, *tail, ws)
        xin = oracle.norm(x, host["gamma"], W, tokens)
    else:
        ws = backend.alloc_bytes(backend.moe_workspace_bytes(tokens, W, F, E, topk))
        backend.moe_layer(X, tokens, *tail, ws)
        xin = x
    eY, eids, ew = oracle.moe_layer(xin, tokens, host["Wr"], host["arena"], host["stride"], host["shared"], host["Wsg"],
                                    W, F, E, topk)
    layer.free()
    assert np.array_equal(backend.read(ids), eids)
    assert weights_ok(tokens, backend.read(w), ew)
    got, want = backend.read(Y), x + eY if block else eY
    assert tol_ok(got, want), "max abs err %g" % np.abs(got - want).max()


@pytest.mark.parametrize("W,F,E,topk", [(1024, 256, 64, 6), (512, 384, 24, 3), (2560, 640, 12, 2), (2048, 512, 64, 6)])
def test_equal_tokens_equal_results(backend, W, F, E, topk):
    """Equal tokens get equal bits in every 16-row tile, the full ones and the
    last one of 1 or 8 rows (of the shared segment, at least), and in calls of
    up to 384 tokens and of more."""
    layer = wl.DeviceLayer(backend, layer=0, width=W, ff=F, experts=E, base_seed=31)
    rows = []
    for tokens in (65, 200, 385):  # (from 512 tokens the weights come from the certified router)
        x = backend.read(device_inputs(backend, tokens, W, 43, False)).reshape(tokens, W).copy()
        x[-20:] = x[1]  # (the same values for every token count)
        X, Y = backend.alloc(x.reshape(-1)), backend.alloc(tokens * W)
        ids, w = backend.alloc(tokens * topk, "i32"), backend.alloc(tokens * topk)
        ws = backend.alloc_bytes(backend.moe_workspace_bytes(tokens, W, F, E, topk))
        backend.moe_layer(X, tokens, layer.Wr, layer.arena, layer.stride, layer.shared, layer.Wsg, W, F, E, topk, Y, ids, w, ws)
        rows.append(backend.read(Y).view(np.uint32).reshape(tokens, W)[-20:])
    layer.free()
    rows = np.concatenate(rows)
    assert np.array_equal(rows, np.broadcast_to(rows[0], rows.shape))
