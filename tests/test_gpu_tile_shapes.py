"""The tile shapes and K chunks that a batch's size selects on the MFMA path
(tile_shape and down_chunks in k_mfma.hip), against float64: token counts on
both sides of every threshold, ragged last tiles, a K that leaves a short last
chunk, and the layer types that differ (a dense layer's chunked down
projection, a routed layer whose shared expert's K is chunked beside the whole
K of the routed experts).  Tolerance: the MFMA path's (conftest)."""
import dataclasses

import numpy as np
import pytest

from conftest import MAX_ABS, MEAN_REL, announce, layer_error

pytestmark = pytest.mark.gpu


def _f64(bits):
    return (np.asarray(bits).astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def _ffn(x, gate, up, down):
    a = x @ _f64(gate).T
    return (a / (1.0 + np.exp(-a)) * (x @ _f64(up).T)) @ _f64(down).T


@pytest.fixture(scope="module")
def dense():
    from litemind_amd import Context
    from litemind_amd import workload as wl
    d = dataclasses.replace(wl.V2_LITE, hidden=416, dense_inter=2880)  # 90 K stages: chunks of 12, the last of 6
    weights = wl.dense_ffn(71, 0, d)
    with Context(d.moe_config(num_layers=1)) as ctx:
        ctx.upload_dense(0, *weights)
        ctx.finalize_layer(0)
        yield ctx, d, weights


@pytest.mark.parametrize("T", [3, 64, 65, 192, 193, 256, 257, 600])
def test_dense_shapes(dense, T):
    from litemind_amd import PATH_MFMA
    from litemind_amd import workload as wl
    ctx, d, weights = dense
    announce(f"dense tile shapes T={T}")
    x = wl.tokens(72, T, d.hidden)
    dx, dy = ctx.to_device(x), ctx.to_device(np.full((T, d.hidden), np.nan, np.float32))
    ctx.dense_forward(0, dx, T, dy, path=PATH_MFMA)
    ctx.synchronize()
    y = dy.download()
    dx.free()
    dy.free()
    mx, rel = layer_error(y, _ffn(x.astype(np.float64), *weights))
    print(f"dense T={T}: max_abs={mx:.3e} mean_rel={rel:.3e}")
    assert mx <= MAX_ABS and rel <= MEAN_REL


# 16 experts, top-4: 64-row tiles of 128 columns up to 32 tokens, of 256 up to
# 256, 128-row tiles above; three shared experts chunk their K in three
@pytest.mark.parametrize("T", [5, 32, 33, 256, 257])
def test_routed_shapes(T):
    from litemind_amd import workload as wl
    _routed(dataclasses.replace(wl.V2_LITE, hidden=320, inter=256, experts=16, top_k=4, n_shared=3), T)


# small groups by their gate/up tiles of 64 x 256 (16 experts x columns / 256)
@pytest.mark.parametrize("hidden,inter,n_shared", [
    (736, 704, 0),    # 96: one per CU or none, 64 x 128
    (736, 1408, 2),   # 198, but the shared expert's K in two chunks: 64 x 128
    (2560, 704, 1),   # 102: 64 x 128
    (2560, 1408, 0),  # 176: one per CU, 64 x 256
    (736, 2112, 0),   # 272: more, 64 x 128
    (736, 512, 1),    # 68 of a short K in down: 64 x 256
])
@pytest.mark.parametrize("T", [13, 32])
def test_routed_shapes_by_tiles(hidden, inter, n_shared, T):
    from litemind_amd import workload as wl
    _routed(dataclasses.replace(wl.V2_LITE, hidden=hidden, inter=inter, experts=16, top_k=4, n_shared=n_shared), T)


def _routed(d, T):
    from litemind_amd import PATH_MFMA, Context
    from litemind_amd import workload as wl
    L = wl.moe_layer(73, 0, d)
    announce(f"routed tile shapes hidden={d.hidden} inter={d.inter} shared={d.n_shared} T={T}")
    x = wl.tokens(74, T, d.hidden)
    with Context(d.moe_config(num_layers=1)) as ctx:
        wl.upload_moe_layer(ctx, 0, L)
        dx, dy = ctx.to_device(x), ctx.to_device(np.full((T, d.hidden), np.nan, np.float32))
        di, dw = ctx.empty((T, d.top_k), np.int32), ctx.empty((T, d.top_k))
        ctx.moe_forward(0, dx, T, dy, idx=di, w=dw, path=PATH_MFMA)
        ctx.synchronize()
        y, idx, w = dy.download(), di.download(), dw.download()
    x = x.astype(np.float64)
    want = _ffn(x, L.shared_gate, L.shared_up, L.shared_down) if d.n_shared else np.zeros_like(x)
    for e in range(d.experts):
        t, r = np.nonzero(idx == e)
        if t.size:
            want[t] += w[t, r, None] * _ffn(x[t], L.gate[e], L.up[e], L.down[e])
    mx, rel = layer_error(y, want)
    print(f"routed T={T}: max_abs={mx:.3e} mean_rel={rel:.3e}")
    assert mx <= MAX_ABS and rel <= MEAN_REL


# heads of other widths than the one-launch core's run the projections and the
# core as GEMMs of the same grouped kernel: split K with few tiles, 64 x 128 and
# 128 x 256 tiles
@pytest.mark.parametrize("q_lora,T", [(0, 40), (96, 40), (0, 300)])
def test_attention_other_head_widths(q_lora, T):
    from litemind_amd import PATH_MFMA
    from litemind_amd import workload as wl
    from test_gpu_attention import ATT_MAX_ABS, ATT_MEAN_REL, Mla, tokens
    d = dataclasses.replace(wl.V2_LITE_MLA, hidden=512, heads=4, q_lora_rank=q_lora, kv_lora_rank=256, qk_nope=64,
                            qk_rope=32, v_head=96, max_positions=T + 8)
    announce(f"attention MFMA path, other head widths q_lora={q_lora} T={T}")
    m = Mla(d, 401, path=PATH_MFMA)
    try:
        x = tokens(402, T + 5, d.hidden)
        for lo, hi in ((0, 5), (5, T + 5)):
            y = m.forward(x[lo:hi], lo)
            want, n = m.oracle(x[lo:hi], lo)
            assert n == hi - lo
            mx, rel = layer_error(y, want)
            print(f"q_lora={q_lora} {lo}..{hi}: max_abs={mx:.3e} mean_rel={rel:.3e}")
            assert mx <= ATT_MAX_ABS and rel <= ATT_MEAN_REL
    finally:
        m.close()
