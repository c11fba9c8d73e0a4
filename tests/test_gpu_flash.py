"""The one-launch attention core (flash_kernel) at DeepSeek-V2-Lite's head widths,
through lm_attention_forward on the MFMA path, against float64 attention over
the same cache: a wave owns 32 query tokens, a tile 64 keys, and few query
tokens over many keys split the keys over several workgroups.

The reference is fed the cache entries that the call itself wrote (read back),
so only the core and the query / output projections differ: fp16 operands
(2^-11 relative each) through a 2048-term product, a softmax over scores of a
few units and a second product, then the output projection; their independent
errors stay near 1e-3 of the output's scale, and the bounds are the path's own
(mean relative 5e-3, maximum 5e-2 at outputs of magnitude 1).
"""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from conftest import announce, layer_error
from test_gpu_attention import ATT_MAX_ABS, ATT_MEAN_REL, Mla, tokens

pytestmark = pytest.mark.gpu


def _f32(bits):
    return (np.asarray(bits).astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def _reference(m, x, cached, rotated=True, rows=None):
    """float64 attention of x [T, H] at positions cached.. over the layer's cache (past the
    rotary table the channels stay as they are), of the given rows only or all."""
    from litemind_amd import mla_softmax_scale, rope_tables
    from litemind_amd import workload as wl
    d, L, T = m.d, m.L, x.shape[0]
    n = cached + T
    at = np.arange(T) if rows is None else np.asarray(rows)
    kn, kr, v = (a.astype(np.float64) for a in m.ctx.kv_cache_read(0, n))
    cfg = wl.mla_config(d)
    cos, sin = (t[cached:n][at].astype(np.float64)[:, None] for t in rope_tables(cfg, n))
    q = (x[at].astype(np.float64) @ _f32(L.q_proj).T).reshape(len(at), d.heads, d.qk_head)
    even, odd = q[..., d.qk_nope::2], q[..., d.qk_nope + 1::2]
    rot = np.concatenate([even * cos - odd * sin, odd * cos + even * sin], axis=-1) if rotated else q[..., d.qk_nope:]
    scale = float(mla_softmax_scale(cfg))
    hidden = np.arange(n)[None] > cached + at[:, None]
    ctx = np.empty((len(at), d.heads, d.v_head))
    for h in range(d.heads):
        s = scale * (q[:, h, :d.qk_nope] @ kn[:, h].T + rot[:, h] @ kr.T)
        s[hidden] = -np.inf
        p = np.exp(s - s.max(axis=1, keepdims=True))
        ctx[:, h] = (p / p.sum(axis=1, keepdims=True)) @ v[:, h]
    return ctx.reshape(len(at), -1) @ _f32(L.o_proj).T


@pytest.mark.parametrize("heads,cached,T", [
    (16, 0, 16),      # one wave, half of it past the last token
    (16, 5, 33),      # one token in the second wave
    (16, 63, 65),     # the diagonal crosses tiles, a third wave
    (3, 0, 97),       # heads that are no multiple of the eight XCDs
    (16, 2048, 16),   # keys split over workgroups
    (16, 1500, 40),   # split, ragged last tile, queries masked in whole tiles
    (5, 0, 1029),     # nine query blocks, the last of five tokens
    (16, 130, 1100),  # nine query blocks after cached tokens
])
def test_flash_core(heads, cached, T):
    from litemind_amd import PATH_MFMA
    from litemind_amd import workload as wl
    d = dataclasses.replace(wl.V2_LITE_MLA, heads=heads, max_positions=cached + T + 3)
    announce(f"attention one-launch core heads={heads} cached={cached} T={T}")
    m = Mla(d, 301 + heads, path=PATH_MFMA)
    try:
        rng = np.random.default_rng(T)
        if cached:
            m.ctx.kv_cache_write(0, 0, *(rng.standard_normal(s).astype(np.float32) for s in (
                (cached, heads, d.qk_nope), (cached, d.qk_rope), (cached, heads, d.v_head))))
        x = tokens(302, T, d.hidden)
        y = m.forward(x, cached)
        want = _reference(m, x, cached)
        assert np.all(np.isfinite(y))
        mx, rel = layer_error(y, want)
        print(f"heads={heads} cached={cached} T={T}: max_abs={mx:.3e} mean_rel={rel:.3e}")
        assert mx <= ATT_MAX_ABS and rel <= ATT_MEAN_REL
        for t in (0, T - 1):  # no row is off while the mean is fine
            assert np.abs(y[t] - want[t]).sum() <= 2 * ATT_MEAN_REL * np.abs(want[t]).sum()
    finally:
        m.close()


@pytest.mark.parametrize("T", [700, 1400, 2600])
def test_prompt_projection_tiles(T):
    """The projections' larger tiles at V2-Lite's widths: q and kv_a, then kv_b, as 128 x 128 tiles
    from 641 tokens and 128 x 256 from 1281, o_proj from 1281 and 2561.  Every row of the cache,
    and the outputs of tokens at the edges of waves and tiles."""
    from litemind_amd import PATH_MFMA
    from litemind_amd import workload as wl
    d = dataclasses.replace(wl.V2_LITE_MLA, max_positions=T)
    announce(f"attention prompt, projection tiles T={T}")
    m = Mla(d, 311, path=PATH_MFMA)
    try:
        x = tokens(312, T, d.hidden)
        y = m.forward(x, 0)
        kn, kr, v = m.ctx.kv_cache_read(0, T)
        L, cfg = m.L, wl.mla_config(d)
        kv = x.astype(np.float64) @ _f32(L.kv_a_proj).T
        c = kv[:, :d.kv_lora_rank]
        c = c / np.sqrt((c * c).mean(axis=1, keepdims=True) + d.rms_norm_eps) * L.kv_a_layernorm.astype(np.float64)
        wide = (c @ _f32(L.kv_b_proj).T).reshape(T, d.heads, d.qk_nope + d.v_head)
        from litemind_amd import rope_tables
        cos, sin = (t.astype(np.float64) for t in rope_tables(cfg, T))
        even, odd = kv[:, d.kv_lora_rank::2], kv[:, d.kv_lora_rank + 1::2]
        rotated = np.concatenate([even * cos - odd * sin, odd * cos + even * sin], axis=1)
        for got, want in ((kn, wide[..., :d.qk_nope]), (kr, rotated), (v, wide[..., d.qk_nope:])):
            # fp16 operands in two products: 2^-11 relative each, per row (a wrong row is of order 1)
            off = np.abs(got - want).reshape(T, -1).sum(axis=1) / np.abs(want).reshape(T, -1).sum(axis=1)
            assert off.max() <= ATT_MEAN_REL
        rows = sorted({t for edge in range(0, T + 1, 128) for t in (edge - 1, edge) if 0 <= t < T} | {33, T - 1})
        want = _reference(m, x, 0, rows=rows)
        off = np.abs(y[rows] - want).sum(axis=1) / np.abs(want).sum(axis=1)
        print(f"T={T}: mean_rel by row up to {off.max():.3e}")
        assert np.all(np.isfinite(y)) and off.max() <= 2 * ATT_MEAN_REL
    finally:
        m.close()


def test_flash_past_the_rotary_table():
    """Positions at or past the table: queries and keys stay unrotated."""
    from litemind_amd import PATH_MFMA
    from litemind_amd import workload as wl
    d = dataclasses.replace(wl.V2_LITE_MLA, max_positions=40)
    announce("attention one-launch core past the rotary table")
    m = Mla(d, 305, path=PATH_MFMA)
    try:
        x = tokens(306, 36, d.hidden)
        y = m.forward(x, 40)
        want = _reference(m, x, 0, rotated=False)
        mx, rel = layer_error(y, want)
        assert mx <= ATT_MAX_ABS and rel <= ATT_MEAN_REL
    finally:
        m.close()


def test_flash_core_groups_bit_identical():
    """A score budget that holds part of the query tokens runs the split core in groups: the
    same bits as in one launch (the splits depend on the whole call)."""
    from litemind_amd import PATH_MFMA, attention_plan_core
    from litemind_amd import workload as wl
    cached, T = 1500, 130
    d = dataclasses.replace(wl.V2_LITE_MLA, max_positions=cached + T)
    rng = np.random.default_rng(9)
    cache = [rng.standard_normal(s).astype(np.float32) for s in (
        (cached, d.heads, d.qk_nope), (cached, d.qk_rope), (cached, d.heads, d.v_head))]
    x = tokens(303, T, d.hidden)
    budget = 33_600_000
    plan = attention_plan_core(wl.mla_config(d), cached, T, PATH_MFMA, budget)
    assert plan.mfma_core == 1 and 1 <= plan.query_group < T
    announce("attention one-launch core, split keys, query groups against one group")
    outs = []
    for b in (budget, 0):
        m = Mla(d, 304, path=PATH_MFMA)
        try:
            m.ctx.attention_set_score_budget(b)
            m.ctx.kv_cache_write(0, 0, *cache)
            outs.append(m.forward(x, cached))
        finally:
            m.close()
    np.testing.assert_array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


def _cache(rng, d, cached):
    return [rng.standard_normal(s).astype(np.float32) for s in (
        (cached, d.heads, d.qk_nope), (cached, d.qk_rope), (cached, d.heads, d.v_head))]


def test_flash_partials_past_the_budget():
    """One head after 4200 tokens: 15 splits of 520 bytes a query token, and a budget of twice the
    key and value copies, which holds the partial contexts of some 390 tokens of 600."""
    from litemind_amd import PATH_MFMA, attention_plan_core
    from litemind_amd import workload as wl
    cached, T, budget = 4200, 600, 6_200_000
    d = dataclasses.replace(wl.V2_LITE_MLA, heads=1, max_positions=cached + T)
    cache = _cache(np.random.default_rng(19), d, cached)
    x = tokens(307, T, d.hidden)
    assert attention_plan_core(wl.mla_config(d), cached, T, PATH_MFMA, budget).mfma_core == 1
    announce("attention one-launch core, partial contexts in two groups against one")
    outs = []
    for b in (budget, 0):
        m = Mla(d, 308, path=PATH_MFMA)
        try:
            m.ctx.attention_set_score_budget(b)
            m.ctx.kv_cache_write(0, 0, *cache)
            outs.append(m.forward(x, cached))
            want = _reference(m, x, cached)
        finally:
            m.close()
    np.testing.assert_array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    mx, rel = layer_error(outs[0], want)
    assert mx <= ATT_MAX_ABS and rel <= ATT_MEAN_REL


@pytest.mark.parametrize("cached,T,launches", [
    (2000, 1024, 8),  # copies of the cache, x, q and kv_a, norm, kv_b, core, its splits joined, o_proj
    (2000, 100, 8),
    (0, 1024, 7),     # no cache
    (0, 512, 6),      # nor splits
])
def test_prompt_captured(cached, T, launches):
    """A prompt under stream capture: one launch per step, the core's splits of all query tokens
    at once, and replays between eager calls that give the eager bits."""
    from litemind_amd import PATH_MFMA
    from litemind_amd import workload as wl
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphGetNodes.argtypes = [C.c_void_p, C.c_void_p, C.POINTER(C.c_size_t)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    hip.hipGraphDestroy.argtypes = hip.hipGraphExecDestroy.argtypes = [C.c_void_p]
    d = dataclasses.replace(wl.V2_LITE_MLA, max_positions=cached + T)
    m = Mla(d, 309, path=PATH_MFMA)
    ctx = m.ctx
    try:
        if cached:
            ctx.kv_cache_write(0, 0, *_cache(np.random.default_rng(20), d, cached))
        x = tokens(310, T, d.hidden)
        dx, dout = ctx.to_device(x), ctx.to_device(np.full_like(x, np.nan))
        stream, graph, run, n = C.c_void_p(ctx.stream()), C.c_void_p(), C.c_void_p(), C.c_size_t()

        def eager():
            ctx.kv_cache_truncate(0, cached)
            ctx.attention_forward(0, dx, T, cached, dout)

        announce(f"attention prompt captured cached={cached} T={T}")
        eager()
        ctx.synchronize()
        want = dout.download()
        assert hip.hipStreamBeginCapture(stream, 2) == 0  # hipStreamCaptureModeRelaxed
        eager()
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
        print(f"cached={cached} T={T}: {n.value} launches")
        assert n.value == launches
        assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
        for _ in range(3):
            dout.upload(np.full_like(x, np.nan))
            assert hip.hipGraphLaunch(run, stream) == 0
            ctx.synchronize()
            np.testing.assert_array_equal(dout.download().view(np.uint32), want.view(np.uint32))
            eager()
            ctx.synchronize()
            np.testing.assert_array_equal(dout.download().view(np.uint32), want.view(np.uint32))
        assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
        dx.free()
        dout.free()
    finally:
        m.close()
