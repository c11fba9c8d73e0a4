"""Device memory that a context takes for what it runs: the workspace of its first
call grows with the call's tokens, and the down projection's partial sums (its K
in chunks, on the MFMA path) fit it at every token count up to that."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from conftest import announce, layer_error

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _free():
    """Bytes of device memory that are free."""
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _dims():
    from litemind_amd import workload as wl

    return dataclasses.replace(wl.V2_LITE, hidden=5120, inter=64, experts=8, top_k=2, dense_inter=64)


def test_first_call_of_one_token_stays_small():
    from litemind_amd import Context
    from litemind_amd import workload as wl

    d = _dims()
    layer = wl.moe_layer(41, 0, d)
    x = wl.tokens(42, 1, d.hidden)
    took = 0
    for _ in range(2):  # the first context also loads the kernels
        with Context(d.moe_config(num_layers=1)) as ctx:
            wl.upload_moe_layer(ctx, 0, layer)
            dx, dy = ctx.to_device(x), ctx.empty((1, d.hidden))
            before = _free()
            announce("first call of a context, one token of hidden 5120")
            ctx.moe_forward(0, dx, 1, dy)
            ctx.synchronize()
            took = before - _free()
            dx.free()
            dy.free()
    print(f"one token of hidden {d.hidden}: {took / MB:.1f} MB")
    # 4096 rows of partial sums would be 80 MB; the buffers need 0.5 MB, in pages of up to 2 MB each
    assert took < 40 * MB


def test_head_upload_keeps_no_logits():
    """The head's resident bytes plus what a launch of 64 tokens needs between its kernels: two
    candidates of 12 bytes per 32 rows and token, and the normalised tokens; the logits only in the caller's
    buffer."""
    from litemind_amd import Context, MoeConfig
    from litemind_amd import workload as wl

    V, H = 102400, 64
    rng = np.random.default_rng(46)
    head = wl.f32_to_bf16(rng.standard_normal((V, H)).astype(np.float32))
    norm = np.ones(H, np.float32)
    config = MoeConfig(hidden_size=H, moe_intermediate_size=64, n_routed_experts=8, num_experts_per_tok=2,
                       n_shared_experts=0, intermediate_size=0, norm_topk_prob=0, routed_scaling_factor=1.0,
                       group_limited=0, n_group=1, topk_group=1, rms_norm_eps=1e-6, num_layers=1)
    announce(f"upload of a head of {V} rows")
    for _ in range(2):  # the first upload also takes what copies need
        with Context(config) as ctx:
            before = _free()
            ctx.upload_head(norm, head)
            took = before - _free()
    print(f"head of {head.nbytes / MB:.1f} MB: {took / MB:.1f} MB")
    need = head.nbytes + norm.nbytes + 64 * 4 * H + 12 * 64 * 2 * (V // 32)
    assert took <= need + 8 * MB  # pages of 2 MB; the logits of 64 tokens would be 25 MB


@pytest.mark.parametrize("T", [4, 8, 21, 64])
def test_shared_chunks_fit_a_workspace_of_the_call(T):
    """A shared expert four times as wide as the routed ones: its K in four chunks, up to 8 rows
    per expert."""
    from litemind_amd import PATH_GEMV, PATH_MFMA, Context
    from litemind_amd import workload as wl

    d = dataclasses.replace(wl.V2_LITE, hidden=512, inter=512, experts=16, top_k=2, n_shared=4)
    layer = wl.moe_layer(44, 0, d)
    x = wl.tokens(45, T, d.hidden)
    outs = []
    for path in (PATH_MFMA, PATH_GEMV):
        with Context(d.moe_config(num_layers=1)) as ctx:
            wl.upload_moe_layer(ctx, 0, layer)
            dx, dy = ctx.to_device(x), ctx.empty((T, d.hidden))
            announce(f"MoE layer with a wide shared expert, workspace of {T} tokens, path {path}")
            ctx.moe_forward(0, dx, T, dy, path=path)
            ctx.synchronize()
            outs.append(dy.download())
            dx.free()
            dy.free()
    mx, rel = layer_error(outs[0], outs[1])
    print(f"T={T}: max_abs={mx:.3e} mean_rel={rel:.3e}")
    assert mx <= 2e-2 and rel <= 1e-3


@pytest.mark.parametrize("T", [1, 2, 5, 64, 511, 512, 513])
def test_partial_sums_fit_a_workspace_of_the_call(T):
    """A dense layer of few columns splits K the most.  The workspace is the call's own (a fresh
    context); 8 chunks of 511 and 512 tokens are the most rows, 513 take 7."""
    from litemind_amd import PATH_GEMV, PATH_MFMA, Context
    from litemind_amd import workload as wl

    rng = np.random.default_rng(T)
    d = dataclasses.replace(wl.V2_LITE, hidden=256, inter=64, experts=8, top_k=2, dense_inter=4096)
    bits = lambda shape: wl.f32_to_bf16((0.02 * rng.standard_normal(shape)).astype(np.float32))
    gate, up, down = bits((4096, 256)), bits((4096, 256)), bits((256, 4096))
    x = wl.tokens(43, T, d.hidden)
    outs = []
    for path in (PATH_MFMA, PATH_GEMV):
        with Context(d.moe_config(num_layers=1)) as ctx:
            ctx.upload_dense(0, gate, up, down)
            ctx.finalize_layer(0)
            dx, dy = ctx.to_device(x), ctx.empty((T, d.hidden))
            announce(f"dense layer, workspace of {T} tokens, path {path}")
            ctx.dense_forward(0, dx, T, dy, path=path)
            ctx.synchronize()
            outs.append(dy.download())
            dx.free()
            dy.free()
    mx, rel = layer_error(outs[0], outs[1])
    print(f"T={T}: max_abs={mx:.3e} mean_rel={rel:.3e}")
    assert mx <= 2e-2 and rel <= 1e-3  # the layer tolerance of the MFMA path
