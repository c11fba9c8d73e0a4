"""Batches of tokens through the fp32 matrix cores (matvec_exact_kernel), bit for
bit against the oracle's gemm::rms_norm + gemm::matvec_bf16 (src/Gemm.cpp:46-82,
:139-155, :197-207), through lm_head_forward.

The kernel's tiles are 32 tokens x 32 rows (64-element stages) or 16 tokens x
32 or 16 rows (128-element stages), its ring 6 or 4 stages deep: the shapes
below end inside a tile in both directions, inside a trip of the ring and at
one stage, and pass the 64 tokens of one head launch.  The tiny scale makes
products and sums subnormal: the matrix cores must keep them as fmaf does.
"""
import numpy as np
import pytest

from conftest import announce
from test_gpu_head import _case, _config, _gpu, _oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,H,T,scale", [
    (33, 64, 5, 1.0),        # one stage; widths that are not multiples of 128 take 32-token tiles
    (65, 192, 33, 1.0),      # three stages, a second token tile of one token
    (15, 128, 6, 1.0),       # 16 x 16 tiles, one stage
    (577, 640, 16, 1.0),     # 16 x 16 tiles, five stages of a four-stage ring
    (8200, 2048, 13, 1.0),   # 16 x 32 tiles, a last tile of 8 rows
    (16500, 1152, 32, 1.0),  # 32 x 32 tiles, three trips of the ring
    (20001, 512, 67, 1.0),   # 64 tokens, then three on the few-token kernel
    (1000, 4096, 80, 1.0),   # two launches
    (300, 2048, 20, 1e-37),  # subnormal products and sums
])
def test_head_batches_bit_exact(V, H, T, scale):
    from litemind_amd import Context
    from litemind_amd import workload as wl

    head, norm, hidden = _case(V * 7 + H + T, V, H, T)
    if scale != 1.0:
        wide = (head.astype(np.uint32) << 16).view(np.float32)
        head = wl.f32_to_bf16((wide * np.float32(scale)).astype(np.float32))
    announce(f"head batch V={V} H={H} T={T} scale={scale}")
    with Context(_config(H)) as ctx:
        ctx.upload_head(norm, head)
        logits, token, token2 = _gpu(ctx, hidden, V)
    want = _oracle(head, norm, hidden)
    assert np.array_equal(logits.view(np.uint32), want.view(np.uint32))
    assert token.tolist() == [int(np.argmax(want[t])) for t in range(T)]
    assert token2.tolist() == token.tolist()


@pytest.mark.parametrize("V,H,T", [
    (300, 5120, 4),    # four rows of 20 KB
    (300, 5120, 68),   # 64 tokens, then four
    (300, 7168, 3),
    (300, 8192, 67),   # 64 tokens, then three
    (65, 16384, 2),    # the widest head
    (65, 4160, 4),     # not a multiple of 128: 32-token tiles
])
def test_few_tokens_at_wide_heads(V, H, T):
    """Two to four tokens, alone or left over from a batch, whose rows exceed the 64 KB of LDS
    that the few-token kernel keeps them in."""
    from litemind_amd import Context

    head, norm, hidden = _case(V + H + T, V, H, T)
    announce(f"head few tokens V={V} H={H} T={T}")
    with Context(_config(H)) as ctx:
        ctx.upload_head(norm, head)
        logits, token, token2 = _gpu(ctx, hidden, V)
    want = _oracle(head, norm, hidden)
    assert np.array_equal(logits.view(np.uint32), want.view(np.uint32))
    assert token.tolist() == [int(np.argmax(want[t])) for t in range(T)]
    assert token2.tolist() == token.tolist()
