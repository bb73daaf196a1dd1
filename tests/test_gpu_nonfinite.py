"""Infinities and NaN in attention inputs reach the rows that attend to them and no others, on the
kernels that hold probabilities in fp32 (fp32 caches, 256-wide heads, decode groups above 8, slot
tables) and on the ragged launch."""

import numpy as np
import pytest
import torch

from tests._util import randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pool(NB, KVH, D, dtype, bs=16):
    return [randn((NB * bs, KVH, D), s, dtype).to(DEV) for s in (1, 2)]


def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("dtype,G,D", [(torch.float32, 3, 64), (torch.float32, 1, 8),
                                       (torch.bfloat16, 4, 256), (torch.float16, 4, 256),
                                       (torch.bfloat16, 12, 128)])
@pytest.mark.parametrize("ctx", [[40, 17], [900, 2000]])
@pytest.mark.parametrize("q_len", [1, 5])
def test_nan_queries_give_nan_rows(hip, dtype, G, D, ctx, q_len):
    """A query with a NaN (one head of one token) gives a row of NaN, not of zeros, whether its
    keys are one partition or several; the other rows are what they are without it."""
    from dispec_amd.engine.hip_attn import paged_decode_attention_blocks, paged_mq_attention
    KVH, bs = 2, 16
    kc, vc = _pool(256, KVH, D, dtype)
    bt = torch.randperm(256, generator=torch.Generator().manual_seed(3)).int().to(DEV).view(2, 128)
    q = randn((2 * q_len, G * KVH, D), 4, dtype).to(DEV)
    if q_len == 1:
        def call(x):
            return paged_decode_attention_blocks(x, kc, vc, bt, _i32(ctx), G, block_size=bs,
                                                 max_ctx=max(ctx))
    else:
        def call(x):
            return paged_mq_attention(x, kc, vc, bt, _i32([0, q_len, 2 * q_len]), _i32(ctx), G,
                                      block_size=bs, max_q_len=q_len, max_ctx=max(ctx))
    want = call(q)
    bad = q.clone()
    bad[q_len, G, D // 2] = float("nan")
    got = call(bad)
    assert bool(torch.isnan(got[q_len, G]).all())
    got[q_len, G] = want[q_len, G]
    assert torch.equal(got, want)
