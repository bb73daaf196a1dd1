"""256-wide 16-bit heads and decode groups above 8 on the MFMA kernels, against the generic
kernel that serves the same shapes where the 16-byte vectors are not aligned.

The generic kernel is reached with the same numbers by handing q over with rows of D + 1
elements.  Bound: each output is the 16-bit rounding of a value the two kernels form in fp32
(one unit in the last place apart at most when those straddle a rounding boundary: 2^-7 of
the value in bf16, 2^-10 in fp16) from probabilities held to 2^-16 or better, whose sum with
|v| moves a row by at most 2^-15 max|v|.
"""

import numpy as np
import pytest
import torch

from tests._util import randn, random_block_tables

pytestmark = pytest.mark.gpu
DEV = "cuda"
RTOL = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


def _unaligned(q):
    """q's values in rows of D + 1 elements: no 16-byte vectors, the generic kernel."""
    buf = torch.empty((*q.shape[:-1], q.shape[-1] + 1), dtype=q.dtype, device=q.device)
    buf[..., :-1] = q
    return buf[..., :-1]


def _inputs(q_lens, ctx, G, KVH, D, dtype, seed, bs):
    NB = sum(-(-n // bs) for n in ctx) + 3
    tables = random_block_tables(NB, ctx, bs, seed)
    bt = torch.zeros((len(ctx), max(max(len(t) for t in tables), 1)), dtype=torch.int32)
    for i, t in enumerate(tables):
        bt[i, :len(t)] = torch.tensor(t, dtype=torch.int32)
    kc = randn((NB * bs, KVH, D), seed + 1, dtype).to(DEV)
    vc = randn((NB * bs, KVH, D), seed + 2, dtype).to(DEV)
    q = randn((sum(q_lens), G * KVH, D), seed + 3, dtype).to(DEV)
    cu = torch.tensor([0] + list(np.cumsum(q_lens)), dtype=torch.int32, device=DEV)
    return q, kc, vc, bt.to(DEV), cu, torch.tensor(ctx, dtype=torch.int32, device=DEV)


def _check(fast, slow, vc, dtype, what):
    # not the same launch twice: the two kernels sum in different orders
    fast, slow = fast.float(), slow.float()
    bound = RTOL[dtype] * slow.abs() + 2.0 ** -15 * vc.float().abs().max()
    worst = float(((fast - slow).abs() - bound).max())
    assert worst <= 0 and torch.isfinite(fast).all(), f"{what}: {worst:.3g} over the bound"


def _decode_both(ctx, G, KVH, D, dtype, seed, bs=16, P=0, bad=False, max_ctx=None):
    from dispec_amd.engine.hip_attn import paged_decode_attention_blocks
    q, kc, vc, bt, _, lens = _inputs([1] * len(ctx), ctx, G, KVH, D, dtype, seed, bs)
    if bad:
        bt[0, 1], bt[-1, 0] = 10 ** 6, -3
    outs = [paged_decode_attention_blocks(x, kc, vc, bt, lens, G, block_size=bs, max_ctx=max_ctx,
                                          partition_tokens=P) for x in (q, _unaligned(q))]
    _check(outs[0], outs[1], vc, dtype, f"decode {ctx} G={G} D={D} P={P} bad={bad}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("G,KVH,D", [(1, 4, 256), (8, 2, 256), (16, 1, 256), (17, 2, 256),
                                     (12, 4, 128), (9, 1, 64), (24, 2, 32)])
@pytest.mark.parametrize("P", [0, 64, 96])
def test_decode(hip, dtype, G, KVH, D, P):
    """Unsplit (max_ctx <= 512), balanced (automatic, G <= 16) and fixed partitions; more than
    16 query heads take a second row tile."""
    _decode_both([0, 1, 15, 16, 17, 500], G, KVH, D, dtype, 100 + G + D, P=P)
    _decode_both([1, 33, 700, 2100], G, KVH, D, dtype, 200 + G + D, bs=32, P=P)


@pytest.mark.parametrize("G,D", [(4, 256), (12, 128), (20, 64)])
@pytest.mark.parametrize("ctx", [[60, 200, 40], [900, 200, 1300]])
def test_decode_bad_blocks_are_skipped(hip, G, D, ctx):
    _decode_both(ctx, G, 2, D, torch.bfloat16, 300 + G, bad=True)
    _decode_both(ctx, G, 2, D, torch.bfloat16, 310 + G, bad=True, P=128)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("q_lens,ctx,bs,P", [
    ([5, 1, 3], [600, 17, 3], 16, 0),               # 16-row tiles
    ([5, 1, 3], [600, 17, 3], 16, 128),
    ([127, 1, 64], [127, 900, 65], 16, 0),          # 128-row tiles
    ([130, 200, 1], [1000, 200, 63], 32, 256),
    ([130, 200, 1], [1000, 200, 63], 8, 0),         # blocks too small for them
])
@pytest.mark.parametrize("bad", [False, True])
def test_multi_query(hip, dtype, q_lens, ctx, bs, P, bad):
    from dispec_amd.engine.hip_attn import paged_mq_attention
    G, KVH, D = 3, 2, 256
    q, kc, vc, bt, cu, lens = _inputs(q_lens, ctx, G, KVH, D, dtype, 400 + bs, bs)
    if bad:
        bt[0, 1] = 10 ** 6
    else:
        # a slot past a sequence's context holds whatever its block held before: never read
        last = int(bt[2, (ctx[2] - 1) // bs]) * bs + (ctx[2] - 1) % bs + 1
        if ctx[2] % bs:
            kc[last], vc[last] = float("nan"), float("nan")
    outs = [paged_mq_attention(x, kc, vc, bt, cu, lens, G, block_size=bs, max_q_len=max(q_lens),
                               partition_tokens=P) for x in (q, _unaligned(q))]
    if not bad and ctx[2] % bs:
        vc[last] = 0
    _check(outs[0], outs[1], vc, dtype, f"mq {q_lens} {ctx} bs={bs} P={P} bad={bad}")
