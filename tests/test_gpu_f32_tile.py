"""fp32 attention on the matrix cores' 16-row tiles: row, key and dim remainders, rows of
4-byte-aligned strides, slot tables and skipped block ids, against the float64 oracle.

Tolerance: max-abs 1e-5, cosine 0.999999 (fp32 sums over at most ~1000 keys of N(0, 1) data:
a result of weights that add to 1 errs by ~1e-6; any 16-bit rounding would miss it 100x)."""

import numpy as np
import pytest
import torch

from oracle import ref_cpu
from tests._util import cosine, f64, gen, randn, random_block_tables

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _close(out, ref, what):
    out = f64(out)
    err = float(np.abs(out - ref).max())
    assert err <= 1e-5 and cosine(out, ref) >= 0.999999, f"{what}: max-abs {err:.3g}"


def _padded(t):
    """t's values in rows one element longer: 4-byte alignment only."""
    buf = torch.zeros((*t.shape[:-1], t.shape[-1] + 1), dtype=t.dtype, device=DEV)
    buf[..., :-1] = t.to(DEV)
    return buf[..., :-1]


@pytest.mark.parametrize("D", [8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("G,KVH", [(1, 2), (3, 2), (8, 1), (20, 1)])
@pytest.mark.parametrize("padded", [False, True])
def test_decode_and_multi_query(hip, D, G, KVH, padded):
    from dispec_amd.engine.hip_attn import (batched_paged_decode_attention,
                                            paged_decode_attention_blocks, paged_mq_attention)
    bs = 8
    ctx, q_lens = [1, 15, 17, 64, 333, 1000], [1, 15, 6, 1, 17, 5]
    NB = sum(-(-n // bs) for n in ctx) + 2
    tables = random_block_tables(NB, ctx, bs, D + G)
    bt = torch.zeros((len(ctx), -(-max(ctx) // bs)), dtype=torch.int32)
    st = torch.zeros((len(ctx), max(ctx)), dtype=torch.int32)
    slots = [ref_cpu.context_slots(t, n, bs) for t, n in zip(tables, ctx)]
    for i, t in enumerate(tables):
        bt[i, :len(t)] = torch.tensor(t, dtype=torch.int32)
        st[i, :ctx[i]] = torch.from_numpy(np.asarray(slots[i])).to(torch.int32)
    kc, vc = randn((NB * bs, KVH, D), 1, torch.float32), randn((NB * bs, KVH, D), 2, torch.float32)
    put = _padded if padded else (lambda t: t.to(DEV))
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    q = randn((len(ctx), G * KVH, D), 3, torch.float32)
    ref = ref_cpu.decode_attention(f64(q), f64(kc), f64(vc), slots, ctx, G)
    for P in (0, 64, 100):
        out = paged_decode_attention_blocks(put(q), put(kc), put(vc), bt.to(DEV), lens, G,
                                            block_size=bs, partition_tokens=P)
        _close(out, ref, f"decode P={P}")
    _close(batched_paged_decode_attention(put(q), put(kc), put(vc), st.to(DEV), lens, G), ref, "slots")
    q = randn((sum(q_lens), G * KVH, D), 4, torch.float32)
    cu = torch.tensor([0] + list(np.cumsum(q_lens)), dtype=torch.int32, device=DEV)
    ref = ref_cpu.mq_attention(f64(q), f64(kc), f64(vc), slots, q_lens, G)
    for P in (0, 128):
        out = paged_mq_attention(put(q), put(kc), put(vc), bt.to(DEV), cu, lens, G, block_size=bs,
                                 max_q_len=max(q_lens), partition_tokens=P)
        _close(out, ref, f"multi-query P={P}")


def test_bad_block_ids_are_skipped_and_counted_per_row(hip):
    """One sequence, 3 queries of 4 heads over 40 keys of which block 1 (keys 16..31) is bad:
    every (query, head) that sees key 16 counts once, and attends to the other keys."""
    from dispec_amd.engine.hip_attn import paged_mq_attention
    bs, KVH, D, G = 16, 1, 64, 4
    kc, vc = (randn((64, KVH, D), s, torch.float32) for s in (5, 6))
    q = randn((3, G, D), 7, torch.float32)
    err = torch.zeros(1, dtype=torch.int32, device=DEV)
    out = paged_mq_attention(q.to(DEV), kc.to(DEV), vc.to(DEV),
                             torch.tensor([[2, 77, 1]], dtype=torch.int32, device=DEV),
                             torch.tensor([0, 3], dtype=torch.int32, device=DEV),
                             torch.tensor([40], dtype=torch.int32, device=DEV), G, block_size=bs,
                             max_q_len=3, max_ctx=48, err=err)
    good = np.r_[np.arange(32, 48), np.arange(16, 24)]
    ref = ref_cpu.mq_attention(f64(q), f64(kc), f64(vc), [good], [3], G)
    _close(out, ref, "bad block")
    assert int(err.item()) == 3 * G
