"""Infinities and NaN in attention inputs reach the rows that attend to them and no others, on the
kernels that hold probabilities in fp32 (fp32 caches, 256-wide heads, decode groups above 8, slot
tables) and on the ragged launch."""

import numpy as np
import pytest
import torch

from oracle import ref_cpu
from tests._util import f64, gen, randn

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


# ---- ids outside the cache: no key of theirs is read, not even the pool's slot 0
P_ERR = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


def _close(got, ref, vmax, dtype, what):
    """The output's rounding (half a unit in its last place, at most 2 P_ERR of it) and, where the
    kernel rounds probabilities to 16 bits, P_ERR of each: of max |v| at most."""
    err = np.abs(f64(got) - ref) - 2 * P_ERR[dtype] * np.abs(ref)
    assert np.isfinite(err).all() and err.max() <= P_ERR[dtype] * vmax, \
        f"{what}: {err.max():.3g} over {P_ERR[dtype] * vmax:.3g}"


def _ragged(q, kc, vc, bt, cu, lens, G, max_q, max_ctx, err=None, bs=16):
    from dispec_amd import _lib
    L, out = _lib.lib(), torch.empty_like(q)
    (S, KVH, D), B = kc.shape, lens.numel()
    need = L.dsp_paged_mq_ragged_workspace_bytes(B, G * KVH, KVH, D, max_q, max_ctx)
    ws = torch.full((need // 4,), float("nan"), device=DEV)
    _lib.check(L.dsp_paged_mq_attention_ragged(
        q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), S, kc.stride(0),
        kc.stride(1), bt.data_ptr(), bt.stride(0), bs, cu.data_ptr(), lens.data_ptr(), B, G * KVH,
        KVH, D, D ** -0.5, max_q, max_ctx, ws.data_ptr(), need, out.data_ptr(), out.stride(0),
        out.stride(1), _lib.dtype_code(q.dtype), _lib.ptr(err), _lib.stream_of(q)), "ragged")
    return out


def _spoiled(ctx, KVH, D, dtype, bad, seed=11):
    """A pool whose block 0 is infinite and NaN, tables that never name it, the slots of every
    sequence's keys in good blocks, and the table with ids outside the pool at `bad` = [(sequence,
    block)]."""
    bs = 16
    need = [-(-n // bs) for n in ctx]
    NB = sum(need) + 1
    perm = (1 + torch.randperm(NB - 1, generator=gen(seed))).int()
    kc, vc = (randn((NB * bs, KVH, D), seed + i, dtype).to(DEV) for i in (1, 2))
    kc[:bs], vc[:8], vc[8:bs] = float("nan"), float("inf"), float("nan")
    bt = torch.zeros((len(ctx), max(need)), dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        bt[b, :n] = perm[at:at + n]
        at += n
    keys = [(bt[b].long()[torch.arange(n) // bs] * bs + torch.arange(n) % bs).numpy()
            for b, n in enumerate(ctx)]
    for i, (b, j) in enumerate(bad):
        bt[b, j] = (NB, -1, 2 ** 30)[i % 3]
        keys[b][j * bs:(j + 1) * bs] = -1
    return kc, vc, bt.to(DEV), [k[k >= 0] for k in keys]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("G,KVH,D", [(12, 2, 128), (9, 1, 64), (12, 1, 32), (4, 2, 256), (17, 1, 256)])
@pytest.mark.parametrize("ctx,P", [([300, 77, 33], 0), ([1300, 2000, 40], 0), ([1300, 700, 40], 256)])
def test_decode_skips_bad_blocks(hip, dtype, G, KVH, D, ctx, P):
    from dispec_amd.engine.hip_attn import paged_decode_attention_blocks
    bad = [(0, 0), (0, 5), (0, 18), (1, 1), (1, 4), (2, 2)]
    kc, vc, bt, keys = _spoiled(ctx, KVH, D, dtype, bad)
    q = randn((3, G * KVH, D), 5, dtype).to(DEV)
    out = paged_decode_attention_blocks(q, kc, vc, bt, _i32(ctx), G, max_ctx=max(ctx),
                                        partition_tokens=P)
    ref = ref_cpu.decode_attention(f64(q), f64(kc), f64(vc), keys, [len(k) for k in keys], G)
    _close(out, ref, 6, dtype, f"G={G} D={D} {ctx} P={P}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("G,KVH,D", [(7, 2, 128), (7, 2, 64), (1, 4, 32)])
def test_slot_decode_skips_bad_slots(hip, dtype, G, KVH, D):
    from dispec_amd.engine.hip_attn import batched_paged_decode_attention
    ctx = [1500, 40, 33, 16] + [900] * 12
    kc, vc, bt, keys = _spoiled(ctx, KVH, D, dtype, [])
    st = torch.zeros((16, max(ctx)), dtype=torch.int32)
    for b, k in enumerate(keys):
        st[b, :len(k)] = torch.from_numpy(k).int()
        for i, j in enumerate(sorted({0, 31, 32, len(k) // 2, len(k) - 1} & set(range(len(k))))):
            st[b, j] = (kc.shape[0], -1, 2 ** 31 - 1)[i % 3]
        keys[b] = k[(st[b, :len(k)] >= 0).numpy() & (st[b, :len(k)] < kc.shape[0]).numpy()]
    q = randn((16, G * KVH, D), 5, dtype).to(DEV)
    out = batched_paged_decode_attention(q, kc, vc, st.to(DEV), _i32(ctx), G)
    ref = ref_cpu.decode_attention(f64(q), f64(kc), f64(vc), keys, [len(k) for k in keys], G)
    _close(out, ref, 6, dtype, f"G={G} D={D}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form,D", [("grid", 256), ("ragged", 64), ("ragged", 128), ("ragged", 256)])
@pytest.mark.parametrize("q_lens", [[3, 1, 2], [70, 1, 9]])
def test_multi_query_skips_bad_blocks(hip, dtype, form, D, q_lens):
    """16-row and 128-row tiles (G 3), the grid and the equal shares; no bad block holds a query."""
    from dispec_amd.engine.hip_attn import paged_mq_attention
    ctx, G, KVH = [1000, 200, 63], 3, 2
    kc, vc, bt, keys = _spoiled(ctx, KVH, D, dtype, [(0, 0), (0, 5), (0, 30), (1, 2), (2, 1)])
    q = randn((sum(q_lens), G * KVH, D), 5, dtype).to(DEV)
    cu = _i32([0] + list(np.cumsum(q_lens)))
    if form == "ragged":
        err = _i32([0])
        out = _ragged(q, kc, vc, bt, cu, _i32(ctx), G, max(q_lens), 1008, err)
        assert int(err.item()) > 0
    else:
        out = paged_mq_attention(q, kc, vc, bt, cu, _i32(ctx), G, max_q_len=max(q_lens))
    ref = ref_cpu.mq_attention(f64(q), f64(kc), f64(vc), keys, q_lens, G)
    _close(out, ref, 6, dtype, f"{form} D={D} {q_lens}")



# ---- infinities and NaN in V of keys that every row sees
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form,G,KVH,D,q_lens,ctx", [
    ("slots", 7, 2, 64, [1] * 16, [1100] * 15 + [40]), ("slots", 3, 2, 128, [1] * 16, [1100] * 16),
    ("decode", 12, 2, 128, [1, 1], [300, 77]), ("decode", 12, 2, 128, [1, 1], [2000, 77]),
    ("decode", 4, 2, 256, [1, 1], [300, 77]), ("decode", 4, 2, 256, [1, 1], [2000, 77]),
    ("multi", 3, 2, 256, [5, 2], [900, 77]), ("multi", 3, 2, 256, [50, 2], [900, 77]),
    ("ragged", 3, 2, 64, [5, 2], [900, 77]), ("ragged", 3, 2, 128, [5, 2], [900, 77]),
    ("ragged", 3, 2, 256, [50, 2], [900, 77])])
def test_infinite_values_stay_infinite(hip, dtype, form, G, KVH, D, q_lens, ctx):
    """inf times a row's probability is inf, whatever the split of the probability into operands:
    values at a sequence's keys 0, 20 and, for decode, the last."""
    from dispec_amd.engine.hip_attn import (batched_paged_decode_attention,
                                            paged_decode_attention_blocks, paged_mq_attention)
    kc, vc, bt, keys = _spoiled(ctx, KVH, D, dtype, [])
    clean = vc.clone()
    for k, n in zip(keys, ctx):
        at = torch.from_numpy(k)
        vc[at[0], 0, 3], vc[at[20], 0, D - 1], vc[at[20], 1, 5] = float("inf"), -float("inf"), float("nan")
        clean[at[0], 0, 3], clean[at[20], 0, D - 1], clean[at[20], 1, 5] = 0, 0, 0
        if max(q_lens) == 1:
            vc[at[-1], 1, 7], clean[at[-1], 1, 7] = float("inf"), 0
    q = randn((sum(q_lens), G * KVH, D), 5, dtype).to(DEV)
    lens = _i32(ctx)
    if form == "slots":
        st = torch.zeros((len(ctx), max(ctx)), dtype=torch.int32)
        for b, k in enumerate(keys):
            st[b, :len(k)] = torch.from_numpy(k).int()
        out = batched_paged_decode_attention(q, kc, vc, st.to(DEV), lens, G)
    elif form == "decode":
        out = paged_decode_attention_blocks(q, kc, vc, bt, lens, G, max_ctx=max(ctx))
    else:
        cu = _i32([0] + list(np.cumsum(q_lens)))
        if form == "ragged":
            out = _ragged(q, kc, vc, bt, cu, lens, G, max(q_lens), bt.shape[1] * 16)
        else:
            out = paged_mq_attention(q, kc, vc, bt, cu, lens, G, max_q_len=max(q_lens))
    want = ref_cpu.mq_attention(f64(q), f64(kc), f64(clean), keys, q_lens, G)
    want[:, :G, 3], want[:, :G, D - 1], want[:, G:, 5] = np.inf, -np.inf, np.nan
    if max(q_lens) == 1:
        want[:, G:, 7] = np.inf
    got, odd = f64(out), ~np.isfinite(want)
    assert np.array_equal(got[odd], want[odd], equal_nan=True)
    assert np.abs(got[~odd] - want[~odd]).max() <= 2 * P_ERR[dtype] * 6

# ---- infinities and NaN in a token's V and K: only the rows that see the token get them
@pytest.mark.parametrize("form,dtype,D", [
    ("grid", torch.float32, 8), ("grid", torch.float32, 16), ("grid", torch.float32, 64),
    ("grid", torch.float32, 256), ("grid", torch.bfloat16, 256), ("grid", torch.float16, 256),
    ("ragged", torch.bfloat16, 64), ("ragged", torch.float16, 64), ("ragged", torch.bfloat16, 128),
    ("ragged", torch.float16, 128), ("ragged", torch.bfloat16, 256), ("ragged", torch.float16, 256)])
@pytest.mark.parametrize("q_lens,ctx", [([9, 1, 4], [300, 64, 4]), ([150, 70, 1], [900, 70, 129]),
                                        ([70, 3], [70, 1000])])
@pytest.mark.parametrize("G", [1, 3])
def test_a_token_spoils_the_rows_that_see_it(hip, form, dtype, D, q_lens, ctx, G):
    """Two of each sequence's new tokens (its only one where it has one) hold NaN, inf and -inf in
    some dims of V: the later rows have them there, the earlier ones are as if they were zeros."""
    from dispec_amd.engine.hip_attn import paged_mq_attention
    KVH, bs = 2, 16
    kc, vc, bt, keys = _spoiled(ctx, KVH, D, dtype, [])
    clean = vc.clone()
    first = {}                          # row -> tokens of its sequence that are spoilt and seen
    at = 0
    for n, c, slots in zip(q_lens, ctx, keys):
        spoilt = sorted({n // 2, n - 1})
        for i in spoilt:
            s = int(slots[c - n + i])
            vc[s, 0, 1], vc[s, 0, 3], vc[s, 0, D - 1] = float("nan"), float("inf"), -float("inf")
            vc[s, 1, 2] = float("inf") if i == n - 1 else -float("inf")
            vc[s, 1, 0] = float("inf")
            clean[s, 0, [1, 3, D - 1]], clean[s, 1, :3:2] = 0, 0
        for i in range(n):
            first[at + i] = [t for t in spoilt if t <= i]
        at += n
    q = randn((sum(q_lens), G * KVH, D), 5, dtype).to(DEV)
    cu = _i32([0] + list(np.cumsum(q_lens)))
    if form == "ragged":
        out = _ragged(q, kc, vc, bt, cu, _i32(ctx), G, max(q_lens), bt.shape[1] * bs)
    else:
        out = paged_mq_attention(q, kc, vc, bt, cu, _i32(ctx), G, max_q_len=max(q_lens))
    want = ref_cpu.mq_attention(f64(q), f64(kc), f64(clean), keys, q_lens, G)
    inf = np.inf
    ends = {a - 1 for a in np.cumsum(q_lens)}
    for t, seen in first.items():
        if seen:
            want[t, :G, 1], want[t, :G, 3], want[t, :G, D - 1] = np.nan, inf, -inf
            want[t, G:, 0] = inf
            # the sequence's last token has inf where an earlier one has -inf
            want[t, G:, 2] = -inf if t not in ends else (inf if len(seen) == 1 else np.nan)
    got = f64(out)
    odd = ~np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[odd & ~np.isnan(want)], want[odd & ~np.isnan(want)])
    err = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11 if dtype == torch.float16 else 1e-6
    assert np.abs(got[~odd] - want[~odd]).max() <= err * 6
