"""Ragged batches of long query blocks in equal shares (dsp_paged_mq_attention_ragged) against
the grid of fixed partitions that serves them otherwise, and the rule that chooses.

Bound: both round fp32 results to 16 bits after summing keys in other chunks and orders, with
probabilities rounded to 16 bits against different running maxima: each weight errs by 2^-9
(bf16) or 2^-12 (fp16) of itself, so a row moves by at most that times sum p |v| <= max |v| on
either side, plus one unit in the last place of the output (2^-7, 2^-10 of the value)."""

import numpy as np
import pytest
import torch

from tests._util import randn, random_block_tables

pytestmark = pytest.mark.gpu
DEV = "cuda"
P_ERR = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


def _run(q_lens, ctx, G, KVH, D, dtype, bs=16, max_q=None, spoil=None, strided=False, max_ctx=None):
    """(ragged, grid) outputs and error counts."""
    from dispec_amd import _lib
    seed = len(q_lens) + G + D
    NB = sum(-(-max(n, 1) // bs) for n in ctx) + 2
    tables = random_block_tables(NB, ctx, bs, seed)
    width = max(-(-max(ctx) // bs), 1)
    bt = torch.zeros((len(ctx), width), dtype=torch.int32)
    for i, t in enumerate(tables):
        bt[i, :len(t)] = torch.tensor(t, dtype=torch.int32)
    max_ctx = max_ctx or width * bs
    lens = torch.tensor(ctx, dtype=torch.int32)
    if spoil:
        spoil(bt, lens)
    kc, vc = randn((NB * bs, KVH, D), 1, dtype).to(DEV), randn((NB * bs, KVH, D), 2, dtype).to(DEV)
    T, Hq = sum(q_lens), G * KVH
    q = randn((T, Hq, D), 3, dtype).to(DEV)
    if strided:   # a view of a fused projection: rows 8 elements longer
        buf = torch.zeros((T, Hq * D + 8), dtype=dtype, device=DEV)
        buf[:, :Hq * D] = q.view(T, -1)
        q = buf[:, :Hq * D].unflatten(1, (Hq, D))
    cu = torch.tensor([0] + list(np.cumsum(q_lens)), dtype=torch.int32, device=DEV)
    bt, lens = bt.to(DEV), lens.to(DEV)
    max_q = max_q or max(q_lens)
    L, res = _lib.lib(), []
    for ragged in (True, False):
        out = torch.full((T, Hq, D), 7.0, dtype=dtype, device=DEV)
        err = torch.zeros(1, dtype=torch.int32, device=DEV)
        size = L.dsp_paged_mq_ragged_workspace_bytes if ragged else L.dsp_paged_mq_workspace_bytes
        need = size(len(ctx), Hq, KVH, D, max_q, max_ctx, *(() if ragged else (0,)))
        ws = torch.full((need // 4 + 1,), float("nan"), dtype=torch.float32, device=DEV)
        fn = L.dsp_paged_mq_attention_ragged if ragged else L.dsp_paged_mq_attention
        _lib.check(fn(q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(),
                      NB * bs, kc.stride(0), kc.stride(1), bt.data_ptr(), bt.stride(0), bs,
                      cu.data_ptr(), lens.data_ptr(), len(ctx), Hq, KVH, D, D ** -0.5, max_q,
                      max_ctx, *(() if ragged else (0,)), ws.data_ptr(), need, out.data_ptr(),
                      out.stride(0), out.stride(1), _lib.dtype_code(dtype), err.data_ptr(),
                      _lib.stream_of(q)), "mq")
        res.append((out.float(), int(err.item())))
    v = float(vc.float().abs().max())
    bound = 2 * P_ERR[dtype] * v + 4 * P_ERR[dtype] * res[1][0].abs()
    worst = float(((res[0][0] - res[1][0]).abs() - bound).max())
    assert worst <= 0, f"{q_lens[:5]}.. {ctx[:5]}.. G={G} KVH={KVH} D={D}: {worst:.3g} over"
    return res[0][1], res[1][1]


BATCHES = [  # query lengths, context lengths
    ([1] * 24 + [700], [100 + 90 * i for i in range(24)] + [1501]),
    ([130], [130]), ([64, 1], [64, 5000]), ([200, 0, 1, 333], [200, 0, 1, 900]),
    ([1] * 70 + [150, 1, 1], list(range(1, 71)) + [2000, 63, 65]),       # two groups of lanes
    ([128, 129, 127, 256], [128, 193, 4000, 256]),
    ([1, 2, 3, 1000], [64, 128, 129, 1000]),
]


@pytest.mark.parametrize("q_lens,ctx", BATCHES)
@pytest.mark.parametrize("G,KVH,D", [(1, 2, 128), (2, 8, 128), (7, 2, 64), (7, 4, 128),
                                     (3, 2, 256), (8, 1, 64), (5, 3, 128)])
def test_ragged_is_the_grid(hip, q_lens, ctx, G, KVH, D):
    assert _run(q_lens, ctx, G, KVH, D, torch.bfloat16) == (0, 0)


@pytest.mark.parametrize("q_lens,ctx", [
    ([5] * 33, [200 + 61 * i for i in range(33)]), ([1, 9, 3], [1, 9, 4000]),
    ([9] * 70, list(range(9, 79))), ([18, 2, 0, 17], [18, 65, 0, 3000])])
@pytest.mark.parametrize("G,KVH,D", [(2, 8, 128), (7, 4, 128), (7, 2, 64), (3, 2, 256)])
def test_short_blocks_are_the_16_row_tiles(hip, q_lens, ctx, G, KVH, D):
    """Below 128 rows (one tile, its last chunk cut inside a block)."""
    assert _run(q_lens, ctx, G, KVH, D, torch.bfloat16) == (0, 0)
    assert _run(q_lens, ctx, G, KVH, D, torch.float16, strided=True) == (0, 0)


def test_stale_rows_past_the_context_are_not_read(hip):
    """Slots of a sequence's last block past its context may hold anything, NaN too: one
    sequence's blocks are 0..n, its context ends inside the last."""
    from dispec_amd import _lib
    G, KVH, D, ctx, bs = 5, 2, 128, 200, 16
    kc, vc = (randn((256, KVH, D), i, torch.bfloat16).to(DEV) for i in (1, 2))
    kc[ctx:], vc[ctx:] = float("nan"), float("nan")
    q = randn((5, G * KVH, D), 3, torch.bfloat16).to(DEV)
    bt = torch.arange(16, dtype=torch.int32, device=DEV).view(1, 16)
    cu, lens = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in ([0, 5], [ctx]))
    L = _lib.lib()
    need = L.dsp_paged_mq_ragged_workspace_bytes(1, G * KVH, KVH, D, 5, 256)
    ws, out = torch.empty(need // 4, device=DEV), torch.empty_like(q)
    _lib.check(L.dsp_paged_mq_attention_ragged(
        q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), 256, kc.stride(0),
        kc.stride(1), bt.data_ptr(), 16, bs, cu.data_ptr(), lens.data_ptr(), 1, G * KVH, KVH, D,
        D ** -0.5, 5, 256, ws.data_ptr(), need, out.data_ptr(), out.stride(0), out.stride(1),
        _lib.dtype_code(q.dtype), None, _lib.stream_of(q)), "ragged")
    assert bool(torch.isfinite(out).all())


@pytest.mark.parametrize("bs", [16, 32, 128])
def test_block_sizes_dtype_and_strides(hip, bs):
    assert _run(*BATCHES[0], 4, 2, 128, torch.float16, bs=bs, strided=True) == (0, 0)
    assert _run(*BATCHES[3], 6, 2, 64, torch.float16, bs=bs, strided=True) == (0, 0)


def test_bad_lengths_are_counted_once_and_zeroed(hip):
    def spoil(bt, lens):
        lens[1], lens[3] = 3000, 100     # past max_ctx; shorter than its 333 queries
    assert _run([200, 7, 1, 333], [200, 50, 1, 900], 4, 2, 128, torch.bfloat16, spoil=spoil) == (2, 2)


def test_query_block_longer_than_max_q_len(hip):
    """The first max_q_len rows are computed (whole 128-row tiles of them on the grid)."""
    assert _run([128, 1, 256], [128, 700, 300], 1, 2, 128, torch.bfloat16, max_q=256) == (0, 0)


def test_bad_block_ids_are_counted(hip):
    def spoil(bt, lens):
        bt[0, 1] = 10 ** 6
    got, want = _run([1, 300], [60, 300], 4, 2, 256, torch.bfloat16, spoil=spoil)
    assert got > 0 and want > 0


def test_the_rule_and_its_refusals(hip, monkeypatch):
    """Ragged batches take the equal shares, uniform ones and explicit partitions the grid, and
    a pool the ragged launch refuses (256-wide heads, half a block at its end) the grid."""
    from dispec_amd import _lib
    from dispec_amd.engine import hip_attn
    took = []

    class Spy:
        def __getattr__(self, name):
            fn = getattr(real, name)
            if not name.startswith("dsp_paged_mq_attention"):
                return fn
            return lambda *a: (lambda st: (took.append((name, st)), st)[1])(fn(*a))

    real = _lib.calls()
    monkeypatch.setattr(_lib, "calls", lambda: Spy())

    def call(q_lens, ctx, G=4, KVH=8, D=128, slots=None, **kw):
        took.clear()
        n = len(ctx)
        bt = torch.arange(n * 64, dtype=torch.int32, device=DEV).view(n, 64) % 64
        kc = torch.zeros((slots or 1024, KVH, D), dtype=torch.bfloat16, device=DEV)
        q = torch.zeros((sum(q_lens), G * KVH, D), dtype=torch.bfloat16, device=DEV)
        cu = torch.tensor([0] + list(np.cumsum(q_lens)), dtype=torch.int32, device=DEV)
        hip_attn.paged_mq_attention(q, kc, kc, bt, cu, torch.tensor(ctx, dtype=torch.int32,
                                    device=DEV), G, max_q_len=max(q_lens), max_ctx=1024, **kw)
        torch.cuda.synchronize()
        return [(n.replace("dsp_paged_mq_attention", ""), st) for n, st in took]

    mixed = ([1] * 20 + [512], [600] * 20 + [1000])
    assert call(*mixed) == [("_ragged", 0)]
    assert call(*mixed, partition_tokens=256) == [("", 0)]
    assert call([256] * 4, [1000] * 4) == [("", 0)]
    # verify: above 16 rows and from 256K keys, on whole blocks of the pool
    assert call([5] * 32, [1000] * 32) == [("_ragged", 0)]
    assert call([5] * 31, [1000] * 31) == [("", 0)]
    assert call([4] * 32, [1000] * 32) == [("", 0)]
    assert call([5] * 32, [1000] * 32, slots=1032) == [("", 0)]
    assert call(*mixed, G=2, D=256, slots=1016) == [("_ragged", _lib.DSP_EUNSUPPORTED), ("", 0)]


# ---- a lost, doubled or misplaced chunk shows whatever the length of the row
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("q_lens,ctx,G,KVH,D", [
    *[(*b, 7, 2, 128) for b in BATCHES], *[(*b, 3, 3, 64) for b in BATCHES[:1] + BATCHES[3:5]],
    (*BATCHES[0], 4, 2, 256), ([5] * 33, [200 + 61 * i for i in range(33)], 7, 4, 128),
    ([9, 18, 1], [4000, 18, 3000], 7, 2, 64),
    ([1] * 24 + [1300], [100 + 90 * i for i in range(24)] + [1377], 7, 2, 128),   # 72 tiles
    ([1, 7900, 3], [5000, 8000, 64], 7, 1, 128),                                  # 432 tiles
    ([4000, 1], [4096, 2000], 1, 2, 64)])
def test_every_chunk_counts_once(hip, dtype, q_lens, ctx, G, KVH, D):
    """All scores 0, V the number of the key's chunk as a unit vector: output d of a row is the
    share of its keys that lie in chunk d (turned by the KV head), to half a unit in the last
    place of the type and, against a row sum of 1, that of a probability."""
    from dispec_amd import _lib
    bs, B, T, Hq = 16, len(ctx), sum(q_lens), G * KVH
    need = [-(-c // bs) for c in ctx]
    perm = torch.randperm(sum(need) + 1, generator=torch.Generator().manual_seed(4)).int()
    bt = torch.zeros((B, max(need)), dtype=torch.int32)
    vc = torch.zeros(((sum(need) + 1) * bs, KVH, D), dtype=dtype)
    at = 0
    for b, n in enumerate(need):
        bt[b, :n] = perm[at:at + n]
        at += n
        j = torch.arange(ctx[b])
        for h in range(KVH):
            vc[bt[b].long()[j // bs] * bs + j % bs, h, (j // 64 + 17 * h) % D] = 1
    assert max(ctx) <= 64 * D
    q, kc = torch.zeros((T, Hq, D), dtype=dtype, device=DEV), torch.zeros_like(vc).to(DEV)
    vc, bt = vc.to(DEV), bt.to(DEV)
    cu, lens = (torch.tensor(x, dtype=torch.int32, device=DEV)
                for x in ([0] + list(np.cumsum(q_lens)), ctx))
    L, mq, mc = _lib.lib(), max(q_lens), bt.shape[1] * bs
    size = L.dsp_paged_mq_ragged_workspace_bytes(B, Hq, KVH, D, mq, mc)
    ws = torch.full((size // 4,), float("nan"), device=DEV)
    out = torch.full_like(q, 7.0)
    _lib.check(L.dsp_paged_mq_attention_ragged(
        q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), kc.shape[0],
        kc.stride(0), kc.stride(1), bt.data_ptr(), bt.stride(0), bs, cu.data_ptr(), lens.data_ptr(),
        B, Hq, KVH, D, 1.0, mq, mc, ws.data_ptr(), size, out.data_ptr(), out.stride(0),
        out.stride(1), _lib.dtype_code(dtype), None, _lib.stream_of(q)), "ragged")
    seen = torch.cat([torch.arange(c - n + 1, c + 1) for n, c in zip(q_lens, ctx)]).to(DEV)
    chunk = (seen[:, None] - 64 * torch.arange(D, device=DEV)).clamp(0, 64)
    want = torch.stack([chunk.roll(17 * h, 1) for h in range(KVH)], 1).double() / seen[:, None, None]
    want = want.repeat_interleave(G, 1)
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert bool(((out.double() - want).abs() <= want * (2 * half) + 2.0 ** -25).all())


@pytest.mark.parametrize("q_lens,ctx", [([1] * 24 + [700], [100 + 90 * i for i in range(24)] + [1501]),
                                        ([5] * 40, [3000] * 40)])
def test_a_callers_workspace_serves_the_ragged_launch(hip, q_lens, ctx):
    """mq_workspace covers it, and a call that is handed the buffer allocates nothing."""
    from dispec_amd.engine.hip_attn import _prefer_ragged, mq_workspace, paged_mq_attention
    G, KVH, D, bs = 7, 4, 128, 16
    B, T, mq = len(ctx), sum(q_lens), max(q_lens)
    width = -(-max(ctx) // bs)
    assert _prefer_ragged(T, B, KVH, G, D, mq, width * bs)
    kc, vc = (randn((width * bs, KVH, D), s, torch.bfloat16).to(DEV) for s in (1, 2))
    bt = torch.arange(width, dtype=torch.int32, device=DEV).repeat(B, 1)
    q = randn((T, G * KVH, D), 3, torch.bfloat16).to(DEV)
    cu, lens = (torch.tensor(x, dtype=torch.int32, device=DEV)
                for x in ([0] + list(np.cumsum(q_lens)), ctx))
    ws = mq_workspace(B, G * KVH, KVH, D, mq, width * bs, DEV)
    out, want = torch.empty_like(q), torch.empty_like(q)

    def call(o, w):
        paged_mq_attention(q, kc, vc, bt, cu, lens, G, block_size=bs, max_q_len=mq,
                           max_ctx=width * bs, out=o, workspace=w)

    call(want, None)
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    call(out, ws)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
    assert torch.equal(out, want)
    small = torch.empty(16, device=DEV)     # too small: the call brings its own
    out.zero_()
    call(out, small)
    assert torch.equal(out, want)
