"""Decode by per-token slot tables on the balanced split (batches of 16 sequences and more)
against the VALU kernel that serves explicit partitions of the same tables.

Bound: each output is the 16-bit rounding of fp32 values the two kernels sum in different
orders from probabilities held to 2^-16 or better: one unit in the last place (2^-7 of the
value in bf16, 2^-10 in fp16) plus 2^-15 of the largest |v|."""

import pytest
import torch

from tests._util import gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"
RTOL = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


def _both(lens, G, KVH, D, dtype, seed, bad=()):
    """(balanced, VALU) outputs and error counts; slots in random order, padding entries of a
    row out of range.  bad: (sequence, position) whose slots are set out of range."""
    from dispec_amd import _lib
    S, B, W = sum(lens) + 5, len(lens), max(lens)
    perm = torch.randperm(S, generator=gen(seed)).int()
    st = torch.full((B, W), 2 ** 30, dtype=torch.int32)
    at = 0
    for i, n in enumerate(lens):
        st[i, :n] = perm[at:at + n]
        at += n
    for i, (b, j) in enumerate(bad):
        st[b, j] = (S, -1, 2 ** 31 - 1)[i % 3]
    q = randn((B, G * KVH, D), seed + 1, dtype).to(DEV)
    kc, vc = randn((S, KVH, D), seed + 2, dtype).to(DEV), randn((S, KVH, D), seed + 3, dtype).to(DEV)
    st, cl = st.to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV)
    L, res = _lib.lib(), []
    for P in (0, 128):
        out, err = torch.empty_like(q), torch.zeros(1, dtype=torch.int32, device=DEV)
        need = L.dsp_paged_decode_workspace_bytes(B, G * KVH, KVH, D, W, P)
        ws = torch.empty(need // 4 + 1, dtype=torch.float32, device=DEV)
        _lib.check(L.dsp_paged_decode(
            q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), S, kc.stride(0),
            kc.stride(1), None, 0, 16, st.data_ptr(), st.stride(0), cl.data_ptr(), B, G * KVH, KVH,
            D, D ** -0.5, W, P, ws.data_ptr(), ws.numel() * 4, out.data_ptr(), out.stride(0),
            out.stride(1), _lib.dtype_code(dtype), err.data_ptr(), _lib.stream_of(q)), "decode")
        res.append((out.float(), int(err.item())))
    bound = RTOL[dtype] * res[1][0].abs() + 2.0 ** -15 * vc.float().abs().max()
    worst = float(((res[0][0] - res[1][0]).abs() - bound).max())
    assert worst <= 0, f"{lens[:4]}.. G={G} KVH={KVH} D={D}: {worst:.3g} over the bound"
    return res[0][1], res[1][1]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("G,KVH,D", [(1, 8, 128), (7, 4, 128), (7, 2, 64), (8, 1, 32), (4, 3, 128)])
def test_slot_tables_on_the_balanced_split(hip, dtype, G, KVH, D):
    edges = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 129, 1000, 2047, 1025]
    assert _both(edges, G, KVH, D, dtype, 50 + D + G) == (0, 0)
    assert _both([1100] * 17, G, KVH, D, dtype, 60 + D + G) == (0, 0)


def test_bad_slots_are_skipped_and_counted_alike(hip):
    lens = [1500, 40] + [900] * 14
    bad = [(0, 0), (0, 31), (0, 32), (0, 1499), (1, 39), (1, 16), (5, 450), (15, 899)]
    got, want = _both(lens, 5, 4, 128, torch.bfloat16, 90, bad)
    assert got == want == len(bad) * 4        # once per slot and KV head


@pytest.mark.parametrize("off", [1, 100, 127])
@pytest.mark.parametrize("form", ["slots", "blocks"])
def test_table_entries_past_max_ctx_are_not_read(hip, off, form):
    """A table that is the last columns of a wider one: its last row ends where the buffer ends
    (here a whole 16 MiB allocation), so the window of entries read ahead has to stop at max_ctx
    and not at the row stride."""
    from dispec_amd import _lib
    B, KVH, G, D, S, stride, bs = 16, 1, 4, 64, 4096, 1 << 18, 16
    buf = torch.full((B, stride), 2 ** 30, dtype=torch.int32, device=DEV)
    per = 1 if form == "slots" else bs           # tokens an entry stands for
    width = stride - off
    max_ctx = width * per if form == "slots" else 3000 * bs
    table = buf[:, off:] if form == "slots" else buf[:, stride - 3000:]
    lens = [max_ctx - 3] + [700 + i for i in range(B - 2)] + [max_ctx]
    for b, n in enumerate(lens):
        n = -(-n // per)
        table[b, :n] = torch.randint(0, S // per, (n,), generator=gen(b)).int().to(DEV)
    q = randn((B, G * KVH, D), 1, torch.bfloat16).to(DEV)
    kc, vc = (randn((S, KVH, D), s, torch.bfloat16).to(DEV) for s in (2, 3))
    cl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    at, row = table.data_ptr(), table.stride(0)
    where = (None, 0, bs, at, row) if form == "slots" else (at, row, bs, None, 0)
    L, res = _lib.lib(), []
    for P in (0, 512):
        out, err = torch.empty_like(q), torch.zeros(1, dtype=torch.int32, device=DEV)
        need = L.dsp_paged_decode_workspace_bytes(B, G * KVH, KVH, D, max_ctx, P)
        ws = torch.empty(need // 4 + 1, dtype=torch.float32, device=DEV)
        _lib.check(L.dsp_paged_decode(
            q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), S, kc.stride(0),
            kc.stride(1), *where, cl.data_ptr(), B, G * KVH, KVH, D, D ** -0.5, max_ctx, P,
            ws.data_ptr(), ws.numel() * 4, out.data_ptr(), out.stride(0), out.stride(1),
            _lib.DSP_BF16, err.data_ptr(), _lib.stream_of(q)), "decode")
        assert int(err.item()) == 0
        res.append(out.float())
    bound = 2.0 ** -7 * res[1].abs() + 2.0 ** -8 * vc.float().abs().max()
    assert bool(((res[0] - res[1]).abs() <= bound).all())
