"""Probabilities enter P.V with all 24 bits of fp32 on the kernels that hold them in fp32: decode by
slot tables in batches, 256-wide heads, decode groups above 8.  (A 16-bit cache's own outputs
hide the 17th bit, so the inputs here cancel down to it, or put the sum into a tail of keys
far below the largest.)"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SCALE = 0.5

# route -> (sequences, context, query tokens per sequence, G, head_dim, keyword arguments)
ROUTES = {
    "slots_64": (16, 1500, 1, 4, 64, {}),
    "slots_128": (16, 1500, 1, 7, 128, {}),
    "decode_group_unsplit": (2, 500, 1, 12, 128, {}),
    "decode_group_balanced": (2, 2000, 1, 12, 128, {}),
    "decode_group_partitions": (2, 2000, 1, 20, 64, dict(partition_tokens=1024)),
    "decode_wide_unsplit": (2, 500, 1, 4, 256, {}),
    "decode_wide_balanced": (2, 2000, 1, 16, 256, {}),
    "verify_wide": (2, 2000, 5, 3, 256, {}),
    "prefill_wide": (2, 2000, 100, 2, 256, {}),
    "ragged_wide": (2, 2000, 100, 2, 256, {}),
}


def _attend(route, q, kc, vc):
    """Every sequence reads the pool's first keys in order."""
    from dispec_amd import _lib
    from dispec_amd.engine import hip_attn
    B, ctx, ql, G, D, kw = ROUTES[route]
    lens = torch.full((B,), ctx, dtype=torch.int32, device=DEV)
    if route.startswith("slots"):
        st = torch.arange(ctx, dtype=torch.int32, device=DEV).repeat(B, 1)
        return hip_attn.batched_paged_decode_attention(q, kc, vc, st, lens, G, SCALE)
    bt = torch.arange(-(-ctx // 16), dtype=torch.int32, device=DEV).repeat(B, 1)
    if ql == 1:
        return hip_attn.paged_decode_attention_blocks(q, kc, vc, bt, lens, G, scale=SCALE,
                                                      max_ctx=ctx, **kw)
    cu = torch.arange(B + 1, dtype=torch.int32, device=DEV) * ql
    if route == "ragged_wide":
        L, out = _lib.lib(), torch.empty_like(q)
        need = L.dsp_paged_mq_ragged_workspace_bytes(B, G, 1, D, ql, ctx)
        ws = torch.empty(need // 4, dtype=torch.float32, device=DEV)
        _lib.check(L.dsp_paged_mq_attention_ragged(
            q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), kc.shape[0],
            kc.stride(0), kc.stride(1), bt.data_ptr(), bt.stride(0), 16, cu.data_ptr(),
            lens.data_ptr(), B, G, 1, D, SCALE, ql, ctx, ws.data_ptr(), need, out.data_ptr(),
            out.stride(0), out.stride(1), _lib.dtype_code(q.dtype), None, _lib.stream_of(q)), route)
        return out
    return hip_attn.paged_mq_attention(q, kc, vc, bt, cu, lens, G, scale=SCALE, max_q_len=ql,
                                       max_ctx=ctx, **kw)


@pytest.mark.parametrize("route", ROUTES)
def test_cancelling_sums_keep_24_bits(hip, route):
    """bf16.  Three keys carry values; in dimension d they are chosen for row d % rows so that
    p0 v0 + p1 v1 + p2 v2 cancels to about 2^-18 of its terms.  A score errs by the roundings of
    its exponent (below 2^-22 of p here) and of exp2 (2^-23), a sum of three by 2^-23: below 2^-21
    in all, of sum p |v|.  16 bits of p would err by 2^-17."""
    B, ctx, ql, G, D, _ = ROUTES[route]
    bf, f64 = torch.bfloat16, torch.float64
    g = torch.Generator().manual_seed(7)
    rows = ql * G
    q = torch.zeros((ql, G, D), dtype=f64)
    q[..., :2] = torch.rand((ql, G, 2), generator=g) * 3 - 1.5
    q[..., 2] = 4
    q = q.to(bf)
    kc = torch.zeros((-(-ctx // 16) * 16, D), dtype=bf)
    kc[1, 0], kc[2, 1], kc[3:, 2] = 2, 2, -8          # scores 0, q0, q1, then -16
    s = SCALE * (q.to(f64).view(rows, D) @ kc[:3].to(f64).t())
    p = s.exp()                                        # (rows, 3)
    vc = torch.zeros((kc.shape[0], D), dtype=bf)
    mine = torch.arange(D) % rows                      # the row that dimension d is chosen for
    pd = p[mine]
    vc[0] = 1
    vc[1] = (-pd[:, 0] / pd[:, 1]).to(bf)
    vc[2] = (-(pd[:, 0] + pd[:, 1] * vc[1].to(f64)) / pd[:, 2]).to(bf)
    seen = ctx - ql + 1 + torch.arange(ql).repeat_interleave(G)
    total = p.sum(1) + (seen - 3) * math.exp(-16)
    want = (pd * vc[:3].to(f64).t()).sum(1) / total[mine]
    size = (pd * vc[:3].to(f64).t().abs()).sum(1) / total[mine]
    got = _attend(route, q.repeat(B, 1, 1).to(DEV), kc[:, None].to(DEV), vc[:, None].to(DEV))
    got = got.to(f64).cpu().view(B, rows, D)[:, mine, torch.arange(D)]
    worst = float(((got - want).abs() / size).max())
    assert worst <= 2.0 ** -20, f"{route}: 2^{math.log2(worst):.2f}"


@pytest.mark.parametrize("route", ROUTES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gap", [9.0, 12.0, 15.0, 18.0])
def test_a_tail_below_a_sink_key_counts(hip, route, dtype, gap):
    """One key scores `gap` above all others; its value is 0, theirs 1.  The result is the tail's
    share, n e^-gap / (1 + n e^-gap), rounded to the cache's type (half a unit in the last of 8
    or 11 bits: 2^-8 or 2^-11 of it, 2^-25 at fp16's end), after sums of n equal terms in fp32 (n
    2^-24)."""
    B, ctx, ql, G, D, _ = ROUTES[route]
    kc = torch.zeros((-(-ctx // 16) * 16, 1, D), dtype=dtype, device=DEV)
    vc = torch.ones_like(kc)
    kc[0, 0, 1], vc[0] = 2 * gap, 0
    q = torch.zeros((B * ql, G, D), dtype=dtype, device=DEV)
    q[..., 1] = 1
    got = _attend(route, q, kc, vc).double().cpu().view(B, ql, G * D)
    n = (ctx - ql + torch.arange(ql)).double()[None, :, None]
    want = n * math.exp(-gap) / (1 + n * math.exp(-gap))
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = want * (half + ctx * 2.0 ** -24) + (2.0 ** -25 if dtype == torch.float16 else 0)
    assert bool(((got - want).abs() <= bound).all()), \
        f"{route}: {float(((got - want).abs() / want).max()):.3g} of the result off"
