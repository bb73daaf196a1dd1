"""All dense layer maps of a prompt in one launch (dsp_kv_map_group, what CrossModelKVMap.map
and map_into run) against the same maps applied one layer at a time, bit for bit; and the
vector form of the RoPE kernel against torch's elementwise ops.

Both sides round at the same points and accumulate K in the same 32-wide steps, so no
tolerance is needed."""

from types import SimpleNamespace

import pytest
import torch

from tests._util import gen

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _map(n_src, n_tgt, H, D, seed, fan=lambda i: 1, low_rank=()):
    from dispec_amd.kv.transfer import CrossModelKVMap, LayerMap
    g, kv = gen(seed), H * D

    def one(i):
        k = kv * fan(i)
        w, b = torch.randn(k, kv, generator=g) * k ** -0.5, torch.randn(kv, generator=g) * 0.1
        layers = tuple((i + j) % n_src for j in range(fan(i)))
        if i in low_rank:
            return LayerMap(layers, b, factors=(w[:, :64].contiguous(),
                                                torch.randn(64, kv, generator=g) / 8))
        return LayerMap(layers, b, weight=w)

    def cfg(n):
        return SimpleNamespace(num_key_value_heads=H, head_dim=D, vocab_size=7, num_hidden_layers=n)

    return CrossModelKVMap([one(i) for i in range(n_tgt)], [one(i) for i in range(n_tgt)],
                           cfg(n_src), cfg(n_tgt)).to(DEV, torch.bfloat16)


def _inputs(n_src, T, H, D, seed):
    g = gen(seed)
    k, v = (torch.randn((n_src, T, H, D), generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    ang = torch.rand((T, D), generator=g) * 6.28
    return k, v, (ang.cos().to(DEV), ang.sin().to(DEV))


def _one_by_one(m, k, v, src_rope, tgt_rope):
    """The layer loop: one map launch per layer, then the rotation."""
    from dispec_amd.kv.transfer import _rope
    content = _rope(k, *src_rope, direction=-1, out_dtype=torch.bfloat16)
    return (m._apply(content, m.keys, True, rope=tgt_rope), m._apply(v, m.values, True))


CASES = [  # tokens, heads, head_dim, source layers, target layers
    (1, 8, 128, 3, 4), (100, 8, 128, 3, 40), (127, 2, 64, 2, 3), (128, 4, 128, 2, 3),
    (129, 8, 128, 2, 5), (256, 8, 128, 4, 36), (257, 8, 64, 2, 3), (300, 1, 64, 2, 90),
    (700, 8, 128, 5, 6), (333, 4, 32, 2, 3),   # head_dim 32: no fused rotation, layer loop
]


@pytest.mark.parametrize("T,H,D,n_src,n_tgt", CASES)
@pytest.mark.parametrize("form", ["one", "two", "mixed"])
def test_map_is_the_layer_loop(hip, T, H, D, n_src, n_tgt, form):
    fan = {"one": lambda i: 1, "two": lambda i: 2, "mixed": lambda i: 1 + i % 2}[form]
    m = _map(n_src, n_tgt, H, D, 11, fan, low_rank=(1,) if form == "mixed" else ())
    k, v, rope = _inputs(n_src, T, H, D, 12)
    tgt = (rope[1].clone(), rope[0].clone())
    keys, vals = m.map(k, v, rope, tgt)
    want = _one_by_one(m, k, v, rope, tgt)
    assert torch.equal(keys, want[0]) and torch.equal(vals, want[1])


@pytest.mark.parametrize("T,H,D,n_src,n_tgt", [c for c in CASES if c[3] < 5])
@pytest.mark.parametrize("bs", [1, 16, 64])
def test_map_into_is_map_and_import(hip, T, H, D, n_src, n_tgt, bs):
    from dispec_amd.kv.paged_cache import PagedKVCache
    m = _map(n_src, n_tgt, H, D, 21, lambda i: 1 + (i == 0))
    k, v, rope = _inputs(n_src, T, H, D, 22)
    need = -(-T // bs)
    ids = torch.randperm(need + 3, generator=gen(23))[:need].tolist()
    got, want = (PagedKVCache(n_tgt, need + 3, bs, H, D, dtype=torch.bfloat16) for _ in range(2))
    for c in (got, want):
        c.key.fill_(3.0)
        c.value.fill_(-3.0)
    m.map_into(k, v, rope, rope, got, ids)
    want.import_contiguous(ids, *_one_by_one(m, k, v, rope, rope))
    got.check_errors()
    assert torch.equal(got.key, want.key) and torch.equal(got.value, want.value)


@pytest.mark.parametrize("L,T,H,D", [(1, 1, 1, 16), (3, 257, 2, 64), (2, 33, 8, 128),
                                     (2, 19, 3, 256), (2, 40, 3, 48), (2, 17, 3, 24)])
@pytest.mark.parametrize("ti", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("to", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("direction", [-1, 1])
def test_rope_forms(hip, L, T, H, D, ti, to, direction):
    """D 24 takes the element form, the others the vector form; a layer stride off the
    16-byte grid takes the element form too.  Same fp32 products and sums as torch's ops."""
    from dispec_amd.kv.transfer import _rope
    g = gen(31)
    x = torch.randn((L, T, H, D), generator=g).to(DEV, ti)
    cos, sin = (torch.randn((T, D), generator=g).to(DEV) for _ in range(2))
    f = x.float()
    rot = torch.cat([-f[..., D // 2:], f[..., :D // 2]], dim=-1)
    want = f * cos[:, None] + direction * (rot * sin[:, None])
    assert torch.equal(_rope(x, cos, sin, direction, out_dtype=to), want.to(to))
    flat = torch.zeros(L * (T * H * D + 1), dtype=ti, device=DEV)
    odd = flat.as_strided((L, T, H, D), (T * H * D + 1, H * D, D, 1))
    odd.copy_(x)
    assert torch.equal(_rope(odd, cos, sin, direction, out_dtype=to), want.to(to))
