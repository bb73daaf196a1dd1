"""PagedKVCache.block_table hands out a table that any stream may read: its copy has ended on
return.  (The cache's own exports and imports, which stay on one stream, do not wait.)"""

import pytest
import torch

from dispec_amd.kv.paged_cache import PagedKVCache


@pytest.mark.parametrize("tables,width", [([[3, 1], [7]], None), ([[]], None), ([[5], [2]], 4)])
def test_block_table_copy_waits(tables, width, monkeypatch):
    cache = object.__new__(PagedKVCache)
    cache.key = torch.zeros(1)          # only its device is read
    seen = []
    to = torch.Tensor.to

    def spy(self, *args, **kw):
        seen.append((self.is_pinned(), kw.get("non_blocking", False)))
        return to(self, *args, **kw)

    monkeypatch.setattr(torch.Tensor, "to", spy)
    got = cache.block_table(tables, width)
    w = width or max(len(t) for t in tables) or 1
    assert got.dtype == torch.int32
    assert got.tolist() == [t + [0] * (w - len(t)) for t in tables]
    assert seen == [(False, False)]


def test_block_table_too_wide():
    cache = object.__new__(PagedKVCache)
    cache.key = torch.zeros(1)
    with pytest.raises(ValueError, match="sequence 1 has 3 blocks, table width 2"):
        cache.block_table([[1], [1, 2, 3]], 2)
