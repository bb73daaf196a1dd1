"""The ragged launch's size on 256 CUs (what the library assumes without a GPU), and the rule that
chooses it on shapes that were timed on both launches."""

import pytest


@pytest.fixture(scope="module")
def lib():
    from dispec_amd import _lib
    if not _lib.LIB_PATH.exists():
        from dispec_amd.build import build
        build()
    return _lib.lib()


@pytest.mark.parametrize("D,per_cu", [(64, 3), (128, 2), (256, 1)])
def test_workers_are_the_workgroups_that_fit(lib, D, per_cu):
    """Every worker has two partials of 128 rows (values, maximum and sum) and a descriptor.  The
    kernel is compiled for `per_cu` workgroups of four waves a CU: more would wait for a second
    round behind the first one's equal shares."""
    for B, ql, ctx in ((25, 700, 3000), (1, 64, 64), (512, 5, 1000)):
        assert lib.dsp_paged_mq_ragged_workspace_bytes(B, 28, 4, D, ql, ctx) == \
            256 * per_cu * 4 * (2 * 128 * (D + 2) + 4)


# head shape, queries of each sequence (count x tokens), longest context; us on the grid / in shares
SLOWER = [
    ((14, 2, 64), [(31, 1), (1, 159)], 672, "20 / 26"),
    ((32, 8, 128), [(58, 1), (1, 148)], 1232, "52 / 93"),
    ((32, 8, 128), [(39, 1), (3, 152)], 2064, "62 / 101"),
    ((28, 4, 128), [(61, 1), (1, 111)], 784, "25 / 38"),
    ((32, 8, 128), [(56, 1), (2, 143)], 4928, "178 / 256"),
    ((28, 4, 64), [(39, 1), (3, 60)], 5440, "58 / 78"),
    ((16, 8, 128), [(64, 1), (3, 46)], 1680, "101 / 163"),
    ((16, 8, 128), [(1, 9), (2, 3)], 11360, "25 / 42"),
    ((32, 8, 128), [(4, 5)], 9024, "24 / 40"),
    ((32, 8, 64), [(10, 3), (9, 4)], 5664, "20 / 28"),
    ((16, 8, 256), [(32, 10)], 1500, "every second one"),
]
FASTER = [
    ((28, 4, 128), [(24, 1), (1, 700)], 2864, "117 / 58"),
    ((14, 2, 64), [(24, 1), (1, 700)], 3008, "46 / 31"),
    ((32, 8, 128), [(30, 1), (2, 1000)], 3008, "318 / 114"),
    ((28, 4, 128), [(32, 5)], 4000, "93 / 48"),
    ((12, 2, 128), [(64, 6)], 4000, "87 / 47"),
    ((32, 8, 128), [(24, 5)], 4000, "92 / 48"),
]


@pytest.mark.parametrize("shape,blocks,max_ctx,us", SLOWER + FASTER)
def test_the_choice_on_timed_shapes(lib, shape, blocks, max_ctx, us):
    from dispec_amd.engine.hip_attn import _prefer_ragged
    (Hq, KVH, D), n = shape, sum(c for c, _ in blocks)
    got = _prefer_ragged(sum(c * q for c, q in blocks), n, KVH, Hq // KVH, D,
                         max(q for _, q in blocks), -(-max_ctx // 16) * 16)
    assert got == ((shape, blocks, max_ctx, us) in FASTER), us


def test_up_to_16_rows_stay_on_the_grid(lib):
    from dispec_amd.engine.hip_attn import _prefer_ragged
    assert not _prefer_ragged(160, 32, 8, 2, 128, 5, 1 << 20)
    assert not _prefer_ragged(0, 0, 8, 2, 128, 5, 4096)
    assert not _prefer_ragged(5, 1, 8, 4, 96, 5, 1 << 20)      # no ragged kernel for the head
