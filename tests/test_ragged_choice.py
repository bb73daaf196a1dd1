"""The ragged launch's size on 256 CUs (what the library assumes without a GPU)."""

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
