"""Query splits of the summary dK/dV pass: every split holds a query, for stages
of 64 and of 32 queries (the kernel takes ceil(ceil(n / stage) / splits) stages a
split)."""
import pytest

from pack3d_amd.core import _splits


@pytest.mark.parametrize("rep", [1, 2, 4, 5, 8, 16])
def test_every_split_holds_a_query(rep):
    for n in (1, 31, 63, 64, 65, 1000, 1024, 4096, 4099, 16384, 18711, 30000, 65536, 131072, 262144):
        for m in (1, 64, 128, 129, 300, 693, 1024, 4096):
            for bg in (1, 2, 3, 4, 8, 12):
                for resident in (512, 256):
                    splits = _splits(n, m, bg, rep, resident)
                    assert splits >= 1
                    for stage in (64, 32):
                        per = -(-(-(-n // stage)) // splits) * stage
                        assert (splits - 1) * per < n, (n, m, bg, rep, splits, stage)


def test_large_problems_keep_their_splits():
    assert _splits(262144, 4096, 4, 1) == 16 and _splits(262144, 128, 1, 4) == 512 and _splits(18711, 693, 4, 1) == 21
