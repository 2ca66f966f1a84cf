"""GPU tests of kernel edges: tile remainders of the score product, bin
lengths of the row sort.  Every value is compared bit for bit with the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(msg):
    print(f"[case] {msg}", flush=True)


@pytest.mark.parametrize("U,I,d", [(1, 2, 1), (127, 129, 15), (128, 128, 16), (129, 131, 17), (130, 260, 3),
                                   (257, 1025, 33), (1030, 259, 150)])
def test_score_product_tiles(orc, U, I, d):
    """Scores at the edges of the 128 x 128 tile, of the 16-term chunk and of 16-byte rows."""
    _case(f"score product U={U} I={I} d={d}")
    import rkr
    rng = np.random.default_rng(U + I + d)
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    with rkr.Index(0) as idx:
        idx.set_data(users, items)
        got = idx.sorted_scores()
    assert np.array_equal(got, orc.sorted_score_rows(orc.normalize_users(users), items))


@pytest.mark.parametrize("copies", [2, 8, 9, 16, 17, 64, 65, 192, 193])
@pytest.mark.parametrize("odd", [0, 1])
def test_row_sort_bin_lengths(orc, copies, odd):
    """Bins of every length class of the row sort, whole 16-byte rows and odd ones,
    more rows than the device has workgroups for."""
    _case(f"row sort with bins of {copies}, odd={odd}")
    import rkr
    rng = np.random.default_rng(copies)
    d, U, I = 6, 300, 4000 + odd
    base = rng.standard_normal((max(2, I // copies), d), dtype=np.float32)
    items = np.concatenate([np.repeat(base, copies, axis=0)[:I],
                            rng.standard_normal((max(0, I - len(base) * copies), d), dtype=np.float32)])
    users = rng.standard_normal((U, d), dtype=np.float32)
    with rkr.Index(0) as idx:
        idx.set_data(users, items)
        got = idx.sorted_scores()
    assert np.array_equal(got, orc.sorted_score_rows(orc.normalize_users(users), items))
