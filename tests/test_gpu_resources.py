"""GPU tests of calls that run short of something: a wait, a memory budget, an
allocation.  What was accepted is answered, and an index stays as usable as it was."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(msg):
    print(f"[case] {msg}", flush=True)


@pytest.mark.parametrize("I,Q,n_sample", [(400, 33, 20), (6000, 530, 40), (9000, 1015, 25)])
def test_sample_rank_dp_without_waiting(I, Q, n_sample):
    """The DP whose workgroups give up on each other at once (0 looks, 3 looks)
    answers layer by layer what it answers in one launch."""
    _case(f"DP without waiting Q={Q}")
    import rkr
    from rkr import train
    from test_gpu_train import _synthetic_distribution
    rng = np.random.default_rng(Q)
    accu = _synthetic_distribution(rng, 40, I, Q, I // 2)
    kth, order = train.sort_kth_rank(accu, 5)
    got = []
    with rkr.Index(0) as idx:
        for looks in (1 << 20, 0, 3, 1 << 20):
            idx.set_option(1001, looks)
            ranks, cost = train.find_optimal_sample(idx, 40, I, kth, accu[order], n_sample, "OptimalPart")
            got.append((ranks.tolist(), cost))
    assert got[1:] == got[:1] * 3
