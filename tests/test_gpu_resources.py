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


def _smallest_budget(works, lo=1 << 10, hi=1 << 28, step=1 << 10):
    """The smallest memory budget (to `step` bytes) that works(budget) accepts."""
    from rkr import _lib
    while hi - lo > step:
        mid = (lo + hi) // 2
        try:
            works(mid)
            hi = mid
        except _lib.RkrError as e:
            assert e.status == _lib.RKR_ERR_NOMEM, e
            lo = mid
    return hi


def test_users_that_do_not_fit():
    """Inserts of users refused for memory, with every budget between one that
    holds the index and one that holds the larger one beside it: the index still
    answers, and the next insert is answered or refused for memory again."""
    _case("insert users without memory")
    import rkr
    from rkr import _lib
    rng = np.random.default_rng(1)
    users = rng.standard_normal((20_000, 8), dtype=np.float32)
    more = rng.standard_normal((9000, 8), dtype=np.float32)
    items = rng.standard_normal((500, 8), dtype=np.float32)
    ranks = rkr.Index.uniform_sample_ranks(500, 16)
    with rkr.Index(0) as idx:
        idx.set_data(users, items)
        idx.build_table(ranks)
        want = idx.query(items[:9], 12)

    def index(budget):
        idx = rkr.Index(0, budget)
        idx.set_option(8, 0)  # RKR_OPT_DENSE_TOP: the sampled table alone
        idx.set_data(users, items)
        idx.set_option(4, 64)  # RKR_OPT_BUILD_BATCH
        idx.build_table(ranks)
        return idx

    def built(budget):
        index(budget).close()

    def grown(budget):
        idx = index(budget)
        try:
            idx.insert_users(more)
        finally:
            idx.close()

    low, high = _smallest_budget(built), _smallest_budget(grown)
    assert high > low
    refused = 0
    for budget in range(low, high, max(1 << 18, (high - low) // 24)):
        idx = index(budget)
        for n in (9000, 1, 1):
            try:
                idx.insert_users(more[:n])
            except _lib.RkrError as e:
                assert e.status == _lib.RKR_ERR_NOMEM, e
                refused += 1
        n_user = idx.counts()["n_user"]
        if n_user == 20_000 and budget > low + (4 << 20):  # room for a query
            got = idx.query(items[:9], 12)
            assert np.array_equal(got.users, want.users) and np.array_equal(got.ranks, want.ranks)
        idx.close()
    assert refused > 0


def test_data_that_does_not_fit():
    """set_data refused for memory at each of its allocations: nothing is freed
    twice, other indexes are not disturbed."""
    _case("set_data without memory")
    import rkr
    from rkr import _lib
    rng = np.random.default_rng(1)
    users = rng.standard_normal((3000, 20), dtype=np.float32)
    items = rng.standard_normal((900, 20), dtype=np.float32)
    ranks = rkr.Index.uniform_sample_ranks(900, 16)
    answers = []
    for budget in list(range(0, 2_000_000, 50_000)) + [0]:
        with rkr.Index(0, budget) as idx, rkr.Index(0) as other:
            try:
                idx.set_data(users, items)
            except _lib.RkrError as e:
                assert e.status == _lib.RKR_ERR_NOMEM, e
            other.set_data(users, items)
            other.build_table(ranks)
            answers.append(other.query(items[:5], 7))
    for a in answers[1:]:
        assert np.array_equal(a.users, answers[0].users) and np.array_equal(a.ranks, answers[0].ranks)
@pytest.mark.parametrize("I,ns", [(4000, 4000), (4001, 3999), (3000, 700)])
def test_rank_distribution_in_little_memory(orc, I, ns):
    """The distribution is answered wherever its inputs, its counts, one row of
    scores, one of sort scratch and one of sample scores fit the budget."""
    _case(f"rank distribution in little memory I={I} ns={ns}")
    import rkr
    from rkr import train
    rng = np.random.default_rng(I)
    users = rng.standard_normal((30, 6), dtype=np.float32)
    items = rng.standard_normal((I, 6), dtype=np.float32)
    ids = rng.choice(I, ns, replace=False).astype(np.int32)

    def loaded(budget):
        with rkr.Index(0, budget) as idx:
            idx.set_data(users, items)

    base = _smallest_budget(loaded, step=256)
    ld = 8
    need = base + 4 * ns * ld + 8 * ns + 4 * ns * (I + 1) + 3 * 4 * I
    want = orc.query_rank_distribution(orc.normalize_users(users), items, ids)
    for spare in (1 << 10, 1 << 13, 1 << 16, 1 << 20):
        with rkr.Index(0, need + spare) as idx:
            idx.set_data(users, items)
            accu, _ = train.query_rank_distribution(idx, ids)
        assert np.array_equal(accu, want)


@pytest.mark.parametrize("call", ["insert_users", "query", "find_optimal_sample"])
def test_scratch_is_given_back(call):
    """A call in a budget that just holds it is answered whether or not sorted
    scores, whose scratch takes two thirds of what is free, came before."""
    _case(f"{call} after sorted scores")
    import rkr
    from rkr import train
    from test_gpu_train import _synthetic_distribution
    rng = np.random.default_rng(3)
    users = rng.standard_normal((4000, 8), dtype=np.float32)
    more = rng.standard_normal((5000, 8), dtype=np.float32)
    items = rng.standard_normal((600, 8), dtype=np.float32)
    accu = _synthetic_distribution(rng, 40, 6000, 700, 3000)
    kth, order = train.sort_kth_rank(accu, 5)
    queries = items[:1]

    def run(budget, sorted_before):
        with rkr.Index(0, budget) as idx:
            idx.set_option(8, 0)  # RKR_OPT_DENSE_TOP: the sampled table alone
            idx.set_option(9, 0)  # RKR_OPT_COARSE
            idx.set_data(users, items)
            if call != "find_optimal_sample":
                idx.build_table(rkr.Index.uniform_sample_ranks(600, 16))
            if sorted_before:
                idx.sorted_scores(0, 100)
                idx.sorted_scores()
            if call == "insert_users":
                idx.insert_users(more)
            elif call == "query":
                return idx.query(queries, 10).users.tolist()
            else:
                return train.find_optimal_sample(idx, 40, 6000, kth, accu[order], 300, "OptimalPart")[0].tolist()

    budget = _smallest_budget(lambda b: run(b, False))
    for spare in (1 << 12, 1 << 18, 1 << 20):
        assert run(budget + spare, True) == run(0, False)


@pytest.mark.parametrize("dense", [0, 2])
def test_table_without_room_for_guard_columns(dense):
    """A table is built, and its queries are answered, wherever it fits with 64
    guard values a user and two rows of scores, whatever else would be faster."""
    _case(f"table in little memory, dense={dense}")
    import rkr
    rng = np.random.default_rng(5)
    U, I, S = 30_000, 700, 20
    users = rng.standard_normal((U, 12), dtype=np.float32)
    items = rng.standard_normal((I, 12), dtype=np.float32)
    ranks = rkr.Index.uniform_sample_ranks(I, S)
    more = rng.standard_normal((500, 12), dtype=np.float32)
    with rkr.Index(0) as idx:
        idx.set_option(8, dense)  # RKR_OPT_DENSE_TOP
        idx.set_data(users, items)
        idx.build_table(ranks)
        want = idx.query(items[:20], 9)
        table = idx.get_table()
        idx.insert_users(more)
        later = idx.query(items[:20], 9)

    def loaded(budget):
        with rkr.Index(0, budget) as idx:
            idx.set_data(users, items)

    base = _smallest_budget(loaded)
    cols = S + (I if dense else 0)
    need = base + 4 * U * cols + 4 * (3 * S + I) + 256 * U + 2 * 4 * I
    for spare in (1 << 12, 4 << 20, 8 << 20, 16 << 20, 32 << 20):
        with rkr.Index(0, need + spare) as idx:
            idx.set_option(8, dense)
            idx.set_data(users, items)
            idx.build_table(ranks)
            assert np.array_equal(idx.get_table(), table)
            if spare < 4 << 20:
                continue
            for form in ("plain", "screened"):
                if form == "screened" and spare < 32 << 20:
                    continue  # its recheck list alone takes 16 MB
                idx.set_form(form)
                got = idx.query(items[:20], 9)
                assert np.array_equal(got.users, want.users) and np.array_equal(got.ranks, want.ranks)
    with rkr.Index(0, need + 4 * U * (cols + 100) + (40 << 20)) as idx:  # grown, perhaps without columns
        idx.set_option(8, dense)
        idx.set_data(users, items)
        idx.build_table(ranks)
        idx.insert_users(more)
        got = idx.query(items[:20], 9)
        assert np.array_equal(got.users, later.users) and np.array_equal(got.ranks, later.ranks)
