"""GPU tests of threshold lists that outgrow their arrays: the answers are those
of the search over every user, and no stage reads the list."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(msg):
    print(f"[case] {msg}", flush=True)


def _sampled(U):
    """The users that the list thresholds are taken from: one of every stride, at a hashed place."""
    stride = max(1, U // min(max(U // 16, 16384), 65536))
    r = np.arange((U + stride - 1) // stride, dtype=np.uint64)
    h = r * np.uint64(0x9E3779B1) & np.uint64(0xFFFFFFFF)
    h = (h ^ (h >> np.uint64(15))) * np.uint64(0x85EBCA6B) & np.uint64(0xFFFFFFFF)
    return np.minimum(r * np.uint64(stride) + (h * np.uint64(stride) >> np.uint64(32)), U - 1).astype(np.int64)


def _same_answers(got, want, ks):
    for i, k in enumerate(ks):
        for f in ("users", "ranks", "qips"):
            assert np.array_equal(getattr(got, f)[i, :k], getattr(want, f)[i, :k]), f"query {i}: {f} differ"


@pytest.mark.parametrize("form", ["plain", "screened"])
@pytest.mark.parametrize("nq", [9, 16, 17, 200])
def test_list_overflow(gpu_index_factory, form, nq):
    """Every user but the sampled ones ranks the queries first: the lists are
    many times longer than the sample lets expect.  Batches searched whole and
    ordered by query, after a larger batch whose pairs the arrays still hold."""
    _case(f"list overflow {form} nq={nq}")
    rng = np.random.default_rng(nq)
    U, I, d = 200_001, 800, 16
    items = rng.standard_normal((I, d), dtype=np.float32)
    users = items[7] + np.float32(0.02) * rng.standard_normal((U, d), dtype=np.float32)
    at = _sampled(U)
    users[at] = rng.standard_normal((len(at), d), dtype=np.float32)
    queries = items[7] + np.float32(1e-3) * rng.standard_normal((nq, d), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 48)
    idx.set_form(form)
    before = idx.query(rng.standard_normal((280, d), dtype=np.float32), 10)  # leaves room for 1.1M pairs
    assert before.timing["n_listed"] > 0
    ks = [int(k) for k in rng.integers(1, 50, nq)]
    got = idx.query(queries, ks)
    assert got.timing["n_fallback"] == nq and got.timing["n_listed"] == 0
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    _same_answers(got, idx.query(queries, ks), ks)
    idx.close()


@pytest.mark.parametrize("form", ["plain", "screened"])
def test_more_listed_pairs_than_31_bits_count(gpu_index_factory, form):
    """1024 queries whose lists hold 2.2 million users each, 2.29e9 pairs in all,
    where the sample shows a dozen users a query."""
    _case(f"2.3e9 listed pairs, {form}")
    rng = np.random.default_rng(1)
    U, I, d, nq = 2_300_000, 300, 8, 1024
    items = rng.standard_normal((I, d), dtype=np.float32)
    items /= np.linalg.norm(items, axis=1, keepdims=True)
    pool = rng.standard_normal((40_000, d), dtype=np.float32)
    rank = (pool @ items.T > (pool @ items[7])[:, None]).sum(axis=1)
    users = pool[rng.choice(np.flatnonzero(rank < 100), U)]
    at = _sampled(U)
    users[at] = pool[rng.choice(np.flatnonzero(rank >= 280), len(at))]
    users[at[100:112]] = pool[np.flatnonzero((rank >= 100) & (rank < 110))[:12]]
    queries = items[7] + np.float32(1e-4) * rng.standard_normal((nq, d), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 64, dense_top=0)
    idx.set_form(form)
    ks = [10] * nq
    got = idx.query(queries, ks)
    # lists from exact scores and the search, before them from one and three products
    assert got.timing["n_batches"] == {"plain": 2, "screened": 4}[form]
    assert got.timing["n_fallback"] == nq and got.timing["n_listed"] == 0
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    _same_answers(got, idx.query(queries, ks), ks)
    idx.close()


@pytest.mark.parametrize("form", ["plain", "screened"])
@pytest.mark.parametrize("U", [66_000, 300_000])
def test_users_in_a_periodic_order(gpu_index_factory, form, U):
    """Users of as many clusters as the sample's stride, in turn, and queries near
    all clusters but the first: every list fits, as the sample says."""
    _case(f"periodic user order {form} U={U}")
    rng = np.random.default_rng(U)
    I, d, nq = 700, 24, 64
    stride = U // max(U // 16, 16384)
    centre = rng.standard_normal((stride, d), dtype=np.float32)
    users = np.float32(0.7) * centre[np.arange(U) % stride] + rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    near = centre[rng.integers(1, stride, nq // 2)] + np.float32(0.5) * rng.standard_normal((nq // 2, d), dtype=np.float32)
    queries = np.concatenate([items[:nq // 2], near]) * np.float32(0.9)
    ks = [int(k) for k in rng.integers(1, 50, nq)]
    idx, _ = gpu_index_factory(users, items, 64)
    idx.set_form(form)
    got = idx.query(queries, ks)
    assert got.timing["n_listed"] > 0 and got.timing["n_fallback"] == 0
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    _same_answers(got, idx.query(queries, ks), ks)
    idx.close()


@pytest.mark.parametrize("form", ["plain", "screened"])
@pytest.mark.parametrize("scale", [0.01, 0.1, 0.3])
def test_one_deep_query_among_ordinary_ones(gpu_index_factory, form, scale):
    """A short query that no user ranks high beside 19 ordinary ones: four
    neighbours in the order of thresholds share one, and the ordinary ones'
    lists would hold most users at the short one's."""
    _case(f"one query scaled by {scale}, {form}")
    rng = np.random.default_rng(11)
    U, I, d, nq = 100_000, 800, 16, 20
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    queries = items[:nq].copy()
    queries[3] *= np.float32(scale)
    idx, _ = gpu_index_factory(users, items, 48)
    idx.set_form(form)
    ks = [20] * nq
    got = idx.query(queries, ks)
    assert got.timing["n_listed"] > 0 and got.timing["n_fallback"] <= 1
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    _same_answers(got, idx.query(queries, ks), ks)
    idx.close()


@pytest.mark.parametrize("form", ["plain", "screened"])
@pytest.mark.parametrize("deep,popular", [(5, 60), (60, 5), (0, 200), (200, 0), (70, 70)])
def test_batches_that_do_not_fit_at_once(gpu_index_factory, form, deep, popular):
    """Popular queries whose lists find no room at first, short ones that no
    list answers and ordinary ones, in one batch: each is answered on its own
    terms, also when the same batch comes again and finds the room there."""
    _case(f"{deep} deep and {popular} popular queries of 200, {form}")
    rng = np.random.default_rng(deep + popular)
    U, I, d, nq = 70_001, 800, 16, 200
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    queries = items[rng.choice(I, nq, replace=False)].copy()
    at = rng.permutation(nq)
    queries[at[:deep]] *= np.float32(0.003)
    queries[at[deep:deep + popular]] *= np.float32(1.7)
    ks = [int(k) for k in rng.integers(1, 60, nq)]
    idx, _ = gpu_index_factory(users, items, 48)
    idx.set_form(form)
    got = [idx.query(queries, ks) for _ in range(2)]
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    want = idx.query(queries, ks)
    for g in got:
        print({f: g.timing[f] for f in ("n_batches", "n_listed", "n_fallback")}, flush=True)
        _same_answers(g, want, ks)
        for f in ("n_candidate", "n_refine_user", "n_prune_user", "n_result_user", "query_id"):
            assert [s[f] for s in g.stats] == [s[f] for s in want.stats], f
        # long lists join a search that other queries need
        assert g.timing["n_listed"] > 0 and g.timing["n_fallback"] <= deep + popular // 2
    idx.close()


@pytest.mark.parametrize("U,nq", [(17_000, 8), (40_001, 37), (90_000, 600)])
@pytest.mark.parametrize("d,noise", [(40, 1.0), (40, 0.3), (40, 0.1), (40, 0.03), (40, 0.01), (20, 0.02), (90, 0.02), (120, 0.02),
                                     (150, 0.02), (190, 0.02), (220, 0.02), (256, 0.02)])
def test_items_that_share_a_common_part(gpu_index_factory, U, nq, d, noise):
    """Items = mean + noise: the less noise, the more users one BF16 product
    cannot tell apart.  Every row width of the three-product scores."""
    _case(f"items = mean + {noise} noise, U={U} nq={nq} d={d}")
    rng = np.random.default_rng(d + nq)
    I = 900
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal(d, dtype=np.float32) + np.float32(noise) * rng.standard_normal((I, d), dtype=np.float32)
    queries = items[rng.choice(I, nq, replace=False)]
    ks = [int(k) for k in rng.integers(1, 60, nq)]
    idx, _ = gpu_index_factory(users, items, 64)
    idx.set_form("screened")
    got = idx.query(queries, ks)
    print({f: got.timing[f] for f in ("n_batches", "n_listed", "n_fallback")}, flush=True)
    assert got.timing["n_listed"] > 0 and got.timing["n_fallback"] <= nq // 8
    if noise <= 0.02 and d >= 90:
        assert got.timing["n_batches"] > 1
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    want = idx.query(queries, ks)
    _same_answers(got, want, ks)
    for f in ("n_candidate", "n_refine_user", "n_prune_user", "n_result_user", "query_id"):
        assert [s[f] for s in got.stats] == [s[f] for s in want.stats], f
    idx.close()


def test_stage_times(gpu_index_factory):
    """Stage times of batches on two streams at once: a query's top-k workgroup
    can end before the batch's first one has stamped the start."""
    _case("stage times")
    rng = np.random.default_rng(2)
    users = rng.standard_normal((300_001, 32), dtype=np.float32)
    items = rng.standard_normal((3000, 32), dtype=np.float32) * np.exp(0.5 * rng.standard_normal((3000, 1), dtype=np.float32))
    idx, _ = gpu_index_factory(users, items, 48)
    for form in ("screened", "plain"):
        idx.set_form(form)
        for _ in range(40):
            t = idx.query(items[:2600], 20).timing
            for f in ("ip_ms", "bound_ms", "prune_ms", "refine_ms", "recheck_ms", "topk_ms", "h2d_ms", "d2h_ms"):
                assert 0 <= t[f] <= 3 * t["total_ms"], f  # of three batches
    idx.close()


@pytest.mark.parametrize("form", ["plain", "screened"])
@pytest.mark.parametrize("U,nq", [(64, 300), (1000, 64), (1000, 400), (5000, 20)])
def test_k_on_either_side_of_a_quarter_of_the_users(gpu_index_factory, form, U, nq):
    """Batches that want less and more than a quarter of all users on average."""
    _case(f"k about U / 4, {form} U={U} nq={nq}")
    rng = np.random.default_rng(U)
    users = rng.standard_normal((U, 14), dtype=np.float32)
    items = rng.standard_normal((700, 14), dtype=np.float32)
    queries = items[rng.choice(700, nq, replace=False)]
    idx, _ = gpu_index_factory(users, items, 30)
    idx.set_form(form)
    for k in (U // 4 - 1, U // 4, U // 4 + 1, U // 2, U):
        ks = [min(k, 4096)] * nq
        idx.set_option(9, 1)  # RKR_OPT_COARSE
        got = idx.query(queries, ks)
        idx.set_option(9, 0)
        _same_answers(got, idx.query(queries, ks), ks)
    idx.close()


def test_queries_left_without_room_are_counted_once(gpu_index_factory):
    """Lists of a little more than a quarter of all users in a batch that wants less on
    average: the ones without room are searched, and are one query each of n_fallback."""
    _case("long lists without room")
    rng = np.random.default_rng(5)
    U, I, nq = 12_000, 3000, 64
    users = rng.standard_normal((U, 24), dtype=np.float32)
    items = rng.standard_normal((I, 24), dtype=np.float32)
    items /= np.linalg.norm(items, axis=1, keepdims=True)
    queries = items[rng.choice(I, nq, replace=False)]
    ks = [10] * 4 + [3010] * 60
    idx, _ = gpu_index_factory(users, items, 64)
    idx.set_form("screened")
    got = idx.query(queries, ks)
    assert 0 < got.timing["n_fallback"] <= nq
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    _same_answers(got, idx.query(queries, ks), ks)
    idx.close()


def test_more_candidates_than_32_bits_count(gpu_index_factory):
    """2000 queries that each of 2.2 million users ranks first, 4.4e9 candidates
    in one batch: refused, as from 2^31 candidates on, whatever a 32-bit sum says."""
    _case("4.4e9 candidates")
    from rkr import _lib
    rng = np.random.default_rng(1)
    U, nq, d = 2_200_000, 2000, 4
    users = np.abs(rng.standard_normal((U, d), dtype=np.float32)) + np.float32(0.1)
    items = -np.abs(rng.standard_normal((60, d), dtype=np.float32))
    queries = np.abs(rng.standard_normal((nq, d), dtype=np.float32)) + np.float32(0.1)
    idx, _ = gpu_index_factory(users, items, 16, dense_top=0)
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    idx.set_option(3, 2000)  # RKR_OPT_QUERY_BATCH
    with pytest.raises(_lib.RkrError) as e:
        idx.query(queries, 5)
    assert e.value.status == _lib.RKR_ERR_NOMEM and "lower the query batch" in str(e.value)
    idx.set_option(3, 200)
    idx.set_option(9, 1)
    assert np.array_equal(idx.query(queries[:300], 5).users, np.tile(np.arange(5), (300, 1)))
    idx.close()
