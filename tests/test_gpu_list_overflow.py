"""GPU tests of threshold lists that outgrow their arrays: the answers are those
of the search over every user, and no stage reads the list."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(msg):
    print(f"[case] {msg}", flush=True)


def _sampled(U):
    """The users that the list thresholds are taken from."""
    n = min(max(U // 16, 16384), 65536)
    return np.arange(0, U, max(1, U // n))


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
    U, I, d = 70_001, 800, 16
    items = rng.standard_normal((I, d), dtype=np.float32)
    users = items[7] + np.float32(0.02) * rng.standard_normal((U, d), dtype=np.float32)
    at = _sampled(U)
    users[at] = rng.standard_normal((len(at), d), dtype=np.float32)
    queries = items[7] + np.float32(1e-3) * rng.standard_normal((nq, d), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 48)
    idx.set_form(form)
    before = idx.query(rng.standard_normal((700, d), dtype=np.float32), 10)
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
    assert got.timing["n_batches"] == 2 and got.timing["n_fallback"] == nq and got.timing["n_listed"] == 0
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    _same_answers(got, idx.query(queries, ks), ks)
    idx.close()
