"""GPU tests of kernel edges: tile remainders of the score product, bin
lengths of the row sort, threshold lists.  Every value is compared bit for bit
with the oracle or with the search over every user."""
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


def _lists_and_search(idx, queries, ks):
    """The answers with threshold lists and those of the search over every user."""
    idx.set_option(9, 0)  # RKR_OPT_COARSE
    full = idx.query(queries, ks)
    idx.set_option(9, 1)
    got = idx.query(queries, ks)
    for i, k in enumerate(ks):
        for f in ("users", "ranks", "qips"):
            assert np.array_equal(getattr(full, f)[i, :k], getattr(got, f)[i, :k]), f"query {i}: {f} differ"
        for f in ("n_candidate", "n_refine_user", "n_prune_user", "n_result_user"):
            assert full.stats[i][f] == got.stats[i][f], f"query {i}: {f}"
    return got


@pytest.mark.parametrize("form", ["plain", "screened"])
@pytest.mark.parametrize("U,nq,d,dense", [(1, 9, 5, 2), (255, 8, 33, 2), (257, 65, 64, 0), (4097, 17, 150, 2),
                                          (16385, 64, 31, 1), (40003, 5, 161, 2), (70001, 1, 40, 2), (70001, 600, 20, 0)])
def test_threshold_lists(gpu_index_factory, form, U, nq, d, dense):
    """Lists against the full search: user counts at the edges of a unit and of
    the sample, batches of one query to more than a slice, k from 1 to thousands,
    queries that are items, that nobody and that everybody ranks first."""
    _case(f"threshold lists {form} U={U} nq={nq} d={d} dense={dense}")
    rng = np.random.default_rng(U + nq + d)
    I = 1500
    users = rng.standard_normal((U, d), dtype=np.float32)
    users[U // 2] = 0.0
    items = (rng.standard_normal((I, d), dtype=np.float32) * rng.lognormal(0, 0.5, (I, 1))).astype(np.float32)
    queries = items[rng.integers(0, I, nq)].copy()
    if nq > 4:
        queries[1] = 0.0
        queries[2] *= 50.0
        queries[3] = -queries[3]
        queries[4] *= 1e-3
    ks = [int(min(U, k)) for k in np.exp(rng.uniform(0, np.log(3000), nq))]
    idx, _ = gpu_index_factory(users, items, 64, dense_top=dense)
    idx.set_form(form)
    res = _lists_and_search(idx, queries, ks)
    if U >= 70000 or (nq >= 8 and (form == "screened" or U >= 4096)):  # the calls that take lists
        assert res.timing["n_listed"] > 0 or res.timing["n_fallback"] > 0
    idx.close()


@pytest.mark.parametrize("form", ["plain", "screened"])
def test_threshold_lists_eps_and_sample(gpu_index_factory, form):
    """A table with eps > 0, and users ordered so that no sampled one is among a
    query's best: the threshold is too tight or the list too long, and the query
    is answered all the same."""
    _case(f"threshold lists {form}: eps, unrepresentative sample")
    rng = np.random.default_rng(3)
    U, I, d = 70001, 800, 16
    items = rng.standard_normal((I, d), dtype=np.float32)
    users = rng.standard_normal((U, d), dtype=np.float32)
    users[::4] = -items[7] + 0.05 * rng.standard_normal((len(users[::4]), d), dtype=np.float32)  # every fourth is sampled
    users[1:400:4] = items[7] + 0.01 * rng.standard_normal((100, d), dtype=np.float32)
    queries = np.concatenate([items[:12], -items[:12]])
    ks = [int(k) for k in rng.integers(1, 300, len(queries))]
    idx, ranks = gpu_index_factory(users, items, 48)
    idx.set_form(form)
    _lists_and_search(idx, queries, ks)
    T = idx.get_table()
    idx.set_table(ranks, T + np.float32(5e-5), eps=1e-4)  # off by less than eps
    res = _lists_and_search(idx, queries, ks)
    assert res.users.shape == (24, max(ks))
    idx.close()


@pytest.mark.parametrize("U,nq,dense", [(1, 1, 2), (63, 5, 0), (1024, 7, 2), (4096, 64, 2), (4096, 65, 0), (4097, 3, 2)])
def test_few_users(orc, gpu_index_factory, U, nq, dense):
    """Calls on either side of the one-kernel selection's limits (4096 users,
    2^18 pairs), with ties, a zero user and k up to every user, against brute force."""
    _case(f"few users U={U} nq={nq} dense={dense}")
    rng = np.random.default_rng(U + nq)
    I, d = 600, 12
    users = rng.standard_normal((U, d), dtype=np.float32)
    users[U // 3] = 0.0
    items = rng.standard_normal((I, d), dtype=np.float32)
    items[100:140] = items[0]
    queries = np.concatenate([items[rng.integers(0, 160, (nq + 1) // 2)],
                              rng.standard_normal((nq // 2, d), dtype=np.float32)])
    ks = [int(min(U, k)) for k in rng.integers(1, 200, nq)]
    ks[0] = min(U, 4096)
    idx, _ = gpu_index_factory(users, items, 40, dense_top=dense)
    res = idx.query(queries, ks)
    bu, br, bq = orc.bruteforce(orc.normalize_users(users), items, queries, max(ks))
    for i, k in enumerate(ks):
        assert np.array_equal(res.users[i, :k], bu[i, :k]) and np.array_equal(res.ranks[i, :k], br[i, :k])
        assert np.array_equal(res.qips[i, :k], bq[i, :k])
        assert np.all(res.users[i, k:] == -1)
    idx.close()


@pytest.mark.parametrize("U,S,nq", [(300, 600, 1), (3000, 40, 2), (12_000, 4, 3)])
def test_refine_group_sizes(orc, gpu_index_factory, U, S, nq):
    """Refinement with few rows (a unit is one item tile), some, and more than a full group for every workgroup."""
    _case(f"refine groups U={U} S={S} nq={nq}")
    rng = np.random.default_rng(U)
    users = rng.standard_normal((U, 18), dtype=np.float32)
    items = rng.standard_normal((5001, 18), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, S)
    queries = items[rng.choice(5001, nq, replace=False)]
    res = idx.query(queries, 10)
    bu, br, _ = orc.bruteforce(orc.normalize_users(users), items, queries, 10)
    for i in range(nq):
        print(f"refined {res.stats[i]['n_refine_user']} users", flush=True)
        assert np.array_equal(res.users[i], bu[i]) and np.array_equal(res.ranks[i], br[i])


@pytest.mark.parametrize("U,which", [(500, "first"), (500, "middle"), (500, "last"), (500, "all_but_one"),
                                     (70_000, "first_and_last")])
def test_delete_users_in_place(orc, gpu_index_factory, U, which):
    """Users leave from every place (also more rows than one move block holds,
    and a tail that is not touched), with inserted and deleted items pending."""
    _case(f"delete users U={U} {which}")
    from test_gpu_update import Mirror
    rng = np.random.default_rng(U)
    d, I = 20, 600
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 300)
    m = Mirror(orc, users, items)
    new = rng.standard_normal((40, d), dtype=np.float32)
    idx.insert_items(new)
    m.insert_items(new)
    idx.delete_items(np.array([3, 50], np.int64))
    m.delete_items([3, 50])
    queries = items[rng.choice(I, 5, replace=False)]
    gone = {"first": np.arange(0, 70), "middle": np.array([130, 131, 200]), "last": np.arange(440, 500),
            "all_but_one": np.arange(1, 500), "first_and_last": np.array([0, 33_000, U - 1])}[which].astype(np.int64)
    for form in ("plain", "screened"):
        m.check(idx, queries, min(10, len(m.users)), form)
    idx.delete_users(gone)
    m.delete_users(gone)
    for form in ("plain", "screened"):
        m.check(idx, queries, min(10, len(m.users)), form)
    more = rng.standard_normal((90, d), dtype=np.float32)
    idx.insert_users(more)
    m.insert_users(more)
    m.check(idx, queries, 12, "screened")


@pytest.mark.parametrize("gone", ["first", "some", "all"])
@pytest.mark.parametrize("reserved", [False, True])
def test_delete_inserted_items(orc, gpu_index_factory, gone, reserved):
    """Inserted items leave again while no base item has, then others come and
    a base item goes too."""
    _case(f"delete inserted items: {gone}, reserved={reserved}")
    from test_gpu_update import Mirror
    rng = np.random.default_rng(7)
    d, U, I = 24, 3000, 700
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 40)
    m = Mirror(orc, users, items)
    if reserved:
        idx.reserve(4000, 300)
    queries = items[rng.choice(I, 9, replace=False)]
    for n in (60, 130):
        new = rng.standard_normal((n, d), dtype=np.float32) * np.float32(1.3)
        idx.insert_items(new)
        m.insert_items(new)
        n_ins = len(m.ins)
        ids = I + {"first": np.arange(1), "some": np.arange(1, n_ins, 3), "all": np.arange(n_ins)}[gone].astype(np.int64)
        idx.delete_items(ids)
        m.delete_items(ids)
        for form in ("plain", "screened"):
            m.check(idx, queries, 20, form)
    new = rng.standard_normal((20, d), dtype=np.float32)
    idx.insert_items(new)
    m.insert_items(new)
    idx.delete_items(np.array([0, 5, I + 2], np.int64))
    m.delete_items([0, 5, I + 2])
    m.check(idx, queries, 20, "screened")


@pytest.mark.parametrize("form", ["plain", "screened"])
@pytest.mark.parametrize("nq,dense", [(16, 2), (17, 2), (200, 0)])
def test_popular_queries(orc, gpu_index_factory, form, nq, dense):
    """Queries that thousands of users rank first (more candidates of one rank
    than k), a list searched whole (16 queries) and one ordered by query."""
    _case(f"popular queries {form} nq={nq} dense={dense}")
    rng = np.random.default_rng(5)
    U, I, d = 30_000, 2000, 16
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    queries = items[rng.choice(I, nq, replace=False)]
    queries[::2] *= np.float32(2.6)
    ks = [int(k) for k in np.exp(rng.uniform(0, np.log(400), nq))]
    idx, _ = gpu_index_factory(users, items, 64, dense_top=dense)
    idx.set_form(form)
    res = _lists_and_search(idx, queries, ks)
    assert res.timing["n_listed"] > 0 and max(s["n_candidate"] for s in res.stats) > 1024
    bu, br, _ = orc.bruteforce(orc.normalize_users(users), items, queries[:8], max(ks[:8]))
    for i in range(8):
        assert np.array_equal(res.users[i, :ks[i]], bu[i, :ks[i]]) and np.array_equal(res.ranks[i, :ks[i]], br[i, :ks[i]])
    idx.close()


def test_list_of_a_large_batch(gpu_index_factory):
    """More queries in one device batch than the list's order counts at a time."""
    _case("list of 4500 queries")
    rng = np.random.default_rng(9)
    users = rng.standard_normal((900, 12), dtype=np.float32)
    items = rng.standard_normal((700, 12), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 32)
    idx.set_option(3, 8192)  # RKR_OPT_QUERY_BATCH
    idx.set_form("screened")
    queries = rng.standard_normal((4500, 12), dtype=np.float32)
    res = _lists_and_search(idx, queries, [int(k) for k in rng.integers(1, 60, 4500)])
    assert res.timing["n_batches"] == 1 and res.timing["n_listed"] > 0
    idx.close()


@pytest.mark.parametrize("d", [5, 33, 70, 100, 130, 161, 200, 256])
@pytest.mark.parametrize("U,I", [(40, 31), (3000, 1031), (700, 20_001)])
def test_screened_refinement(orc, gpu_index_factory, d, U, I):
    """The screen at every row width, with a last stage of one item, fewer and
    more row blocks than workgroups, both row counts per wavefront."""
    _case(f"screened refinement d={d} U={U} I={I}")
    rng = np.random.default_rng(d + U)
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    queries = np.concatenate([items[:6], rng.standard_normal((6, d), dtype=np.float32)])
    idx, _ = gpu_index_factory(users, items, 6, dense_top=0)
    idx.set_form("screened")
    k = min(U, 30)
    bu, br, _ = orc.bruteforce(orc.normalize_users(users), items, queries, k)
    for rows in (32, 64):
        idx.set_option(7, rows)  # RKR_OPT_SCREEN_ROWS
        res = idx.query(queries, k)
        assert res.timing["n_refined"] > 0
        assert np.array_equal(res.users[:, :k], bu) and np.array_equal(res.ranks[:, :k], br)
    idx.close()


@pytest.mark.parametrize("U,nq,k,max_k", [(1, 1, 1, 1), (65, 16, 20, 33), (3000, 17, 5, 300), (9000, 600, 40, 1500)])
def test_results_written_to_the_host(orc, gpu_index_factory, U, nq, k, max_k):
    """Outputs written by the top-k itself (up to 8 MB, the last one is past it):
    padding past k, stats and counters, twice in a row."""
    _case(f"host results U={U} nq={nq} k={k} max_k={max_k}")
    rng = np.random.default_rng(U)
    users = rng.standard_normal((U, 10), dtype=np.float32)
    items = rng.standard_normal((500, 10), dtype=np.float32)
    queries = rng.standard_normal((nq, 10), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 20)
    n = min(8, nq)
    bu, br, bq = orc.bruteforce(orc.normalize_users(users), items, queries[:n], min(k, U))
    for form in ("plain", "screened"):
        idx.set_form(form)
        for _ in range(2):
            res = idx.query(queries, min(k, U), max_k=max_k)
            m = min(k, U)
            assert np.array_equal(res.users[:n, :m], bu) and np.array_equal(res.ranks[:n, :m], br)
            assert np.array_equal(res.qips[:n, :m], bq)
            assert np.all(res.users[:, m:] == -1) and np.all(res.ranks[:, m:] == -1) and np.all(res.qips[:, m:] == -1)
            assert all(s["n_candidate"] >= m and s["n_prune_user"] == U - s["n_candidate"] for s in res.stats)
            assert res.timing["total_ms"] > 0 and res.timing["topk_ms"] > 0
    idx.close()


def _sample_rank_dp(n_user, kth, accu, n_sample):
    """Cost and path of the sample-rank DP over prefix sums, 64-bit whole numbers."""
    Q = len(kth)
    rank = np.array(sorted({int(k) for k in kth} | {int(k) - 1 for k in kth if k > 0}))
    pos = np.searchsorted(kth, rank, side="right")
    S = np.zeros((Q + 1, len(rank)), np.int64)  # S[x, j] = sum of accu[q][rank_j] over q < x
    S[1:] = np.cumsum(accu[:, rank].astype(np.int64), axis=0)
    j = np.arange(len(rank))
    end = (Q - pos) * n_user - (S[Q] - S[pos, j])
    between = (S[pos, j][:, None] - S[pos][:, j].T) - (S[pos][:, j] - S[pos, j][None, :])
    between[(pos[None, :] >= pos[:, None]) | (pos[None, :] >= Q)] = 0
    T = -end[None, :] + between + end[:, None]
    T[j[None, :] >= j[:, None]] = 1 << 60
    dp, path = S[pos, j] + end, [j.copy()]
    for _ in range(1, n_sample):
        c = dp[None, :] + T
        p = c.argmin(axis=1)
        better = c[j, p] < dp
        path.append(np.where(better, p, path[-1]))
        dp = np.where(better, c[j, p], dp)
    i = int(dp.argmin())
    cost, out = int(dp[i]), []
    for p in reversed(path):
        out.append(int(rank[i]))
        i = int(p[i])
    return out[::-1], cost


@pytest.mark.parametrize("I,Q,n_sample", [(60, 3, 2), (400, 33, 20), (3000, 120, 12), (6000, 530, 40), (9000, 1015, 25),
                                          (14_000, 2100, 9), (30_000, 2300, 6)])
def test_sample_rank_dp_sizes(orc, I, Q, n_sample):
    """The DP of sample-rank training at every number of ranks it holds in
    registers (up to 512, 1024, 2048) and past it."""
    from rkr import train
    from test_gpu_train import _synthetic_distribution
    import rkr
    rng = np.random.default_rng(Q)
    accu = _synthetic_distribution(rng, 40, I, Q, I // 2)
    kth, order = train.sort_kth_rank(accu, 5)
    acc_s = accu[order]
    want, cost = _sample_rank_dp(40, kth, acc_s, n_sample)
    n_rank = len(set(kth.tolist()) | {int(k) - 1 for k in kth if k > 0})
    _case(f"sample-rank DP Q={Q}: {n_rank} ranks, {n_sample} layers")
    if n_rank < 200:  # the oracle's own DP is cubic
        oranks, ocost = orc.find_optimal_sample_fast(40, I, kth, acc_s, 0, n_sample)
        assert ocost == cost and (len(set(want)) < n_sample or list(oranks) == want)
    with rkr.Index(0) as idx:
        for _ in range(2):
            ranks, got = train.find_optimal_sample(idx, 40, I, kth, acc_s, n_sample, "OptimalPart")
            assert got == cost
            if len(set(want)) == n_sample:  # a rank kept for several samples is filled up from others
                assert ranks.tolist() == want


@pytest.mark.parametrize("I", [2, 255, 1617, 7168, 7169, 7172, 14_336, 14_340, 28_672, 28_676])
def test_row_sort_thread_counts(orc, I):
    """Rows on either side of the lengths that take 256, 512 and 1024 threads, some with equal values only."""
    _case(f"row sort I={I}")
    import rkr
    rng = np.random.default_rng(I)
    users = rng.standard_normal((70, 5), dtype=np.float32)
    users[3] = 0.0
    items = rng.standard_normal((I, 5), dtype=np.float32)
    with rkr.Index(0) as idx:
        idx.set_data(users, items)
        got = idx.sorted_scores()
    assert np.array_equal(got, orc.sorted_score_rows(orc.normalize_users(users), items))


@pytest.mark.parametrize("I,S", [(4000, 100), (9000, 4096), (20_000, 4096), (20_001, 700), (52_000, 4096)])
@pytest.mark.parametrize("ties", [0, 1])
def test_select_gather_sizes(orc, I, S, ties):
    """Target bins that fill less and more than half of the gather buffer, rows
    in registers and not, rows whose values crowd into few bins."""
    _case(f"select I={I} S={S} ties={ties}")
    import rkr
    rng = np.random.default_rng(I + S)
    users = rng.standard_normal((9, 7), dtype=np.float32)
    items = rng.standard_normal((I, 7), dtype=np.float32)
    if ties:
        items[I // 3:] = items[rng.integers(0, I // 3, I - I // 3)]
        items[:50] *= 1e4
    with rkr.Index(0) as idx:
        idx.set_option(8, 0)  # RKR_OPT_DENSE_TOP: the sampled table alone
        idx.set_data(users, items)
        ranks = np.unique(np.concatenate([np.arange(S // 2), rng.choice(I, S, replace=False)]))[:S].astype(np.int32)
        idx.build_table(ranks)
        got = idx.get_table()
    want = orc.sorted_score_rows(orc.normalize_users(users), items)[:, ranks]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("U,nq,dense", [(65, 3, 2), (4100, 24, 2), (4100, 25, 0), (1, 1, 0)])
def test_update_bounds_by_guards(orc, gpu_index_factory, U, nq, dense):
    """Bounds with updates pending on either side of the guard rows' limit of
    24 queries, with inserts and deletes, users at the edge of a block of 64."""
    _case(f"update bounds U={U} nq={nq} dense={dense}")
    from test_gpu_update import Mirror
    rng = np.random.default_rng(U + nq)
    d, I = 14, 900
    users = rng.standard_normal((U, d), dtype=np.float32)
    items = rng.standard_normal((I, d), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 200, dense_top=dense)
    m = Mirror(orc, users, items)
    new = rng.standard_normal((30, d), dtype=np.float32) * np.float32(1.2)
    idx.insert_items(new)
    m.insert_items(new)
    idx.delete_items(np.array([0, 7, 9, I + 2], np.int64))
    m.delete_items([0, 7, 9, I + 2])
    queries = np.concatenate([items[:nq // 2], rng.standard_normal((nq - nq // 2, d), dtype=np.float32)])
    for form in ("plain", "screened"):
        m.check(idx, queries, min(U, 12), form)
    idx.close()


@pytest.mark.parametrize("n_new", [1, 2, 63, 64, 65, 128, 129, 256, 257, 511, 512, 513, 1000, 1024, 1025])
def test_inserted_score_rows(orc, gpu_index_factory, n_new):
    """Inserted items' scores sorted in one wavefront at every length, placed,
    merged with those there, and taken out again."""
    _case(f"insert {n_new} items")
    from test_gpu_update import Mirror
    rng = np.random.default_rng(n_new)
    d = 9
    users = rng.standard_normal((300, d), dtype=np.float32)
    users[5] = 0.0
    items = rng.standard_normal((400, d), dtype=np.float32)
    idx, _ = gpu_index_factory(users, items, 30)
    m = Mirror(orc, users, items)
    queries = items[:9]
    for n in (n_new, 77):
        new = rng.standard_normal((n, d), dtype=np.float32)
        new[n // 2:] = new[: n - n // 2]  # equal scores
        idx.insert_items(new)
        m.insert_items(new)
        for form in ("plain", "screened"):
            m.check(idx, queries, 40, form)
    gone = (400 + np.arange(0, n_new, 2)).astype(np.int64)
    idx.delete_items(gone)
    m.delete_items(gone)
    more = rng.standard_normal((3, d), dtype=np.float32)
    idx.insert_users(more)
    m.insert_users(more)
    m.check(idx, queries, 40)
    idx.close()


def test_rebuild_reuses_buffers(orc):
    """Tables built one after the other on the same data: equal sizes, other
    sizes, without and with a query table, after users came."""
    _case("rebuild with equal and other sizes")
    import rkr
    rng = np.random.default_rng(4)
    users = rng.standard_normal((500, 11), dtype=np.float32)
    items = rng.standard_normal((900, 11), dtype=np.float32)
    queries = items[:12]
    nu = orc.normalize_users(users)
    with rkr.Index(0) as idx:
        idx.set_data(users, items)
        for S, dense in ((40, 2), (40, 2), (41, 2), (41, 0), (41, 0), (40, 1), (40, 2)):
            idx.set_option(8, dense)  # RKR_OPT_DENSE_TOP
            ranks = np.sort(rng.choice(900, S, replace=False)).astype(np.int32)
            idx.build_table(ranks)
            assert np.array_equal(idx.get_table(), orc.sorted_score_rows(nu, items)[:, ranks])
            for form in ("plain", "screened"):
                idx.set_form(form)
                res = idx.query(queries, 15)
                bu, br, _ = orc.bruteforce(nu, items, queries, 15)
                assert np.array_equal(res.users, bu) and np.array_equal(res.ranks, br)
        more = rng.standard_normal((30, 11), dtype=np.float32)
        idx.insert_users(more)
        nu = np.concatenate([nu, orc.normalize_users(more)])
        for _ in range(2):
            idx.build_table(ranks)
            assert np.array_equal(idx.get_table(), orc.sorted_score_rows(nu, items)[:, ranks])
        bu, br, _ = orc.bruteforce(nu, items, queries, 15)
        res = idx.query(queries, 15)
        assert np.array_equal(res.users, bu) and np.array_equal(res.ranks, br)


@pytest.mark.parametrize("n", [63, 64, 65, 192, 193, 250])
def test_narrow_column_tiles(orc, gpu_index_factory, n):
    """A last column block on either side of 64 columns: items of sorted rows, queries of a plain batch."""
    _case(f"narrow tiles n={n}")
    import rkr
    rng = np.random.default_rng(n)
    users = rng.standard_normal((4300, 21), dtype=np.float32)
    items = rng.standard_normal((n, 21), dtype=np.float32)
    with rkr.Index(0) as idx:
        idx.set_data(users[:200], items)
        assert np.array_equal(idx.sorted_scores(), orc.sorted_score_rows(orc.normalize_users(users[:200]), items))
    catalogue = rng.standard_normal((400, 21), dtype=np.float32)
    idx, _ = gpu_index_factory(users, catalogue, 30)
    res = idx.query(items, 9)
    bu, br, bq = orc.bruteforce(orc.normalize_users(users), catalogue, items, 9)
    assert np.array_equal(res.users, bu) and np.array_equal(res.ranks, br) and np.array_equal(res.qips, bq)
    idx.close()
