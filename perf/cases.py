"""Workloads of the reverse k-ranks library, each one call sequence of a user's program.

Every case is a dict of plain values.  ``path`` names the call sequence:

query    ``Index.query`` on a built index: from one query at a time (latency) to ten thousand in one call.
build    ``Index.build_table`` over the users and items, and the sampled table read back, as an index build does
         before it saves the table.
scores   every item's score, sorted, for a range of users, into device memory (``rkr_sorted_scores_noalloc``).
update   one round of a live index: items and users inserted, a batch answered with those updates pending, and the
         same items and users deleted again.
train    the QS sample-rank training (``rkr.train.train_sample_ranks``).

Users are N(0, 1)/sqrt(d) rows (the library normalises them), items the same with lognormal(0, 0.5) norms, as the
benchmark draws them; queries are items.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "reverse-k-ranks_amd"))

import rkr  # noqa: E402
from rkr import _lib  # noqa: E402
from rkr.train import train_sample_ranks  # noqa: E402


def listed():
    return [
        # a small catalogue, one query at a time: launches and waits are all there is
        dict(name="one_query_small", path="query", n_user=1000, n_item=5000, dim=30, n_sample=128, n_query=1,
             k_lo=10, k_hi=10, form="plain", output="exact", zipf=False),
        # interactive: a single query against the full-size index
        dict(name="one_query_1m", path="query", n_user=1_000_000, n_item=50_000, dim=150, n_sample=512, n_query=1,
             k_lo=50, k_hi=50, form="screened", output="exact", zipf=False),
        # a handful of queries at once with the default form, odd sizes, one eighth of the serving shape's users
        dict(name="few_queries", path="query", n_user=249_989, n_item=100_003, dim=128, n_sample=512, n_query=7,
             k_lo=10, k_hi=200, form="plain", output="exact", zipf=False),
        # the batch size a serving loop reaches under load
        dict(name="serving_batch", path="query", n_user=500_000, n_item=50_000, dim=128, n_sample=512, n_query=64,
             k_lo=10, k_hi=200, form="screened", output="exact", zipf=False),
        # offline batch against the middle-size index, screened form
        dict(name="batch_100k", path="query", n_user=100_000, n_item=20_000, dim=150, n_sample=512, n_query=1000,
             k_lo=10, k_hi=100, form="screened", output="exact", zipf=False),
        # the same kind of batch with the default FP32 form, an odd dimension
        dict(name="batch_plain", path="query", n_user=100_003, n_item=20_011, dim=145, n_sample=512, n_query=300,
             k_lo=50, k_hi=50, form="plain", output="exact", zipf=False),
        # the headline benchmark's batch
        dict(name="batch_1m", path="query", n_user=1_000_000, n_item=50_000, dim=150, n_sample=512, n_query=1000,
             k_lo=50, k_hi=50, form="screened", output="exact", zipf=False),
        # many queries in one call, popular items repeated, every query with a k of its own
        dict(name="batch_zipf_1m", path="query", n_user=1_000_000, n_item=50_000, dim=150, n_sample=512,
             n_query=10_000, k_lo=10, k_hi=200, form="screened", output="exact", zipf=True),
        # an index build
        dict(name="build_table", path="build", n_user=150_000, n_item=50_000, dim=150, n_sample=512),
        # full sorted score rows kept on the device
        dict(name="sorted_scores", path="scores", n_user=12_000, n_item=20_000, dim=150, n_rows=10_007),
        # a round of live updates with a batch in between
        dict(name="update_round", path="update", n_user=100_000, n_item=20_000, dim=150, n_sample=512, n_query=64,
             k_lo=10, k_hi=100, form="screened", n_new_item=500, n_new_user=2000),
        # sample-rank training
        dict(name="train_ranks", path="train", n_user=50_000, n_item=10_000, dim=150, n_sample=512,
             n_sample_query=1000, sample_topk=600),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["query", "query", "query", "query", "build", "scores", "update", "train"])
    dim = rng.randint(30, 192)
    if path == "query":
        case = dict(path=path, n_user=_log_int(rng, 1000, 1_000_000), n_item=_log_int(rng, 5000, 50_000), dim=dim,
                    n_sample=rng.choice([128, 256, 512]), n_query=_log_int(rng, 1, 4000), k_lo=10,
                    k_hi=_log_int(rng, 10, 200), form=rng.choice(["plain", "screened", "screened"]), output="exact",
                    zipf=rng.random() < 0.3)
        if case["form"] == "plain":
            # the plain form's work grows with every (user, query) pair
            case["n_query"] = max(1, min(case["n_query"], 60_000_000 // case["n_user"]))
            case["output"] = rng.choice(["exact", "exact", "reference"])
            if case["output"] == "reference":
                case["n_user"] = min(case["n_user"], 50_000)
                case["n_query"] = min(case["n_query"], 128)
        return case
    if path == "build":
        n_item = _log_int(rng, 5000, 50_000)
        return dict(path=path, n_user=min(_log_int(rng, 1000, 300_000), 6_000_000_000 // n_item), n_item=n_item,
                    dim=dim, n_sample=rng.choice([128, 256, 512]))
    if path == "scores":
        n_item = _log_int(rng, 1000, 50_000)
        n_rows = min(_log_int(rng, 64, 20_000), 200_000_000 // n_item)
        return dict(path=path, n_user=n_rows + rng.randint(0, 5000), n_item=n_item, dim=dim, n_rows=n_rows)
    if path == "update":
        return dict(path=path, n_user=_log_int(rng, 5000, 150_000), n_item=_log_int(rng, 5000, 30_000), dim=dim,
                    n_sample=rng.choice([128, 512]), n_query=_log_int(rng, 1, 128), k_lo=10,
                    k_hi=_log_int(rng, 10, 200), form=rng.choice(["plain", "screened"]),
                    n_new_item=_log_int(rng, 10, 1000), n_new_user=_log_int(rng, 10, 4000))
    return dict(path=path, n_user=_log_int(rng, 5000, 60_000), n_item=_log_int(rng, 4000, 12_000), dim=dim,
                n_sample=rng.choice([128, 256, 512]), n_sample_query=_log_int(rng, 100, 1000),
                sample_topk=_log_int(rng, 100, 1000))


def _inputs(case, seed):
    """The case's users and items (and the ones an update adds) on the device, and its queries and their k."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    d = case["dim"]

    def rows(n, lognorm):
        x = torch.randn(n, d, generator=g, device="cuda") / math.sqrt(d)
        if lognorm:
            x *= torch.exp(0.5 * torch.randn(n, 1, generator=g, device="cuda"))
        return x

    data = {"users": rows(case["n_user"], False), "items": rows(case["n_item"], True)}
    if case["path"] == "update":
        data["new_users"] = rows(case["n_new_user"], False)
        data["new_items"] = rows(case["n_new_item"], True)
    if "n_query" in case:
        rng = np.random.default_rng(seed)
        n, n_item = case["n_query"], case["n_item"]
        if case.get("zipf"):
            # popular items (the ones with the largest norms) are asked for most: Zipf(1.1) over the norm order
            order = torch.argsort(data["items"].double().norm(dim=1), descending=True, stable=True).cpu().numpy()
            cdf = np.cumsum(1.0 / np.arange(1, n_item + 1) ** 1.1)
            pick = order[np.minimum(np.searchsorted(cdf / cdf[-1], rng.random(n)), n_item - 1)]
        else:
            pick = rng.choice(n_item, size=n, replace=n > n_item)
        data["queries"] = data["items"][torch.from_numpy(np.ascontiguousarray(pick)).cuda()]
        data["topk"] = rng.integers(case["k_lo"], case["k_hi"] + 1, size=n).astype(np.int32)
    return data


def prepare(case, seed):
    data = _inputs(case, seed)
    host = {k: v.cpu().numpy() if torch.is_tensor(v) else v for k, v in data.items()}
    path = case["path"]
    state = {"case": case, "host": host}
    index = state["index"] = rkr.Index(0)
    index.set_data(host["users"], host["items"])
    if path in ("query", "update"):
        index.set_form(case["form"])
        index.build_table(rkr.Index.uniform_sample_ranks(case["n_item"], case["n_sample"]))
        if path == "update":
            index.reserve(case["n_user"] + case["n_new_user"], case["n_new_item"])
        else:
            index.set_output(case["output"])
    elif path == "build":
        state["ranks"] = rkr.Index.uniform_sample_ranks(case["n_item"], case["n_sample"])
    elif path == "scores":
        state["rows"] = torch.empty(case["n_rows"], case["n_item"], device="cuda")
    for name in ("users", "items"):  # the library holds its own copies
        del host[name]
    return state


def run(state):
    case, host, index = state["case"], state["host"], state["index"]
    path = case["path"]
    if path == "query":
        res = index.query(host["queries"], host["topk"], max_k=case["k_hi"])
        return {"users": res.users, "ranks": res.ranks, "qips": res.qips}
    if path == "build":
        index.build_table(state["ranks"])
        return {"table": index.get_table()}
    if path == "scores":
        first = case["n_user"] - case["n_rows"]
        for rc in (index.lib.rkr_sorted_scores_noalloc(index.ctx, first, case["n_rows"], state["rows"].data_ptr()),
                   index.lib.rkr_sync(index.ctx)):  # the rows are complete once the context's stream is
            if rc != _lib.RKR_OK:
                raise _lib.RkrError(rc, index.lib.rkr_last_error(index.ctx).decode())
        return {"rows": state["rows"]}
    if path == "update":
        n_user, n_item = case["n_user"], case["n_item"]
        index.insert_items(host["new_items"])
        index.insert_users(host["new_users"])
        res = index.query(host["queries"], host["topk"], max_k=case["k_hi"])
        index.delete_users(np.arange(n_user, n_user + case["n_new_user"]))
        index.delete_items(np.arange(n_item, n_item + case["n_new_item"]))
        return {"users": res.users, "ranks": res.ranks, "qips": res.qips}
    got = train_sample_ranks(index, case["n_sample"], case["n_sample_query"], case["sample_topk"])
    return {k: got[k] for k in ("ranks", "train_io_cost", "sample_item_ids", "sort_kth_rank", "accu_sorted")}


def work(case):
    """Bytes of the inputs and outputs, each once, and the operations of the inner products a pass is defined by."""
    path, d, n_user, n_item = case["path"], case["dim"], case["n_user"], case["n_item"]
    vectors = 4.0 * d * (n_user + n_item)
    if path == "query":
        n = case["n_query"]
        return {"bytes": 4.0 * d * (n_user + n) + 12.0 * n * case["k_hi"], "flops": 2.0 * d * n_user * n}
    if path == "build":
        return {"bytes": vectors + 4.0 * n_user * (case["n_sample"] + min(4096, n_item)),
                "flops": 2.0 * d * n_user * n_item}
    if path == "scores":
        n = case["n_rows"]
        return {"bytes": 4.0 * d * (n + n_item) + 4.0 * n * n_item, "flops": 2.0 * d * n * n_item}
    if path == "update":
        nu, ni, n = case["n_new_user"], case["n_new_item"], case["n_query"]
        return {"bytes": vectors + 4.0 * d * (nu + ni + n) + 4.0 * n_user * ni + 12.0 * n * case["k_hi"],
                "flops": 2.0 * d * (float(n_user + nu) * (ni + n) + float(nu) * n_item)}
    n = case["n_sample_query"]
    return {"bytes": vectors + 4.0 * n * (n_item + 1), "flops": 2.0 * d * n_user * n_item}


def _sorted_rows(users, items):
    """Scores of every (user, item) in 64 bits, each row descending."""
    return torch.sort(users @ items.T, dim=1, descending=True).values


def exact(case, seed):
    path = case["path"]
    if path == "train":  # whole numbers only
        return None
    # 64-bit sorts of every score row: a few seconds up to this many scores
    n_rows = case["n_rows"] if path == "scores" else case["n_user"]
    if float(n_rows) * case["n_item"] > 8e9 or case.get("output") == "reference":
        return None
    data = _inputs(case, seed)
    users, items = data["users"].double(), data["items"].double()
    if path == "update":
        users = torch.cat([users, data["new_users"].double()])
        items = torch.cat([items, data["new_items"].double()])
    norm = users.norm(dim=1, keepdim=True)
    users = torch.where(norm > 0.001, users / norm, users)
    step = max(1, 100_000_000 // items.shape[0])
    if path == "scores":
        users = users[case["n_user"] - case["n_rows"]:]
        out = torch.empty(users.shape[0], items.shape[0], dtype=torch.float64)
        for a in range(0, users.shape[0], step):
            out[a:a + step] = _sorted_rows(users[a:a + step], items)
        return {"rows": out}
    if path == "build":
        ranks = torch.floor(torch.arange(case["n_sample"], dtype=torch.float64)
                            * ((case["n_item"] - 1) / case["n_sample"])).long().cuda()
        return {"table": torch.cat([_sorted_rows(users[a:a + step], items)[:, ranks].cpu()
                                    for a in range(0, users.shape[0], step)])}
    # queries: <u, q> of the max k users of smallest (rank, user); a query is an item, and does not beat itself
    queries, k = data["queries"].double(), case["k_hi"]
    ips, ranks = [], []
    for a in range(0, users.shape[0], step):
        u = users[a:a + step]
        ip = u @ queries.T
        ascending = -_sorted_rows(u, items)
        ips.append(ip)
        ranks.append(torch.searchsorted(ascending, -(ip + 1e-12)))
    ips, ranks = torch.cat(ips), torch.cat(ranks)
    order = torch.sort(ranks, dim=0, stable=True).indices[:k].T
    qips = torch.gather(ips.T, 1, order).cpu()
    for i, n in enumerate(data["topk"]):
        qips[i, int(n):] = -1.0  # past a query's own k
    return {"users": None, "ranks": None, "qips": qips}
