"""The lowering of plans (``kernels.prepare``): what each work item holds, read back from its
metadata the way the kernels read it."""
import random

import pytest
import torch

from tree_attention import _native
from tree_attention.kernels import XTAIL_FIELDS, prepare
from tree_attention.schedule import Job, Plan


def held(p, group, kvheads):
    """Per (request, KV head): the sorted tokens its work items attend, from the device metadata."""
    qids, kstart, qlen, klen = (t.tolist() for t in (p.qids, p.kids[:, 0], p.qlen, p.klen))
    out = {}

    def add(reqs, head, t0, n):
        for r in reqs:
            out.setdefault((r, head), []).extend(range(t0, t0 + n))

    for kind in range(_native.TA_NKINDS):
        items = p.items[kind].view(-1, 3).tolist()
        for i, (j, row0, head) in enumerate(items):
            rows = _native.KIND_ROWS.get(kind, 16)
            per = rows // group if rows >= group else 1
            add(qids[j][:qlen[j]][row0 // group:row0 // group + per], head, kstart[j], klen[j])
            if kind == _native.TA_LARGE256 and p.xtail is not None:
                rec = p.xtail[i].tolist()
                for k in range(rec[0]):
                    t0, n, lrow, nrows = rec[1 + XTAIL_FIELDS * k:1 + XTAIL_FIELDS * (k + 1)]
                    assert row0 <= lrow and lrow + nrows <= min(row0 + 256, qlen[j] * group)
                    add(qids[j][lrow // group:(lrow + nrows) // group], head, t0, n)
    return {key: sorted(v) for key, v in out.items()}


def check_covers(plan, p, nreq, group, kvheads):
    want = [[] for _ in range(nreq)]
    for job in plan.jobs:
        for r in job.requests:
            want[r].extend(job.tokens)
    got = held(p, group, kvheads)
    for r in range(nreq):
        for h in range(kvheads):
            assert got.get((r, h), []) == sorted(want[r]), (r, h)


def random_plan(rng, nreq):
    """A random prefix tree's jobs: a root, uneven branches, nodes of a few requests, tails."""
    jobs, base = [], rng.randrange(0, 9)

    def job(reqs, n):
        nonlocal base
        jobs.append(Job(tuple(reqs), tuple(range(base, base + n))))
        base += n + rng.choice((0, 0, 3))

    def split(reqs, depth):
        job(reqs, rng.choice((5, 64, 300, 2100) if depth else (64, 700, 4096)))
        if depth < 3 and len(reqs) > 1 and rng.random() < 0.9:
            cuts = sorted(rng.sample(range(1, len(reqs)), min(len(reqs) - 1, rng.choice((1, 1, 2, 5)))))
            for a, b in zip([0] + cuts, cuts + [len(reqs)]):
                split(reqs[a:b], depth + 1)

    split(list(range(nreq)), 0)
    for r in range(nreq):
        job([r], rng.choice((1, 40, 64, 64, 130)))
    return Plan(jobs, "x", 0.0, dict(kvheads=2))


def test_attachments_follow_their_items_past_attached_nodes():
    """A node of 8 requests attaches to the root's items and leaves the list of large jobs; the
    256-row jobs after it keep their own attachments (they are named by their place)."""
    jobs = [Job(tuple(range(64)), tuple(range(0, 4096))), Job(tuple(range(8)), tuple(range(4096, 4160))),
            Job(tuple(range(8, 64)), tuple(range(4160, 6208)))]
    jobs += [Job((r,), tuple(range(6208 + 64 * r, 6272 + 64 * r))) for r in range(64)]
    plan = Plan(jobs, "x", 0.0, dict(kvheads=8))
    p = prepare(plan, torch.empty(64, 32, 128, dtype=torch.bfloat16))
    assert any(len(seg.requests) == 8 for segs in p.attached.values() for seg, _ in segs)
    assert {p.jobs[j].requests[0] for j, _ in p.attached} == {0, 8}
    check_covers(plan, p, 64, 4, 8)


@pytest.mark.parametrize("seed", range(40))
def test_random_trees_cover_every_token(seed):
    """Every request's work items hold its path once, per KV head."""
    rng = random.Random(seed)
    nreq = rng.choice((1, 3, 17, 40, 72, 130))
    plan = random_plan(rng, nreq)
    group = rng.choice((4, 4, 8))
    q = torch.empty(nreq, 2 * group, 128, dtype=torch.bfloat16)
    for opts in ({}, dict(attach_tails=False), dict(tile_rows=64)):
        check_covers(plan, prepare(plan, q, **opts), nreq, group, 2)


@pytest.mark.parametrize("seed", range(60))
def test_native_lowering_equals_python(seed):
    """tp_lower gives the jobs and attachments of kernels._lower_py, in the same order, over random
    trees, head groups and every option."""
    from tree_attention import _planner, kernels
    assert _planner.available()
    rng = random.Random(1000 + seed)
    nreq = rng.choice((1, 3, 17, 40, 72, 130))
    plan = random_plan(rng, nreq)
    tokens = max(j.tokens[-1] for j in plan.jobs)
    group = rng.choice((1, 2, 4, 4, 8, 16, 24))
    opts = dict(kvheads=rng.choice((1, 2, 8)), group=group, tile_rows=rng.choice((256, 256, 128, 64)),
                fixed_from=rng.choice((None, None, 0, tokens // 2)), attach_tails=rng.random() < 0.8,
                route_items=rng.choice((0, 768, 5000)), fuse_rows=rng.choice((0, 64, 256)),
                consolidate_rows=rng.choice((0, 128, 256)), large_target=rng.choice((0, 1, 64, 256)),
                small_target=rng.choice((0, 64, 2048)), large_min_tiles=rng.choice((1, 2, 4)))
    jobs = list(plan.jobs)
    if rng.random() < 0.5:  # jobs over one token run, split by requests, and chunks of one group
        wide = jobs[0]
        cut = len(wide.requests) // 2
        half = len(wide.tokens) // 2
        jobs = [Job(r, t) for r in (wide.requests[:cut], wide.requests[cut:]) if r
                for t in (wide.tokens[:half], wide.tokens[half:]) if t] + jobs[1:]
    want = kernels._lower_py(jobs, 256, **opts)
    got = kernels._lower(jobs, nreq, 256, **opts)
    assert got[1] == want[1] and got[0] == want[0]
    assert list(got[2].items()) == list(want[2].items())


def test_native_lowering_leaves_bad_requests_to_prepare():
    plan = Plan([Job((0, 5), (0, 1, 2))], "x", 0.0, dict(kvheads=1))
    with pytest.raises(ValueError, match="names request 5"):
        prepare(plan, torch.empty(2, 4, 32, dtype=torch.float16))


@pytest.mark.parametrize("opts", [dict(fixed_from=-1), dict(fixed_from=-7), dict(fixed_from=64.0),
                                  dict(large_target=200.5, small_target=float("inf")), dict(large_target=10 ** 20),
                                  dict(consolidate_rows=None)])
def test_options_that_are_not_small_ints(opts):
    """Targets and limits may be any numbers; a negative fixed_from keeps every job as it is."""
    from tree_attention import kernels
    plan = random_plan(random.Random(7), 40)
    q = torch.empty(40, 8, 128, dtype=torch.bfloat16)
    p = prepare(plan, q, **opts)
    full = {**dict(tile_rows=256, fixed_from=None, attach_tails=True, route_items=kernels.ROUTE_ITEMS,
                   fuse_rows=kernels.FUSE_ROWS, consolidate_rows=kernels.CONSOLIDATE_ROWS, large_target=256,
                   small_target=2048, large_min_tiles=kernels.LARGE_MIN_TILES), **opts}
    jobs, small, attached = kernels._lower_py(list(plan.jobs), 256, kvheads=2, group=4, **full)
    assert p.jobs == jobs and p.small_jobs == small
    assert p.attached == {(j + small, row0): segs for (j, row0), segs in attached.items()}
