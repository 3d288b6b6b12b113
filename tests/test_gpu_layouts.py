"""The segment kernels over pools of any capacity and over token-major K/V.

Pools whose capacity is not a multiple of 8 bring K into LDS through registers
(its rows start at any 2-byte address); ``attention`` reads token-major K and V
where they lie.  Both run every work-item kind: small and 64/128/256-row items,
several kinds in one launch, tails that merge their request.  Sizes sit at the
edges: capacities below one 8-token chunk, last tiles that end with the pool,
jobs that start anywhere.  Bars as in test_gpu_parity (0.3 % relative L2 against
the FP32 oracle, atol .008 / rtol .03).
"""
import math

import pytest
import torch

from oracle.attention_oracle import relative_l2, request_attention
from tree_attention import CostModel, KVTree, schedule, shapes
from tree_attention import _native, kernels
from tree_attention.kernels import attention, attention_matrix, pack_kv, prepare
from tree_attention.schedule import Job, Plan

pytestmark = pytest.mark.gpu


def say(*args):
    print(*args, flush=True)


# (tree spec, methods): what kinds they lower to is asserted below
TREES = {
    "tiny": ([-1, 0, 0], [1, 2, 0], [1, 2]),                                        # 3 tokens in all
    "one_chunk": ([-1, 0, 0], [5, 1, 3], [1, 2]),                                   # 9 tokens
    "ragged_tails": shapes.shared_prefix(33, 130, [1 + (29 * r) % 131 for r in range(33)]),
    "wide_root": shapes.shared_prefix(70, 643, [1 + r % 9 for r in range(70)]),     # 256-row items
    "branches": ([-1] + [0] * 3 + [1 + i % 3 for i in range(45)], [300, 77, 130, 65] + [3 + 11 * i for i in range(45)],
                 list(range(4, 49))),                                               # 64-row items and small ones
}


@pytest.mark.parametrize("hq,hk,d,dtype", [(32, 8, 128, torch.bfloat16), (8, 2, 64, torch.float16),
                                           (8, 2, 32, torch.bfloat16)])
@pytest.mark.parametrize("name", list(TREES))
def test_any_capacity_and_token_major(name, hq, hk, d, dtype, device):
    """Every method's plan over pools of 8n + 1 .. 8n + 7 tokens and over token-major K/V."""
    tree = shapes.tree(TREES[name])
    t = tree.storage_tokens
    pads = [p for p in (0, 1, 4) if (t + p) % 8] or [1]
    g = torch.Generator().manual_seed(d + t)
    q = torch.randn(len(tree.paths), hq, d, generator=g).to(dtype)
    k = torch.randn(t + max(pads), hk, d, generator=g).to(dtype)
    v = torch.randn(t + max(pads), hk, d, generator=g).to(dtype)
    ref = request_attention(q.float(), k[:t].float(), v[:t].float(), tree)
    qd, kd, vd = q.to(device), k.to(device), v.to(device)
    kinds = set()
    for method in ("request", "fixed", "cube"):
        for tile_rows in (256, 128, 64):
            plan = schedule(tree, hq, hk, d, method, CostModel(kv_split=200, max_query_rows=512))
            p = prepare(plan, qd, tile_rows=tile_rows, route_items=0)  # the large jobs stay large
            outs = {f"token-major {tile_rows}": attention(qd, kd[:t], vd[:t], p).clone()}
            for pad in pads:
                kp, vp = pack_kv(kd[:t + pad], vd[:t + pad])
                assert kp.shape[2] % 8
                outs[f"capacity {t + pad} {tile_rows}"] = attention_matrix(qd, kp, vp, p).clone()
                kinds |= {i for i in range(_native.TA_NKINDS) if p.for_pools(kp).abi.n_items[i]}
            torch.cuda.synchronize()
            for what, out in outs.items():
                say(name, method, what, list(p.abi.n_items))
                torch.testing.assert_close(out.cpu(), ref.to(dtype), atol=0.008, rtol=0.03,
                                           msg=lambda m: f"{method} {what}: {m}")
                assert relative_l2(out.cpu(), ref) <= 3e-3, (method, what)
    if name == "wide_root":
        assert {_native.TA_LARGE64, _native.TA_LARGE128, _native.TA_LARGE256} <= kinds
    if name == "branches":
        assert {_native.TA_SMALL, _native.TA_LARGE64} <= kinds


def _rounding_case(nreq, n, device):
    """One job of ``nreq`` requests over ``n`` tokens whose probabilities lie between two bf16
    values: one token scores 0, the others p = 0.5013, which bf16 rounds to 0.5."""
    q = torch.zeros(nreq, 32, 128)
    q[..., 0] = 8.0
    k = torch.zeros(n, 8, 128)
    k[1:, :, 0] = -0.9765625
    p = math.exp(-8 * 0.9765625 / math.sqrt(128))
    lse = math.log(1 + (n - 1) * p)
    assert lse - math.log(1 + (n - 1) * float(torch.tensor(p).bfloat16())) > 1e-3  # what rounded P would give
    jobs = [Job(tuple(range(nreq)), tuple(range(n)))]
    return q.bfloat16().to(device), k.bfloat16().to(device), Plan(jobs, "x", 0.0, dict(kvheads=8)), lse


@pytest.mark.parametrize("nreq,tile_rows,kind", [(3, 256, _native.TA_SMALL), (14, 256, _native.TA_LARGE64),
                                                 (30, 128, _native.TA_LARGE128), (40, 256, _native.TA_LARGE256),
                                                 (64, 256, _native.TA_LARGE256)])
@pytest.mark.parametrize("n", [29, 197])
def test_odd_capacity_sums_fp32_probabilities(n, nreq, tile_rows, kind, device):
    """The log-sum-exp of pools of other capacities carries no rounding of the probabilities
    (they are summed in FP32, as in the reference's kernel); 1e-4 is ten times what 197 FP32
    additions and the exponential's last bit can move it."""
    q, k, plan, lse = _rounding_case(nreq, n, device)
    v = torch.randn(n, 8, 128, device=device).bfloat16()
    prepared = prepare(plan, q, tile_rows=tile_rows, route_items=0, consolidate_rows=0, large_target=1, small_target=1)
    say("fp32 sums", n, nreq, list(prepared.abi.n_items))
    assert prepared.abi.n_items[kind] and len(prepared.jobs) == 1
    for layer in (lambda: attention_matrix(q, *pack_kv(k, v), prepared), lambda: attention(q, k, v, prepared)):
        prepared.lse.zero_()
        layer()
        assert (prepared.lse[..., 0].cpu() - lse).abs().max() < 1e-4


@pytest.mark.parametrize("n", [5, 45, 75, 333])
@pytest.mark.parametrize("nreq", [2, 14, 40, 64])
def test_odd_capacity_same_bits_in_every_kind(n, nreq, device):
    """A row's result on pools of other capacities does not depend on the kind of work item it
    is in, and an infinite value counts once (its row also pads the job's last tile)."""
    g = torch.Generator().manual_seed(n)
    q = torch.randn(nreq, 32, 128, generator=g).mul(4).bfloat16().to(device)
    k = torch.randn(n, 8, 128, generator=g).bfloat16().to(device)
    v = torch.randn(n, 8, 128, generator=g).bfloat16().to(device)
    inf = v.clone()
    inf[-1, :, 3] = float("inf")
    plan = Plan([Job(tuple(range(nreq)), tuple(range(n)))], "x", 0.0, dict(kvheads=8))
    outs, kinds = [], set()
    for tile_rows in (64, 128, 256):
        p = prepare(plan, q, tile_rows=tile_rows, route_items=0, consolidate_rows=0, large_target=1, small_target=1)
        kinds |= {i for i in range(_native.TA_NKINDS) if p.abi.n_items[i]}
        outs.append(attention_matrix(q, *pack_kv(k, v), p).clone())
        attention_matrix(q, *pack_kv(k, inf), p)
        assert not p.part.isnan().any() and int(p.part.isposinf().sum()) == nreq * 32
    say("kinds", n, nreq, kinds)
    assert all(torch.equal(outs[0], o) for o in outs[1:])
    ref = request_attention(q.float().cpu(), k.float().cpu(), v.float().cpu(), KVTree([], [tuple(range(n))] * nreq))
    assert relative_l2(outs[0].cpu(), ref) <= 3e-3


@pytest.mark.parametrize("start", [2 ** 31 - 400, 2 ** 31 - 100])
@pytest.mark.parametrize("nreq", [4, 14, 40, 64])
def test_a_job_far_beyond_the_pool_adds_nothing(nreq, start, device):
    """Jobs whose tokens all lie past the pool, up to the largest ids there are, contribute
    nothing in any kind (no sum of ids and tile sizes may wrap around)."""
    n = 333
    g = torch.Generator().manual_seed(nreq)
    q = torch.randn(nreq, 32, 128, generator=g).bfloat16().to(device)
    k = torch.randn(n, 8, 128, generator=g).bfloat16().to(device)
    v = torch.randn(n, 8, 128, generator=g).bfloat16().to(device)
    everyone = tuple(range(nreq))
    jobs = [Job(everyone, tuple(range(n))), Job(everyone, tuple(range(start, start + 90)))]
    for pad in (0, 3):
        kp, vp = pack_kv(torch.cat([k, k[:pad + 3]]), torch.cat([v, v[:pad + 3]]))
        for tile_rows in (64, 128, 256):
            opts = dict(tile_rows=tile_rows, route_items=0, consolidate_rows=0, large_target=1, small_target=1)
            out = []
            for js in (jobs, jobs[:1]):
                p = prepare(Plan(js, "x", 0.0, dict(kvheads=8)), q, **opts)
                say("beyond", nreq, start, pad, tile_rows, list(p.abi.n_items))
                out.append(attention_matrix(q, kp, vp, p).clone())
            assert torch.equal(*out)


@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("nreq,tile_rows", [(3, 256), (14, 256), (30, 128), (64, 256)])
def test_a_job_without_requests_writes_nothing(nreq, tile_rows, pad, device):
    """``ta_segment`` on a job whose qlen is 0 (a C caller's, ``prepare`` makes none): no row is
    read or written for it, and the other jobs' partials are the same."""
    n = 96
    jobs = [Job(tuple(range(nreq)), tuple(range(n * i, n * i + 90 - i))) for i in range(3)]
    g = torch.Generator().manual_seed(nreq)
    q = torch.randn(nreq, 32, 128, generator=g).bfloat16().to(device)
    k = torch.randn(3 * n + pad, 8, 128, generator=g).bfloat16().to(device)
    v = torch.randn(3 * n + pad, 8, 128, generator=g).bfloat16().to(device)
    kp, vp = pack_kv(k, v)
    p = prepare(Plan(jobs, "x", 0.0, dict(kvheads=8)), q, tile_rows=tile_rows, route_items=0, consolidate_rows=0,
                large_target=1, small_target=1, attach_tails=False)
    abi, lib = p.abi, _native.load()
    kind = next(i for i in range(_native.TA_NKINDS) if abi.n_items[i])
    qlen = p.qlen.clone()
    say("no requests", nreq, kind, pad, list(abi.n_items), qlen.tolist())

    def run():
        p.part.zero_()
        _native.check(lib.ta_segment(q.data_ptr(), kp.data_ptr(), vp.data_ptr(), abi.qids, abi.kstart, qlen.data_ptr(),
                                     abi.klen, abi.rowbase, abi.items[kind], abi.n_items[kind], kind, abi.part,
                                     abi.lse, abi.nreq, abi.hq, abi.hk, abi.d, kp.shape[2], abi.maxr, abi.dtype,
                                     torch.cuda.current_stream().cuda_stream))
        return p.part.clone()

    whole = run()
    for job in (0, len(p.jobs) - 1):
        qlen.copy_(p.qlen)
        qlen[job] = 0
        a = int(p.rowbase[job])
        part = run()
        assert not part[a:a + nreq].any() and whole[a:a + nreq].any()
        whole_rest = whole.clone()
        whole_rest[a:a + nreq] = 0
        assert torch.equal(part, whole_rest)


def test_token_major_equals_packed(device):
    """Token-major K/V give the bits of the packed pools of an aligned capacity (same tiles, same
    order), attachments included; views that are not contiguous are packed as before."""
    tree = KVTree.synthetic([-1] + [0] * 96, [2043] + [1 + (37 * r) % 200 for r in range(96)], list(range(1, 97)))
    t = -(-tree.storage_tokens // 8) * 8
    g = torch.Generator().manual_seed(8)
    q = torch.randn(96, 32, 128, generator=g).bfloat16().to(device)
    k = torch.randn(t, 8, 128, generator=g).bfloat16().to(device)
    v = torch.randn(t, 8, 128, generator=g).bfloat16().to(device)
    p = prepare(schedule(tree, 32, 8, 128, "cube", CostModel.mi355x()), q)
    assert p.attached
    a = attention(q, k, v, p).clone()
    b = attention_matrix(q, *pack_kv(k, v), p).clone()
    strided = torch.stack([k, k], dim=1)[:, 0]
    assert not strided.is_contiguous()
    c = attention(q, strided, v, p).clone()
    torch.cuda.synchronize()
    assert torch.equal(a, b) and torch.equal(a, c)
    with pytest.raises(ValueError):
        attention(q, k.half(), v, p)
    with pytest.raises(ValueError):
        attention(q[:3], k, v, p)


@pytest.mark.parametrize("hq,hk,d,dtype", [(32, 8, 128, torch.bfloat16), (8, 2, 64, torch.float16),
                                           (8, 8, 32, torch.bfloat16)])
@pytest.mark.parametrize("shared,nreq", [(2043, 96), (77, 9), (0, 300)])
def test_token_major_of_any_count_equals_packed(shared, nreq, hq, hk, d, dtype, device):
    """Numbers of tokens that are no multiple of 8: the bits of the packed pools, also under a
    plan with attachments (both run it without) and with tails of their own, without packing."""
    spec = shapes.shared_prefix(nreq, shared, [1 + (37 * r) % 60 for r in range(nreq)])
    tree = shapes.tree(spec)
    t = tree.storage_tokens + (1 if tree.storage_tokens % 8 == 0 else 0)
    g = torch.Generator().manual_seed(shared)
    q = torch.randn(nreq, hq, d, generator=g).to(dtype).to(device)
    k = torch.randn(t, hk, d, generator=g).to(dtype).to(device)
    v = torch.randn(t, hk, d, generator=g).to(dtype).to(device)
    for method in ("cube", "request"):
        p = prepare(schedule(tree, hq, hk, d, method, CostModel.mi355x()), q)
        a = attention(q, k, v, p).clone()
        b = attention_matrix(q, *pack_kv(k, v), p).clone()
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        attention(q, k, v, p)
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before  # nothing packed
        say("any count", t, method, list(p.abi.n_items), len(p.attached))
        assert torch.equal(a, b)


@pytest.mark.parametrize("hk,d,nreq,pad,packed", [(32, 32, 120, 0, True), (32, 32, 40, 0, False), (24, 32, 120, 0, True),
                                                  (32, 32, 120, 1, False), (16, 32, 120, 0, False),
                                                  (32, 64, 120, 0, False)])
def test_narrow_rows_read_often_are_packed(hk, d, nreq, pad, packed, device, monkeypatch):
    """Token-major K and V of head dim 32 under a plan that reads them many times over: packed
    (PACK_READS), with the bits of the call in place; any other call stays in place."""
    tree = shapes.tree(shapes.shared_prefix(nreq, 2400, 4))
    t = -(-tree.storage_tokens // 8) * 8 + pad
    g = torch.Generator().manual_seed(hk + nreq)
    q = torch.randn(nreq, hk, d, generator=g).bfloat16().to(device)
    k = torch.randn(t, hk, d, generator=g).bfloat16().to(device)
    v = torch.randn(t, hk, d, generator=g).bfloat16().to(device)
    p = prepare(schedule(tree, hk, hk, d, "request", CostModel.mi355x()), q)
    calls = []
    monkeypatch.setattr(kernels, "pack_kv", lambda *kv: calls.append(1) or pack_kv(*kv))
    a = attention(q, k, v, p).clone()
    say("narrow", hk, d, nreq, t, p.narrow_reads, bool(calls))
    assert bool(calls) == packed
    monkeypatch.setattr(kernels, "PACK_READS", 10 ** 9)
    assert torch.equal(a, attention(q, k, v, p)) and len(calls) == packed


@pytest.mark.parametrize("hk", [8, 4])
@pytest.mark.parametrize("small", [1, 31, 43, 60])
def test_one_wave_items_in_any_order(small, hk, device):
    """Launches of one-wave items on both sides of one round of the GPU (1,280 items), alone and
    beside 64-row items, over requests that are consecutive or not: every item runs once."""
    d, group = 128, 4
    nreq = 2 * small + 16
    jobs = [Job((r, r + 2) if r % 3 == 0 and r % 4 < 2 and r + 2 < 2 * small else (r,),
                tuple(range(40 * r, 40 * r + 17 + r % 13))) for r in range(2 * small)]
    jobs += [Job((r,), tuple(range(40 * r + 31, 40 * r + 34 + r % 4))) for r in range(2 * small)]
    base = 40 * 2 * small
    wide = [Job(tuple(range(2 * small, nreq)), tuple(range(base, base + 150)))]
    rest = [Job((r,), tuple(range(base + 160 + 8 * i + o, base + 161 + 8 * i + o)))
            for i, r in enumerate(range(2 * small, nreq)) for o in (0, 3)]
    g = torch.Generator().manual_seed(small)
    t = base + 160 + 8 * nreq
    q = torch.randn(nreq, group * hk, d, generator=g).bfloat16()
    k = torch.randn(t, hk, d, generator=g).bfloat16()
    v = torch.randn(t, hk, d, generator=g).bfloat16()
    kp, vp = pack_kv(k.to(device), v.to(device))
    for plan_jobs in (jobs + rest, jobs + rest + wide):
        paths = [sum((list(j.tokens) for j in plan_jobs if r in j.requests), []) for r in range(nreq)]
        p = prepare(Plan(plan_jobs, "x", 0.0, dict(kvheads=hk)), q.to(device), route_items=0)
        say("one-wave", small, hk, list(p.abi.n_items), -1 in p.qbase_host)
        assert p.abi.n_items[_native.TA_TAIL] == 0 and (p.abi.n_items[_native.TA_SMALL] > 1280) == (hk == 8 and small > 40)
        out = attention_matrix(q.to(device), kp, vp, p).cpu()
        ref = request_attention(q.float(), k.float(), v.float(), KVTree([], [tuple(x) for x in paths]))
        torch.testing.assert_close(out, ref.bfloat16(), atol=0.008, rtol=0.03)
        assert relative_l2(out, ref) <= 3e-3


@pytest.mark.parametrize("d,hk,group,per", [(128, 8, 1, 63), (128, 8, 1, 64), (128, 8, 2, 97), (64, 8, 1, 70),
                                            (64, 4, 4, 33), (32, 2, 8, 33), (64, 12, 4, 61), (128, 16, 8, 5)])
def test_one_wave_items_beside_64_row_items_in_any_order(d, hk, group, per, device):
    """Small items of one or more rows a head beside 64-row items, on both sides of the line from
    which they go to the XCDs by KV head (2,048 items of one or two rows): every item runs once."""
    nreq = -(-64 // group) + per
    base = 8 * per
    jobs = [Job((r,), tuple(range(8 * r + 4 * h, 8 * r + 4 * h + 1 + (r + h) % 3))) for h in (0, 1) for r in range(per)]
    wide = range(per, nreq)
    jobs += [Job((r,), tuple(range(base + 8 * i + o, base + 8 * i + o + 2))) for i, r in enumerate(wide) for o in (0, 3)]
    root = base + 8 * len(wide)
    jobs.append(Job(tuple(wide), tuple(range(root, root + 77))))
    t = -(-(root + 77) // 8) * 8
    g = torch.Generator().manual_seed(per)
    q = torch.randn(nreq, group * hk, d, generator=g).bfloat16()
    k = torch.randn(t, hk, d, generator=g).bfloat16()
    v = torch.randn(t, hk, d, generator=g).bfloat16()
    p = prepare(Plan(jobs, "x", 0.0, dict(kvheads=hk)), q.to(device), route_items=0, attach_tails=False)
    say("one-wave beside 64 rows", d, hk, group, list(p.abi.n_items))
    assert p.abi.n_items[_native.TA_SMALL] == 2 * nreq * hk and p.abi.n_items[_native.TA_LARGE64]
    out = attention_matrix(q.to(device), *pack_kv(k.to(device), v.to(device)), p).cpu()
    paths = [sum((tuple(j.tokens) for j in jobs if r in j.requests), ()) for r in range(nreq)]
    ref = request_attention(q.float(), k.float(), v.float(), KVTree([], paths))
    torch.testing.assert_close(out, ref.bfloat16(), atol=0.008, rtol=0.03)
    assert relative_l2(out, ref) <= 3e-3


@pytest.mark.parametrize("d,cap", [(32, 2 ** 28 + 8), (64, 2 ** 28), (64, 2 ** 28 + 8)])
def test_pools_past_the_short_offsets(d, cap, device):
    """Pools of more than 2**28 tokens (34 and 69 GB here) take 64-bit lane addresses in one-wave
    items and leave the spread copies of 256-row items: the bits of the same tokens in a small
    pool, at the end of the large one and across its 2**28-th token."""
    n, nreq, group = 700, 40, 8
    first = cap - 1024
    g = torch.Generator().manual_seed(d)
    q = torch.randn(nreq, group, d, generator=g).bfloat16().to(device)
    small = [torch.randn(1, d, 1024, generator=g).bfloat16().to(device),
             torch.randn(1, 1024, d, generator=g).bfloat16().to(device)]
    kp = torch.empty(1, d, cap, dtype=torch.bfloat16, device=device)
    vp = torch.empty(1, cap, d, dtype=torch.bfloat16, device=device)
    kp[:, :, first:] = small[0]
    vp[:, first:] = small[1]
    for attach in (True, False):
        outs = []
        for base, pools in ((first, (kp, vp)), (0, small)):
            jobs = [Job(tuple(range(nreq)), tuple(range(base + 3, base + 3 + n)))]
            jobs += [Job((r,), tuple(range(base + 710 + 7 * r, base + 715 + 7 * r))) for r in range(nreq)]
            p = prepare(Plan(jobs, "x", 0.0, dict(kvheads=1)), q, attach_tails=attach, route_items=0, large_target=1)
            say("large pool", d, cap, list(p.abi.n_items), len(p.attached))
            outs += [attention_matrix(q, *pools, p).clone()]
            plain = prepare(Plan(jobs[1:], "x", 0.0, dict(kvheads=1)), q, small_target=1)
            jobs2 = [Job((r,), tuple(range(base + 9 * r + o, base + 9 * r + o + 4))) for o in (0, 5) for r in range(nreq)]
            pair = prepare(Plan(jobs2, "x", 0.0, dict(kvheads=1)), q, small_target=1)
            assert pair.abi.n_items[_native.TA_SMALL] == 2 * nreq
            outs += [attention_matrix(q, *pools, plain).clone(), attention_matrix(q, *pools, pair).clone()]
        assert all(torch.equal(a, b) for a, b in zip(outs[:3], outs[3:]))
    del kp, vp, pools
    torch.cuda.empty_cache()


@pytest.mark.parametrize("hk", [2 ** 18 - 1, 2 ** 18, 270_000])
def test_token_major_rows_past_the_short_offsets(hk, device):
    """Token-major rows so wide that 64 of them pass 4 GiB (d = 128, 2**18 heads): the bits of
    the packed pools."""
    n, d = 64, 128
    q = torch.randn(1, hk, d, dtype=torch.bfloat16, device=device)
    k = torch.randn(n, hk, d, dtype=torch.bfloat16, device=device)
    v = torch.randn(n, hk, d, dtype=torch.bfloat16, device=device)
    p = prepare(Plan([Job((0,), tuple(range(30))), Job((0,), tuple(range(31, n)))], "x", 0.0, dict(kvheads=hk)), q,
                small_target=1)
    say("wide rows", hk, list(p.abi.n_items))
    assert p.abi.n_items[_native.TA_SMALL] == 2 * hk
    a = attention(q, k, v, p).clone()
    assert torch.equal(a, attention_matrix(q, *pack_kv(k, v), p))
    del k, v
    torch.cuda.empty_cache()


@pytest.mark.parametrize("d,hq,hk,dtype", [(128, 32, 8, torch.bfloat16), (64, 8, 2, torch.float16)])
@pytest.mark.parametrize("n", [319, 320, 321, 384, 385, 449, 1000])
def test_copies_spread_over_steps(n, d, hq, hk, dtype, device):
    """256-row items of packed pools from just under five whole tiles (the ring) on: the loop that
    starts a tile's copies inside the steps (pools) gives the bits of the one that starts them behind
    the barrier (token-major), at starts on and off a tile chunk, with idle waves, with attachments."""
    g = torch.Generator().manual_seed(n)
    for start, nreq, attach in ((0, 64, False), (3, 70, False), (8, 66, True), (16, 34, False)):
        jobs = [Job(tuple(range(nreq)), tuple(range(start, start + n)))]
        base = start + n + 5
        jobs += [Job((r,), tuple(range(base + 20 * r, base + 20 * r + 9 + r % 11))) for r in range(nreq)]
        t = -(-(base + 20 * nreq) // 8) * 8
        q = torch.randn(nreq, hq, d, generator=g).to(dtype)
        k = torch.randn(t, hk, d, generator=g).to(dtype)
        v = torch.randn(t, hk, d, generator=g).to(dtype)
        qd, kd, vd = q.to(device), k.to(device), v.to(device)
        p = prepare(Plan(jobs, "x", 0.0, dict(kvheads=hk)), qd, route_items=0, consolidate_rows=0, large_target=1,
                    attach_tails=attach)
        say("spread", n, start, nreq, list(p.abi.n_items), len(p.attached))
        assert p.abi.n_items[_native.TA_LARGE256]
        out = attention_matrix(qd, *pack_kv(kd, vd), p).cpu()
        assert torch.equal(out, attention(qd, kd, vd, p).cpu())
        paths = [sum((list(j.tokens) for j in jobs if r in j.requests), []) for r in range(nreq)]
        ref = request_attention(q.float(), k.float(), v.float(), KVTree([], [tuple(x) for x in paths]))
        torch.testing.assert_close(out, ref.to(dtype), atol=0.008, rtol=0.03)
        assert relative_l2(out, ref) <= 3e-3
