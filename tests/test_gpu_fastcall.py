"""The host entry of the per-layer calls (csrc/fastcall.cpp) against the general path.

Every form that the calls accept -- contiguous or not, any slot type, one RoPE row or one per
request, an output given or not, another stream -- gives the bits that the ctypes path gives,
and what was refused is refused with the same error.
"""
import ctypes

import pytest
import torch

from tree_attention import CostModel, schedule, shapes
from tree_attention import _native
from tree_attention.kernels import (CachedDecodePlan, attention, attention_matrix, decode_append, launch_durations_us,
                                    pack_kv, prepare)

pytestmark = pytest.mark.gpu


class _General:
    """Stands in for the module: every call takes the general path."""
    attention = decode_append = fill = staticmethod(lambda *a: None)


@pytest.fixture
def general(monkeypatch):
    def run(fn):
        _native.load()
        with monkeypatch.context() as m:
            m.setattr(_native, "fastcall", _General)
            out = fn()
        torch.cuda.synchronize()
        return out
    return run


def test_attention_matrix_forms(device, general):
    tree = shapes.tree(shapes.shared_prefix(32, 2048, 64))
    g = torch.Generator().manual_seed(2)
    q = torch.randn(32, 32, 128, generator=g).bfloat16().to(device)
    k = torch.randn(tree.storage_tokens, 8, 128, generator=g).bfloat16().to(device)
    v = torch.randn(tree.storage_tokens, 8, 128, generator=g).bfloat16().to(device)
    kp, vp = pack_kv(k, v)
    odd = pack_kv(torch.cat([k, k[:3]]), torch.cat([v, v[:3]]))
    p = prepare(schedule(tree, 32, 8, 128, "cube", CostModel.mi355x()), q)
    assert p.attached
    side = torch.cuda.Stream()
    for what, qx, pools in (("plain", q, (kp, vp)), ("strided q", q.transpose(0, 1).contiguous().transpose(0, 1), (kp, vp)),
                            ("odd capacity", q, odd)):
        fast = attention_matrix(qx, *pools, p).clone()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            on_side = attention_matrix(qx, *pools, p).clone()
        torch.cuda.current_stream().wait_stream(side)
        want = general(lambda: attention_matrix(qx, *pools, p).clone())
        assert torch.equal(fast, want) and torch.equal(on_side, want), what
    for bad in ((q.half(), kp, vp), (q[:5], kp, vp), (q, kp.transpose(1, 2), vp), (q, kp, vp[:, :-8]), (q.cpu(), kp, vp),
                (q, kp.cpu(), vp), (q, kp[0], vp)):
        with pytest.raises(ValueError) as fast_error:
            attention_matrix(*bad, p)
        with pytest.raises(ValueError) as general_error:
            general(lambda: attention_matrix(*bad, p))
        assert str(fast_error.value) == str(general_error.value)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rope_rows", [1, 6])
def test_decode_append_forms(dtype, rope_rows, device, general):
    nreq, hq, hk, d, cap = 6, 8, 2, 64, 40
    g = torch.Generator().manual_seed(rope_rows)

    def randn(*shape):
        return torch.randn(*shape, generator=g).to(dtype).to(device)

    q, k, v = randn(nreq, 1, hq, d), randn(nreq, 1, hk, d), randn(nreq, 1, hk, d)
    cos, sin = randn(rope_rows, 1, d), randn(rope_rows, 1, d)
    kp, vp = randn(hk, d, cap), randn(hk, cap, d)
    slots = torch.randperm(cap, generator=g)[:nreq]
    flat = [t.reshape(nreq, -1, d) for t in (q, k, v)]
    strided = [torch.stack([t, t], dim=-1)[..., 0] for t in (q, k, v)]
    for what, qkv, sl in (("plain", (q, k, v), slots.int().to(device)), ("3-d", flat, slots.int().to(device)),
                          ("strided", strided, slots.int().to(device)), ("int64", (q, k, v), slots.to(device)),
                          ("host", (q, k, v), slots.tolist())):
        for given in (False, True):
            got, pools = [], []
            for run in (lambda f: f(), general):
                a, b = kp.clone(), vp.clone()
                out = torch.empty(nreq, hq, d, device=device, dtype=dtype) if given else None
                got.append(run(lambda: decode_append(*qkv, cos, sin, sl, a, b, out)))
                pools.append((a, b))
            torch.cuda.synchronize()
            assert torch.equal(got[0], got[1]) and got[0].shape == (nreq, hq, d), what
            assert all(torch.equal(x, y) for x, y in zip(*pools)), what
    for bad in (dict(k=k[:, :, :1]), dict(kp=kp.transpose(1, 2)), dict(cos=cos.float()), dict(v=v[:3])):
        args = {**dict(q=q, k=k, v=v, cos=cos, sin=sin, slots=slots.int().to(device), kp=kp, vp=vp), **bad}
        errors = []
        for run in (lambda f: f(), general):
            with pytest.raises((ValueError, RuntimeError)) as e:
                run(lambda: decode_append(**args))
            errors.append((type(e.value), str(e.value)))
        assert errors[0] == errors[1], bad.keys()


@pytest.mark.parametrize("requests", [1, 3, 70])
def test_fill_growing(requests, device, general):
    """Every word of the metadata after an update equals the torch op's."""
    tree = shapes.tree(shapes.shared_prefix(requests, 700, 5))
    q = torch.empty(requests, 32, 128, dtype=torch.bfloat16, device=device)
    c = CachedDecodePlan(schedule(tree, 32, 8, 128, "cube", CostModel.mi355x()), q, tree.storage_tokens, 9)
    for n in (9, 0, 4):
        fast = c.update(n).metadata.clone()
        c.update(7)
        want = general(lambda: c.update(n).metadata.clone())
        assert torch.equal(fast, want)


def test_attention_calls_that_the_module_takes(device):
    """The ordinary call is handled by the module itself (it returns the library's code), on any
    stream; every other form is left to the general path (None)."""
    tree = shapes.tree(shapes.shared_prefix(32, 2043, 60))
    for dtype in (torch.bfloat16, torch.float16):
        g = torch.Generator().manual_seed(3)
        q = torch.randn(32, 32, 128, generator=g).to(dtype).to(device)
        k = torch.randn(tree.storage_tokens + 5, 8, 128, generator=g).to(dtype).to(device)
        v = torch.randn(tree.storage_tokens + 5, 8, 128, generator=g).to(dtype).to(device)
        assert k.shape[0] % 8 == 0
        plan = schedule(tree, 32, 8, 128, "cube", CostModel.mi355x())
        attached, plain = prepare(plan, q), prepare(plan, q, attach_tails=False)
        assert attached.attached
        _native.load()
        call = _native.fastcall.attention

        def run(p, q, k, v, tokens=False):
            return call(q, k, v, ctypes.addressof(p.abi), p.out, tokens)

        even, odd = (k, v), (k[:-3], v[:-3])
        side = torch.cuda.Stream()
        for p in (attached, plain):
            assert run(p, q, *pack_kv(*even)) == 0 and run(p, q, *even, True) == 0
            with torch.cuda.stream(side):
                assert run(p, q, *pack_kv(*even)) == 0
        assert run(plain, q, *pack_kv(*odd)) == 0 and run(plain, q, *odd, True) == 0
        torch.cuda.synchronize()
        # attachments on a count that is no multiple of 8: the unattached variant is the caller's to choose
        assert run(attached, q, *pack_kv(*odd)) is None and run(attached, q, *odd, True) is None
        kp, vp = pack_kv(*even)
        strided = q.transpose(0, 1).contiguous().transpose(0, 1)
        other = torch.float16 if dtype == torch.bfloat16 else torch.bfloat16
        for bad in ((strided, kp, vp), (q[:5], kp, vp), (q.to(other), kp, vp), (q, kp.to(other), vp), (q, kp, vp[:, :-8]),
                    (q, kp.transpose(1, 2), vp), (q.cpu(), kp, vp), (q, kp.cpu(), vp), (q, kp[0], vp), (q, kp, None)):
            assert run(plain, *bad) is None
        for bad in ((q, kp, vp), (q, k[:, :, :64], v), (q, k.transpose(0, 1), v), (q, k[:-8], v)):
            assert run(plain, *bad, True) is None
        shifted = torch.empty(k.numel() + 1, dtype=dtype, device=device)[1:].view(k.shape).copy_(k)
        assert run(plain, q, shifted, v, True) is None  # 2 bytes off: a packed copy is aligned


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rope_rows", [1, 6])
def test_decode_append_calls_that_the_module_takes(dtype, rope_rows, device):
    nreq, hq, hk, d, cap = 6, 8, 2, 64, 40
    q, k, v = (torch.randn(nreq, 1, h, d, device=device).to(dtype) for h in (hq, hk, hk))
    cos, sin = (torch.randn(rope_rows, 1, d, device=device).to(dtype) for _ in range(2))
    kp, vp = torch.zeros(hk, d, cap, dtype=dtype, device=device), torch.zeros(hk, cap, d, dtype=dtype, device=device)
    slots = torch.arange(nreq, dtype=torch.int32, device=device)
    _native.load()
    call = _native.fastcall.decode_append
    flat = [t.reshape(nreq, -1, d) for t in (q, k, v)]
    for args in ((q, k, v, cos, sin, slots, kp, vp), (*flat, cos[:, 0], sin[:, 0], slots, kp, vp)):
        out = call(*args)
        assert isinstance(out, torch.Tensor) and out.shape == (nreq, hq, d)
        with torch.cuda.stream(torch.cuda.Stream()):
            assert isinstance(call(*args), torch.Tensor)
    torch.cuda.synchronize()
    strided = torch.stack([q, q], dim=-1)[..., 0]
    for bad in ((strided, k, v, cos, sin, slots, kp, vp), (q, k, v, cos, sin, slots.long(), kp, vp),
                (q, k, v, cos, sin, slots[:3], kp, vp), (q, k, v, cos.float(), sin, slots, kp, vp),
                (q, k[:3], v, cos, sin, slots, kp, vp), (q, k, v, cos, sin, slots.cpu(), kp, vp),
                (q, k, v, cos, sin, slots, kp.transpose(1, 2), vp), (q, k, v, cos, sin, slots, kp, vp[:, :-1]),
                (q, k, v, cos, sin, slots.tolist(), kp, vp)):
        assert call(*bad) is None


def test_fill_calls_that_the_module_takes(device):
    _native.load()
    call = _native.fastcall.fill
    meta = torch.zeros(12, dtype=torch.int32, device=device)
    at = torch.tensor([1, 5, 11], device=device)
    assert call(meta, at, 7) == 0
    with torch.cuda.stream(torch.cuda.Stream()):
        assert call(meta, at[:0], 7) == 0
    torch.cuda.synchronize()
    assert meta.tolist() == [0, 7, 0, 0, 0, 7, 0, 0, 0, 0, 0, 7]
    for bad in ((meta, at, -1), (meta, at, 2 ** 31), (meta, at, 1.5), (meta, at.int(), 7), (meta.long(), at, 7),
                (meta.cpu(), at, 7), (meta, at.cpu(), 7), (meta, [1], 7)):
        assert call(*bad) is None
    assert meta.tolist() == [0, 7, 0, 0, 0, 7, 0, 0, 0, 0, 0, 7]


def test_plans_with_attachments_on_any_count_stay_on_the_module(device, monkeypatch):
    """attention_matrix and attention on a count that is no multiple of 8 under a plan with
    attachments: the module runs the unattached variant, the Python path is not taken."""
    tree = shapes.tree(shapes.shared_prefix(64, 2000, 5))
    t = tree.storage_tokens + (tree.storage_tokens % 8 == 0)
    q = torch.randn(64, 8, 64, device=device).half()
    k, v = (torch.randn(t, 2, 64, device=device).half() for _ in range(2))
    p = prepare(schedule(tree, 8, 2, 64, "cube", CostModel.mi355x()), q)
    assert p.attached
    codes = []
    _native.load()

    class Spy:
        @staticmethod
        def attention(*args):
            codes.append(_native_call(*args))
            return codes[-1]

    _native_call = _native.fastcall.attention
    kp, vp = pack_kv(k, v)
    monkeypatch.setattr(_native, "fastcall", Spy)
    a = attention_matrix(q, kp, vp, p).clone()
    assert codes == [None, 0]
    assert torch.equal(a, attention(q, k, v, p)) and codes == [None, 0] * 2
    with pytest.raises(ValueError, match="share dtype"):
        attention_matrix(q.bfloat16(), kp, vp, p)


def test_timing_hook_passes_over_the_tails_update(device):
    """launch_durations_us of a step that sets the tails' lengths first stamps the layer's kernel
    (25 us and more here), not the update's (4 us, what any stamp of an empty kernel reads)."""
    tree = shapes.tree(shapes.headline())
    q = torch.randn(128, 32, 128, device=device).bfloat16()
    cached = CachedDecodePlan(schedule(tree, 32, 8, 128, "cube", CostModel.mi355x()), q, tree.storage_tokens, 8)
    t = tree.storage_tokens + 128 * 8
    kp, vp = (torch.randn(*s, device=device).bfloat16() for s in ((8, 128, t), (8, t, 128)))
    us = launch_durations_us(lambda i: attention_matrix(q, kp, vp, cached.update(i % 8)), 16)
    assert min(us) > 15.0
