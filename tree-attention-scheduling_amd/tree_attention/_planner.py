"""ctypes binding of ``libtree_plan.so``, the host planner library (include/tree_plan.h).

``grouped_decisions`` hands the tree to ``tp_grouped_plan`` in CSR form and
returns, per node, whether its parent pushes it (the subset-DP / greedy
decision of the reference's schedule.py:94-131).  ``attach_tails`` runs the
tail-attachment step of ``kernels.prepare`` (``tp_attach_tails``) and
``build_metadata`` its device metadata (``tp_build_metadata``).  The
library is a plain host library (g++), loaded on first use; ``TREE_PLAN_LIB``
selects another build.
"""
from __future__ import annotations

import ctypes
import os
import threading
from array import array
from itertools import accumulate, chain
from pathlib import Path

import numpy as np

LIB_PATH = Path(__file__).with_name("libtree_plan.so")
EXPORTS = ("tp_grouped_plan", "tp_attach_tails", "tp_build_metadata", "tp_lower", "tp_lower_take")
METHODS = {"greedy": 0, "cube": 1}

_lib = None
_missing = False
_lock = threading.Lock()
_p = ctypes.c_void_p


def load(required: bool = True):
    """Return the loaded library; ``None`` if it is not built and not ``required``."""
    global _lib, _missing
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            target = Path(os.environ.get("TREE_PLAN_LIB", LIB_PATH))
            if not target.exists():
                _missing = True
                if required:
                    raise RuntimeError(f"planner library not found at {target}; build it with "
                                       "`python tree-attention-scheduling_amd/csrc/build.py`")
                return None
            lib = ctypes.CDLL(str(target))
            lib.tp_grouped_plan.restype = ctypes.c_int
            lib.tp_grouped_plan.argtypes = [ctypes.c_int32, ctypes.c_int32] + [_p] * 11
            i32 = ctypes.c_int32
            lib.tp_attach_tails.restype = ctypes.c_int
            lib.tp_attach_tails.argtypes = ([i32, _p, _p, _p, _p, i32, i32, _p, _p, _p, _p, i32, i32, i32, i32, i32]
                                            + [_p] * 5)
            lib.tp_build_metadata.restype = ctypes.c_int
            lib.tp_build_metadata.argtypes = [i32, i32, _p, _p, _p, _p, i32, i32, i32, i32, i32, _p, _p, _p, i32,
                                              _p, _p, ctypes.c_int64]
            lib.tp_lower.restype = _p
            lib.tp_lower.argtypes = [i32, _p, _p, _p, _p, i32, _p, _p]
            lib.tp_lower_take.restype = None
            lib.tp_lower_take.argtypes = [_p, _p]
            _lib = lib
    return _lib


def available() -> bool:
    return load(required=False) is not None


def _ptr(a: np.ndarray):
    """The address of ``a``'s data; the caller keeps ``a`` alive until the library has used it."""
    return a.__array_interface__["data"][0]  # (an int: ctypes.data_as costs four times as much)


def lower(jobs, nreq, options):
    """``tp_lower`` over job objects: (jobs as (requests, first token, tokens) triples, small jobs,
    attachments as ``(large job, first row, [(requests, first token, tokens, first job row)])``), or
    ``None`` for arguments it does not take."""
    lib = load()
    off = array("i", accumulate((len(j.requests) for j in jobs), initial=0))
    req = array("i", chain.from_iterable(j.requests for j in jobs))
    start = array("i", (j.tokens[0] for j in jobs))
    ntok = array("i", (len(j.tokens) for j in jobs))
    opts = array("q", options)
    sizes = array("i", bytes(28))
    at = [a.buffer_info()[0] for a in (off, req, start, ntok, opts, sizes)]
    handle = lib.tp_lower(len(jobs), at[0], at[1], at[2], at[3], nreq, at[4], at[5])
    if not handle:
        return None
    n, small, n_groups, n_req, n_att, n_seg, total = sizes
    out = array("i", bytes(4 * total))
    lib.tp_lower_take(handle, out.buffer_info()[0])
    o = out.tolist()
    p = 3 * n
    groups, q = [], p + n_groups
    for size in o[p:q]:
        groups.append(tuple(o[q:q + size]))
        q += size
    triples = [(groups[g], t0, k) for g, t0, k in zip(o[:n], o[n:2 * n], o[2 * n:p])]
    att, s = [], q + 3 * n_att
    for i in range(q, q + 3 * n_att, 3):
        segs = []
        for _ in range(o[i + 2]):
            segs.append((groups[o[s]], o[s + 1], o[s + 2], o[s + 3]))
            s += 4
        att.append((o[i], o[i + 1], segs))
    return triples, small, att


def grouped_decisions(tree, method: str, model, qheads: int, kvheads: int, dim: int, node_runs):
    """Per-node push flags and the root estimate from the native planner.

    ``node_runs[v]`` are node v's tokens as ``((start, length), ...)`` runs.
    """
    lib = load()
    nodes = tree.nodes
    n = len(nodes)
    parent = array("i", [nd.parent for nd in nodes])
    child_off = array("i", accumulate((len(nd.children) for nd in nodes), initial=0))
    child_idx = array("i", [c for nd in nodes for c in nd.children] or [0])
    nreq = array("i", [len(nd.requests) for nd in nodes])
    run_off = array("q", accumulate(map(len, node_runs), initial=0))
    run_start = array("q", [s for runs in node_runs for s, _ in runs] or [0])
    run_len = array("q", [k for runs in node_runs for _, k in runs] or [0])
    fparams = array("d", (model.bandwidth, model.cube_flops, model.task_us, model.merge_us))
    iparams = array("q", (model.cube_rows, model.key_tile, model.kv_split, model.max_query_rows, qheads, kvheads, dim))
    pushed = array("b", bytes(n))
    total = array("d", (0.0,))
    rc = lib.tp_grouped_plan(METHODS[method], n, *(a.buffer_info()[0] for a in (
        parent, child_off, child_idx, nreq, run_off, run_start, run_len, fparams, iparams, pushed, total)))
    if rc != 0:
        raise ValueError(f"tp_grouped_plan rejected its arguments (code {rc})")
    return pushed, total[0]


def attach_tails(large, small, group, is256, large_tiles, small_tiles, fixed, nreq, xtail_max, wave_rows,
                 item_rows, min_cap):
    """``tp_attach_tails`` over job lists; returns (item per candidate job or -1, its first row, item keys)."""
    lib = load()
    nl, ns = len(large), len(small)
    req_off = np.zeros(nl + 1, dtype=np.int32)
    np.cumsum([len(j.requests) for j in large], out=req_off[1:])
    req = np.fromiter(chain.from_iterable(j.requests for j in large), dtype=np.int32, count=int(req_off[-1]))
    is256 = np.asarray(is256, dtype=np.int32)
    tiles = np.asarray(large_tiles, dtype=np.int32)
    sreq_off = np.zeros(ns + 1, dtype=np.int32)
    np.cumsum([len(j.requests) for j in small], out=sreq_off[1:])
    sreq = np.fromiter(chain.from_iterable(j.requests for j in small), dtype=np.int32, count=int(sreq_off[-1]))
    tiles_s = np.asarray(small_tiles, dtype=np.int32)
    fixed = np.asarray(fixed, dtype=np.int8) if ns else np.zeros(1, dtype=np.int8)
    cap = int(sum(-(-len(j.requests) * group // item_rows) for j, b in zip(large, is256) if b))
    item = np.zeros(max(ns, 1), dtype=np.int32)
    lrow = np.zeros(max(ns, 1), dtype=np.int32)
    item_job = np.zeros(max(cap, 1), dtype=np.int32)
    item_row0 = np.zeros(max(cap, 1), dtype=np.int32)
    n_items = np.zeros(1, dtype=np.int32)
    one = np.zeros(1, dtype=np.int32)
    ptr = lambda a: _ptr(a if a.size else one)  # noqa: E731
    rc = lib.tp_attach_tails(nl, ptr(is256), ptr(tiles), _ptr(req_off), ptr(req), group, ns, _ptr(sreq_off), ptr(sreq),
                             ptr(tiles_s), _ptr(fixed), nreq, xtail_max,
                             wave_rows, item_rows, min_cap, _ptr(item), _ptr(lrow), _ptr(item_job), _ptr(item_row0),
                             _ptr(n_items))
    if rc != 0:
        raise ValueError(f"tp_attach_tails rejected its arguments (code {rc})")
    keys = list(zip(item_job[:n_items[0]].tolist(), item_row0[:n_items[0]].tolist()))
    return item[:ns].tolist(), lrow[:ns].tolist(), keys


def build_metadata(qlen, req, kstart, klen, small_jobs, nreq, group, kvheads, tile_rows, att_job, att_row0, att_rec,
                   xstride):
    """``tp_build_metadata``: (sizes, one int32 buffer of every metadata section)."""
    lib = load()
    one = np.zeros(1, dtype=np.int32)
    ptr = lambda a: _ptr(a if a.size else one)  # noqa: E731
    sizes = np.zeros(13, dtype=np.int32)
    att_rec = np.ascontiguousarray(att_rec, dtype=np.int32).reshape(-1)
    args = (len(qlen), small_jobs, ptr(qlen), ptr(req), ptr(kstart), ptr(klen), nreq, group, kvheads, tile_rows,
            len(att_job), ptr(att_job), ptr(att_row0), ptr(att_rec), xstride,
            _ptr(sizes))
    if lib.tp_build_metadata(*args, None, 0) != 0:
        raise ValueError("tp_build_metadata rejected its arguments")
    buf = np.empty(int(sizes[11]), dtype=np.int32)
    if lib.tp_build_metadata(*args, _ptr(buf), buf.size) != 0:
        raise ValueError("tp_build_metadata rejected its arguments")
    return sizes.tolist(), buf
