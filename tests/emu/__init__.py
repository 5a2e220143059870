"""Test tool: the cell tiers' device code on the CPU.  csrc/pg_cell.hip is
compiled by g++ against a stand-in for the HIP header and its lanes run as
coroutines (rt.cpp), in an order that changes at every operation across lanes.
Checked on the way: array indexes (the compiler's bounds checks), that all lanes
of a group come to the same operations, that a cell ends within a number of
them, and that two lanes touch a word of LDS only with a fence in between."""
from __future__ import annotations

import os
import shutil
import struct
import subprocess
from dataclasses import dataclass

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(os.path.dirname(HERE)), "paragram_amd", "csrc")
TIERS = {"0": 0, "m": 1, "1": 2, "2": 3}


def build(out_dir: str) -> str:
    """Compiles the emulated cells into ``out_dir``; returns the program's path."""
    cxx = os.environ.get("CXX") or shutil.which("g++")
    base = [cxx, "-std=c++17", "-O1", "-U_FORTIFY_SOURCE", "-ffp-contract=off", "-Wno-attributes", f"-I{HERE}"]
    # loads and stores are reported to rt.cpp; an index out of an array's bounds traps
    checked = ["-fsanitize=thread", "--param", "tsan-instrument-func-entry-exit=0",
               "-fsanitize=bounds", "-fsanitize-undefined-trap-on-error"]
    rt, cells, prog = (os.path.join(out_dir, f) for f in ("rt.o", "cells.o", "cells"))
    for cmd in ([*base, "-c", os.path.join(HERE, "rt.cpp"), "-o", rt],
                [*base, *checked, "-c", os.path.join(HERE, "cells.cpp"), "-o", cells],
                [cxx, cells, rt, "-o", prog]):
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("emulator build failed:\n" + r.stderr)
    return prog


@dataclass
class Cells:
    kept: np.ndarray      # the tier built the cell (else it left it to the next)
    vertices: np.ndarray
    planes: np.ndarray
    status: np.ndarray
    open_tests: np.ndarray  # removal tests taken by their FP32 sign (tier 0)
    clips: np.ndarray
    rows: list            # neighbours, in the caller's numbering
    held: list            # owners of the planes held at the end, in plane order (negative: the box)
    unordered: list       # exchanges through LDS without a fence


def morton_order(p):
    q = p.astype(np.float64) - p.min(0)
    q = np.minimum((q * (1023.0 / max(q.max(), 1e-30))).astype(np.uint64), 1023)
    key = np.zeros(len(p), np.uint64)
    for b in range(10):
        for a in range(3):
            key |= ((q[:, a] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + a)
    return np.argsort(key, kind="stable")


def run(prog, points, weights=None, cells=None, tier="0", knn=16, fanout=12, binary_below=0, seed=1,
        limit=3_000_000, order=None, guesses=None, use_d2=True) -> Cells:
    """Builds ``cells`` (default: all) of the diagram in ``tier``, from ``knn``
    nearest neighbours (or ``guesses``, an int array [n, k] in the index's order)
    and then a walk of wide records of ``fanout`` children; subtrees of fewer
    than ``binary_below`` points are binary."""
    import oracle

    pts = np.ascontiguousarray(points, np.float32)
    n = pts.shape[0]
    w = np.zeros(n, np.float32) if weights is None else np.asarray(weights, np.float32)
    order = morton_order(pts) if order is None else np.asarray(order)
    inv = np.empty(n, np.int64)
    inv[order] = np.arange(n)
    p4 = np.concatenate([pts, w[:, None]], 1)[order].astype(np.float32)
    sel = np.arange(n) if cells is None else np.asarray(cells)
    if guesses is None and knn > 0:
        d = p4[:, None, :3] - p4[None, :, :3]
        d2 = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1] + d[..., 2] * d[..., 2]).astype(np.float32)
        np.fill_diagonal(d2, np.inf)
        near = np.argsort(d2, axis=1, kind="stable")[:, :knn].astype(np.int32)
        last = np.take_along_axis(d2, near[:, -1:], 1)[:, 0]
    else:
        near = np.zeros((n, 0), np.int32) if guesses is None else np.asarray(guesses, np.int32)
        last, use_d2 = np.zeros(n, np.float32), False
    has_d2 = 1 if use_d2 and near.shape[1] else 0
    lo, hi = oracle.box(pts)
    req = struct.pack("8iq", n, TIERS[tier], len(sel), near.shape[1], fanout, binary_below, seed, has_d2, limit)
    req += p4.tobytes() + inv[sel].astype(np.int32).tobytes() + near.tobytes()
    req += last.astype(np.float32).tobytes() if has_d2 else b""
    req += np.concatenate([lo, hi]).astype(np.float32).tobytes()
    r = subprocess.run([prog], input=req, capture_output=True, timeout=300)
    err = r.stderr.decode(errors="replace")
    assert r.returncode == 0, f"the emulated cells stopped ({r.returncode}): {err}"
    a = np.frombuffer(r.stdout, np.int32)
    m = len(sel)
    info = a[:6 * m].reshape(m, 6)
    at, lists = 6 * m, []
    for _ in range(2 * m):
        k = int(a[at])
        lists.append(a[at + 1:at + 1 + k])
        at += 1 + k
    named = lambda v: np.where(v >= 0, order[np.maximum(v, 0)], v)
    return Cells(info[:, 0] != 0, info[:, 1], info[:, 2], info[:, 3], info[:, 4], info[:, 5],
                 [np.sort(order[r]) for r in lists[:m]], [named(h) for h in lists[m:]],
                 [s for s in err.splitlines() if s.startswith("unordered")])
