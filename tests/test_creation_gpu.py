"""What a context is made from: rows in any order, with self loops and repeated
neighbours, are the same model as their canonical form, and a topology is taken
as symmetric only if every link has its reverse of the same weight."""
import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi
from pliscuda_amd import workloads as W
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _rows(topo):
    rp, col = topo["row_ptr"].astype(np.int64), topo["col"].astype(np.int64)
    w = topo.get("w")
    w = np.ones(len(col)) if w is None else np.asarray(w, dtype=np.float64)
    return [list(zip(col[rp[v]:rp[v + 1]], w[rp[v]:rp[v + 1]])) for v in range(topo["N"])]


def _topo(rows):
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    flat = [e for r in rows for e in r]
    return {"N": len(rows), "row_ptr": rp, "col": np.array([u for u, _ in flat], dtype=np.uint32),
            "w": np.array([w for _, w in flat], dtype=np.float32)}


def _run(topo, x0, steps=12):
    ctx = capi.Context(W.abc_network(), [topo], [x0], eps=0.1, seed=5)
    ctx.run(np.inf, step_limit=steps)
    out = ctx.get_state(0), ctx.stats(0)
    blob = ctx.checkpoint()
    ctx.close()
    return out, blob


@pytest.mark.parametrize("kind", ["grid", "mesh", "asym"])
def test_rows_in_any_form_are_the_canonical_model(kind):
    """Each row reversed, rotated, with a self loop, or one link given as two halves
    (their sum is exact): the same trajectory, and a checkpoint of one form
    restores into the other."""
    base = {"grid": lambda: W.cubic_grid(13, 11, 15, periodic=False), "mesh": lambda: W.random_mesh(14, 12, 10, 3),
            "asym": lambda: H.asym_topology(2003, 6)}[kind]()
    rows = _rows(base)
    other = []
    for v, r in enumerate(rows):
        r = list(r)
        if v % 5 == 1:
            r.reverse()
        elif v % 5 == 2 and len(r) > 1:
            r = r[1:] + r[:1]
        elif v % 5 == 3:
            r.insert(len(r) // 2, (v, 1.0))
        elif v % 5 == 4 and r:
            u, w = r[-1]
            r = [(u, np.float32(w) / 2)] + r[:-1] + [(u, np.float32(w) / 2)]
        other.append(r)
    x0 = W.poisson_state(3, base["N"], 40.0, 4)
    (xa, sa), blob = _run(base, x0)
    (xb, sb), _ = _run(_topo(other), x0)
    assert np.array_equal(xa, xb) and sa == sb
    ctx = capi.Context(W.abc_network(), [_topo(other)], [x0], eps=0.1, seed=5)
    ctx.restore(blob)
    assert np.array_equal(ctx.get_state(0), xa)
    ctx.close()


def _changed(kind):
    rows = _rows(W.cubic_grid(13, 11, 9, periodic=False))
    if kind == "first_out":
        rows[0] = rows[0][1:]
    elif kind == "first_in":
        u = rows[0][0][0]
        rows[u] = [e for e in rows[u] if e[0] != 0]
    elif kind == "last_out":
        rows[-1] = rows[-1][:-1]
    elif kind == "last_in":
        u = rows[-1][0][0]
        rows[u] = [e for e in rows[u] if e[0] != len(rows) - 1]
    elif kind == "weight":
        rows[700] = [(u, 1.5 if i == 2 else w) for i, (u, w) in enumerate(rows[700])]
    elif kind == "moved":  # the row sums of a symmetric topology, but one link turned round a triangle
        a, b, c = 5, 6, 400
        rows[a] = sorted(rows[a] + [(c, 1.0)])
        rows[c] = sorted(rows[c] + [(b, 1.0)])
        rows[b] = sorted(rows[b] + [(a, 1.0)] if a not in [u for u, _ in rows[b]] else rows[b] + [(c + 9, 1.0)])
    return _topo(rows)


@pytest.mark.parametrize("kind", ["first_out", "first_in", "last_out", "last_in", "weight", "moved"])
def test_one_link_without_its_reverse(kind):
    topo = _changed(kind)
    x0 = W.poisson_state(3, topo["N"], 60.0, 4)
    (x, st), _ = _run(topo, x0, steps=20)
    xo = np.array(x0, dtype=np.uint32).copy()
    so = ffi.run(ffi.Model(W.abc_network(), topo), xo, 0.1, 10, 5, np.inf, step_limit=20)
    assert np.array_equal(x, xo) and st["t"] == so.t and st["firings"] == so.firings


@pytest.mark.parametrize("bad,message", [("id", "neighbour id"), ("weight", "edge weight"), ("nan", "edge weight")])
def test_bad_rows_are_refused(bad, message):
    """In the first, a middle and the last entry of a row that is in order otherwise."""
    for at in (0, 2, -1):
        topo = _topo(_rows(W.cubic_grid(5, 4, 3, periodic=False)))
        q = int(topo["row_ptr"][31]) + at if at >= 0 else int(topo["row_ptr"][32]) - 1
        if bad == "id":
            topo["col"][q] = topo["N"]
        else:
            topo["w"][q] = 0.0 if bad == "weight" else np.nan
        with pytest.raises(capi.PlisError, match=message):
            capi.Context(W.abc_network(), [topo], [W.poisson_state(3, topo["N"], 40.0, 4)])
