"""The traversals' FP32 screen: outside its range every node takes the exact
test, so neighbour lists equal the oracle's at extreme scales; groups of a
few particles and gather tiles (Newton-h) at several sizes, scales, a common
offset, with a position that is not a number and beside a dense clump."""
import ctypes as C
import os

import numpy as np
import pytest

from flecsph_amd import BodySystem, _abi, generators

pytestmark = pytest.mark.gpu


def scaled(n, scale, offset, n_ngb):
    parts, prm = generators.random_box(n, seed=n, h_spread=0.6, n_ngb=n_ngb)
    for k in ("x", "y", "z"):
        parts[k] = parts[k] * scale + offset
    parts["h"] = parts["h"] * scale
    return parts, prm


@pytest.mark.parametrize("scale", [1e-151, 1e-149, 1e149, 1e152])
@pytest.mark.parametrize("n", [9, 700, 5000])
def test_lists_at_extreme_scales(oracle_mod, n, scale):
    parts, prm = scaled(n, scale, 0.0, 20)
    p = _abi.default_params(**prm)
    g, o = BodySystem(p), oracle_mod.OracleSystem(p, threads=8)
    for s in (g, o):
        s.upload(parts)
        s.update_iteration()
    og, ig = g.neighbor_lists()
    oo, io = o.neighbor_lists()
    assert np.array_equal(og, oo)
    io = np.concatenate([np.sort(io[oo[i]:oo[i + 1]]) for i in range(n)])
    assert np.array_equal(ig, io)
    o.close()
    g.close()


def test_lists_where_fp32_squares_overflow(oracle_mod):
    """h^2 just below the largest FP32 number; two rows of particles far
    from the tile's first one, each a little closer than h to its partner in
    the other row, where rounding to FP32 takes every such pair beyond h: the
    squared distance is infinite there, h^2 is not."""
    rng = np.random.default_rng(3)
    f32 = np.float32
    far, h = 1e23, float(np.sqrt(np.finfo(f32).max)) * (1 - 1e-6)
    m = 60
    rows = []
    while len(rows) < m:
        y0 = 0.5 * far - h * rng.uniform(0.1, 0.9)
        y1 = y0 + h * (1 - 1e-5)
        with np.errstate(over="ignore"):
            if np.isinf((f32(y1) - f32(y0)) * (f32(y1) - f32(y0))):
                rows.append((y0, y1))
    rows = np.array(rows)
    x = np.linspace(0.0, far, m)
    x = np.concatenate([[0.0, far], x, x])
    y = np.concatenate([[0.0, far], rows[:, 0], rows[:, 1]])
    n = x.size
    z = np.zeros(n)
    parts = dict(x=x, y=y, z=z, vx=z, vy=z, vz=z, u=z + 1, m=z + 1,
                 h=z + h, id=np.arange(n))
    p = _abi.default_params()
    g, o = BodySystem(p), oracle_mod.OracleSystem(p, threads=8)
    for s in (g, o):
        s.upload(parts)
        s.update_iteration()
    og, ig = g.neighbor_lists()
    oo, io = o.neighbor_lists()
    assert oo[n] == n + 2 * m
    assert np.array_equal(og, oo)
    io = np.concatenate([np.sort(io[oo[i]:oo[i + 1]]) for i in range(n)])
    assert np.array_equal(ig, io)
    o.close()
    g.close()


def within_h(g, rows=slice(None)):
    """#{b : r < h} of the particles `rows` at the context's own h, by all
    pairs."""
    x, y, z, h = (g.get(f) for f in ("x", "y", "z", "h"))
    d2 = sum((c[rows, None] - c) ** 2 for c in (x, y, z))
    return (d2 < (h * h)[rows, None]).sum(axis=1)


@pytest.mark.parametrize("n,n_target,scale,offset", [
    (65, 10, 1.0, 0.0), (1000, 40, 1.0, 0.0), (3000, 40, 1e9, 0.0),
    (3000, 40, 1.0, 1e4)])
@pytest.mark.parametrize("tile_rows", [64, 128])
@pytest.mark.parametrize("edge", [False, True])
def test_newton_h_over_gather_tiles(oracle_mod, n, n_target, scale, offset,
                                    tile_rows, edge):
    """Both solvers stop within newton_tol * h of the same root, and the
    neighbours within the result are all counted; with `edge` the roots lie
    just inside the gather radius (h_search times the starting h), so that
    the candidates at its end count."""
    parts, prm = scaled(n, scale, offset, n_target)
    prm.update(h_mode=_abi.H_NEWTON, n_target=n_target,
               precision=_abi.PREC_FP64)
    p = _abi.default_params(**prm)
    g, o = BodySystem(p), oracle_mod.OracleSystem(p, threads=8)
    g._call("set_tuning", tile_rows, 128)
    if edge:
        o.upload(parts)
        for _ in range(4):
            o.update_iteration()
            o.update_h()
        parts = dict(parts, h=np.empty(n))
        parts["h"][o.get("id")] = o.get("h") / (p.h_search * 0.998)
    for s in (g, o):
        s.upload(parts)
        s.update_iteration()
        s.update_h()
    assert np.allclose(g.get("h"), o.get("h"), rtol=2e-4, atol=0)
    assert np.array_equal(g.get("hngb"), within_h(g))
    o.close()
    g.close()


@pytest.mark.parametrize("tile_rows", [64, 128])
def test_gather_tile_of_a_nan_position(tile_rows):
    """A tile whose first particle has no position takes the exact test: its
    other particles find their neighbours, that one finds none."""
    n = 3000
    parts, prm = scaled(n, 1.0, 0.0, 40)
    prm.update(h_mode=_abi.H_NEWTON, n_target=40)
    for k in ("x", "y", "z"):
        parts[k][7] = np.nan
    g = BodySystem(_abi.default_params(**prm))
    g._call("set_tuning", tile_rows, 128)
    g.upload(parts)
    g.update_iteration()
    assert g.get("id")[0] == 7  # (the lowest key)
    g.update_h()
    ok = np.arange(n) != 0
    assert np.array_equal(g.get("hngb")[ok], within_h(g)[ok])
    assert g.get("hngb")[0] == 0
    g.close()


@pytest.mark.parametrize("clump", [6000, 280_000])
@pytest.mark.parametrize("k", [2, 4, 6])
@pytest.mark.parametrize("wide", [False, True])
def test_a_clump_beside_a_diffuse_tile(clump, k, wide):
    """A dense clump among 20,000 particles: its particles lie within the
    sphere about some eight of a neighbouring tile but near none of the
    eight, and are no candidates of that tile.  Starting with the clump's h,
    the particles around it are tested one by one and the capacity stays as
    it was; with a wider one it may grow to 16,384, not by the clump."""
    rng = np.random.default_rng(k)
    v = rng.standard_normal((clump, 3))
    v *= (rng.random(clump) ** (1 / 3) / np.linalg.norm(v, axis=1))[:, None]
    mid, rad = 0.15 + 0.06 * k, 0.004
    h0, gap = rad * (40 / clump) ** (1 / 3), 0.03 if wide else 1.5 * rad
    a = rng.random((20_000, 3))
    a = a[np.linalg.norm(a - mid, axis=1) > gap]
    X = np.concatenate([mid + rad * v, a])
    n = len(X)
    z = np.zeros(n)
    h = z + h0
    if wide:
        h[clump:] = 0.015
    parts = dict(x=X[:, 0], y=X[:, 1], z=X[:, 2], vx=z, vy=z, vz=z, u=z + 1,
                 m=z + 1 / n, h=h, id=np.arange(n))
    _, prm = generators.random_box(100)
    prm.update(h_mode=_abi.H_NEWTON, n_target=40)
    g = BodySystem(_abi.default_params(**prm))
    g.upload(parts)
    g.update_iteration()
    print(clump, "particles within", rad, "of", mid, flush=True)
    g.update_h()
    sizes = (C.c_int64 * 2)()
    lib = C.CDLL(os.path.join(os.path.dirname(_abi.__file__),
                              "libfsph_probe.so"))
    lib.fsph_probe_gather(g._h, sizes)
    assert sizes[0] == 4096 or (wide and sizes[0] <= 16384)
    x, y, zz = (g.get(f) for f in ("x", "y", "z"))
    d = np.sqrt((x - mid) ** 2 + (y - mid) ** 2 + (zz - mid) ** 2)
    outside = np.flatnonzero(d > 1.2 * rad)
    rows = outside[np.argsort(d[outside])[:100]]
    assert np.array_equal(g.get("hngb")[rows], within_h(g, rows))
    g.close()
