"""The two forms of the radix sort (one workgroup, three launches per pass)
at the edges of their ranges and of their tiles:
keys and ids in the oracle's order, and a batch in its instances' own."""
import ctypes as C
import os

import numpy as np
import pytest

from flecsph_amd import BatchSystem, BodySystem, _abi, generators

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 63, 65, 1025, 2048, 2049, 4096, 4097,
                               8192, 8193, 12288, 12289, 63489])
def test_sorted_keys_equal_the_oracles(oracle_mod, n):
    parts, prm = generators.random_box(n, seed=n)
    if 3 < n < 20000:  # half of them in a corner: equal high digits
        for k in ("x", "y", "z", "h"):
            parts[k][: n // 2] *= 0.03
    p = _abi.default_params(**prm)
    g, o = BodySystem(p), oracle_mod.OracleSystem(p, threads=8)
    for s in (g, o):
        s.upload(parts)
        s.update_iteration()
    for f in ("key", "id", "x", "h"):
        assert np.array_equal(g.get(f), o.get(f)), f
    o.close()
    g.close()


@pytest.mark.parametrize("sizes", [(2, 3, 40), (700, 1349), (3000, 5192),
                                   (3000, 9286, 2), (3000, 9287, 2),
                                   (40000, 91072, 2)])
def test_sorted_keys_of_a_batch(sizes):
    sets = [generators.random_box(n, seed=n + i) for i, n in enumerate(sizes)]
    prm = sets[0][1]
    prm["eta"] = 1.2
    b = BatchSystem(_abi.default_params(**prm), len(sizes))
    b.upload([parts for parts, _ in sets])
    b.update_iteration()
    key, ids = b.get("key"), b.get("id")
    o = 0
    for parts, _ in sets:
        n = len(parts["x"])
        s = BodySystem(_abi.default_params(**prm))
        s.upload(parts)
        s.update_iteration()
        assert np.array_equal(key[o:o + n], s.get("key"))
        assert np.array_equal(ids[o:o + n], s.get("id"))
        s.close()
        o += n
    b.close()


def with_cluster(n, m):
    """n random particles, m of them on a lattice of neighbouring keys that
    share the 32 bits by which the sort's passes order them, in random
    order (at 40,000 and 200 some lie in the next such cell)."""
    parts, prm = generators.random_box(n, seed=n + m)
    side = int(np.ceil(m ** (1.0 / 3.0)))
    q = np.random.default_rng(m).permutation(side ** 3)[:m]
    for d, k in enumerate(("x", "y", "z")):
        parts[k][1:2 * m:2] = 0.4 + 2e-6 * (q // side ** d % side)
    return parts, prm


@pytest.mark.parametrize("m", [2, 27, 32, 33, 34, 600])
@pytest.mark.parametrize("n", [1500, 12288, 12289, 40000])
def test_runs_of_equal_prefixes(oracle_mod, n, m):
    parts, prm = with_cluster(n, m)
    p = _abi.default_params(**prm)
    g, o = BodySystem(p), oracle_mod.OracleSystem(p, threads=8)
    for s in (g, o):
        s.upload(parts)
        s.update_iteration()
        s.update_iteration()  # (of sorted particles)
    for f in ("key", "id", "x", "h"):
        assert np.array_equal(g.get(f), o.get(f)), f
    o.close()
    g.close()


@pytest.mark.parametrize("sizes,m", [((1300, 700, 900), 25),
                                     ((1300, 700, 900), 200),
                                     ((9000, 7000), 25), ((9000, 7000), 200)])
def test_runs_of_equal_prefixes_in_a_batch(sizes, m):
    sets = [with_cluster(n, m) for n in sizes]
    prm = sets[0][1]
    b = BatchSystem(_abi.default_params(**prm), len(sizes))
    b.upload([parts for parts, _ in sets])
    b.update_iteration()
    key, ids = b.get("key"), b.get("id")
    o = 0
    for parts, _ in sets:
        n = len(parts["x"])
        s = BodySystem(_abi.default_params(**prm))
        s.upload(parts)
        s.update_iteration()
        assert np.array_equal(key[o:o + n], s.get("key"))
        assert np.array_equal(ids[o:o + n], s.get("id"))
        s.close()
        o += n
    b.close()


@pytest.mark.parametrize("n", [1500, 12288, 12289])
def test_a_full_sort_is_remembered_until_the_next_upload(n):
    """Both forms: once a run of equal prefixes was too long, the following
    sorts take all key bits at once."""
    full = C.CDLL(os.path.join(os.path.dirname(_abi.__file__),
                               "libfsph_probe.so")).fsph_probe_sort_full
    full.restype = C.c_int64
    long_run, prm = with_cluster(n, 600)
    short_run, _ = with_cluster(n, 27)
    g = BodySystem(_abi.default_params(**prm))
    for parts, want in ((long_run, 1), (short_run, 0), (long_run, 1)):
        g.upload(parts)
        assert full(g._h) == 0
        for _ in range(3):
            g.update_iteration()
            assert full(g._h) == want
            assert np.all(np.diff(g.get("key").astype(np.int64)) > 0)
    g.close()
