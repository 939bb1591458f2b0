"""State checks (check_nans, check_negativity, default_physics.h:918-979):
the driver's step returns FSPH_E_NAN / FSPH_E_NEG as the reference's
asserts would stop the run, and the oracle agrees on the same input."""
import ctypes as C
import os

import numpy as np
import pytest

from flecsph_amd import BodySystem, FsphError, _abi, generators

pytestmark = pytest.mark.gpu


def _case():
    parts, prm = generators.random_box(3000, seed=41, h_spread=0.5)
    return dict(parts), dict(prm, precision=_abi.PREC_FP32)


def test_nan_in_u_stops_the_step(oracle_mod):
    parts, prm = _case()
    parts["u"] = parts["u"].copy()
    parts["u"][1234] = np.nan
    p = _abi.default_params(**prm)
    print("nan in u of particle 1234, initial iteration", flush=True)
    g = BodySystem(p)
    g.upload(parts)
    with pytest.raises(FsphError) as e:
        g.step()  # the initial iteration (no drift: positions stay finite)
    assert e.value.code == _abi.FSPH_E_NAN
    g.close()
    o = oracle_mod.OracleSystem(p, threads=4)
    o.upload(parts)
    o.step()
    assert oracle_mod.load().fo_check_state(o._h) == _abi.FSPH_E_NAN


def test_negative_internal_energy_is_reported(oracle_mod):
    parts, prm = _case()
    parts["u"] = parts["u"].copy()
    parts["u"][17] = -1.0
    p = _abi.default_params(**prm)
    g = BodySystem(p)
    g.upload(parts)
    with pytest.raises(FsphError) as e:
        g.check_state()
    assert e.value.code == _abi.FSPH_E_NEG
    assert "id 17" in str(e.value)
    g.close()
    o = oracle_mod.OracleSystem(p, threads=4)
    o.upload(parts)
    assert oracle_mod.load().fo_check_state(o._h) == _abi.FSPH_E_NEG


def test_clean_state_passes_and_checks_can_be_turned_off():
    parts, prm = _case()
    g = BodySystem(_abi.default_params(**prm))
    g.upload(parts)
    for _ in range(3):
        g.step()
    g.check_state()
    parts["u"] = parts["u"].copy()
    parts["u"][5] = -1.0
    g.upload(parts)
    g.set_checks(False)
    g.step()  # not checked
    with pytest.raises(FsphError):
        g.check_state()
    g.close()


def test_a_drift_needs_a_new_tree_before_the_neighbour_passes():
    """After fsph_integrate drifts the particles, the tree and tiles no
    longer describe them: the passes that use them (density, the Newton-h
    and learned-h updates) fail with FSPH_E_ARG until
    fsph_update_iteration, the order of hydro/main_driver.cc:187-193; a
    kick alone leaves them valid."""
    parts, prm = _case()
    g = BodySystem(_abi.default_params(**dict(prm, h_mode=_abi.H_NEWTON)))
    g.upload(parts)
    g.step()
    g.integrate(_abi.KICK_V)
    g.density_eos()
    g.integrate(_abi.DRIFT)
    for call in (g.density_eos, g.update_h):
        with pytest.raises(FsphError) as e:
            call()
        assert e.value.code == _abi.FSPH_E_ARG
    g.update_iteration()
    g.density_eos()
    g.update_h()
    g.close()


def _probe(name, g, *args):
    """A function of libfsph_probe.so (flecsph_amd/host/ctx_probe.cpp) on
    g's context."""
    lib = C.CDLL(os.path.join(os.path.dirname(_abi.__file__),
                              "libfsph_probe.so"))
    fn = getattr(lib, "fsph_probe_" + name)
    fn.restype = C.c_int64
    return fn(g._h, *args)


@pytest.mark.parametrize("n", [5000, 280_001])
def test_nan_position_under_newton_h_is_reported(n):
    """A particle whose position is not a number (its key is the lowest, so
    it is the first of a tile) meets nothing: the solver's gather tiles stay
    as small as without it, the step reports the NaN, and the context works
    after an upload of sound data."""
    parts, prm = generators.random_box(n, seed=5, h_spread=0.3)
    prm.update(h_mode=_abi.H_NEWTON, n_target=40)
    bad = dict(parts)
    for k in ("x", "y", "z"):
        bad[k] = parts[k].copy()
        bad[k][n // 2] = np.nan
    sizes = []
    for p in (parts, bad):
        g = BodySystem(_abi.default_params(**prm))
        g.upload(p)
        if p is bad:
            print("one particle of", n, "without a position", flush=True)
            with pytest.raises(FsphError) as e:
                g.step()
            assert e.value.code == _abi.FSPH_E_NAN
        else:
            g.step()
        sizes.append((C.c_int64 * 2)())
        _probe("gather", g, sizes[-1])
    assert list(sizes[1]) == list(sizes[0])
    g.upload(parts)
    g.step()
    h = g.get("h")
    assert np.all(np.isfinite(h)) and np.all(h > 0)
    g.close()


def test_check_state_keeps_an_unread_scan_stall():
    """A stalled scan whose result nothing has read yet stays on record
    through a state check, until the next update_iteration: the next call
    that needs a scan fails."""
    parts, prm = _case()
    g = BodySystem(_abi.default_params(**prm))
    g.upload(parts)
    g.step()
    assert _probe("scan_stall", g, 1) == 1
    g.check_state()
    assert _probe("scan_stall", g, 0) == 1
    with pytest.raises(FsphError) as e:
        g.neighbor_lists()
    assert e.value.code == _abi.FSPH_E_HIP
    g.update_iteration()
    assert _probe("scan_stall", g, 0) == 0
    g.neighbor_lists()
    g.check_state()
    g.close()


def test_upload_needs_no_memory_beyond_the_fields():
    """rho, P and c are converted through the fields' own scratch."""
    parts, prm = _case()
    for given in ((), ("rho", "P", "c")):
        q = dict(parts)
        for k in ("rho", "P", "c"):
            q[k] = np.linspace(1.0, 2.0, len(q["x"])) if k in given else None
        g = BodySystem(_abi.default_params(**prm))
        g.upload(q)
        assert _probe("scratch_bytes", g) == 0
        for k in ("rho", "P", "c"):
            want = q[k] if k in given else np.zeros(len(q["x"]))
            assert np.array_equal(g.get(k), want.astype(np.float32))
        g.close()


@pytest.mark.parametrize("thermokinetic", [0, 1])
def test_phase_times_are_the_phases_own(thermokinetic):
    """With the timers on, each phase of a single simulation's step is timed
    by itself (the smoothing-length update is no part of the time step's),
    and the state is that of a step without timers."""
    parts, prm = _case()
    prm.update(thermokinetic=thermokinetic)
    runs = []
    for timed in (False, True):
        g = BodySystem(_abi.default_params(**prm))
        g.upload(parts)
        g.enable_timing(timed)
        for _ in range(3):
            g.step()
            if timed:
                t = g.phase_times()
                assert t["h"] > 0 and t["dt"] > 0 and t["integrate"] > 0
        runs.append([g.get(f) for f in ("x", "vx", "u", "e", "h", "rho")] +
                    [np.array(g.time())])
        g.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)
