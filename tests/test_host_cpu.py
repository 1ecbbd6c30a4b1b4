"""The library's host logic on a HIP runtime of host memory whose kernels do not
run (host_hip.hip): allocations and launches that are refused, list builds that
overflow or are refused.  Each case is a process of its own, in which that
runtime is loaded before the library."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NOMEM, UNSUPPORTED, DEVICE = -3, -4, -2
REBUILD = 1  # skin flag


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_hip")
    obj, so = str(d / "host_hip.o"), str(d / "libhost_hip.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-std=c++17",
                    "-O1", "-fPIC", "-c", os.path.join(ROOT, "tests", "host_hip.hip"), "-o", obj],
                   check=True)
    subprocess.run(["g++", "-shared", "-o", so, obj], check=True)
    return so


def _child(runtime, case, *args, **env):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), runtime, case,
                        *map(str, args)], capture_output=True, text=True, timeout=120, cwd=ROOT,
                       env={**os.environ, **env})
    assert r.returncode == 0, r.stdout + r.stderr


def _refused(code, f, *a):
    from parm_amd import capi
    try:
        f(*a)
    except (capi.ParmError, capi.ParmValueError) as e:
        assert e.code == code, e
    else:
        raise AssertionError("not refused")


# ------------------------------------------------------------------- batches
def _batch(hh, n=300, nsys=2):
    from parm_amd import capi
    b = capi.Batch(3, [n] * nsys, [[9.0] * 3] * nsys, 0.2)
    b.set_state(x=np.random.default_rng(0).uniform(0, 9, (n * nsys, 3)))
    return b


def _set_pair(b):
    b.set_repulsion([1.0], [1.0], [2.0], np.zeros(b.n, np.int32))


def case_batch_list_refused(hh, where):
    b = _batch(hh)
    if where == "set":      # the interaction's own list allocation
        hh.hh_alloc_limit(16 * b.n * 4 - 1)
        _refused(NOMEM, _set_pair, b)
        hh.hh_reset()
        _refused(-6, b.initialize)  # no interaction set
        _set_pair(b)
    else:                   # the growth of a list that overflowed
        _set_pair(b)
        hh.hh_overflows(1)
        hh.hh_fail_at(1)
        _refused(NOMEM, b.initialize)
        assert len(b.pairs(0)[0]) == 0
        hh.hh_reset()
    b.initialize()
    assert "k_batch_build" in hh.hh_log().decode()
    b.damped(0.01, 1.0, 12)
    assert hh.hh_bad() == 0
    b.close()


@pytest.mark.parametrize("where", ["set", "grow"])
def test_batch_list_refused(runtime, where):
    _child(runtime, "case_batch_list_refused", where)


# a list that grew in place (the freed block's address given out again): the
# captured run of steps holds the capacity that was
def case_graph_follows_the_list(hh):
    b = _batch(hh)
    _set_pair(b)
    b.initialize()
    b.damped(0.01, 1.0, 17)  # 16 steps in graphs, then the last
    b.damped(0.01, 1.0, 17)
    assert hh.hh_graphs() == 1
    hh.hh_overflows(1)
    b.initialize()
    b.damped(0.01, 1.0, 17)
    assert hh.hh_graphs() == 2 and hh.hh_bad() == 0
    b.close()


def test_graph_follows_the_list(runtime):
    _child(runtime, "case_graph_follows_the_list", PARM_TPA="4")


# ------------------------------------------------------------- single systems
def _system(n=20000, **kw):
    from parm_amd import capi
    s = capi.System(3, np.ones(n))
    s.set_box([40.0] * 3)
    s.nlist_set(0.3, np.ones(n))
    s.set_repulsion([1.0], [1.0], [2.0], np.zeros(n, np.int32))
    s.set_state(x=np.random.default_rng(0).uniform(0, 40, (n, 3)))
    return s


def _log(hh):
    out = hh.hh_log().decode()
    hh.hh_clear_log()
    return out


# every allocation of a first list build refused in turn, and of one with more
# cells and tiles (a larger box): no launch goes through what is not there
def case_list_allocations_refused(hh, edge):
    refused = 0
    for k in range(1, 40):
        s = _system()
        if float(edge) > 0:
            s.update_list(True)
            s.set_box([float(edge)] * 3)
        hh.hh_fail_at(k)
        try:
            s.update_list(True)
            done = True
        except RuntimeError as e:
            assert e.code == NOMEM
            done = False
            refused += 1
        hh.hh_fail_at(0)
        s.update_list(True)
        s.set_forces()
        s.verlet(0.001, 5)
        assert hh.hh_bad() == 0, k
        s.close()
        if done:
            break
    assert refused >= (8 if float(edge) == 0 else 5), refused


@pytest.mark.parametrize("edge", [0, 60])
def test_list_allocations_refused(runtime, edge):
    _child(runtime, "case_list_allocations_refused", edge)


# a rebuild inside a run, queued with step launches behind it or not, and the
# relaying of a list, whose row no lane could hold: the list is gone, and the
# next call that needs it builds one or is refused again
def case_refused_list_comes_back(hh, call):
    s = _system()
    s.update_list(True)
    s.update_list(True)  # (with the plan of the one before: built speculatively)
    built = s.which()
    assert built == 2
    if call == "set_pair":
        hh.hh_row(10 ** 7)
        _refused(UNSUPPORTED, s.set_repulsion, [1.0], [1.0], [2.0], np.zeros(s.n, np.int32))
    else:
        s.ignore([0], [1])  # an update that is due
        hh.hh_row(10 ** 7)
        _refused(UNSUPPORTED, s.verlet, 0.001, 6)
    assert s.which() == built and s.numpairs() == 0
    _log(hh)
    calls = dict(forces=s.set_forces, add=s.add_pair_forces, sums=s.pair_sums,
                 verlet=lambda: s.verlet(0.001, 4), damped=lambda: s.damped(0.001, 0.1, 4),
                 update=lambda: s.update_list(False), init=s.initialize,
                 tune=lambda: s.autotune(0.001), set_pair=s.set_forces)
    hh.hh_row(10 ** 7)
    _refused(UNSUPPORTED, calls[call])
    assert "k_force" not in _log(hh)
    calls[call]()
    first = [k for k in _log(hh).split() if "k_build" in k or "k_force" in k][0]
    assert "k_build" in first
    assert s.which() == built + 1 and s.numpairs() == 1
    s.update_list(False)
    assert s.which() == built + 1 and hh.hh_bad() == 0
    s.close()


@pytest.mark.parametrize("tiled", ["0", "1"])
@pytest.mark.parametrize("call", ["forces", "add", "sums", "verlet", "damped", "update", "init",
                                  "tune", "set_pair"])
def test_refused_list_comes_back(runtime, call, tiled):
    _child(runtime, "case_refused_list_comes_back", call, PARM_TILED=tiled, PARM_TPA="4")


# the minimiser's force launches, and the sums that may not allocate
def case_refused_list_nlcg(hh):
    from parm_amd import capi
    s = _system()
    c = capi.NLCG(s, 0.1, 1e-3)
    hh.hh_row(10 ** 7)
    _refused(UNSUPPORTED, s.update_list, True)
    out = C.c_void_p()
    assert capi.lib().parm_pair_sums_noalloc(s.h, C.byref(out)) == -6  # no list, by rule
    hh.hh_row(10 ** 7)
    _refused(UNSUPPORTED, c.timestep)
    _log(hh)
    c.timestep(1)
    assert "k_build" in [k for k in _log(hh).split() if "k_build" in k or "k_force" in k][0]
    assert hh.hh_bad() == 0


def test_refused_list_nlcg(runtime):
    _child(runtime, "case_refused_list_nlcg")


# a refused launch whose sums the host would read: the error of the force kernel is
# not lost in the launch of its reduction
def case_refused_sums_launch(hh, what):
    from parm_amd import capi
    s = _system()
    s.update_list(True)
    s.set_forces()
    c = capi.NLCG(s, 0.1, 1e-3) if what == "nlcg" else None
    hh.hh_refuse("7k_force" if os.environ["PARM_TILED"] == "0" else "k_force_tiled")
    _refused(DEVICE, s.pair_sums if what == "sums" else c.timestep)
    hh.hh_refuse("")
    (s.pair_sums if what == "sums" else c.timestep)()
    s.close()


@pytest.mark.parametrize("tiled", ["0", "1"])
@pytest.mark.parametrize("what", ["sums", "nlcg"])
def test_refused_sums_launch(runtime, what, tiled):
    _child(runtime, "case_refused_sums_launch", what, PARM_TILED=tiled, PARM_TPA="4")


# lanes given, layout by rule (mixed LJ of few atoms: untiled): the rule holds for
# the rebuilds after the tuning too
def case_tuned_layout_stays(hh):
    from parm_amd import capi
    n = 2000
    s = capi.System(3, np.ones(n), capi.MIXED)
    s.set_box([14.0] * 3)
    s.nlist_set(0.3, np.full(n, 2.5))
    s.set_lj([[1.0]], [1.0], [2.5], np.zeros(n, np.int32))
    s.set_state(x=np.random.default_rng(0).uniform(0, 14, (n, 3)))
    s.update_list(True)
    assert s.list_info()["tiled"]
    s.verlet(0.001, 16)
    assert not s.list_info()["tiled"]
    s.update_list(True)
    assert not s.list_info()["tiled"]
    s.close()


@pytest.mark.parametrize("tpa", ["", "4"])
def test_tuned_layout_stays(runtime, tpa):
    _child(runtime, "case_tuned_layout_stays", PARM_TPA=tpa)


# mixed repulsion of many atoms: the candidates that add up alike, unless rows
# are long, where more lanes are the faster
def case_repulsion_candidates(hh, row):
    from parm_amd import capi
    n = 100000
    s = capi.System(3, np.ones(n), capi.MIXED)
    s.set_box([60.0] * 3)
    s.nlist_set(0.3, np.ones(n))
    s.set_repulsion([1.0], [1.0], [2.0], np.zeros(n, np.int32))
    s.set_state(x=np.random.default_rng(0).uniform(0, 60, (n, 3)))
    hh.hh_entries(int(row) * n)
    s.update_list(True)
    _log(hh)
    s.autotune(0.001)
    lanes = {int(k.split("EEEv")[0].split("ELi")[-1]) for k in _log(hh).split()
             if "7k_forceI" in k}
    assert lanes == ({1, 2} if int(row) <= 16 else {1, 2, 4, 8}), lanes
    s.close()


@pytest.mark.parametrize("row", [6, 16, 17, 90])
def test_repulsion_candidates(runtime, row):
    _child(runtime, "case_repulsion_candidates", row)


# the most lanes per atom on both sides of the sizes where they change (lanes asked
# for beyond them leave the default of four)
def case_most_lanes(hh, n, lanes):
    s = _system(int(n))
    s.update_list(True)
    assert s.list_info()["lanes"] == int(lanes)
    s.set_forces()
    s.verlet(0.001, 3)
    assert hh.hh_bad() == 0
    s.close()


@pytest.mark.parametrize("n,ask,lanes", [(8192, 32, 32), (8193, 32, 4), (8193, 16, 16),
                                         (16384, 16, 16), (16385, 16, 4), (16385, 8, 8)])
def test_most_lanes(runtime, n, ask, lanes):
    _child(runtime, "case_most_lanes", n, lanes, PARM_TPA=str(ask), PARM_TILED="0")


# rows that one lane's 16-bit count cannot hold: fewer lanes are no candidate; and
# a candidate whose layout is refused leaves the lanes and the layout as they were
def case_tuning_long_rows(hh, refused):
    s = _system()
    if refused == "no":
        hh.hh_row(80000)
        s.update_list(True)
        assert s.list_info()["capacity"] >= 80000
        s.verlet(0.001, 16)
        assert s.list_info()["lanes"] > 1
    else:
        s.update_list(True)
        was = s.list_info()
        hh.hh_row(10 ** 7)
        _refused(UNSUPPORTED, s.verlet, 0.001, 16)
        assert s.list_info() == was
        s.verlet(0.001, 8)
        assert s.which() == 2  # (the list that was lost)
    assert hh.hh_bad() == 0
    s.close()


@pytest.mark.parametrize("refused", ["no", "yes"])
@pytest.mark.parametrize("tiled", ["", "0"])
def test_tuning_long_rows(runtime, tiled, refused):
    _child(runtime, "case_tuning_long_rows", refused, **({"PARM_TILED": tiled} if tiled else {}))


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    hh = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    hh.hh_log.restype = C.c_char_p
    hh.hh_alloc_limit.argtypes = [C.c_size_t]
    hh.hh_row.argtypes = hh.hh_entries.argtypes = [C.c_ulonglong]
    from parm_amd import capi
    assert capi.device_count() == 1 and hh.hh_bad() == 0
    globals()[sys.argv[2]](hh, *sys.argv[3:])
