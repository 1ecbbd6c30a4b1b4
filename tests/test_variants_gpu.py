"""The kernels' size-dependent variants at the sizes where they change over
(edges of slices, groups and rounds, remainders), against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from parm_amd import capi
from tests import systems as S
from tests import test_batch_gpu as B

pytestmark = pytest.mark.gpu


def _device_or_fail():
    if capi.device_count() < 1:
        pytest.fail("no GPU visible: the -m gpu tests need an MI355X")


# build slices of 8 and 16 atoms and their multiples: one less, equal, one more
@pytest.mark.parametrize("ndim", [2, 3])
@pytest.mark.parametrize("lj", [False, True])
def test_batch_build_slice_edges(ndim, lj):
    _device_or_fail()
    print(f"batch build edges ndim={ndim} lj={lj}", flush=True)
    sizes = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 600]
    systems = B.packings(sizes, 0.4 if lj else 0.64, ndim, seed=11 + ndim)
    b = B.make_batch(systems, ndim, 0.25, lj=lj)
    refs = B.oracle_systems(systems, ndim, 0.25, lj=lj)
    b.initialize()
    for s, r in enumerate(refs):
        r.initialize()
        fd, ld = b.pairs(s)
        fr, lr = r.pairs()
        assert np.array_equal(fd, fr) and np.array_equal(ld, lr), (s, sizes[s])
    b.close()


# the sort: from registers (up to 4096 atoms, 64 to a cell), by chunks (a cell of
# more: boxes of fewer than three cells per edge; a system of more), and a
# workgroup or a wavefront per system in the skin test; slices of 8 to 64 atoms
# (32, 16, 8 and 4 build lanes); runs shorter and longer than a graph's eight steps
@pytest.mark.parametrize("sizes,ndim,lj", [
    ([4097, 1, 64, 65, 66, 130], 3, False), ([4096, 8200, 2], 2, False),
    ([200, 3, 1000, 4500], 3, True), ([5] * 200 + [400], 3, True),
    ([4000] * 67 + [70], 3, False), ([4000] * 263 + [70], 2, False)])
def test_batch_sort_and_worklist(sizes, ndim, lj):
    _device_or_fail()
    print(f"batch sort {len(sizes)} systems ndim={ndim} lj={lj}", flush=True)
    if lj:
        systems = []
        for k, n in enumerate(sizes):
            x, L = S.jittered_lattice(n, 0.5, 3, seed=90 + k)
            systems.append(dict(n=n, L=float(L[0]), x=x, v=np.zeros((n, 3)),
                                types=np.zeros(n, np.int32), sig=np.ones(n)))
    else:
        systems = B.packings(sizes, 0.5, ndim, seed=31)
    b = B.make_batch(systems, ndim, 0.3, lj=lj)
    b.initialize()
    look = sorted({0, len(sizes) // 2, len(sizes) - 2, len(sizes) - 1})
    refs = dict(zip(look, B.oracle_systems([systems[k] for k in look], ndim, 0.3, lj=lj)))
    for r in refs.values():
        r.initialize()
    for steps in (0, 1, 10, 19):
        if steps:
            b.damped(0.004, 1.0, steps)
            for r in refs.values():
                r.damped(0.004, 1.0, steps)
        w, npairs = b.lists()
        for s, r in refs.items():
            fd, ld = b.pairs(s)
            fr, lr = r.pairs()
            assert np.array_equal(fd, fr) and np.array_equal(ld, lr), (s, steps)
            assert w[s] == r.which() and npairs[s] == len(fr), (s, steps)
    assert w.max() > 1
    b.close()


# the step loop queues launches ahead of the flags that may stop them: rebuilds
# at every step, at none, and on both sides of the run-ahead's size limit
@pytest.mark.parametrize("n,skin,steps", [(1, 0.3, 3), (300, 0.0, 1), (300, 0.0, 2),
                                          (300, 1e-3, 7), (1000, 0.05, 40),
                                          (33000, 0.02, 6)])
@pytest.mark.parametrize("damped", [False, True])
def test_step_loop_rebuild_schedule(n, skin, steps, damped):
    _device_or_fail()
    print(f"step loop n={n} skin={skin} steps={steps} damped={damped}", flush=True)
    x, L = S.jittered_lattice(n, 0.7, 3, seed=n) if n > 1 else (np.zeros((1, 3)), np.full(3, 9.0))
    v = S.gaussian_velocities(n, 3, 1.0, seed=n) if n > 1 else np.ones((1, 3))
    p = S.lj_params(n)
    t = O.PairTable(O.LJ_ATTRACT_REPULSE, p["eps"], p["sigma"], p["third"], p["types"])
    r = O.System(np.ones(n), L, t, p["diam"], skin, ndim=3, brute=False)
    s = capi.System(3, np.ones(n))
    s.set_box(L)
    s.nlist_set(skin, p["diam"])
    s.set_lj(p["eps"], p["sigma"], p["third"], p["types"])
    for q in (r, s):
        q.set_state(x=x, v=v, a=np.zeros_like(x))
        q.initialize()
    s.profile_enable(True)
    for _ in range(2):
        if damped:
            r.damped(0.002, 0.3, steps)
            s.damped(0.002, 0.3, steps)
        else:
            r.verlet(0.002, steps)
            s.verlet(0.002, steps)
    assert s.which() == r.which()
    assert s.profile_read()["step_launches"] == 2 * (steps - 1)
    xr, vr = r.state()[:2]
    xd, vd = s.state()[:2]
    assert np.abs(xd - xr).max() <= 1e-11 * max(1.0, np.abs(xr).max())
    assert np.abs(vd - vr).max() <= 1e-9 * max(1.0, np.abs(vr).max())
    s.close()


def test_step_loop_stops_at_nonfinite():
    _device_or_fail()
    n = 2000
    x, L = S.jittered_lattice(n, 0.7, 3, seed=4)
    s = capi.System(3, np.ones(n))
    s.set_box(L)
    s.nlist_set(0.3, np.full(n, 2.5))
    s.set_lj([[1.0]], [1.0], [2.5], np.zeros(n, np.int32))
    v = np.zeros_like(x)
    v[17, 1] = np.inf
    s.set_state(x=x, v=v, a=np.zeros_like(x))
    s.initialize()
    with pytest.raises(capi.ParmError) as e:
        s.verlet(0.002, 8)
    assert e.value.code == capi.E_NONFINITE and "step 0" in str(e.value)
    s.close()


# atoms falling together: rebuilds inside a run whose rows outgrow the list's
# capacity and whose stencils outgrow the build's bound, with step launches
# already queued behind the build that does not stand
@pytest.mark.parametrize("tiled", ["0", "1"])
@pytest.mark.parametrize("n,ndim,steps", [(600, 3, 60), (600, 2, 15), (6000, 3, 40)])
def test_rebuilds_outgrow_the_list_inside_a_run(monkeypatch, tiled, n, ndim, steps):
    _device_or_fail()
    print(f"outgrow tiled={tiled} n={n} ndim={ndim} steps={steps}", flush=True)
    monkeypatch.setenv("PARM_TILED", tiled)
    monkeypatch.setenv("PARM_TPA", "4")
    rng = np.random.default_rng(n + ndim)
    edge = 2.2 * n ** (1.0 / ndim)
    L = np.full(ndim, edge)
    x = rng.uniform(0, edge, (n, ndim))
    v = -(x - edge / 2) * 0.85  # all but together at t = 1
    t = O.PairTable(O.REPULSION, [1e-6], [1.0], [2.0], np.zeros(n, np.int32))
    r = O.System(np.ones(n), L, t, np.ones(n), 0.4, ndim=ndim, brute=False)
    s = capi.System(ndim, np.ones(n))
    s.set_box(L)
    s.nlist_set(0.4, np.ones(n))
    s.set_repulsion([1e-6], [1.0], [2.0], np.zeros(n, np.int32))
    for q in (r, s):
        q.set_state(x=x, v=v, a=np.zeros_like(x))
        q.initialize()
    cap = s.list_info()["capacity"]
    for _ in range(2):
        for q in (r, s):
            q.verlet(0.5 / steps, steps)
        assert s.which() == r.which()
        fd, ld = s.pairs()
        fr, lr = r.pairs()
        assert np.array_equal(fd, fr) and np.array_equal(ld, lr)
        xr, xd = r.state()[0], s.state()[0]
        assert np.abs(xd - xr).max() <= 1e-12 * np.abs(xr).max()
    assert s.list_info()["capacity"] > cap and s.which() > 10
    s.close()


# the tiled LJ pair loop: several types (table and type bytes in LDS), counts
# that are no multiple of a group, folded (small box) and plain offsets, and
# pairs at the cutoff itself
@pytest.mark.parametrize("tpa", [1, 4, 8])
@pytest.mark.parametrize("ntypes", [1, 3, 16])
@pytest.mark.parametrize("n", [65, 500, 6000])
def test_tiled_lj_group_edges(monkeypatch, tpa, ntypes, n):
    _device_or_fail()
    print(f"tiled lj tpa={tpa} ntypes={ntypes} n={n}", flush=True)
    monkeypatch.setenv("PARM_TPA", str(tpa))
    monkeypatch.setenv("PARM_TILED", "1")
    x, L = S.jittered_lattice(n, 0.75, 3, seed=n + ntypes)
    rng = np.random.default_rng(ntypes)
    types = rng.integers(0, ntypes, n).astype(np.int32)
    eps = rng.uniform(0.5, 1.5, (ntypes, ntypes))
    eps = (eps + eps.T) / 2
    sigma = rng.uniform(0.8, 1.0, ntypes)
    cut = rng.uniform(1.5, 2.2, ntypes)
    # pairs of atoms exactly at their cutoff along x (inside: d2 / sig2 > cut2 is false)
    if ntypes == 1:
        x[1] = x[0] + [sigma[0] * cut[0], 0, 0]
    diam = (sigma * cut)[types]
    t = O.PairTable(O.LJ_ATTRACT_REPULSE, eps, sigma, cut, types)
    s = capi.System(3, np.ones(n))
    s.set_box(L)
    s.nlist_set(0.3, diam)
    s.set_lj(eps, sigma, cut, types)
    s.set_state(x=x)
    s.update_list(True)
    s.set_forces(False)
    assert s.list_info()["tiled"]
    first, last = O.nlist(x, L, diam, 0.3)
    S.assert_fp64_forces(s.forces(), O.forces(x, L, t, first, last), x, L, t, first, last)
    s.close()


# LJ of so many types that LDS has no room for their table beside the stencil
# (FP64: from about 25 on, mixed: 45): the tiled list all the same, rows from memory
@pytest.mark.parametrize("prec", [capi.FP64, capi.MIXED])
@pytest.mark.parametrize("ndim,n,tpa", [(3, 500, 4), (3, 6000, 8), (2, 3000, 1)])
@pytest.mark.parametrize("ntypes", [20, 33, 64])
def test_tiled_lj_many_types(monkeypatch, ntypes, ndim, n, tpa, prec):
    _device_or_fail()
    print(f"tiled lj ntypes={ntypes} ndim={ndim} n={n} tpa={tpa} prec={prec}", flush=True)
    monkeypatch.setenv("PARM_TPA", str(tpa))
    monkeypatch.setenv("PARM_TILED", "1")
    x, L = S.jittered_lattice(n, 0.75, ndim, seed=n + ntypes)
    rng = np.random.default_rng(ntypes)
    types = rng.integers(0, ntypes, n).astype(np.int32)
    types[:ntypes] = np.arange(ntypes)
    eps = rng.uniform(0.5, 1.5, (ntypes, ntypes))
    eps = (eps + eps.T) / 2
    sigma = rng.uniform(0.8, 1.0, ntypes)
    cut = rng.uniform(1.5, 2.2, ntypes)
    diam = (sigma * cut)[types]
    t = O.PairTable(O.LJ_ATTRACT_REPULSE, eps, sigma, cut, types)
    v = S.gaussian_velocities(n, ndim, 0.5, seed=n)
    s = capi.System(ndim, np.ones(n), prec)
    s.set_box(L)
    s.nlist_set(0.3, diam)
    s.set_lj(eps, sigma, cut, types)
    s.set_state(x=x, v=v, a=np.zeros_like(x))
    s.update_list(True)
    s.set_forces(False)
    assert s.list_info()["tiled"]
    first, last = O.nlist(x, L, diam, 0.3)
    ref = O.forces(x, L, t, first, last)
    u = s.pair_sums()["U"]
    if prec == capi.FP64:
        S.assert_fp64_forces(s.forces(), ref, x, L, t, first, last)
        assert abs(u - ref["U"]) <= 1e-12 * max(1.0, abs(ref["U"]))
        r = O.System(np.ones(n), L, t, diam, 0.3, ndim=ndim, brute=False)
        r.set_state(x=x, v=v, a=np.zeros_like(x))
        for q in (r, s):
            q.initialize()
            q.verlet(0.001, 5)
        assert np.abs(s.positions() - r.state()[0]).max() <= 1e-12 * max(1.0, np.abs(x).max())
    else:
        # two offsets of up to ~10 sigma rounded to FP32 (half an ulp: 5e-7 each)
        # move a pair force by 14 |dr| / r = 1.6e-5 of its terms; three times that
        scale = S.pair_term_scale(x, L, t, first, last)
        d = np.sqrt(((s.forces() - ref["f"]) ** 2).sum(1))
        assert np.all(d <= 5e-5 * scale + 1e-12)
    s.close()


# 16 and 32 lanes per atom: rows shorter than the lanes, rows of more than the
# entries in flight per lane, both pair kinds, the largest system of either
@pytest.mark.parametrize("lanes,n", [(16, 2), (16, 700), (16, 1 << 14), (32, 2), (32, 700),
                                     (32, 1 << 13)])
@pytest.mark.parametrize("lj", [True, False])
def test_wide_untiled_lanes(monkeypatch, lanes, n, lj):
    _device_or_fail()
    print(f"wide lanes={lanes} n={n} lj={lj}", flush=True)
    monkeypatch.setenv("PARM_TPA", str(lanes))
    monkeypatch.setenv("PARM_TILED", "0")
    x, L = S.jittered_lattice(n, 0.8, 3, seed=n) if n > 2 else (np.array([[0.1, 0, 0], [1.2, 0, 0]]),
                                                               np.full(3, 6.0))
    v = S.gaussian_velocities(n, 3, 0.5, seed=n)
    s = capi.System(3, np.ones(n))
    s.set_box(L)
    if lj:
        p = S.lj_params(n, sigcut=3.2 if n == 700 else 2.5)
        t = O.PairTable(O.LJ_ATTRACT_REPULSE, p["eps"], p["sigma"], p["third"], p["types"])
        s.nlist_set(0.3, p["diam"])
        s.set_lj(p["eps"], p["sigma"], p["third"], p["types"])
    else:
        p = S.bidisperse_repulsion(n, n)
        t = O.PairTable(O.REPULSION, p["eps"], p["sigma"], p["third"], p["types"])
        s.nlist_set(0.3, p["diam"])
        s.set_repulsion(p["eps"], p["sigma"], p["third"], p["types"])
    s.set_state(x=x, v=v, a=np.zeros_like(x))
    s.update_list(True)
    s.set_forces(False)
    assert s.list_info()["lanes"] == lanes
    first, last = O.nlist(x, L, p["diam"], 0.3)
    ref = O.forces(x, L, t, first, last)
    S.assert_fp64_forces(s.forces(), ref, x, L, t, first, last)
    fd, ld = s.pairs()
    assert np.array_equal(fd, first) and np.array_equal(ld, last)
    assert abs(s.pair_sums()["U"] - ref["U"]) <= 1e-12 * max(1.0, abs(ref["U"]))
    r = O.System(np.ones(n), L, t, p["diam"], 0.3, ndim=3, brute=n < 1000)
    r.set_state(x=x, v=v, a=np.zeros_like(x))
    for q in (r, s):
        q.initialize()
        q.verlet(0.001, 5)
    assert s.which() == r.which()
    xr, xd = r.state()[0], s.state()[0]
    assert np.abs(xd - xr).max() <= 1e-12 * max(1.0, np.abs(xr).max())
    s.close()


# mixed precision with a lane's first entries in flight ahead of the loop (8 lanes
# and more)
@pytest.mark.parametrize("lanes,n", [(8, 2), (8, 701), (16, 2), (16, 701), (32, 2), (32, 701),
                                     (32, 1 << 13)])
@pytest.mark.parametrize("form", ["lj", "harmonic", "hertz"])
def test_wide_untiled_lanes_mixed(monkeypatch, lanes, n, form):
    _device_or_fail()
    print(f"wide mixed lanes={lanes} n={n} {form}", flush=True)
    monkeypatch.setenv("PARM_TPA", str(lanes))
    monkeypatch.setenv("PARM_TILED", "0")
    x, L = S.jittered_lattice(n, 0.8, 3, seed=n) if n > 2 else (np.array([[0.1, 0, 0], [1.2, 0, 0]]),
                                                               np.full(3, 6.0))
    s = capi.System(3, np.ones(n), capi.MIXED)
    s.set_box(L)
    if form == "lj":
        p = S.lj_params(n, sigcut=3.2 if n == 701 else 2.5)
        t = O.PairTable(O.LJ_ATTRACT_REPULSE, p["eps"], p["sigma"], p["third"], p["types"])
        s.nlist_set(0.3, p["diam"])
        s.set_lj(p["eps"], p["sigma"], p["third"], p["types"])
    else:
        e = 2.0 if form == "harmonic" else 2.5
        p = S.bidisperse_repulsion(n, n, exponent=(e, e))
        t = O.PairTable(O.REPULSION, p["eps"], p["sigma"], p["third"], p["types"])
        s.nlist_set(0.3, p["diam"])
        s.set_repulsion(p["eps"], p["sigma"], p["third"], p["types"])
    s.set_state(x=x)
    s.update_list(True)
    s.set_forces(False)
    assert s.list_info()["lanes"] == lanes
    first, last = O.nlist(x, L, p["diam"], 0.3)
    ref = O.forces(x, L, t, first, last)
    d = np.sqrt(((s.forces() - ref["f"]) ** 2).sum(1))
    assert np.all(d <= 2e-5 * ref["fabs"] + 1e-6), np.max(d - 2e-5 * ref["fabs"])
    s.close()


# the autotuner's candidates for mixed repulsion of many atoms differ in time only:
# one lane adds the even and the odd entries apart, as two lanes do
@pytest.mark.parametrize("ndim,n", [(2, 63), (2, 3001), (3, 2), (3, 1500)])
@pytest.mark.parametrize("exponent", [2.0, 2.5])
def test_mixed_repulsion_one_lane_adds_as_two(monkeypatch, ndim, n, exponent):
    _device_or_fail()
    print(f"one lane as two ndim={ndim} n={n} exponent={exponent}", flush=True)
    monkeypatch.setenv("PARM_TILED", "0")
    rng = np.random.default_rng(n)
    p = S.bidisperse_repulsion(n, n, exponent=(exponent, exponent))
    L = np.full(ndim, max(4.5, (0.9 * n) ** (1 / ndim)))
    x = rng.uniform(0, 1, (n, ndim)) * L
    v = rng.normal(size=(n, ndim)) * 0.1
    out = []
    for tpa in ("1", "2"):
        monkeypatch.setenv("PARM_TPA", tpa)
        s = capi.System(ndim, np.ones(n), capi.MIXED)
        s.set_box(L)
        s.nlist_set(0.3, p["diam"])
        s.set_repulsion(p["eps"], p["sigma"], p["third"], p["types"])
        s.set_state(x=x, v=v, a=np.zeros_like(x))
        s.initialize()
        f = s.forces()
        s.damped(0.02, 0.5, 12)
        assert s.list_info()["lanes"] == int(tpa)
        out.append((f, *s.state()))
        s.close()
    assert n < 10 or np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# 16 and 32 lanes per atom in a batch: systems smaller than a group, odd sizes
@pytest.mark.parametrize("prec", [capi.FP64, capi.MIXED])
@pytest.mark.parametrize("lj", [False, True])
@pytest.mark.parametrize("lanes", [16, 32])
def test_batch_wide_lanes(monkeypatch, lanes, lj, prec):
    _device_or_fail()
    print(f"batch lanes={lanes} lj={lj} prec={prec}", flush=True)
    monkeypatch.setenv("PARM_TPA", str(lanes))
    if lj:
        systems = []
        for k, n in enumerate([3, 33, 300, 701]):
            x, L = S.jittered_lattice(n, 0.5, 3, seed=70 + k)
            systems.append(dict(n=n, L=float(L[0]), x=x, v=S.gaussian_velocities(n, 3, 0.5, seed=k),
                                types=np.zeros(n, np.int32), sig=np.ones(n)))
    else:
        systems = B.packings([1, 2, 31, 33, 300, 701], 0.64, 3, seed=8)
    b = B.make_batch(systems, 3, 0.25, prec=prec, lj=lj)
    refs = B.oracle_systems(systems, 3, 0.25, lj=lj)
    b.initialize()
    for s, r in enumerate(refs):
        r.initialize()
        fd, ld = b.pairs(s)
        fr, lr = r.pairs()
        assert np.array_equal(fd, fr) and np.array_equal(ld, lr), s
    if prec == capi.FP64:
        B._compare(b, refs, systems, 1e-12, 0)
        for q in (b, *refs):
            q.damped(0.004, 0.5, 10)
        B._compare(b, refs, systems, 1e-12, 10)
    else:
        f, off = b.state()[3], b.offsets
        for s, (q, r) in enumerate(zip(systems, refs)):
            t = (O.PairTable(O.LJ_ATTRACT_REPULSE, [[1.0, 1.0], [1.0, 1.0]], [1.0, 1.4],
                             [2.5, 2.5], q["types"]) if lj else
                 O.PairTable(O.REPULSION, B.REP["eps"], B.REP["sigma"], B.REP["third"], q["types"]))
            ref = O.forces(q["x"], [q["L"]] * 3, t, *r.pairs())
            d = np.sqrt(((f[off[s]:off[s + 1]] - ref["f"]) ** 2).sum(1))
            assert np.all(d <= 2e-5 * ref["fabs"] + 1e-6), s
    b.close()


# the build of a large sparse 2D system (two lanes of four candidates) with one
# diameter, and with ignored pairs, for either list
@pytest.mark.parametrize("tiled", ["0", "1"])
@pytest.mark.parametrize("one_diameter,ignored", [(True, 0), (True, 3000), (False, 3000)])
def test_flat_build_variants(monkeypatch, tiled, one_diameter, ignored):
    _device_or_fail()
    print(f"flat build tiled={tiled} one={one_diameter} ignored={ignored}", flush=True)
    monkeypatch.setenv("PARM_TILED", tiled)
    n, edge = 100003, 270.0  # (dense enough that no tile is wider than its limit)
    rng = np.random.default_rng(ignored + one_diameter)
    L = np.full(2, edge)
    x = rng.uniform(0, edge, (n, 2))
    x[::2000] += rng.integers(-2, 3, (len(x[::2000]), 2)) * edge
    diam = np.ones(n) if one_diameter else rng.uniform(0.8, 1.0, n)
    first, last = O.nlist(x, L, diam, 0.3)
    pick = rng.permutation(len(first))[:ignored]
    ex = np.stack([first[pick], last[pick]], -1).astype(np.int32)
    s = capi.System(2, np.ones(n))
    s.set_box(L)
    s.nlist_set(0.3, diam)
    if ignored:
        s.ignore(ex[:, 0], ex[:, 1])
        keep = np.ones(len(first), bool)
        keep[pick] = False
        first, last = first[keep], last[keep]
    s.set_repulsion([1.0], [1.0], [2.0], np.zeros(n, np.int32))
    s.set_state(x=x)
    for _ in range(2):
        s.update_list(True)
        fd, ld = s.pairs()
        assert np.array_equal(fd, first) and np.array_equal(ld, last)
    assert s.list_info()["tiled"] == (tiled == "1")
    s.close()


# rebuilds inside a run on the untiled list, step launches queued behind them, with
# ignored pairs and with an ignore between two runs
def test_rebuilds_inside_a_run_with_ignored_pairs(monkeypatch):
    _device_or_fail()
    print("deferred rebuilds, ignored pairs", flush=True)
    monkeypatch.setenv("PARM_TILED", "0")
    monkeypatch.setenv("PARM_TPA", "4")
    n = 6000
    x, L = S.jittered_lattice(n, 0.7, 3, seed=3)
    v = S.gaussian_velocities(n, 3, 1.0, seed=3)
    p = S.lj_params(n)
    t = O.PairTable(O.LJ_ATTRACT_REPULSE, p["eps"], p["sigma"], p["third"], p["types"])
    r = O.System(np.ones(n), L, t, p["diam"], 0.05, ndim=3, brute=False)
    s = capi.System(3, np.ones(n))
    s.set_box(L)
    s.nlist_set(0.05, p["diam"])
    s.set_lj(p["eps"], p["sigma"], p["third"], p["types"])
    first, last = O.nlist(x, L, p["diam"], 0.05)
    pick = np.random.default_rng(1).permutation(len(first))[:800]
    for q in (r, s):
        q.set_state(x=x, v=v, a=np.zeros_like(x))
    for part in (pick[:400], pick[400:]):
        s.ignore(first[part], last[part])
        for k in part:
            r.ignore(first[k], last[k])
        for q in (r, s):
            if part[0] == pick[0]:
                q.initialize()
            q.verlet(0.002, 14)
        assert s.which() == r.which()
        fd, ld = s.pairs()
        fr, lr = r.pairs()
        assert np.array_equal(fd, fr) and np.array_equal(ld, lr)
        xr, xd = r.state()[0], s.state()[0]
        assert np.abs(xd - xr).max() <= 1e-11 * max(1.0, np.abs(xr).max())
    assert s.which() > 6
    s.close()


# the counted order and the tile plan: one workgroup (up to 8192 atoms and cells)
# and several launches, one and several scan tiles of cells,
# several rows to a plan workgroup, crowded cells, empty rows, the build lanes of a
# large 2D system, and a rebuild on
# top of the order of the one before
@pytest.mark.parametrize("n,ndim,edge,clustered", [
    (1, 3, 9.0, False), (2, 2, 9.0, False), (63, 3, 4.0, False), (65, 2, 12.0, True),
    (1500, 3, 40.0, False), (1500, 3, 40.0, True), (3000, 2, 150.0, False),
    (8192, 2, 60.0, False), (8192, 3, 20.0, False), (8193, 3, 20.0, False), (70000, 3, 84.0, False),
    (99999, 2, 400.0, False), (100000, 2, 400.0, False)])
def test_counted_order_and_tile_plan(n, ndim, edge, clustered):
    _device_or_fail()
    print(f"counted order n={n} ndim={ndim} edge={edge} clustered={clustered}", flush=True)
    rng = np.random.default_rng(n + ndim)
    L = np.full(ndim, edge)
    x = rng.uniform(0, edge / (6 if clustered else 1), (n, ndim))
    x += rng.integers(-2, 3, (n, ndim)) * edge
    diam = rng.uniform(0.8, 1.0, n)
    s = capi.System(ndim, np.ones(n))
    s.set_box(L)
    s.nlist_set(0.3, diam)
    t = O.PairTable(O.REPULSION, [1.0], [1.0], [2.0], np.zeros(n, np.int32))
    r = O.System(np.ones(n), L, t, diam, 0.3, ndim=ndim, brute=False)
    for _ in range(2):
        s.set_state(x=x)
        r.set_state(x=x)
        s.update_list(True)
        r.update_list(True)
        fd, ld = s.pairs()
        fr, lr = r.pairs()
        assert np.array_equal(fd, fr) and np.array_equal(ld, lr)
        assert np.array_equal(s.positions(), x)
        x = x + rng.normal(scale=0.4, size=x.shape)
    s.close()


# a slab of more than 131,072 short rows (up to 256 to a plan workgroup): a cubic
# lattice in random order, whose atoms all have 32 neighbours within the list
# radius and no net force
def test_tile_plan_of_many_rows(monkeypatch):
    _device_or_fail()
    print("tile plan of many rows", flush=True)
    monkeypatch.setenv("PARM_TILED", "1")
    m, a = (7, 812, 812), 1.08
    n = m[0] * m[1] * m[2]
    rng = np.random.default_rng(5)
    x = np.stack(np.unravel_index(rng.permutation(n), m), -1) * a + rng.uniform(-9, 9, 3)
    s = capi.System(3, np.ones(n))
    s.set_box(np.array(m) * a)
    s.nlist_set(0.3, np.full(n, 2.1))
    s.set_lj([[1.0]], [1.0], [2.1], np.zeros(n, np.int32))
    s.set_state(x=x)
    for _ in range(2):
        s.update_list(True)
        assert s.list_info()["tiled"] and s.numpairs() == 16 * n
    s.set_forces(False)
    assert np.abs(s.forces()).max() <= 1e-10
    s.close()


# the minimiser's sums out of the force launch: fixed atoms (no dot products,
# a = 0), both list layouts, workgroup edges
@pytest.mark.parametrize("tiled", ["0", "1"])
@pytest.mark.parametrize("ndim,n", [(2, 63), (3, 257), (2, 900), (3, 2000)])
def test_nlcg_point_sums(monkeypatch, tiled, ndim, n):
    _device_or_fail()
    print(f"nlcg sums tiled={tiled} ndim={ndim} n={n}", flush=True)
    monkeypatch.setenv("PARM_TILED", tiled)
    p = B.packings([n], 0.6, ndim, seed=n)[0]
    m = np.ones(n)
    m[::7] = np.inf
    x, L = p["x"], [p["L"]] * ndim
    t = O.PairTable(O.REPULSION, B.REP["eps"], B.REP["sigma"], B.REP["third"], p["types"])
    r = O.System(m, L, t, p["sig"], 0.3, ndim=ndim)
    s = capi.System(ndim, m)
    s.set_box(L)
    s.nlist_set(0.3, p["sig"])
    s.set_repulsion(B.REP["eps"], B.REP["sigma"], B.REP["third"], p["types"])
    for q in (r, s):
        q.set_state(x=x, v=np.zeros_like(x), a=np.ones_like(x))
    c, cr = capi.NLCG(s, 0.1, 1e-2), O.NLCG(r, 0.1, 1e-2)
    for q in (c, cr):
        q.set_limits(stepmax=1e-2)
        q.timestep(4)
    d, dr = c.info(), cr.info()
    assert d["sec"] == dr["sec"] and d["k"] == dr["k"]
    for key in ("alpha", "dxsum", "vl", "fl", "al", "Knew", "beta"):
        assert abs(d[key] - dr[key]) <= 1e-9 * (abs(dr[key]) + 1e-12), key
    for a, b in zip(s.state(), r.state()):
        assert np.abs(a - b).max() <= 1e-9 * max(1.0, np.abs(b).max())
    c.close()
    s.close()
