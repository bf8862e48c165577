"""GPU parity of the WCSPH path (libdemsph.so on the MI355X) against the
FP64 oracle and the reference's own output frames.

Bit-exact: cell hashes, sort permutation, cell ranges, neighbour counts and
pair lists (as the reference's objectPointing arrays, in its order).
Tolerances (FP32 pair arithmetic, FP64 integration) are stated per test.
"""
from pathlib import Path

import numpy as np
import pytest

import oracle
import this_studio_amd as ts
from this_studio_amd import scenes

pytestmark = pytest.mark.gpu
GOLDEN = Path(__file__).resolve().parent / "golden"


def make_gpu(spec, capacity=None):
    s = ts.SPHScene()
    s.set_eos(spec.eos, spec.gamma)
    if capacity:
        s.set_capacity(*capacity)
    s.add_fluid(spec.fluid_pos, spec.fluid_vel, *spec.fluid_props())
    if spec.nd:
        s.add_dummy(spec.dummy_pos, spec.dummy_vel, spec.c0, spec.dx, spec.rho0, spec.nu)
    s.initialize(spec.min_bound, spec.max_bound, spec.gravity)
    return s


@pytest.mark.parametrize("n", [50000, 100000, 300000])
def test_build_cells_raw_matches_oracle(n):
    """Sizes cover the sort's two ways to its scatter bases: derived in the
    scatter from the digit table (up to 32 tiles of 2,048 keys) and a device
    scan of the table (49 and 147 tiles)."""
    import torch

    rng = np.random.default_rng(11)
    pos = rng.uniform(-0.1, 1.1, (n, 3))  # some points outside the domain exercise the clamps
    g = oracle.grid_set([0, 0, 0], [1.0, 0.7, 0.4], 0.021)
    ng = g.num_grids
    hv = oracle.hash_points(g, pos)
    sh, si = oracle.sort_by_hash(hv, ng)
    cs, ce = oracle.cell_ranges(sh, ng)
    dev = torch.device("cuda:0")
    dpos = torch.from_numpy(pos.reshape(-1)).to(dev)
    hidx = torch.empty(n, dtype=torch.int32, device=dev)
    hval = torch.empty(n, dtype=torch.int32, device=dev)
    dcs = torch.empty(ng, dtype=torch.int32, device=dev)
    dce = torch.empty(ng, dtype=torch.int32, device=dev)
    torch.cuda.synchronize()
    ts.build_cells(dpos.data_ptr(), hidx.data_ptr(), hval.data_ptr(), dcs.data_ptr(), dce.data_ptr(),
                   [g.minx, g.miny, g.minz], [g.maxx, g.maxy, g.maxz], [g.cx, g.cy, g.cz], [g.nx, g.ny, g.nz], ng, n)
    torch.cuda.synchronize()
    assert np.array_equal(hval.cpu().numpy(), sh)
    assert np.array_equal(hidx.cpu().numpy(), si)
    assert np.array_equal(dcs.cpu().numpy(), cs)
    assert np.array_equal(dce.cpu().numpy(), ce)


@pytest.fixture(scope="module")
def small():
    spec = scenes.small_dam_break()
    return spec


def test_neighbor_search_bit_exact(small):
    o = oracle.OracleSPH(small)
    s = make_gpu(small)
    o.neighbor_search()
    s.neighbor_search()
    assert np.array_equal(s.get("hashValue"), np.sort(o.get("hash"), kind="stable"))
    assert np.array_equal(s.get("hashIndex"), o.get("index"))
    # The reference re-hashes the dummies into the same cell arrays after the
    # fluid list is written (WCSPHSolver.h:218-231), so the oracle's final
    # cell arrays hold dummy ranges; the fluid ranges come from its fluid sort.
    g = o.grid()
    sh, _ = oracle.sort_by_hash(o.get("hash"), g.num_grids)
    cs, ce = oracle.cell_ranges(sh, g.num_grids)
    assert np.array_equal(s.get("cellHashStart"), cs)
    assert np.array_equal(s.get("cellHashEnd"), ce)
    assert np.array_equal(s.get("neighborCount"), o.get("count_ff"))
    assert np.array_equal(s.get("objectPointing"), o.get("pointing_ff"))
    assert np.array_equal(s.get("dummyNeighborCount"), o.get("count_fd"))
    assert np.array_equal(s.get("dummyObjectPointing"), o.get("pointing_fd"))


def test_dummy_normals_match_oracle(small):
    o = oracle.OracleSPH(small)
    s = make_gpu(small)
    # normals are stored in FP32: 1e-6 absolute on unit vectors
    np.testing.assert_allclose(s.get("dummyNormal"), o.get("dnormal"), atol=1e-6)


def _compare(s, o, pos_tol, vel_tol, rho_tol):
    dp = np.abs(s.get("position") - o.get("pos")).max()
    dv = np.abs(s.get("velocity") - o.get("vel")).max()
    dr = np.abs(s.get("density") - o.get("rho")).max()
    assert dp < pos_tol, dp
    assert dv < vel_tol, dv
    assert dr < rho_tol, dr
    return dp, dv, dr


def test_one_step_matches_oracle(small):
    o = oracle.OracleSPH(small)
    s = make_gpu(small)
    o.step(small.dt, 1)
    s.step(small.dt, 1)
    # one step: FP32 pair sums against FP64 -> |dv| <= 1e-6 m/s, |dx| <= dt*|dv|
    _compare(s, o, 1e-9, 1e-6, 1e-4)


def test_split_halves_equal_fused_step(small):
    a = make_gpu(small)
    b = make_gpu(small)
    for _ in range(3):
        a.neighbor_search()
        a.first_half(small.dt)
        a.second_half(small.dt)
    b.step(small.dt, 3)
    assert np.array_equal(a.get("position"), b.get("position"))
    assert np.array_equal(a.get("velocity"), b.get("velocity"))


def test_200_steps_match_oracle(small):
    o = oracle.OracleSPH(small)
    s = make_gpu(small)
    o.step(small.dt, 200)
    s.step(small.dt, 200)
    # 200 steps (0.037 s of collapse): relative to dx = 1e-2 m, <= 1e-5
    dp, dv, dr = _compare(s, o, 1e-7, 1e-4, 1e-2)
    assert dp / small.dx < 1e-5


def test_graph_replays_equal_eager_steps(small):
    """Two-step graph replays against eager launches, bit for bit, over
    several blocks with host work and extra neighbour searches (which flip
    the buffer parity and so exercise a second captured graph) in between."""
    a = make_gpu(small)
    b = make_gpu(small)
    b.set_graphs(False)
    for nsteps in (6, 5, 8, 3, 4):
        a.step(small.dt, nsteps)
        b.step(small.dt, nsteps)
        for f in ("position", "velocity", "densityChange"):
            assert np.array_equal(a.get(f), b.get(f)), (nsteps, f)
        a.neighbor_search()
        b.neighbor_search()
    assert a.graph_captures() >= 2
    assert b.graph_captures() == 0


def test_lane_settings_build_identical_lists_and_agree(small):
    """Every listLanes setting builds the same lists (entries and order);
    pairLanes settings differ only by FP32 summation order and each is
    deterministic."""
    ref = None
    for L in (1, 2, 4, 8):
        s = make_gpu(small)
        s.tune("listLanes", L)
        assert s.tuned("listLanes") == L
        s.neighbor_search()
        got = [s.get(f) for f in ("neighborCount", "objectPointing", "dummyNeighborCount", "dummyObjectPointing")]
        if ref is None:
            ref = got
        for a, b in zip(got, ref):
            assert np.array_equal(a, b), L
    base = None
    for L in (1, 2, 4, 8):
        runs = []
        for _ in range(2):
            s = make_gpu(small)
            s.tune("pairLanes", L)
            s.step(small.dt, 30)
            runs.append(s.get("position"))
        assert np.array_equal(runs[0], runs[1]), L
        if base is None:
            base = runs[0]
        # 30 steps of FP32 sums in another order: far below the spacing
        assert np.abs(runs[0] - base).max() < 1e-6 * small.dx, L


def test_gather_records_agree_with_fp64_records():
    """The pair passes gather 32-byte records holding each fluid neighbour's
    position in 32-bit fixed point (pairRecords 1), or the FP64 positions
    themselves (pairRecords 0).  The lists are the same; the steps agree to
    FP32 rounding, and both stay deterministic."""
    spec = scenes.dam_break(dx=0.01)  # 40 x 40 x 20 fluid
    runs, lists = {}, {}
    for mode in (1, 0, 1):
        s = make_gpu(spec)
        s.tune("pairRecords", mode)
        assert s.tuned("pairRecords") == mode
        s.neighbor_search()
        got = [s.get(f) for f in ("neighborCount", "objectPointing")]
        s.step(spec.dt, 40)
        res = [s.get(f) for f in ("position", "velocity", "densityChange")]
        if mode in runs:
            for a, b in zip(res, runs[mode]):
                assert np.array_equal(a, b), mode
        runs[mode], lists[mode] = res, got
    for a, b in zip(lists[0], lists[1]):
        assert np.array_equal(a, b)
    assert np.abs(runs[0][0] - runs[1][0]).max() < 1e-6 * spec.dx
    assert np.abs(runs[0][1] - runs[1][1]).max() < 1e-4


def test_gather_records_outside_the_grid_match_oracle():
    """With the grid's top face below the column's top row and the tank's
    upper dummies, those particles hash into the top layer of cells
    (clamped) while lying outside it, and a stencil centre can differ from the
    hashed cell.
    Both record forms still match the FP64 oracle over 50 steps."""
    spec = scenes.small_dam_break()
    spec.max_bound = np.array(spec.max_bound, dtype=float)
    spec.max_bound[2] = 0.085  # the column's top row is at z = 0.09
    o = oracle.OracleSPH(spec)
    o.step(spec.dt, 50)
    for mode in (1, 0):
        s = make_gpu(spec)
        s.tune("pairRecords", mode)
        assert s.tuned("pairRecords") == mode
        s.step(spec.dt, 50)
        _compare(s, o, 1e-7, 1e-4, 1e-2)


def test_autotune_restores_state_and_keeps_results(small):
    """Autotuning times its trials from a checkpoint and restores it: a tuned
    scene steps exactly like an untuned one.  In "exact" mode the result
    is bit-identical to the default knobs; in "pairs" mode it is
    bit-identical to a scene given the chosen knobs by hand."""
    ts.SPHScene.clear_autotune_cache()
    ref = make_gpu(small)
    ref.step(small.dt, 7)
    ref.step(small.dt, 20)
    a = make_gpu(small)
    a.step(small.dt, 7)  # tune mid-run, not only right after initialisation
    rep = a.autotune(small.dt, trial_steps=2, mode="exact", use_cache=False)
    print("[autotune] exact:", rep, flush=True)
    assert rep["configs"] == 7 and rep["cached"] == 0
    assert rep["listLanes"] in (1, 2, 4, 8) and rep["listPrefilter"] in (0, 1)
    assert a.tuned("listLanes") == rep["listLanes"]
    assert a.tuned("listPrefilter") == rep["listPrefilter"]
    assert a.tuned("pairLanes") == rep["pairLanes"] == rep["rulesPairLanes"]
    assert rep["listUs"] > 0 and rep["pairUs"] > 0 and rep["rulesListUs"] > 0
    a.step(small.dt, 20)
    for f in ("position", "velocity", "densityChange"):
        assert np.array_equal(a.get(f), ref.get(f)), f

    b = make_gpu(small)
    rep = b.autotune(small.dt, trial_steps=2, mode="pairs", use_cache=False)
    print("[autotune] pairs:", rep, flush=True)
    assert rep["configs"] == 11
    b.step(small.dt, 25)
    c = make_gpu(small)
    c.tune("listLanes", rep["listLanes"])
    c.tune("listPrefilter", rep["listPrefilter"])
    c.tune("pairLanes", rep["pairLanes"])
    c.step(small.dt, 25)
    for f in ("position", "velocity", "densityChange"):
        assert np.array_equal(b.get(f), c.get(f)), f

    # the size class is cached: a second scene takes the choice untimed
    d = make_gpu(small)
    rep2 = d.autotune(small.dt, mode="pairs")
    assert rep2["cached"] == 1 and rep2["configs"] == 0
    assert (rep2["listLanes"], rep2["listPrefilter"], rep2["pairLanes"]) == \
        (rep["listLanes"], rep["listPrefilter"], rep["pairLanes"])
    assert d.tuned("pairLanes") == rep["pairLanes"]
    ts.SPHScene.clear_autotune_cache()


def test_prefilter_keeps_pairs_at_the_cut_exact():
    """Shells of particles at |r| = cut (1 + u 1e-6), u in [-1, 1], around
    seeded centres: every decision falls inside the FP32 prefilter's band and
    is taken by the exact FP64 test, so the lists equal the oracle's with the
    prefilter on and off, at every lane count."""
    rng = np.random.default_rng(123)
    dx = 0.01
    cut = 2.0 * 1.3 * dx
    pts = []
    for c in rng.uniform(0.1, 0.4, (12, 3)):
        d = rng.normal(size=(60, 3))
        d /= np.linalg.norm(d, axis=1)[:, None]
        r = cut * (1.0 + rng.uniform(-1e-6, 1e-6, 60))
        pts.append(c)
        pts.append(c + d * r[:, None])
    pos = np.concatenate([np.atleast_2d(p) for p in pts])
    spec = scenes.SPHSceneSpec(fluid_pos=pos, dummy_pos=np.zeros((0, 3)), dx=dx, rho0=1000.0, c0=10.0, nu=1e-6,
                               min_bound=np.zeros(3), max_bound=np.full(3, 0.5), gravity=np.array([0.0, 0.0, -9.81]),
                               dt=1e-5)
    o = oracle.OracleSPH(spec)
    o.neighbor_search()
    want = o.get("pointing_ff")
    for pre in (1, 0):
        for L in (2, 4, 8):
            s = make_gpu(spec)
            s.tune("listPrefilter", pre)
            s.tune("listLanes", L)
            s.neighbor_search()
            assert np.array_equal(s.get("neighborCount"), o.get("count_ff")), (pre, L)
            assert np.array_equal(s.get("objectPointing"), want), (pre, L)


@pytest.mark.parametrize("two_h", [False, True])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 7, 8, 9, 31, 33, 65, 300, 6001])
def test_lists_at_slot_edges_and_outside_the_grid(n, two_h):
    """Particle counts about the list build's wave widths (4, 8, 16, 32 and 64
    slots; 6,001 is past its four-slot rule) with one particle in five outside
    the grid: a fraction of a cell to 20 cells off, on both sides of the 10.5
    and 12 cells at which a point stops taking plain tests, in tight pairs
    there, and on the maximum faces.  Whole numbers: lists equal the oracle's
    at every lane count, one and two smoothing lengths."""
    rng = np.random.default_rng(1000 + n)
    dx = 0.01
    cell = 2.0 * 1.3 * dx
    side = max(3.2 * cell, 0.75 * dx * n ** (1.0 / 3.0))
    pos = rng.uniform(0.0, side, (n, 3))
    off = np.flatnonzero(rng.random(n) < 0.2)
    ax = rng.integers(0, 3, len(off))
    d = cell * rng.choice([0.3, 1.2, 2.0, 4.0, 10.45, 10.55, 11.9, 12.1, 20.0], len(off)) * rng.uniform(0.97, 1.03, len(off))
    up = rng.random(len(off)) < 0.5
    pos[off, ax] = np.where(up, side + d, -d)
    pos[off[1::2]] = pos[off[:len(off) // 2 * 2:2]] + rng.uniform(-0.4, 0.4, (len(off) // 2, 3)) * cell
    if n > 8:
        pos[off[0], :2] = side
    g = np.arange(0.0, side, dx)
    dummy = np.stack(np.meshgrid(g, g, [0.5 * dx], indexing="ij"), -1).reshape(-1, 3)
    spec = scenes.SPHSceneSpec(fluid_pos=pos, dummy_pos=dummy, dx=dx, rho0=1000.0, c0=10.0, nu=1e-6, min_bound=np.zeros(3),
                               max_bound=np.full(3, side), gravity=np.array([0.0, 0.0, -9.81]), dt=1e-5)
    if two_h:
        w = rng.random(n) < 0.5
        spec.fluid_dx = np.where(w, dx, 0.8 * dx)
        spec.fluid_rho0 = np.where(w, 1000.0, 900.0)
    o = oracle.OracleSPH(spec)
    o.neighbor_search()
    for L in (0, 1, 2, 4, 8):
        s = make_gpu(spec)
        s.tune("listLanes", L)
        s.neighbor_search()
        assert np.array_equal(s.get("neighborCount"), o.get("count_ff")), L
        assert np.array_equal(s.get("objectPointing"), o.get("pointing_ff")), L
        assert np.array_equal(s.get("dummyNeighborCount"), o.get("count_fd")), L
        assert np.array_equal(s.get("dummyObjectPointing"), o.get("pointing_fd")), L


@pytest.mark.parametrize("thin", [(0,), (1,), (2,), (0, 1), (0, 2), (1, 2), (0, 1, 2)])
def test_lists_on_axes_of_one_cell(thin):
    """Domains of one cell on some axes, of 1.4 supports, with particles and
    dummies past the faces and on them: fluid and dummy lists and the dummy
    normals (1e-6 on unit vectors in FP32) against the oracle."""
    rng = np.random.default_rng(10 * len(thin) + thin[0])
    dx = 0.01
    cut = 2.0 * 1.3 * dx
    side = np.full(3, 3.3 * cut)
    side[list(thin)] = 1.4 * cut

    def points(n):
        p = rng.uniform(0.0, 1.0, (n, 3)) * side
        off = rng.random((n, 3))
        p += np.where(off < 0.1, -1.0, np.where(off > 0.85, 1.0, 0.0)) * rng.uniform(0.0, 1.5, (n, 3)) * cut
        for k in range(3):
            p[10 * k:10 * k + 10, k] = side[k]
        return p

    spec = scenes.SPHSceneSpec(fluid_pos=points(400), dummy_pos=points(200), dx=dx, rho0=1000.0, c0=10.0, nu=1e-6,
                               min_bound=np.zeros(3), max_bound=side, gravity=np.array([0.0, 0.0, -9.81]), dt=1e-5)
    o = oracle.OracleSPH(spec)
    o.neighbor_search()
    s = make_gpu(spec)
    s.neighbor_search()
    assert np.array_equal(s.get("hashIndex"), o.get("index"))
    assert np.array_equal(s.get("neighborCount"), o.get("count_ff"))
    assert np.array_equal(s.get("objectPointing"), o.get("pointing_ff"))
    assert np.array_equal(s.get("dummyNeighborCount"), o.get("count_fd"))
    assert np.array_equal(s.get("dummyObjectPointing"), o.get("pointing_fd"))
    np.testing.assert_allclose(s.get("dummyNormal"), o.get("dnormal"), atol=1e-6)


@pytest.mark.parametrize("two_h", [False, True])
@pytest.mark.parametrize("side", [0.3, 0.5, 0.7, 0.95])
def test_lists_in_a_domain_smaller_than_a_support(side, two_h):
    """A domain of `side` supports on every axis is one cell whose edges are
    shorter than the cut.  Particles up to 30 of these edges outside it,
    thickest at 8 to 14 of them: lists equal the oracle's at every lane
    count."""
    rng = np.random.default_rng(int(100 * side))
    dx = 0.01
    cut = 2.0 * 1.3 * dx
    edge = side * cut
    pos = [rng.uniform(0.0, edge, (20, 3))]
    for d in np.concatenate([np.arange(8.0, 14.0, 0.25), rng.uniform(0.0, 30.0, 20)]):
        c = rng.uniform(0.0, edge, 3)
        c[rng.integers(3)] += edge * d * rng.choice([-1.0, 1.0])
        pos.append(c + rng.uniform(-0.4, 0.4, (6, 3)) * cut)
    # a line of close neighbours through all of the limits
    t = np.arange(-16.0 * edge, 17.0 * edge, 0.3 * cut)
    pos.append(np.stack([t, np.full(len(t), 0.5 * edge), np.full(len(t), 0.4 * edge)], -1))
    pos = np.concatenate(pos)
    g = np.arange(-15.0 * edge, 16.0 * edge, 0.5 * cut)
    dummy = np.stack([g, np.full(len(g), 0.6 * edge), np.full(len(g), 0.3 * edge)], -1)
    spec = scenes.SPHSceneSpec(fluid_pos=pos, dummy_pos=dummy, dx=dx, rho0=1000.0, c0=10.0, nu=1e-6, min_bound=np.zeros(3),
                               max_bound=np.full(3, edge), gravity=np.array([0.0, 0.0, -9.81]), dt=1e-5)
    if two_h:
        spec.fluid_dx = np.where(rng.random(len(pos)) < 0.5, dx, 0.8 * dx)
    o = oracle.OracleSPH(spec)
    o.neighbor_search()
    for L in (0, 1, 2, 4, 8):
        s = make_gpu(spec)
        s.tune("listLanes", L)
        s.neighbor_search()
        assert np.array_equal(s.get("neighborCount"), o.get("count_ff")), L
        assert np.array_equal(s.get("objectPointing"), o.get("pointing_ff")), L
        assert np.array_equal(s.get("dummyNeighborCount"), o.get("count_fd")), L
        assert np.array_equal(s.get("dummyObjectPointing"), o.get("pointing_fd")), L


@pytest.mark.parametrize("ops", [
    ["search", "search", "step", "first", "second", "step"],
    ["search", "first", "step", "second"],
    ["search", "first", "second", "step", "first", "second"],
    ["step", "first", "step", "velocity", "first", "second"],
])
def test_halves_after_replayed_blocks(ops, small):
    """Searches and halves between replays of captured step graphs, at every
    parity of the buffers that the sequence passes through (its fourth round
    replays graphs captured in the earlier ones): bit for bit what eager steps
    give, and within the rounding of the two forms of the pair passes (1e-5 of
    the largest value, as above) of the FP64 records."""
    rng = np.random.default_rng(5)
    kick = 0.05 * rng.uniform(-1.0, 1.0, (small.nf, 3))
    runs = []
    for graphs, rec in ((True, 1), (False, 1), (True, 0)):
        s = make_gpu(small)
        s.set_graphs(graphs)
        s.tune("pairRecords", rec)
        s.step(small.dt, 2)
        for _ in range(4):
            for op in ops:
                if op == "search":
                    s.neighbor_search()
                elif op == "first":
                    s.first_half(small.dt)
                elif op == "second":
                    s.second_half(small.dt)
                elif op == "velocity":
                    s.set("velocity", s.get("velocity") + kick)
                else:
                    s.step(small.dt, 2)
        s.first_half(small.dt)
        s.second_half(small.dt)
        assert (s.graph_captures() > 0) == graphs
        runs.append([s.get(f) for f in ("position", "velocity", "densityChange")])
    for a, b, c in zip(*runs):
        assert np.array_equal(a, b)
        assert np.abs(a - c).max() < 1e-5 * np.abs(c).max()


@pytest.mark.parametrize("cells", [0.5, 20.0, 64.0, 128.0, 1e6])
@pytest.mark.parametrize("n", [2, 300])
def test_a_particle_that_flies_off_in_one_step(n, cells):
    """One particle drifts `cells` supports in the first half (64 and 128 are
    multiples of the period of the records' positions), after which the second
    half must not see it beside its former neighbours.  Records against the
    FP64 records over the other particles: rounding of FP32 sums, 1e-5 of the
    largest value."""
    rng = np.random.default_rng(n)
    dx, dt = 0.01, 1e-4
    side = max(0.1, 0.8 * dx * n ** (1.0 / 3.0))
    pos = 0.5 * side + rng.uniform(-0.5, 0.5, (n, 3)) * (0.4 * dx if n == 2 else side)
    vel = rng.uniform(-0.1, 0.1, (n, 3))
    vel[0, 0] = cells * 2.0 * 1.3 * dx / dt
    spec = scenes.SPHSceneSpec(fluid_pos=pos, fluid_vel=vel, dummy_pos=np.zeros((0, 3)), dx=dx, rho0=1000.0, c0=10.0,
                               nu=0.0, min_bound=np.zeros(3), max_bound=np.full(3, side),
                               gravity=np.array([0.0, 0.0, -9.81]), dt=dt)
    got = []
    for rec in (1, 0):
        s = make_gpu(spec)
        s.tune("pairRecords", rec)
        s.neighbor_search()
        s.first_half(dt)
        s.second_half(dt)
        got.append([s.get(f)[1:] for f in ("position", "velocity", "densityChange")])
    for a, b in zip(*got):
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_pairs_across_the_ends_of_the_coordinate_range(axis):
    """A grid of 140 supports on one axis, with the ends of the records' 32-bit
    range at 64 supports (largest and smallest value side by side) and 128 (zero):
    lists there against the oracle's, and a step within the tolerances of one
    step."""
    rng = np.random.default_rng(axis)
    dx = 0.01
    cut = 2.0 * 1.3 * dx
    side = np.full(3, 4.0 * cut)
    side[axis] = 140.0 * cut
    pos = rng.uniform(0.0, 1.0, (1200, 3)) * side
    g = np.arange(6) * dx
    block = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) + rng.uniform(-0.1, 0.1, (216, 3)) * dx
    pos = [pos]
    for at in (32.0, 64.0, 96.0, 128.0):
        c = np.full(3, 0.5 * cut)
        c[axis] = at * cut - 2.5 * dx
        pos.append(block + c)
    pos = np.concatenate(pos)
    dummy = pos[-216:] + 0.4 * dx
    spec = scenes.SPHSceneSpec(fluid_pos=pos, dummy_pos=dummy, dx=dx, rho0=1000.0, c0=10.0, nu=1e-6, min_bound=np.zeros(3),
                               max_bound=side, gravity=np.array([0.0, 0.0, -9.81]), dt=1e-6)
    o = oracle.OracleSPH(spec)
    o.neighbor_search()
    s = make_gpu(spec)
    s.neighbor_search()
    assert np.array_equal(s.get("neighborCount"), o.get("count_ff"))
    assert np.array_equal(s.get("objectPointing"), o.get("pointing_ff"))
    assert np.array_equal(s.get("dummyObjectPointing"), o.get("pointing_fd"))
    o = oracle.OracleSPH(spec)
    s = make_gpu(spec)
    o.step(spec.dt, 1)
    s.step(spec.dt, 1)
    _compare(s, o, 1e-9, 1e-6, 1e-4)


@pytest.mark.parametrize("ratio", [0.5, 1.0, 1.3, 2.5, 4.0])
def test_records_lose_nothing_beside_dummies(ratio):
    """A layer of fluid on dummies of another spacing, where every particle has
    as many dummy as fluid neighbours: after 20 steps the pair passes on
    records are as close to the oracle as those on FP64 records.  Both round
    to FP32; twice the error of the FP64 records allows for chance, and 2e-7 of
    the change (three roundings of 6e-8) where those happen to cancel."""
    rng = np.random.default_rng(1)
    dx = 0.01
    side = 0.3
    g = np.arange(0.5 * dx, side, dx)
    pos = np.stack(np.meshgrid(g, g, [0.5 * dx], indexing="ij"), -1).reshape(-1, 3)
    pos = pos + rng.uniform(-0.2, 0.2, pos.shape) * dx
    vel = rng.uniform(-0.05, 0.05, pos.shape)
    wide = ratio * dx
    g = np.arange(0.5 * wide, side, wide)
    dummy = np.stack(np.meshgrid(g, g, -wide * (0.5 + np.arange(3)), indexing="ij"), -1).reshape(-1, 3)
    spec = scenes.SPHSceneSpec(fluid_pos=pos, fluid_vel=vel, dummy_pos=dummy, dx=wide, rho0=1000.0, c0=10.0, nu=1e-3,
                               min_bound=np.array([0.0, 0.0, -4.0 * wide]), max_bound=np.array([side, side, 0.5]),
                               gravity=np.array([0.0, 0.0, -9.81]), dt=0.01 * 1.3 * dx)
    spec.fluid_dx = np.full(len(pos), dx)
    o = oracle.OracleSPH(spec)
    o.step(spec.dt, 20)
    dv, dr = o.get("vel") - vel, o.get("rho") - 1000.0
    err = []
    for rec in (1, 0):
        s = make_gpu(spec)
        s.tune("pairRecords", rec)
        assert s.tuned("pairRecords") == rec
        s.step(spec.dt, 20)
        err.append((np.linalg.norm(s.get("velocity") - vel - dv) / np.linalg.norm(dv),
                    np.linalg.norm(s.get("densityChange") - dr) / np.linalg.norm(dr)))
    print("[records] ratio", ratio, "records", err[0], "FP64", err[1], flush=True)
    for a, b in zip(*err):
        assert a <= max(2.0 * b, 2e-7)


@pytest.mark.parametrize("first_only", [False, True])
def test_fluid_without_support(first_only):
    """Fluid particles of spacing zero (all of them, or the first one) over
    dummies: they have no support of their own, lists equal the oracle's and a
    step gives what the FP64 records give (1e-5 of the largest value, as for
    FP32 sums in another order) and no infinities."""
    rng = np.random.default_rng(2)
    dx = 0.01
    pos = rng.uniform(0.0, 0.1, (300, 3)) * [1.0, 1.0, 0.3]
    g = np.arange(0.0, 0.1, dx)
    dummy = np.stack(np.meshgrid(g, g, [-0.5 * dx], indexing="ij"), -1).reshape(-1, 3)
    spec = scenes.SPHSceneSpec(fluid_pos=pos, dummy_pos=dummy, dx=dx, rho0=1000.0, c0=10.0, nu=1e-6,
                               min_bound=np.array([0.0, 0.0, -dx]), max_bound=np.full(3, 0.1),
                               gravity=np.array([0.0, 0.0, -9.81]), dt=1e-6)
    spec.fluid_dx = np.zeros(300) if not first_only else np.where(np.arange(300) == 0, 0.0, dx)
    o = oracle.OracleSPH(spec)
    o.neighbor_search()
    got = []
    for rec in (1, 0):
        s = make_gpu(spec)
        s.tune("pairRecords", rec)
        s.neighbor_search()
        assert np.array_equal(s.get("neighborCount"), o.get("count_ff"))
        assert np.array_equal(s.get("objectPointing"), o.get("pointing_ff"))
        assert np.array_equal(s.get("dummyObjectPointing"), o.get("pointing_fd"))
        s.step(spec.dt, 1)
        got.append([s.get(f) for f in ("position", "velocity", "density")])
    for a, b in zip(*got):
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()


@pytest.mark.parametrize("field", ["velocity", "densityChange"])
def test_records_follow_a_field_set_between_search_and_halves(field, small):
    """A field set after the search reaches the records that the passes
    gather.  The two forms of the pair passes differ by the rounding of FP32
    sums over about 80 pairs, 80 x 6e-8 of the largest term: 1e-5 of the
    largest value bounds it, and a stale field would miss by its change."""
    rng = np.random.default_rng(9)
    got = []
    value = None
    for rec in (1, 0):
        s = make_gpu(small)
        s.tune("pairRecords", rec)
        s.neighbor_search()
        if value is None:
            old = s.get(field)
            value = old + rng.uniform(-0.5, 0.5, old.shape)
        s.set(field, value)
        s.first_half(small.dt)
        s.second_half(small.dt)
        got.append([s.get(f) for f in ("velocity", "density")])
    for a, b in zip(*got):
        assert np.abs(a - b).max() < 1e-5 * np.abs(b).max()


@pytest.mark.parametrize("n", [1, 85, 256, 257])
def test_read_back_in_insertion_order(n):
    """Values come back in insertion order, unchanged, from sorted particles
    (counts about the read-back kernel's blocks); a too small output is
    refused; reading between the calls of a step leaves the step alone."""
    import ctypes as C

    rng = np.random.default_rng(n)
    pos, vel = rng.uniform(0.0, 0.2, (n, 3)), rng.uniform(-1.0, 1.0, (n, 3))
    spec = scenes.SPHSceneSpec(fluid_pos=pos, fluid_vel=vel, dummy_pos=np.zeros((0, 3)), dx=0.01, rho0=1000.0, c0=10.0,
                               nu=1e-6, min_bound=np.zeros(3), max_bound=np.full(3, 0.2),
                               gravity=np.array([0.0, 0.0, -9.81]), dt=1e-6)
    a, b = make_gpu(spec), make_gpu(spec)
    for s in (a, b):
        s.neighbor_search()
    assert np.array_equal(a.get("position"), pos) and np.array_equal(a.get("velocity"), vel)
    assert a.get("density").shape == a.get("pressure").shape == a.get("densityChange").shape == (n,)
    out, cnt = np.empty(3 * n), C.c_size_t()
    for f in (b"position", b"velocity"):
        assert ts.lib().demsph_sph_get(a._h, f, out.ctypes.data_as(C.c_void_p), 3 * n - 1, C.byref(cnt)) != 0
    for s in (a, b):
        s.first_half(spec.dt)
    a.get("velocity")
    for s in (a, b):
        s.second_half(spec.dt)
    for f in ("position", "velocity", "density", "densityChange"):
        assert np.array_equal(a.get(f), b.get(f)), f


def read_from_threads(scene, fields, rounds):
    """Fields of one scene read by a thread each, at the same time: the reads
    that differ from the same fields read in turn."""
    import threading

    want = {f: scene.get(f) for f in fields}
    wrong = []

    def reader(f):
        for k in range(rounds):
            if not np.array_equal(scene.get(f), want[f]):
                wrong.append((f, k))

    threads = [threading.Thread(target=reader, args=(f,)) for f in fields]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    return wrong


@pytest.mark.parametrize("n", [100, 30000])
def test_fields_read_from_several_threads(n):
    rng = np.random.default_rng(n)
    spec = scenes.SPHSceneSpec(fluid_pos=rng.uniform(0.0, 0.4, (n, 3)), fluid_vel=rng.uniform(-1.0, 1.0, (n, 3)),
                               dummy_pos=np.zeros((0, 3)), dx=0.01, rho0=1000.0, c0=10.0, nu=1e-6, min_bound=np.zeros(3),
                               max_bound=np.full(3, 0.4), gravity=np.array([0.0, 0.0, -9.81]), dt=1e-6)
    s = make_gpu(spec)
    s.step(spec.dt, 2)
    assert read_from_threads(s, ["position", "velocity", "density", "densityChange"], 150) == []


def test_two_phases_match_oracle():
    """Two fluid phases of different spacing, density and viscosity side by
    side (the kernels' non-uniform paths: per-pair cuts, phase lookups,
    averaged smoothing lengths): lists bit-exact at every lane setting, 30
    steps within the single-phase tolerances."""
    spec = scenes.two_phase_tank()
    o = oracle.OracleSPH(spec)
    o.neighbor_search()
    for L in (1, 2, 8):
        s = make_gpu(spec)
        s.tune("listLanes", L)
        s.neighbor_search()
        assert np.array_equal(s.get("neighborCount"), o.get("count_ff")), L
        assert np.array_equal(s.get("objectPointing"), o.get("pointing_ff")), L
        assert np.array_equal(s.get("dummyObjectPointing"), o.get("pointing_fd")), L
    o2 = oracle.OracleSPH(spec)
    s = make_gpu(spec)
    o2.step(spec.dt, 30)
    s.step(spec.dt, 30)
    _compare(s, o2, 1e-7, 1e-4, 1e-2)


def test_tait_eos_matches_oracle():
    spec = scenes.small_dam_break(eos=1)
    o = oracle.OracleSPH(spec)
    s = make_gpu(spec)
    o.step(spec.dt, 100)
    s.step(spec.dt, 100)
    _compare(s, o, 1e-7, 1e-4, 1e-2)
    p_o, p_s = o.get("p"), s.get("pressure")
    assert np.abs(p_s - p_o).max() < 1e-3 * max(1.0, np.abs(p_o).max())


def test_list_overflow_replays_exactly(small):
    a = make_gpu(small)
    b = make_gpu(small, capacity=(4, 2))  # forces overflow, regrow and replay from the checkpoint
    a.step(small.dt, 20)
    b.step(small.dt, 20)
    assert np.array_equal(a.get("position"), b.get("position"))
    assert np.array_equal(a.get("velocity"), b.get("velocity"))
    assert np.array_equal(a.get("densityChange"), b.get("densityChange"))
    # neighbour_search alone also regrows
    c = make_gpu(small, capacity=(3, 3))
    c.neighbor_search()
    o = oracle.OracleSPH(small)
    o.neighbor_search()
    assert np.array_equal(c.get("objectPointing"), o.get("pointing_ff"))


def test_reference_dam_break_frame1():
    """The reference's damBreak.cpp scene, 670 steps, against the reference's
    own frame at step 670 (tests/golden/dam_break_frames.npz)."""
    spec = scenes.reference_dam_break()
    ref = np.load(GOLDEN / "dam_break_frames.npz")
    s = make_gpu(spec)
    s.step(spec.dt, 670)
    err = np.abs(s.get("position") - ref["pos1"]).max()
    # FP32 pair arithmetic over 670 steps: within 1e-5 of the spacing (5e-3 m)
    assert err < 5e-8 + 1e-5 * spec.dx, err
    assert np.abs(s.get("velocity") - ref["vel1"]).max() < 1e-3
    assert np.abs(s.get("density") - ref["rho1"]).max() < 0.05


def test_full_size_dam_break_cells_and_counts():
    """256,000-particle dam break: hash, permutation, cell ranges and
    per-particle neighbour counts are bit-exact against the oracle."""
    spec = scenes.dam_break()
    s = make_gpu(spec)
    s.neighbor_search()
    g = oracle.grid_set(spec.min_bound, spec.max_bound, 2.0 * 1.3 * spec.dx)
    hv = oracle.hash_points(g, spec.fluid_pos)
    sh, si = oracle.sort_by_hash(hv, g.num_grids)
    cs, ce = oracle.cell_ranges(sh, g.num_grids)
    assert np.array_equal(s.get("hashIndex"), si)
    assert np.array_equal(s.get("cellHashStart"), cs)
    assert np.array_equal(s.get("cellHashEnd"), ce)
    cnt = s.get("neighborCount")
    assert cnt.max() == 80 and cnt.sum() > 70 * spec.nf
    h = np.full(spec.nf, 1.3 * spec.dx)
    ocnt = np.zeros(spec.nf, dtype=np.int32)
    oracle.lib().o_sph_count(oracle.Grid.from_buffer_copy(g), oracle.d(spec.fluid_pos), oracle.d(h), spec.nf,
                             oracle.d(spec.fluid_pos), oracle.d(h), oracle.i(si), oracle.i(cs), oracle.i(ce), 1,
                             oracle.i(ocnt))
    assert np.array_equal(cnt, ocnt)


def test_background_frame_is_a_snapshot(small, tmp_path):
    """A fluid frame written in the background equals, byte for byte, the
    blocking write of the same state, although the scene steps on before
    the frame thread writes it."""
    s = make_gpu(small)
    s.step(small.dt, 10)
    s.write_vtu(tmp_path / "now", 1, 10, 0.5, dummies=False)
    s.write_vtu(tmp_path / "bg", 1, 10, 0.5, dummies=False, background=True)
    s.step(small.dt, 30)
    ts.frames_wait()
    a = (tmp_path / "now" / "SPH_0001.vtu").read_bytes()
    b = (tmp_path / "bg" / "SPH_0001.vtu").read_bytes()
    assert a == b
    s.write_vtu(tmp_path / "later", 2, 40, 1.0, dummies=False)
    assert (tmp_path / "later" / "SPH_0002.vtu").read_bytes() != a


def test_exported_state_resumes_bit_for_bit(small):
    """A scene evicted to host memory and restored into a freshly built scene
    of the same particles continues exactly as the scene that kept running,
    with graphs on and off; a state of other particle counts is refused."""
    a = make_gpu(small)
    a.step(small.dt, 13)
    state = a.export_state()
    for graphs in (True, False):
        b = make_gpu(small)
        b.set_graphs(graphs)
        b.step(small.dt, 3)  # the state replaces whatever b held
        b.import_state(state)
        ref = make_gpu(small)
        ref.step(small.dt, 13)
        assert ref.export_state() == state
        ref.step(small.dt, 21)
        b.step(small.dt, 21)
        for f in ("position", "velocity", "density", "pressure", "densityChange"):
            assert np.array_equal(ref.get(f), b.get(f)), (graphs, f)
    with pytest.raises(ts.DemsphError):
        b.import_state(state[:-4])
    other = scenes.small_dam_break()
    assert other.fluid_vel is None and other.fluid_c0 is None
    other.fluid_pos = other.fluid_pos[:-1]
    with pytest.raises(ts.DemsphError):
        make_gpu(other).import_state(state)


def test_reference_dam_break_full_series():
    """The reference's damBreak.cpp scene over all of its recorded frames:
    46,900 steps (3.5 s), compared frame by frame (every 670 steps) with the
    front position, column height and mean density of the reference's own
    71 SPH_*.vtu frames (tests/golden/dam_break_series.npz).  Front within
    half a particle spacing and mean density within 0.05 kg/m^3 over the
    whole run; column height within 1 mm through the collapse and the run-up
    on the far wall (t <= 0.7 s), after which the splash is chaotic and only
    bounded."""
    spec = scenes.reference_dam_break()
    ser = np.load(GOLDEN / "dam_break_series.npz")["series"]
    s = make_gpu(spec)
    front, zmax, rho = [], [], []
    for k in range(1, ser.shape[0]):
        s.step(spec.dt, 670)
        p = s.get("position")
        front.append(p[:, 0].max())
        zmax.append(p[:, 2].max())
        rho.append(s.get("density").mean())
    front, zmax, rho = map(np.array, (front, zmax, rho))
    assert int(ser[-1, 1]) == 670 * (ser.shape[0] - 1)
    assert np.abs(front - ser[1:, 2]).max() < 0.5 * spec.dx
    early = ser[1:, 0] <= 0.7
    assert np.abs(zmax[early] - ser[1:, 3][early]).max() < 1e-3
    assert np.abs(zmax - ser[1:, 3]).max() < 0.2
    assert np.abs(rho - ser[1:, 5]).max() < 0.05


def test_full_size_dam_break_lists_and_steps_match_oracle():
    """The 256,000-particle dam break at full size: the fluid-fluid and
    fluid-dummy lists (19.5M and 0.5M entries) bit-exact against the
    oracle's, in the reference's order, then 20 steps within the FP32
    pair-arithmetic tolerances (positions 1e-9 m, velocities 1e-5 m/s,
    densities 1e-3 kg/m^3)."""
    spec = scenes.dam_break()
    o = oracle.OracleSPH(spec)
    s = make_gpu(spec)
    o.neighbor_search()
    s.neighbor_search()
    for f, of in (("neighborCount", "count_ff"), ("dummyNeighborCount", "count_fd"),
                  ("objectPointing", "pointing_ff"), ("dummyObjectPointing", "pointing_fd")):
        assert np.array_equal(s.get(f), o.get(of)), f
    assert o.get("pointing_ff").size > 19_000_000
    o.step(spec.dt, 20)
    s.step(spec.dt, 20)
    _compare(s, o, 1e-9, 1e-5, 1e-3)
