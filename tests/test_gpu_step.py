"""Joined integrator steps (k_advance) and the one-launch forces of small systems with the lists they
keep (k_forces), against the oracle: the edges of the size rule, both integrators, partitions, and a
list that outgrows its rows in the middle of a segment."""
import dataclasses
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
pytestmark = pytest.mark.gpu


def _follow(spec, steps, precision=0, tol=1e-8, lists=True, rebuilds=True):
    """Positions, velocities, forces and the neighbour sets after `steps` steps against the oracle, which
    takes the same noise.  1e-8 is the bar of the FP64 trajectories (rounding grows by less than 1e4 over
    a few hundred steps of these systems).  rebuilds: the steps must have rebuilt lists (the builds of the
    set-up do not count)."""
    import oracle
    from mjolnir_amd import capi
    e, o = capi.Engine(spec, precision), oracle.OracleEngine(spec)
    built = e.counters()[1]
    for n in (steps // 3, steps - steps // 3):          # two calls: segments start from a stored state
        e.step(n)
        o.step(n)
    x, v, f = e.state()
    xo, vo, fo = o.state()
    d = x - xo
    if spec.boundary == "periodic":
        w = spec.upper - spec.lower
        d -= w * np.round(d / w)
    scale = np.abs(fo).max()
    print(f"[gpu] {spec.name}: dx {np.abs(d).max():.1e} dv {np.abs(v - vo).max():.1e} "
          f"df {np.abs(f - fo).max() / scale:.1e} rebuilds {e.counters()[1] - built}", flush=True)
    assert np.abs(d).max() < tol and np.abs(v - vo).max() < tol and np.abs(f - fo).max() < tol * max(1.0, scale)
    assert e.counters()[0] == steps
    assert not rebuilds or e.counters()[1] > built
    for g in range(len(spec.global_) if lists else 0):
        same = np.array_equal(e.pairs(len(spec.local) + g), o.pairs(g))   # the oracle counts globals alone
        assert same, spec.global_[g].potential
    return e


def _gjf(spec):
    it = dataclasses.replace(spec.integrator, type="GJFNVTLangevin", coefs=spec.integrator.coefs * spec.mass)
    return dataclasses.replace(spec, integrator=it)


@pytest.mark.parametrize("n,steps,margin", [(65, 150, 0.15), (257, 150, 0.15), (1000, 150, 0.5), (4096, 110, 0.5),
                                            (4097, 110, 0.5), (4200, 70, 0.19), (4200, 70, 0.2)])
def test_fluids_at_the_edges_of_the_size_rule(n, steps, margin):
    """Lists kept by the force kernel up to 4096 participants; above, inner lists from a margin of 0.2 on."""
    from mjolnir_amd import workloads
    spec = workloads.lj_fluid(n=n, seed=n, margin=margin)
    _follow(spec, steps)


@pytest.mark.parametrize("partition", ["CellList", "VerletList", "Naive"])
def test_partitions(partition):
    from mjolnir_amd import workloads
    spec = _gjf(workloads.cg_chain(130, seed=8, max_bend_deg=150.0, margin=0.1))
    spec.global_ = [dataclasses.replace(g, partition=partition) for g in spec.global_]
    _follow(spec, 120, tol=1e-7, rebuilds=partition != "Naive")


def test_list_outgrows_its_rows_inside_a_segment():
    """Two clusters of 48 that drift together: a row holds 47 partners at the start (capacity 64) and 95
    once the clusters see each other.  The segment then runs again from a list rebuilt at its start, so
    the later rebuilds fall on other steps than the oracle's and only the trajectory is compared."""
    from mjolnir_amd import workloads
    from mjolnir_amd.spec import GlobalSpec, IntegratorSpec, SystemSpec
    g = np.stack(np.meshgrid(np.arange(4), np.arange(4), np.arange(3), indexing="ij"), -1).reshape(-1, 3) * 1.3
    pos = np.concatenate([g, g + [16.0, 0.6, 0.6]])
    vel = np.zeros_like(pos)
    vel[:48, 0], vel[48:, 0] = 3.5, -3.5
    n = len(pos)
    lj = GlobalSpec(potential="LennardJones", participants=np.arange(n), params=np.tile([1.0, 0.02], (n, 1)), cutoff=2.5,
                    partition="CellList", margin=1.5)
    spec = SystemSpec(boundary="unlimited", mass=np.ones(n), pos=pos, vel=vel, attributes={"temperature": 1.0},
                      global_=[lj], integrator=IntegratorSpec("BAOABLangevin", 0.01, np.full(n, 0.01), seed=3),
                      name="two_clusters")
    e = _follow(spec, 165, lists=False)
    per = np.bincount(e.pairs(0).ravel(), minlength=n)
    assert per.max() > 64


@pytest.mark.parametrize("system", ["chain", "dna"])
def test_mixed_small_systems_follow_fp64(system):
    """The mixed precision through the same kernels: forces along the way within the mixed bar of the FP64
    engine's (1e-5 of the RMS force) after 60 steps of one noise stream."""
    from mjolnir_amd import capi, workloads
    spec = workloads.cg_chain(700, seed=9, max_bend_deg=150.0) if system == "chain" else workloads.dna_duplex(40, seed=5)
    a, b = capi.Engine(spec, capi.FP64), capi.Engine(spec, capi.FP32_FIXED)
    a.step(60)
    b.step(60)
    fa, fb = a.state()[2], b.state()[2]
    rms = np.sqrt(np.mean(fa ** 2))
    print(f"[gpu] {system} mixed vs FP64: {np.sqrt(np.mean((fa - fb) ** 2)) / rms:.1e}", flush=True)
    assert np.sqrt(np.mean((fa - fb) ** 2)) < 1e-5 * rms


@pytest.mark.parametrize("n_bp", [6, 40])
def test_duplex_rows(n_bp):
    """Base pairing, cross stacking (four lanes a pair) and the lists' base rules, through rebuilds."""
    from mjolnir_amd import workloads
    _follow(workloads.dna_duplex(n_bp, seed=4, margin=0.1), 120)


def test_exclusions_far_apart_in_index():
    """A hub excluded from 150 particles far from it in index: more than a rebuild keeps in LDS for a row."""
    from mjolnir_amd.spec import GlobalSpec, IntegratorSpec, LocalSpec, SystemSpec
    rng = np.random.default_rng(12)
    n = 216
    g = np.stack(np.meshgrid(*[np.arange(6)] * 3, indexing="ij"), -1).reshape(-1, 3) * 4.5
    pos = g + rng.uniform(-0.3, 0.3, size=g.shape)
    other = np.arange(60, 210)
    hub = LocalSpec("BondLength", "GoContact", "contact", np.stack([np.zeros_like(other), other], 1),
                    np.stack([np.full(len(other), 1e-3), np.full(len(other), 8.0)], 1))
    ev = GlobalSpec(potential="ExcludedVolume", participants=np.arange(n), params=np.full((n, 1), 1.2), cutoff=2.0,
                    epsilon=0.2, partition="CellList", margin=0.2, ignore_within={"contact": 1})
    spec = SystemSpec(boundary="unlimited", mass=np.ones(n), pos=pos, vel=rng.normal(size=pos.shape) * 0.7,
                      attributes={"temperature": 300.0}, local=[hub], global_=[ev],
                      integrator=IntegratorSpec("BAOABLangevin", 0.01, np.full(n, 0.1), seed=2), name="hub")
    _follow(spec, 120)


def test_replica_block_shapes_agree():
    """FP64 replicas of 257 to 1024 particles run 1024 threads while there are no more of them than CUs
    (256), else 512; larger ones 1024.  Forces are integer sums, so a trajectory is the same bit for bit
    in both shapes, and it follows the oracle's."""
    import oracle
    from mjolnir_amd import capi, workloads
    targets = [workloads.cg_chain(n, seed=n, max_bend_deg=150.0) for n in (257, 700, 1024, 1025, 2048)]
    filler = [workloads.cg_chain(258, seed=1, max_bend_deg=150.0)] * 254      # 257 replicas of the middle class
    out = []
    for specs in (targets, targets + filler):
        b = capi.Batch(capi.FP64)
        ids = [b.add(s) for s in specs][:len(targets)]
        b.initialize()
        b.step(60)
        out.append([b.state(r) for r in ids])
        b.close()
    for spec, few, many in zip(targets, *out):
        assert all(np.array_equal(a, c) for a, c in zip(few, many)), spec.name
        o = oracle.OracleEngine(spec)
        o.step(60)
        xo, vo, fo = o.state()
        # as the other FP64 replica trajectories (fixed-point sums in units of 2^-32)
        assert np.abs(few[0] - xo).max() < 1e-7 and np.abs(few[1] - vo).max() < 1e-7, spec.name


def test_cell_grid_of_participants_far_apart():
    """An open box whose participants span 1e13 A in every direction (an exploded chain reaches 1e10): the
    one-workgroup rebuild widens its cells until they fit its tables, and the list is the all-pairs list.
    The list's cells would have to be 1e8 times the list radius wide to fit after a bounded widening."""
    from mjolnir_amd import capi
    from mjolnir_amd.spec import GlobalSpec, IntegratorSpec, SystemSpec
    rng = np.random.default_rng(7)
    g = np.stack(np.meshgrid(*[np.arange(2)] * 3, indexing="ij"), -1).reshape(-1, 3) * 1.1
    far = np.concatenate([np.zeros((1, 3)), rng.uniform(-1e13, 1e13, size=(20, 3))])
    pos = np.concatenate([g + c for c in far])
    n = len(pos)

    def engine(partition):
        lj = GlobalSpec(potential="LennardJones", participants=np.arange(n), params=np.tile([1.0, 0.02], (n, 1)),
                        cutoff=2.5, partition=partition, margin=0.5)
        return capi.Engine(SystemSpec(boundary="unlimited", mass=np.ones(n), pos=pos, vel=np.zeros_like(pos),
                                      attributes={"temperature": 1.0}, global_=[lj],
                                      integrator=IntegratorSpec("BAOABLangevin", 0.01, np.full(n, 0.01), seed=3),
                                      name=f"far_{partition}"))

    cells, plain = engine("CellList"), engine("VerletList")
    assert len(cells.pairs(0)) >= 28 and np.array_equal(cells.pairs(0), plain.pairs(0))
    fc, fp = cells.state()[2], plain.state()[2]
    # the same pairs in another order: rounding of sums of up to 7 partners
    assert np.abs(fc - fp).max() <= 1e-14 * np.abs(fp).max()


def _fluid(potential, n, margin, seed, box=None):
    """n particles of one pair potential on a jittered lattice in a periodic box (cubic unless given)."""
    from mjolnir_amd import workloads
    from mjolnir_amd.spec import GlobalSpec, IntegratorSpec, SystemSpec
    rng = np.random.default_rng(seed)
    spacing = {"LennardJones": 4.74, "ExcludedVolume": 5.0, "DebyeHuckel": 6.0, "3SPN2ExcludedVolume": 5.5}[potential]
    if box is None:
        side = int(np.ceil(n ** (1 / 3) - 1e-9))
        sites = (side, side, side)
    else:
        sites = tuple(int(w / spacing) for w in box)
    g = np.stack(np.meshgrid(*[np.arange(k) for k in sites], indexing="ij"), -1).reshape(-1, 3)[:n]
    upper = np.array(box if box is not None else [s * spacing for s in sites], dtype=float)
    pos = (g + 0.5) * (upper / np.array(sites)) + rng.uniform(-0.3, 0.3, size=g.shape)
    n = len(pos)
    par, kw = {"LennardJones": (np.tile([4.0, 0.2], (n, 1)), {}),
               "ExcludedVolume": (rng.uniform(1.6, 2.0, size=(n, 1)), {"epsilon": 0.2}),
               "DebyeHuckel": (rng.choice([-1.0, 1.0], size=(n, 1)), {"cutoff": 2.0}),
               "3SPN2ExcludedVolume": (rng.integers(0, 6, size=(n, 1)).astype(float), {})}[potential]
    pair = GlobalSpec(potential=potential, participants=np.arange(n), params=par, partition="CellList", margin=margin, **kw)
    mass = np.ones(n)
    return SystemSpec(boundary="periodic", mass=mass, pos=pos, vel=workloads.maxwell_boltzmann(rng, mass, 300.0),
                      lower=np.zeros(3), upper=upper, attributes={"temperature": 300.0, "ionic_strength": 0.5},
                      global_=[pair], integrator=IntegratorSpec("BAOABLangevin", 0.01, np.full(n, 0.1), seed=seed),
                      name=f"{potential}_{n}")


THIN = (62.0, 60.0, 27.0)      # r_list = 15: the third axis' three cells are 9 A wide


def test_mixed_forces_in_a_box_narrower_than_three_list_radii(monkeypatch):
    """An axis clamped to three cells: a pair of neighbouring cells can be nearer through the other side of the
    box, which the mixed cell-tile kernel's staging (one image a cell) would miss.  Bar: the mixed path's
    1e-5 of the RMS force."""
    from mjolnir_amd import capi
    monkeypatch.setenv("MJG_TILE_MIN_NP", "0")
    spec = _fluid("LennardJones", 10 ** 6, 0.5, 3, THIN)
    e = capi.Engine(spec, capi.FP32_FIXED)
    for steps in (0, 40):
        e.step(steps)
        x, _, f = e.state()
        ref = capi.Engine(dataclasses.replace(spec, pos=x), capi.FP64, with_integrator=False)
        ref.calc_force()
        want = ref.state()[2]
        rms = float(np.sqrt(np.mean((f - want) ** 2) / np.mean(want ** 2)))
        print(f"[gpu] thin box N={spec.n} after {steps} steps: mixed RMS error {rms:.1e}", flush=True)
        assert rms < 1e-5


def _crossing_clusters(boundary, filler, remove=False):
    """Two clusters of 48 that fly through each other within 100 steps: the rows hold 47 partners before and
    after and up to 95 in between, above the first row length of 64.  The filler (a lattice of single
    particles beyond each other's list radius) only makes the interaction large."""
    from mjolnir_amd.spec import GlobalSpec, IntegratorSpec, SystemSpec
    g = np.stack(np.meshgrid(np.arange(4), np.arange(4), np.arange(3), indexing="ij"), -1).reshape(-1, 3) * 1.3
    centre = np.array([48.0, 48.0, 121.0])
    pos = np.concatenate([g - [6.0, 0, 0], g + [6.0, 0.6, 0.6]]) + centre
    vel = np.zeros_like(pos)
    vel[:48, 0], vel[48:, 0] = 12.0, -12.0
    if filler:
        f = np.stack(np.meshgrid(np.arange(16), np.arange(16), np.arange(17), indexing="ij"), -1).reshape(-1, 3)[:filler]
        pos = np.concatenate([pos, (f + 0.5) * 6.0])
        vel = np.concatenate([vel, np.zeros((filler, 3))])
    n = len(pos)
    lj = GlobalSpec(potential="LennardJones", participants=np.arange(n), params=np.tile([1.0, 0.02], (n, 1)), cutoff=2.5,
                    partition="CellList", margin=1.0)
    return SystemSpec(boundary=boundary, mass=np.ones(n), pos=pos, vel=vel, lower=np.zeros(3),
                      upper=np.array([96.0, 96.0, 140.0]), attributes={"temperature": 1.0}, global_=[lj],
                      integrator=IntegratorSpec("BAOABLangevin", 0.01, np.full(n, 0.01), seed=3,
                                                remove=(remove, False, False)), name=f"crossing_{boundary}_{n}")


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("case", ["open", "periodic", "tile", "small_separate"])
def test_rows_outgrown_by_a_build_between_two_that_fit(case, precision, monkeypatch):
    """Every build of a segment counts, not only its last: the segment runs again with longer rows.  The tile
    case fixes a staging capacity that the neighbourhoods exceed in the middle of the segment as well, so that
    its rows are served from global memory and from the staged tile in turn."""
    import oracle
    from mjolnir_amd import capi
    if case == "tile":
        monkeypatch.setenv("MJG_TILE_MIN_NP", "0")
        monkeypatch.setenv("MJG_TILE_CAP", "70")
    spec = _crossing_clusters("periodic" if case in ("periodic", "tile") else "unlimited",
                              0 if case == "small_separate" else 4200, remove=case == "small_separate")
    e, o = capi.Engine(spec, capi.FP64 if precision == "fp64" else capi.FP32_FIXED), oracle.OracleEngine(spec)
    built = e.counters()[1]
    e.step(100)
    o.step(100)
    (x, v, _), (xo, vo, _) = e.state(), o.state()
    dx, dv = float(np.abs(x - xo).max()), float(np.abs(v - vo).max())
    print(f"[gpu] {spec.name} {case} {precision}: dx {dx:.1e} dv {dv:.1e} rebuilds {e.counters()[1] - built}", flush=True)
    # FP64: rounding; mixed: forces of up to about 10 kcal/mol/A at 1e-6 of themselves over one time unit
    tol = 1e-8 if precision == "fp64" else 1e-4
    assert dx < tol and dv < tol
    assert np.abs(vo[:48, 0] - 12.0).max() > 0.05              # the clusters did feel each other
    assert e.counters()[1] - built >= 5


def _open_crossing_among(extra):
    """The crossing clusters in an open box among 4200 + extra^3 single particles."""
    spec = _crossing_clusters("unlimited", 4200)
    f = np.stack(np.meshgrid(*[np.arange(extra)] * 3, indexing="ij"), -1).reshape(-1, 3)
    more = (f + 0.5) * 6.0 + [0.0, 0.0, 200.0]
    n = spec.n + len(more)
    g = dataclasses.replace(spec.global_[0], participants=np.arange(n), params=np.tile([1.0, 0.02], (n, 1)))
    return dataclasses.replace(spec, pos=np.concatenate([spec.pos, more]), vel=np.concatenate([spec.vel, np.zeros_like(more)]),
                               mass=np.ones(n), global_=[g],
                               integrator=dataclasses.replace(spec.integrator, coefs=np.full(n, 0.01)))


def test_open_system_above_the_one_workgroup_rebuild_is_set_up_through_its_grid():
    """The first build of a large open system finds its own bounding box.  With all 50,000 participants in one
    cell the set-up took 100 s, most of it one lane's sort; through the grid it takes a few milliseconds."""
    import time
    from mjolnir_amd import capi
    spec = _open_crossing_among(36)
    t0 = time.perf_counter()
    e = capi.Engine(spec)
    took = time.perf_counter() - t0
    print(f"[gpu] open system of {spec.n}: set up in {took:.2f} s", flush=True)
    assert took < 10.0
    assert len(e.pairs(0)) > 48 * 40 and e.pairs(0).max() < 96       # the clusters' pairs alone


def _used():
    """Bytes of the device in use, asked of the HIP runtime that the library has loaded."""
    import ctypes
    from mjolnir_amd import capi
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert capi.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return total.value - free.value


def test_grown_rows_give_the_old_ones_back():
    """The crossing clusters among 50,000 single particles: growing the rows (64 words, then about 130, in the
    list and in the inner list) costs the difference, within 8 MB; the old rows are 26 MB."""
    from mjolnir_amd import capi
    spec = _open_crossing_among(36)
    n = spec.n
    e = capi.Engine(spec)
    e.step(20)
    before = _used()
    e.step(80)
    grown = _used() - before
    rows = 95 + 95 // 4 + 16
    print(f"[gpu] {n} particles: {grown / 2 ** 20:.1f} MB more after growing", flush=True)
    assert grown < 2 * n * 4 * (rows - 64) + 8e6


def test_first_rows_of_a_list_that_drops_other_molecules():
    """Most partners within a large list radius belong to other molecules, which the interaction ignores (here
    all of them: rows of 19,000 words would be 1.5 GB, and as much again beside them)."""
    from mjolnir_amd import capi, workloads
    spec = workloads.lj_fluid(n=20000, seed=2, cutoff=12.0)
    spec.global_[0].ignore_molecule = "Others"
    before = _used()
    e = capi.Engine(spec)
    used = _used() - before
    print(f"[gpu] engine of {spec.n} particles: {used / 2 ** 20:.1f} MB", flush=True)
    assert used < 3e8 and len(e.pairs(0)) == 0


@pytest.mark.parametrize("n,margin", [(300, 0.05), (2000, 0.02), (4096, 0.05), (4096, 0.2)])
def test_dilute_fluids_rebuild_with_enough_lanes(n, margin):
    """Short rows and frequent rebuilds: the rows' lanes are chosen for the rebuild too.  With one lane a row a
    step of the 4096 particles at margin 0.05 took 175 us (15 us now; the bar leaves room for a busy host)."""
    import time
    from mjolnir_amd import workloads
    spec = workloads.lj_fluid(n=n, seed=n, rho_reduced=0.05, margin=margin)
    e = _follow(spec, 90)
    best = 1.0
    for _ in range(5):
        t0 = time.perf_counter()
        e.step(100)
        best = min(best, (time.perf_counter() - t0) / 100)
    print(f"[gpu] dilute {n}, margin {margin}: {best * 1e6:.1f} us a step", flush=True)
    assert best < 60e-6


@pytest.mark.parametrize("n", [1, 10922, 10923, 21845, 40000])
def test_state_set_and_read_back_through_the_pinned_halves(n):
    """Sizes around the particles of a half (10922 triples of positions): positions up to a box width outside come
    back wrapped once, as the reference wraps them, velocities as they are, forces zero before the first call."""
    import ctypes as C
    from mjolnir_amd import capi
    rng = np.random.default_rng(n)
    lower, upper = np.array([-3.0, 0.0, 5.0]), np.array([9.0, 11.0, 18.0])
    w = upper - lower
    pos, vel = lower + w * rng.uniform(-0.9, 1.9, size=(n, 3)), rng.normal(size=(n, 3))
    want = np.where(pos < lower, pos + w, np.where(pos >= upper, pos - w, pos))
    L, h = capi.lib(), C.c_void_p()
    assert L.mjg_engine_create(capi.FP64, capi.PERIODIC, lower, upper, n, 0, C.byref(h)) == capi.OK
    try:
        assert L.mjg_system_set_state(h, np.ones(n), pos, vel) == capi.OK
        x, v, f = (np.full((n, 3), 7.0) for _ in range(3))
        assert L.mjg_system_get_state(h, x.ctypes.data, v.ctypes.data, f.ctypes.data) == capi.OK
    finally:
        L.mjg_engine_destroy(h)
    assert np.array_equal(x, want) and np.array_equal(v, vel) and not f.any()


@pytest.mark.parametrize("potential", ["LennardJones", "ExcludedVolume", "DebyeHuckel", "3SPN2ExcludedVolume"])
@pytest.mark.parametrize("kernel", ["tile", "gather"])
def test_inner_lists_of_every_potential(potential, kernel, monkeypatch):
    """Steps on inner lists (written on the first step of a call, walked on the others) through rebuilds: FP64
    against the oracle; mixed forces of the step against the whole list's at the same positions, bit for
    bit (fixed-point sums), on a step that writes the inner list and on steps that walk it."""
    from mjolnir_amd import capi
    if kernel == "tile":
        monkeypatch.setenv("MJG_TILE_MIN_NP", "0")
    spec = _fluid(potential, 4300, 0.25, 11)
    _follow(spec, 60)
    e = capi.Engine(spec, capi.FP32_FIXED)
    built = e.counters()[1]
    for steps in (1, 2, 27, 41):
        e.step(steps)
        f = e.state()[2]
        e.calc_force()
        assert np.array_equal(f, e.state()[2]), steps
    assert e.counters()[1] > built


def test_inner_lists_of_a_fluid_at_the_tile_size():
    """The same for a fluid that the tile kernel serves by its size, at the usual margin."""
    from mjolnir_amd import capi, workloads
    e = capi.Engine(workloads.lj_fluid(n=16390, seed=5), capi.FP32_FIXED)
    for steps in (1, 2, 90):
        e.step(steps)
        f = e.state()[2]
        e.calc_force()
        assert np.array_equal(f, e.state()[2]), steps


@pytest.mark.parametrize("kernel", ["tile", "gather"])
def test_thin_box_steps(kernel, monkeypatch):
    """FP64 in a box with an axis of three cells narrower than the list radius (the list build tests its
    candidates in FP64 there)."""
    if kernel == "tile":
        monkeypatch.setenv("MJG_TILE_MIN_NP", "0")
    _follow(_fluid("LennardJones", 10 ** 6, 0.25, 4, (THIN[0], THIN[1], 25.0)), 60)


def test_cells_of_more_participants_than_a_wave():
    """Three cells an axis with about 160 participants each: sorted by one lane instead of the wave."""
    _follow(_fluid("LennardJones", 4300, 1.2, 6), 60, rebuilds=False)


@pytest.mark.parametrize("n", [500, 4200])
def test_steps_joined_and_separate_in_turn(n):
    """A motion remover set and taken away between calls: joined steps, separate ones, joined again."""
    import oracle
    from mjolnir_amd import capi, workloads
    spec = workloads.lj_fluid(n=n, seed=n, margin=0.25)
    e, o = capi.Engine(spec), oracle.OracleEngine(spec)
    for remove in (0, 1, 0, 1):
        assert capi.lib().mjg_integrator_set_remover(e.h, remove, 0, 0) == capi.OK
        oracle.lib().orc_set_remover(o.h, remove, 0, 0)
        e.step(30)
        o.step(30)
    (x, v, f), (xo, vo, fo) = e.state(), o.state()
    w = spec.upper - spec.lower
    d = x - xo
    d -= w * np.round(d / w)
    assert np.abs(d).max() < 1e-8 and np.abs(v - vo).max() < 1e-8 and np.abs(f - fo).max() < 1e-8 * np.abs(fo).max()


@pytest.mark.parametrize("n", [70, 3000, 4096, 20000])
def test_participants_crowded_into_one_cell(n):
    """A particle far away from all others stretches an open system's cells until one holds the rest: up to 4096 the
    one-workgroup rebuild, above it the counting sort.  The list is the all-pairs list; one lane's
    sort took 1.8 s for 5000 of them and grows with the square."""
    import time
    from mjolnir_amd import capi
    from mjolnir_amd.spec import GlobalSpec, IntegratorSpec, SystemSpec
    rng = np.random.default_rng(n)
    side = int(np.ceil((n - 1) ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n - 1] * 2.0
    pos = np.concatenate([g, [[1e12, -1e12, 1e12]]])[rng.permutation(n)]
    out = []
    for partition in ("CellList", "VerletList"):
        lj = GlobalSpec(potential="LennardJones", participants=np.arange(n), params=np.tile([1.0, 0.02], (n, 1)),
                        cutoff=2.5, partition=partition, margin=0.1)
        t0 = time.perf_counter()
        e = capi.Engine(SystemSpec(boundary="unlimited", mass=np.ones(n), pos=pos, vel=np.zeros_like(pos),
                                   attributes={"temperature": 1.0}, global_=[lj],
                                   integrator=IntegratorSpec("BAOABLangevin", 0.01, np.full(n, 0.01), seed=3),
                                   name=f"crowd_{n}"))
        print(f"[gpu] {n} in one cell, {partition}: set up in {time.perf_counter() - t0:.3f} s", flush=True)
        out.append((e.pairs(0), time.perf_counter() - t0))
    assert len(out[0][0]) > n and np.array_equal(out[0][0], out[1][0])
    assert out[0][1] < 3.0
