"""Edges of how the step's work is split over launches and workgroups: lists
longer than one launch's threads, tiles smaller than the default and grids on
either side of a rule's line. Needs an MI355X."""
import ctypes
import time

import numpy as np
import pytest

from method_amd import engine as eng
from method_amd import initdata as idt
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 40])
def test_retry_of_every_cell_clears_its_list(n):
    """Every cell fails from a guess at |v| = 1 and is recovered by the retry
    from rest: fewer cells than one workgroup's threads, and more than all the
    threads of the launch (64 x 256). A second call finds an empty list, so it
    counts the same failures. The root is found to the Newton tolerance 1e-12,
    which the recovery divides by p's share of the energy, above 1e-2 here."""
    g = idt.kh3d_grid(n)
    p0 = idt.kh_prims(g, seed=3)
    print(f"gpu: retry of all cells, {n}^3", flush=True)
    with eng.Engine(eng.Config(n, n, n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0, quirks=0)) as e:
        e.set_prims(p0)
        true = e.download()[1]
        bad = true.copy()
        bad[1], bad[2], bad[3] = 1.0, 0.0, 0.0
        for call in range(2):
            e.upload(prims=bad)
            rc, st = e.c2p()
            got = e.download()[1]
            assert rc == n**3 and st["failures"] == n**3 and st["fallbacks"] == 0, call
            assert np.abs(got - true).max() <= 1e-10


@pytest.mark.parametrize("nx,ny", [(8, 15), (185, 252), (193, 257), (225, 233)])
@pytest.mark.parametrize("resistive,weno", [(False, 3), (False, 5), (True, 3), (True, 5)])
def test_2d_tiles_equal_separate_sweeps_bitwise(nx, ny, resistive, weno):
    """The 2-D launch on its 8 x 8 tiles (up to 768 of them: 185 x 252 is 24 x 32)
    and on the larger ones beyond, with ragged edges, against the y and x
    launches of plan 0: the same sums in the same order, so the same bits."""
    print(f"gpu: 2-D tiles {nx}x{ny} resistive={resistive} weno={weno}", flush=True)
    g = idt.Grid(nx, ny, 0, 0.0, 1.0, 0.0, 1.0)
    if resistive:
        prims = idt.ot_prims_resistive(g)
        cfg = dict(model=eng.SRRMHD, integrator=eng.SSP2, sigma=10.0)
    else:
        prims = idt.kh_prims(g, seed=9)
        cfg = dict(model=eng.SRMHD, integrator=eng.RK2)
    got = []
    for plan in (3, 0):
        with eng.Engine(eng.Config(nx, ny, 0, 0.0, 1.0, 0.0, 1.0, weno_order=weno,
                                   bc=(eng.OUTFLOW, eng.PERIODIC, eng.PERIODIC), **cfg)) as e:
            e.set_sweep_plan(plan)
            e.set_prims(prims)
            for _ in range(2):
                e.update_time()
            got.append(e.download())
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nx", [5, 31, 32, 33, 97])
@pytest.mark.parametrize("weno,periodic", [(3, 1), (5, 0)])
def test_1d_tiles_match_oracle(nx, weno, periodic):
    """1-D grids around the 32-cell tile against the oracle: three steps, each
    exact to the Newton tolerance 1e-12 times the handful of fields it feeds."""
    ng = 4
    g = idt.Grid(nx, 0, 0, -0.5, 0.5, 0.0, 1.0)
    x = np.linspace(-0.6, 0.6, nx + 2 * ng)
    p = np.zeros((8,) + g.shape)
    p[0, :, 0, 0], p[4, :, 0, 0] = 1.0 + 0.3 * np.sin(5 * x), 1.0 + 0.2 * np.cos(3 * x)
    p[1, :, 0, 0], p[2, :, 0, 0], p[3, :, 0, 0] = 0.3 * np.cos(4 * x), 0.2 * np.sin(x), -0.1
    p[5], p[6, :, 0, 0], p[7] = 0.4, 0.3 * np.sin(2 * x), 0.2
    print(f"gpu: 1-D {nx} weno={weno}", flush=True)
    bounds = dict(nx=nx, ny=0, nz=0, xmin=-0.5, xmax=0.5, ymin=0.0, ymax=1.0)
    with eng.Engine(eng.Config(weno_order=weno, bc=(periodic,) * 3, **bounds)) as e:
        e.set_prims(p)
        for _ in range(3):
            rc, st = e.update_time(stats=True)
            assert rc == 0 and st["cells"] == 2 * nx
        c, q, a = e.download()
    oc, oq, oa, _, _ = orc.Oracle(orc.Case(weno_order=weno, periodic=(periodic,) * 3, **bounds)).run(p, 3)
    for got, ref in ((c, oc), (q, oq), (a, oa)):
        for u, v in zip(got[:, ng:-ng], ref[:, ng:-ng]):
            assert np.abs(u - v).max() <= 1e-11 * max(1.0, np.abs(v).max())


def test_batch_tilings_and_retry_launch():
    """Every tile shape and schedule, with fewer workgroups than tiles on an
    XCD and more than there are tiles, gives the same bits; a member whose
    every cell starts from |v| = 1 is retried by the launch that ends a stage,
    once per stage and step, which it can only count when the list is cleared."""
    sizes = [(17, 33), (8, 8), (40, 31)]
    print("gpu: batch tilings", flush=True)
    prims = [idt.kh_prims(idt.Grid(nx, ny, 0, -0.5, 0.5, -1.0, 1.0), seed=k) for k, (nx, ny) in enumerate(sizes)]
    ref = None
    for tile in ((16, 16), (8, 32), (32, 8), (8, 16)):
        for sched in (0, 1):
            for blocks in (8, 2048):
                with eng.Batch([eng.Instance(nx, ny) for nx, ny in sizes], weno_order=3, quirks=0) as b:
                    for k, p in enumerate(prims):
                        b.set_prims(k, p)
                    b.set_tuning(*tile, sched, blocks)
                    assert b.step(3) == 0
                    out = [b.download(k) for k in range(len(sizes))]
                    c, p, a = b.download(0)
                    bad = p.copy()
                    bad[0] = 1e-310  # the starting root Z = rho h / (1 - v^2) is infinite
                    b.upload(0, c, bad, a)
                    rc, st = b.step(2, stats=True)
                    # both stages of the first step start from the bad prims, the second step from good ones
                    assert st["failures"] == rc == 2 * 17 * 33 and st["fallbacks"] == 0, (tile, sched, blocks)
                if ref is None:
                    ref = out
                for x, y in zip(out, ref):
                    for u, v in zip(x, y):
                        assert np.array_equal(u, v)


@pytest.mark.parametrize("n", [(5, 9, 17), (8, 40, 70), (70, 17, 33), (9, 130, 97)])
@pytest.mark.parametrize("resistive,weno", [(False, 3), (False, 5), (True, 3)])
def test_3d_tiles_equal_separate_sweeps_bitwise(n, resistive, weno):
    """The fused y + z launch and the x sweep on the tiles of small grids (8 x 8,
    up to 256 16 x 16 tiles), of grids short along z (16 x 16) and of long ones
    (8 x 32), with ragged edges, against plan 2's three launches: the same bits."""
    print(f"gpu: 3-D tiles {n} resistive={resistive} weno={weno}", flush=True)
    g = idt.Grid(*n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0)
    prims = idt.kh_prims(g, seed=4)
    prims[5], prims[6] = 0.1, -0.2
    cfg = dict(model=eng.SRMHD, integrator=eng.RK2)
    if resistive:
        v, B = prims[1:4], prims[5:8]
        prims = np.concatenate([prims, -np.cross(v, B, axis=0)])
        cfg = dict(model=eng.SRRMHD, integrator=eng.RK2, sigma=0.1)
    got = []
    for plan in (3, 2):
        with eng.Engine(eng.Config(*n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0, weno_order=weno, **cfg)) as e:
            e.set_sweep_plan(plan)
            e.set_prims(prims)
            for _ in range(2):
                e.update_time()
            got.append(e.download())
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("n", [(50, 131, 129), (17, 190, 190), (16, 181, 182)])
@pytest.mark.parametrize("weno,periodic", [(3, 1), (5, 0), (5, 1)])
def test_marching_x_sweep_equals_tiles_bitwise(n, weno, periodic):
    """The marching x sweep (three segments, one of 17 and one of 16 cells, columns
    that do not fill the last wave) against the tiled one, which finishes the
    stage under plan 0: on a state uniform in y and z the other axes' terms are
    exactly zero, so both give the same bits."""
    ng = 4
    print(f"gpu: marching x sweep {n} weno={weno}", flush=True)
    x = np.linspace(0.0, 1.0, n[0] + 2 * ng)[:, None, None]
    p = np.zeros((8,) + tuple(k + 2 * ng for k in n))
    p[0], p[4] = 1.0 + 0.4 * np.sin(9 * x), 1.0 + 0.3 * np.cos(7 * x)
    p[1], p[2], p[3] = 0.4 * np.cos(5 * x), 0.2 * np.sin(3 * x), -0.1 + 0.1 * x
    p[5], p[6], p[7] = 0.4, 0.3 * np.sin(2 * x), 0.2 * np.cos(x)
    got = []
    for plan in (3, 0):
        with eng.Engine(eng.Config(*n, 0.0, 1.0, 0.0, 1.0, 0.0, 1.0, weno_order=weno, bc=(periodic,) * 3)) as e:
            e.set_sweep_plan(plan)
            e.set_prims(p)
            for _ in range(2):
                e.update_time()
            got.append(e.download())
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("integrator", [eng.RK2B, eng.RK3, eng.RK4])
@pytest.mark.parametrize("n,resistive", [((41, 0, 0), False), ((37, 23, 0), False), ((37, 23, 0), True),
                                         ((230, 229, 0), False), ((9, 14, 11), True)])
def test_rkplus_stages_in_the_sweeps(integrator, n, resistive):
    """RKPlus stages are put together by the last sweep, whichever launch that is:
    the fused one (plan 3) and the separate one that sums in the same order (plan
    2 in 3-D, 0 in 2-D) give the same bits, the aux among them, which for SRMHD
    is formed from the kept root and has to be the one of the downloaded prims:
    h, W and v^2 recomputed from them agree to a few roundings (1e-13)."""
    print(f"gpu: rkplus {integrator} {n} resistive={resistive}", flush=True)
    g = idt.Grid(*n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0)
    p = idt.kh_prims(g, seed=8)
    p[5], p[6] = 0.2, 0.1
    cfg = dict(model=eng.SRMHD, cp=1.0)
    if resistive:
        p = np.concatenate([p, -np.cross(p[1:4], p[5:8], axis=0)])
        cfg = dict(model=eng.SRRMHD, sigma=1.0, cp=1.0)
    got = []
    for plan in (3, 2 if n[2] else 0):
        with eng.Engine(eng.Config(*n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0, integrator=integrator, **cfg)) as e:
            e.set_sweep_plan(plan)
            e.set_prims(p)
            for _ in range(2):
                assert e.update_time() == 0
            got.append(e.download())
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.array_equal(a, b)
    _, q, a = got[0]
    v2 = (q[1:4] ** 2).sum(0)
    assert np.abs(a[9] - v2).max() <= 1e-13
    assert np.abs(a[1] * np.sqrt(1 - v2) - 1).max() <= 1e-12


def failing(true, where):
    """Prims whose guess is at |v| = 1 in the cells `where`, so that they fail there."""
    bad = true.copy()
    bad[1][where], bad[2][where], bad[3][where] = 1.0, 0.0, 0.0
    return bad


def test_failed_cells_marks_run_out():
    """Lists of failed cells follow one another with no flag taken down until the
    255 marks are used up: after 300 and 600 of them, alternating between the two
    colours of a checkerboard and then all cells, each retry still starts from the
    neighbours that did not fail (from rest if all did), so it leaves the bits that
    a new engine's first call does."""
    n = 11  # 1,331 flags: 83 groups of 16 and 3 more
    g = idt.kh3d_grid(n)
    p0 = idt.kh_prims(g, seed=3)
    cfg = eng.Config(n, n, n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0, quirks=0)
    colour = np.indices((n + 2 * 4,) * 3).sum(0) % 2 == 0
    cases = [colour, ~colour, np.ones_like(colour)]
    print("gpu: marks of failed cells", flush=True)
    want = []
    for where in cases:
        with eng.Engine(cfg) as e:
            e.set_prims(p0)
            true = e.download()[1]
            e.upload(prims=failing(true, where))
            assert e.c2p()[1]["fallbacks"] == 0
            want.append(e.download()[1])
    with eng.Engine(cfg) as e:
        e.set_prims(p0)
        for call in range(603):
            e.upload(prims=failing(true, cases[call % 3]))
            e.c2p()
            if call % 300 < 3:
                assert np.array_equal(e.download()[1], want[call % 3]), call


def test_retry_of_every_cell_takes_no_longer_than_the_cells_do():
    """A cons2prim of 128^3 cells that all fail runs every cell's Newton twice, the
    second time on 64 workgroups: 7 times the time of one where none fails.
    Taking two million flags down in one workgroup made that 25 times."""
    n = 128
    g = idt.kh3d_grid(n)
    print("gpu: time of a full retry", flush=True)
    with eng.Engine(eng.Config(n, n, n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0, quirks=0)) as e:
        e.set_prims(idt.kh_prims(g, seed=3))
        true = e.download()[1]
        took = []
        for prims in (true, failing(true, np.ones(true.shape[1:], bool))):
            best = np.inf
            for _ in range(5):
                e.upload(prims=prims)
                t = time.perf_counter()
                e.c2p()
                best = min(best, time.perf_counter() - t)
            took.append(best)
    assert took[1] <= 14 * took[0], took


def test_timed_c2p_leaves_no_failed_cells_behind():
    """The timed cons2prim runs without a retry. Its failed cells are forgotten,
    three lists of every cell among them: the prims stay those of the first pass,
    and the step after it, from good prims, is the step of an engine that timed
    nothing, bit for bit (a cell found on an old list would be solved again, from
    its neighbours' mean root)."""
    n = 10
    g = idt.kh3d_grid(n)
    cfg = eng.Config(n, n, n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0, quirks=0)
    print("gpu: timed cons2prim with failures", flush=True)
    got = []
    for timed in (False, True):
        with eng.Engine(cfg) as e:
            e.set_prims(idt.kh_prims(g, seed=3))
            cons, true, aux = e.download()
            if timed:
                e.upload(prims=failing(true, np.ones(true.shape[1:], bool)))
                _, st, _ = e.timed_c2p(3)
                assert st["failures"] == n**3
                e.upload(cons, true, aux)
            rc, st = e.update_time(stats=True)
            assert rc == 0 and st["failures"] == 0
            got.append(e.download())
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("integrator,stages", [(eng.RK2B, 1), (eng.RK3, 2), (eng.RK4, 4)])
def test_rkplus_engines_hold_no_root_beside_the_aux(integrator, stages):
    """Device memory of an SRMHD RKPlus engine: cons, prims and aux (30 doubles a
    cell), one stage's cons and prims and the net flux (26), 17 per stage state, 9
    for RK4's kept rhs, 9 bytes of the failed cells' list and flags, and less than
    half a double of rounding up to whole pages. The cons2prim root lives in the
    aux array, and the aux formed from it there is the one a fresh array gets."""
    hip = ctypes.CDLL("libamdhip64.so.7")

    def free_memory():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    n = 1024
    print(f"gpu: memory of integrator {integrator}", flush=True)
    eng.Engine(eng.Config(8, 8, 0, 0.0, 1.0, 0.0, 1.0, integrator=integrator)).close()
    free = free_memory()
    with eng.Engine(eng.Config(n, n, 0, -0.5, 0.5, -1.0, 1.0, integrator=integrator)) as e:
        used = (free - free_memory()) / (8 * n * n)
        assert used <= 56 + 17 * stages + (9 if integrator == eng.RK4 else 0) + 9 / 8 + 0.5, used
        e.set_prims(idt.kh_prims(idt.Grid(n, n, 0, -0.5, 0.5, -1.0, 1.0), seed=8))
        assert e.update_time() == 0
        _, q, a = e.download()
        again = e.download()[2]
    v2 = (q[1:4] ** 2).sum(0)
    assert np.abs(a[9] - v2).max() <= 1e-13 and np.abs(a[1] * np.sqrt(1 - v2) - 1).max() <= 1e-12
    assert np.array_equal(a, again)


@pytest.mark.parametrize("n", [(40, 31), (700, 650)])
def test_autotuner_descends_the_workgroup_counts(n):
    """The autotuner takes each tile shape and schedule with the two largest resident
    numbers of workgroups per CU, then down to one or to the first number that is
    2 % slower than the best, and chooses the fastest of all it tried."""
    print(f"gpu: autotuner candidates {n}", flush=True)
    with eng.Batch([eng.Instance(*n)], weno_order=3) as b:
        b.set_prims(0, idt.kh_prims(idt.Grid(*n, 0, -0.5, 0.5, -1.0, 1.0), seed=1))
        best, tried = b.autotune(2)
    rows = {}
    for c in tried:
        rows.setdefault((c["tile_x"], c["tile_y"], c["schedule"]), []).append((c["blocks"], c["ms_per_step"]))
    assert len(rows) == 8  # four shapes, two schedules
    ncu = min(row[1][0] - row[0][0] for row in rows.values())
    for row in rows.values():
        counts, ms = [k // ncu for k, _ in row], [t for _, t in row]
        top = counts[1]
        assert counts == [top - 1, top] + list(range(top - 2, counts[-1] - 1, -1))[:len(row) - 2], rows
        down = [0] + list(range(2, len(row)))  # tried one after the other downwards
        slower = [ms[k] > 1.02 * min(ms[:max(k, 1) + 1]) for k in down]
        assert not any(slower[:-1]) and (1 in counts or slower[-1]), rows
    fastest = min(tried, key=lambda c: c["ms_per_step"])
    assert all(best[k] == fastest[k] for k in ("tile_x", "tile_y", "schedule", "blocks"))


def waves_3d(n, ng=4):
    """SRMHD prims that vary along all three axes, each with its own wavelengths."""
    x, y, z = np.meshgrid(*[np.linspace(0.0, 1.0, k + 2 * ng) for k in n], indexing="ij")
    p = np.zeros((8,) + x.shape)
    p[0], p[4] = 1.0 + 0.3 * np.sin(9 * x + 17 * y + 23 * z), 1.0 + 0.3 * np.cos(7 * x - 13 * y + 19 * z)
    p[1], p[2], p[3] = 0.3 * np.cos(5 * x + 29 * z), 0.2 * np.sin(3 * x + 31 * y), 0.2 * np.cos(11 * y - 8 * z)
    p[5], p[6], p[7] = 0.4 * np.sin(6 * y), 0.3 * np.sin(2 * x + 37 * z), 0.2 * np.cos(x + 21 * y)
    return p


@pytest.mark.parametrize("n", [(50, 131, 129), (17, 190, 190), (48, 127, 129), (6007, 11, 17)])
@pytest.mark.parametrize("weno,periodic", [(3, 1), (3, 0), (5, 1), (5, 0)])
def test_marching_x_sweep_keeps_to_its_columns(n, weno, periodic):
    """The marching x sweep on a state that varies along y and z, with a last wave
    of 3, 4 and 63 columns in use and, on the long thin grid, of 59 and hundreds of
    segments: the net flux against plan 0, whose x sweep is tiled and sums the axes
    the other way round. Same terms in another order: three roundings, 3.4e-16 of
    the terms, which are within ten times the largest net flux."""
    print(f"gpu: marching x sweep with structure {n} weno={weno} periodic={periodic}", flush=True)
    got = []
    for plan in (3, 0):
        with eng.Engine(eng.Config(*n, 0.0, 1.0, 0.0, 1.0, 0.0, 1.0, weno_order=weno, bc=(periodic,) * 3)) as e:
            e.set_sweep_plan(plan)
            e.set_prims(waves_3d(n))
            got.append(e.fnet())
    for v, (a, b) in enumerate(zip(*got)):
        assert np.isfinite(a).all() and np.abs(a - b).max() <= 3.4e-15 * np.abs(got[1]).max(), v


TILES_3D = [(70, 17, 33), (9, 130, 97), (9, 130, 104)]  # 16 x 16, 8 x 32 and, by its aligned rows, 16 x 16 again


@pytest.mark.parametrize("n", TILES_3D)
@pytest.mark.parametrize("kind,weno", [("rk2", 3), ("rk2", 5), ("rk3", 3), ("rk4", 5), ("ssp2", 3), ("ssp2", 5),
                                       ("resistive rk2", 5), ("resistive rk3", 3)])
def test_3d_modes_on_every_tile_bitwise(n, kind, weno):
    """What the fused y + z launch does with a cell (RK2, RKPlus and both SSP2
    stages) on the tiles of grids beyond 256 16 x 16 tiles, against plan 2's
    separate launches: the same bits."""
    print(f"gpu: 3-D {kind} {n} weno={weno}", flush=True)
    p = waves_3d(n)
    cfg = dict(integrator={"rk2": eng.RK2, "rk3": eng.RK3, "rk4": eng.RK4, "ssp2": eng.SSP2}[kind.split()[-1]])
    if kind == "ssp2" or kind.startswith("resistive"):
        p = np.concatenate([p, -np.cross(p[1:4], p[5:8], axis=0)])
        cfg.update(model=eng.SRRMHD, sigma=1.0)
    got = []
    for plan in (3, 2):
        with eng.Engine(eng.Config(*n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0, weno_order=weno, cp=1.0, **cfg)) as e:
            e.set_sweep_plan(plan)
            e.set_prims(p)
            for _ in range(2):
                e.update_time()
            got.append(e.download())
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.array_equal(a, b)
