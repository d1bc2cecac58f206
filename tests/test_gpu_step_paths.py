"""Both ways through a step, each forced and each shown to have run: a chain of
like launches and the graph of stages, for systems above the size of four lanes
a sphere and for ensembles (where timing chooses between them otherwise)."""

import numpy as np
import pytest

from parity import all_fields, compare_all
from sphere_amd import configs

pytestmark = pytest.mark.gpu

MEMBER_FIELDS = ["x", "vel", "angvel", "force", "torque", "angpos", "vel0", "angvel0", "xysum", "es_dot", "es", "ev_dot",
                 "ev", "p", "contacts", "delta_t", "walls_nx", "walls_mvfd", "walls_vel0", "wall_pp", "time"]


def _bits(a):
    return a.view(np.uint64) if a.dtype == np.float64 else a


def _ran(dem, path, steps):
    """The steps counted on the path, and on no other."""
    p = dem.path()
    assert (p["chain_steps"], p["stage_steps"]) == ((steps, 0) if path == "chain" else (0, steps)), p
    assert (p["chain_launches"] >= steps) == (path == "chain")
    return p["lanes"]


def _lattice(nside, seed, moving=0.01, speed=3.0):
    sb = configs.lattice_settle(nside=nside, spacing=2.0e-2, jitter=2e-5, r_lo=0.998e-2, r_hi=1.002e-2, gamma_n=0.0,
                                gamma_t=10.0, nw=1)
    sb.wmode = np.array([1], dtype=np.int32)
    sb.w_devs[0] = 1e3
    sb.w_vel[0] = -0.01
    rng = np.random.default_rng(seed)
    sb.vel = np.where(rng.random((sb.np, 1)) < moving, rng.uniform(-speed, speed, (sb.np, 3)), 0.0)
    return sb


@pytest.mark.parametrize("path", ["chain", "stages"])
@pytest.mark.parametrize("nside,lanes", [((20, 21, 22), 4), ((42, 41, 41), 1)])
def test_one_system_against_the_oracle(nside, lanes, path, tmp_path):
    from oracle_lib import Oracle
    from sphere_amd.dem import DEM

    sb = _lattice(nside, 3)
    dem, orc = DEM(sb, verbosity=0), Oracle.from_spherebin(sb, tmp_path)
    dem.set_path(path)
    done = 0
    for steps in (1, 2, 17):
        dem.step(steps)
        done += steps
        assert orc.step(steps) == 0
        assert _ran(dem, path, done) == lanes
        errs = compare_all(dem, orc, all_fields(orc))
        assert not errs, errs
    dem.close()


@pytest.mark.parametrize("nside", [(20, 21, 22), (42, 41, 41)])
def test_one_system_in_mixed_precision(nside):
    """The two paths against each other (the oracle computes in FP64)."""
    from sphere_amd.dem import DEM

    sb = _lattice(nside, 4)
    got = []
    for path in ("chain", "stages"):
        dem = DEM(sb, verbosity=0)
        dem.set_precision("mixed")
        dem.set_path(path)
        dem.step(1)
        dem.step(24)
        _ran(dem, path, 25)
        got.append({f: dem.get(f) for f in MEMBER_FIELDS})
        dem.close()
    for f in MEMBER_FIELDS:
        assert np.array_equal(_bits(got[0][f]), _bits(got[1][f])), f


@pytest.mark.parametrize("path", ["chain", "stages"])
@pytest.mark.parametrize("sides", [((6, 6, 6), (4, 5, 9), (1, 1, 1)), ((26, 26, 26), (6, 6, 6))])
def test_ensemble_members_against_their_own_handles(sides, path):
    """Members with up to 64 wall-sum blocks, whose walls take one launch of the
    chain, and one with more (17,576 spheres), which takes two."""
    from sphere_amd.dem import DEM, Ensemble

    sbs = [_lattice(s, 10 + k) if np.prod(s) > 1 else configs.lattice_settle(nside=s, spacing=2.1e-2, jitter=0.0, nw=1, periodic=0)
           for k, s in enumerate(sides)]
    ens = Ensemble(sbs)
    ens.set_path(path)
    ens.step(1)
    ens.step(30)
    assert _ran(ens, path, 31) == 1
    for k, sb in enumerate(sbs):
        dem = DEM(sb, verbosity=0)
        dem.step(1)
        dem.step(30)
        for f in MEMBER_FIELDS:
            assert np.array_equal(_bits(ens.get(k, f)), _bits(dem.get(f))), (k, f)
        dem.close()
    ens.close()


@pytest.mark.parametrize("sides", [((6, 6, 6), (4, 5, 9)), ((26, 26, 26), (6, 6, 6))])
def test_ensemble_in_mixed_precision(sides):
    from sphere_amd.dem import Ensemble

    sbs = [_lattice(s, 20 + k) for k, s in enumerate(sides)]
    got = []
    for path in ("chain", "stages"):
        ens = Ensemble(sbs)
        ens.set_precision("mixed")
        ens.set_path(path)
        ens.step(1)
        ens.step(30)
        _ran(ens, path, 31)
        got.append([{f: ens.get(k, f) for f in MEMBER_FIELDS} for k in range(len(sbs))])
        ens.close()
    for a, b in zip(*got):
        for f in MEMBER_FIELDS:
            assert np.array_equal(_bits(a[f]), _bits(b[f])), f


def _pair_about_two_faces():
    """Two touching spheres a cell apart, both turning round a cell face (one
    of them the periodic one) within the lists' reach: b to the left of the
    periodic face in steps 3 to 5 only, a to the right of its own in the steps
    in which b is not."""
    from sphere_amd.spherebin import Spherebin

    D, dt = 0.02, 1e-4
    sb = Spherebin(2, nw=0, sid="two-faces")
    sb.set_walls(0)
    configs._contact_params(sb, k_n=1e3, k_t=1e3, gamma_n=0.0, gamma_t=0.0)
    sb.radius = np.full(2, D / 2)
    sb.x = np.array([[0.028 * D, 2.5 * D, 2.5 * D], [1.026 * D, 2.5 * D, 2.5 * D]])
    sb.vel = np.array([[-0.018 * D / dt, 0.0, 0.0]] * 2)
    configs._grid(sb, [8 * D, 6 * D, 6 * D], 0.999999 * D)
    assert tuple(sb.num) == (8, 6, 6)
    sb.periodic = 1
    sb.g = np.array([0.004 * D / dt ** 2, 0.0, 0.0])
    sb.time_dt = dt
    sb.time_total = sb.time_file_dt = 1.0
    return sb


@pytest.mark.parametrize("switch", ["profiling", "graph"])
def test_stages_between_chain_steps_that_change_an_image(switch):
    """What a chain's search has noted about a sphere's contacts (that none goes
    through a periodic face) does not outlast steps taken as stages."""
    from sphere_amd.dem import Ensemble

    sbs = [_pair_about_two_faces(), _pair_about_two_faces()]
    got = []
    for path in ("chain", "stages"):
        ens = Ensemble(sbs)
        ens.set_path(path)
        ens.step(3)
        ens.set_profiling(switch == "profiling")
        ens.set_graph(switch != "graph")
        ens.step(3)
        ens.set_profiling(False)
        ens.set_graph(True)
        ens.step(1)
        p = ens.path()
        assert (p["chain_steps"], p["stage_steps"]) == ((4, 3) if path == "chain" else (0, 7)), p
        got.append([{f: ens.get(k, f) for f in MEMBER_FIELDS if not f.startswith("wall")} for k in range(2)])
        ens.close()
    assert np.all(got[1][0]["force"][:, 0] != 0.0)  # the pair touches in the last step
    for a, b in zip(*got):
        for f in a:
            assert np.array_equal(_bits(a[f]), _bits(b[f])), f


def test_launches_of_a_long_call_after_a_short_one():
    """One step after new positions sorts and builds lists (six launches); the
    quiet steps of the next call are one launch each."""
    from sphere_amd.dem import DEM

    sb = configs.lattice_settle(nside=(10, 10, 10), spacing=2.1e-2, jitter=0.0, r_lo=1e-2, r_hi=1e-2, gravity=0.0)
    dem = DEM(sb, verbosity=0)
    for _ in range(2):
        dem.set("x", dem.get("x"))
        dem.step(1)
        before = dem.path()["chain_launches"]
        dem.step(300)
        assert dem.path()["chain_launches"] - before <= 310
    dem.close()


def test_block_sizes_of_an_ensemble_are_the_callers():
    """Set sizes are those of the kernels that run: not of a chain, which has
    its own."""
    from sphere_amd.dem import Ensemble

    sbs = [_lattice((6, 6, 6), 1), _lattice((7, 5, 6), 2)]
    got = []
    for blocks in (None, (64, 128)):
        ens = Ensemble(sbs)
        ens.set_path("chain")
        if blocks:
            ens.set_blocks(*blocks)
        ens.step(10)
        i = ens.info()
        if blocks:
            assert (i.force_block, i.search_block) == blocks
        _ran(ens, "stages" if blocks else "chain", 10)
        got.append([ens.get(k, "x") for k in range(2)])
        ens.close()
    for a, b in zip(*got):
        assert np.array_equal(_bits(a), _bits(b))


def _large_among_small(side=17, ratio=6.0):
    """A sphere with more small neighbours within the lists' reach than a list
    holds (48), none of them touching it."""
    from sphere_amd.spherebin import Spherebin

    r, a = 1e-3, 2.2e-3
    L = np.full(3, side * a)
    x = (np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) * a
    R = ratio * r
    x = x[np.linalg.norm(x - L / 2, axis=1) > R + 1.01 * r]
    sb = Spherebin(len(x) + 1, nw=0, sid="large-among-small")
    sb.set_walls(0)
    configs._contact_params(sb, gamma_n=0.0, gamma_t=10.0)
    sb.x = np.concatenate([x, [L / 2]])
    sb.radius = np.concatenate([np.full(len(x), r), [R]])
    configs._grid(sb, L, 2 * R)
    sb.periodic = 1
    sb.g = np.zeros(3)
    sb.time_dt = configs._dt(sb)
    sb.time_total = sb.time_file_dt = 1.0
    sb.vel = np.random.default_rng(1).uniform(-0.5, 0.5, (sb.np, 3))
    return sb


@pytest.mark.parametrize("path", ["chain", "stages"])
def test_neighbour_list_that_overflows(path, tmp_path):
    """Such a list is no use and is built at every step; four lanes a sphere
    against the oracle, one lane (an ensemble) against those."""
    from oracle_lib import Oracle
    from sphere_amd.dem import DEM, Ensemble

    sb = _large_among_small()
    near = np.linalg.norm(sb.x[:-1] - sb.x[-1], axis=1) < sb.radius[0] + sb.radius[-1] + 0.1 * np.min(sb.L / sb.num)
    assert near.sum() > 48
    dem, orc, ens = DEM(sb, verbosity=0), Oracle.from_spherebin(sb, tmp_path), Ensemble([sb, sb])
    dem.set_path(path)
    ens.set_path(path)
    for steps in (1, 9, 30):
        dem.step(steps)
        ens.step(steps)
        assert orc.step(steps) == 0
        errs = compare_all(dem, orc, all_fields(orc))
        assert not errs, errs
    if path == "chain":
        assert dem.timing()["list_builds"] == ens.timing()["list_builds"] == 40
        assert _ran(dem, path, 40) == 4 and _ran(ens, path, 40) == 1
    for f in MEMBER_FIELDS:
        if not f.startswith("wall"):
            assert np.array_equal(_bits(ens.get(1, f)), _bits(dem.get(f))), f
    dem.close()
    ens.close()
