"""The adjoint's two ways of running its steps (a recording chain of launches,
and single steps with hooks when the kernels are chosen by the caller) step the
same bits, so J and the gradient agree to the rounding of their sums; a second
run reuses the first one's buffers."""

import numpy as np
import pytest

from sphere_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("steps,segment", [(1, 1), (10, 3), (9, 16)])
def test_recorded_chain_matches_hooks(precision, steps, segment):
    from sphere_amd.dem import DEM

    sb = configs.fcc_shear(cells=(5, 6, 5))
    w = np.zeros((sb.np, 3))
    w[np.asarray(sb.vel)[:, 0] > 0.0, 0] = -1.0 / (sb.L[0] * sb.L[1])
    got = []
    for variant in (0, 1):
        dem = DEM(sb, verbosity=0)
        dem.set_precision(precision)
        dem.set_force_kernel(variant)
        dem.step(3)
        runs = []
        for _ in range(2):
            J = dem.adjoint_forward(steps, w, segment)
            runs.append((J, dem.adjoint_backward(), dem.get("x"), dem.get("delta_t")))
        got.append(runs)
        dem.close()
    for a, b in zip(*got):
        assert a[0] == pytest.approx(b[0], rel=1e-9)
        assert np.allclose(a[1], b[1], rtol=1e-9, atol=0.0)
        assert np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tape_that_does_not_fit_leaves_nothing_half_made(precision):
    """A segment whose tape is more than the card holds (5.6e8 particle-steps:
    134 GB, which fit, and then springs of 430 GB or, in FP32, 215 GB): the call
    is refused each time it is made, and what follows runs as if it had not been
    made."""
    from sphere_amd.dem import DEM, HipError

    sb = configs.fcc_shear(cells=(5, 6, 5))
    w = np.zeros((sb.np, 3))
    w[np.asarray(sb.vel)[:, 0] > 0.0, 0] = -1.0 / (sb.L[0] * sb.L[1])
    segment = int(5.6e8 / sb.np)
    got = []
    for refused in (True, False):
        dem = DEM(sb, verbosity=0)
        dem.set_precision(precision)
        if refused:
            dem.adjoint_forward(2, w, segment)
            for _ in range(2):
                with pytest.raises(HipError):
                    dem.adjoint_backward()
            dem.adjoint_forward(2, w, segment)
            with pytest.raises(HipError):
                dem.adjoint_backward()
        else:
            dem.step(4)
        dem.step(1)
        got.append((dem.adjoint_forward(3, w, 2), dem.adjoint_backward(), dem.get("x"), dem.get("delta_t")))
        dem.close()
    a, b = got
    assert a[0] == pytest.approx(b[0], rel=1e-9)
    assert np.allclose(a[1], b[1], rtol=1e-9, atol=0.0)
    assert np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3])


def test_plain_launches_are_plain_in_the_adjoint_too():
    """set_graph(False) asks for one kernel per stage; back on, the same handle
    steps as a chain again."""
    from sphere_amd.dem import DEM

    sb = configs.fcc_shear(cells=(5, 6, 5))
    w = np.zeros((sb.np, 3))
    w[np.asarray(sb.vel)[:, 0] > 0.0, 0] = -1.0 / (sb.L[0] * sb.L[1])
    got = []
    for graph in (True, False):
        dem = DEM(sb, verbosity=0)
        dem.set_graph(graph)
        dem.step(3)
        got.append((dem.adjoint_forward(7, w, 3), dem.adjoint_backward(), dem.get("x"), dem.get("delta_t")))
        p = dem.path()
        assert (p["chain_steps"] > 0, p["stage_steps"] > 0) == (graph, not graph), p
        dem.set_graph(True)
        dem.step(5)
        q = dem.path()
        assert q["chain_steps"] == p["chain_steps"] + 5 and q["stage_steps"] == p["stage_steps"], q
        dem.close()
    a, b = got
    assert a[0] == pytest.approx(b[0], rel=1e-9)
    assert np.allclose(a[1], b[1], rtol=1e-9, atol=0.0)
    assert np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3])
