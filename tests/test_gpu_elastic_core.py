"""The fused core of a 2D elastic step, on grids that hold it, against the oracle.

Every case is large enough that the core takes more than half the nodes, with
its block columns and row chunks ending ragged; the frame around it runs the
pair's code. Forward fields and traces are expected to the bit (the core runs
the pair's operations in their order); the gradient, whose reverse march and
adjoint pair run through the core too, within the tolerance of the elastic
tests (1e-4 relative in float32, 1e-10 in float64).
"""

from __future__ import annotations

import numpy as np
import pytest

from helpers import Receivers, elastic_core_nodes, host, rel_max

pytestmark = pytest.mark.gpu

from cuwave_amd import boundary, elastic, utils, wave  # noqa: E402

T, C = boundary.Traction, boundary.Clamped


def _case(n, order, shots, N, precision, walls, layer, faces, plane="strain"):
    from oracle import driver as D
    from oracle import elastic as E

    pml = boundary.Pml(layer, 2.0, 1e-6, 2.0, faces) if layer else None
    sim = elastic.ElasticWave(n, (1.0, 1.1), N, 0.12, precision=precision, space_order=order,
                              density=1.3, wavespeed_p=2.0, wavespeed_s=1.0, plane=plane,
                              boundary=walls, pml=pml)
    rng = np.random.default_rng(sum(n) + order)
    gamma = (0.8 + 0.4 * rng.random(sim.Nx_padded)).astype(sim.np_dtype)
    sig = rng.standard_normal((N, 1)).astype(sim.np_dtype)
    sources = [wave.Source(np.array([[k % 2], [rng.integers(2, n[0] - 3)],
                                     [rng.integers(2, n[1] - 3)]]), sig * (1 + k))
               for k in range(shots)]
    sensors = np.stack([rng.integers(0, 2, 20), rng.integers(2, n[0] - 3, 20),
                        rng.integers(2, n[1] - 3, 20)])
    osim = E.ElSim(sim.Nx, sim.dx, sim.N, sim.dt, sim.precision, sim.space_order, sim.stencil,
                   tuple(tuple(int(c == C) for c in pair) for pair in walls), sim.density,
                   sim.wavespeed_p, sim.wavespeed_s, plane,
                   D.Pml(layer, 2.0, 1e-6, 2.0, faces) if layer else None)
    return sim, osim, gamma, sources, sensors


LINED = ((T, C), (C, C))
CASES = [
    ((131, 157), 4, 3, 12, "float32", LINED, 9, (1, 2, 3)),     # lanes a thread, one block column
    ((140, 333), 2, 1, 12, "float32", ((T, T), (T, T)), 0, ()),  # one lane, two block columns
    ((117, 203), 4, 16, 10, "float32", ((C, C), (C, C)), 8, (0, 1, 2, 3)),
    ((150, 145), 6, 5, 10, "float64", ((T, C), (C, T)), 0, ()),  # no layer, two lanes of eight
    ((163, 170), 8, 2, 10, "float32", ((T, C), (T, C)), 11, (3,)),
    ((128, 128), 4, 33, 8, "float32", LINED, 8, (1, 2, 3)),      # sixteen threads a node
]


@pytest.mark.parametrize("args", CASES, ids=lambda a: f"{a[0][0]}x{a[0][1]}-o{a[1]}-b{a[2]}-{a[4]}")
def test_the_core_steps_to_the_oracle_s_bits(args):
    from oracle import elastic as E

    print(f"case {args}", flush=True)
    sim, osim, gamma, sources, sensors = _case(*args)
    fields, records = wave.simulate_shots(sim, sources, gamma, sensors)
    for k in sorted({0, len(sources) // 2, len(sources) - 1}):
        f, r = E.simulate(osim, sources[k].position, sources[k].signal, gamma, sensors)
        np.testing.assert_array_equal(host(records[k]), r, err_msg=f"shot {k}")
        np.testing.assert_array_equal(host(fields[k]), f, err_msg=f"shot {k}")


@pytest.mark.parametrize("precision, tol", [("float32", 1e-4), ("float64", 1e-10)])
def test_the_core_s_gradient_matches_the_oracle(precision, tol):
    from oracle import elastic as E

    print(f"case gradient {precision}", flush=True)
    sim, osim, gamma, sources, sensors = _case((121, 149), 4, 3, 30, precision, LINED, 8, (1, 2, 3))
    _, records = wave.simulate_shots(sim, sources, gamma, sensors)
    observed = [host(r) * 0.9 for r in records]
    cost, gradient = utils.misfit_gradient(sim, sources, gamma, Receivers(sensors), observed)
    ocost, ograd = E.misfit_gradient(osim, [(s.position, s.signal) for s in sources], gamma,
                                     sensors, observed)
    assert abs(cost - ocost) <= 1e-5 * ocost
    assert rel_max(gradient, ograd) < tol


# the shapes of a core block the cases above leave out: 32 lanes (512 threads) in both
# precisions, 16 of doubles, and 16 and 32 at the long stencils
SHAPES = [
    ((131, 150), 4, 20, 8, "float32", LINED, 8, (1, 2, 3)),
    ((150, 146), 8, 20, 8, "float32", LINED, 6, (1, 2, 3)),
    ((140, 137), 6, 16, 8, "float32", ((T, C), (C, T)), 0, ()),
    ((128, 140), 4, 12, 8, "float64", LINED, 8, (1, 2, 3)),
    ((131, 133), 4, 20, 8, "float64", LINED, 7, (1, 2, 3)),
    ((129, 131), 2, 20, 8, "float64", ((C, T), (T, T)), 0, ()),
]


def _id(a):
    return f"{a[0][0]}x{a[0][1]}-o{a[1]}-b{a[2]}-{a[4]}"


@pytest.mark.parametrize("args", CASES + SHAPES, ids=_id)
def test_a_case_runs_through_the_core(args):
    assert elastic_core_nodes(_case(*args)[0], args[2]) > 0


@pytest.mark.parametrize("args", SHAPES, ids=_id)
def test_every_shape_of_the_core_steps_to_the_oracle_s_bits(args):
    test_the_core_steps_to_the_oracle_s_bits(args)


@pytest.mark.parametrize("n, order, shots, precision", [
    ((121, 149), 2, 5, "float32"), ((133, 149), 8, 6, "float32"), ((125, 141), 4, 16, "float32"),
    ((125, 141), 4, 20, "float32"), ((121, 137), 6, 5, "float64"), ((121, 137), 4, 20, "float64")])
def test_the_core_s_gradient_matches_the_oracle_at_other_shapes(n, order, shots, precision):
    from oracle import elastic as E

    print(f"case gradient {n} order {order} {shots} shots {precision}", flush=True)
    sim, osim, gamma, sources, sensors = _case(n, order, shots, 24, precision, LINED, 6, (1, 2, 3))
    assert elastic_core_nodes(sim, shots) > 0
    _, records = wave.simulate_shots(sim, sources, gamma, sensors)
    observed = [host(r) * 0.9 for r in records]
    cost, gradient = utils.misfit_gradient(sim, sources, gamma, Receivers(sensors), observed)
    ocost, ograd = E.misfit_gradient(osim, [(s.position, s.signal) for s in sources], gamma,
                                     sensors, observed)
    assert abs(cost - ocost) <= 1e-5 * ocost
    assert rel_max(gradient, ograd) < (1e-4 if precision == "float32" else 1e-10)
