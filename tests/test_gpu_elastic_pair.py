"""The two kernels of a 3D elastic step at the edges of their branches, against the oracle.

An axis with no wall near a node takes its derivatives and divergences in one
branch, and a layer reads all its memories before it writes any: the boxes
here are the smallest that have nodes on both sides of either (some axes have
none), at every stencil and count of lanes a thread. Forward fields and traces
are expected to the bit; the gradient within the tolerance of the elastic
tests (1e-4 relative in float32, 1e-10 in float64).
"""

from __future__ import annotations

import numpy as np
import pytest

from helpers import Receivers, host, rel_max

pytestmark = pytest.mark.gpu

from cuwave_amd import boundary, elastic, utils, wave  # noqa: E402

T, C = boundary.Traction, boundary.Clamped
OPEN, LINED, MIXED = ((T, T),) * 3, ((T, C), (C, C), (C, T)), ((C, T), (T, C), (C, C))


def _case(n, order, shots, N, precision, walls, layer, faces):
    from oracle import driver as D
    from oracle import elastic as E

    pml = boundary.Pml(layer, 2.0, 1e-6, 2.0, faces) if layer else None
    sim = elastic.ElasticWave(n, (1.0, 1.1, 0.9), N, 0.1, precision=precision, space_order=order,
                              density=1.3, wavespeed_p=2.0, wavespeed_s=1.0, boundary=walls,
                              pml=pml)
    rng = np.random.default_rng(sum(n) + order)
    gamma = (0.8 + 0.4 * rng.random(sim.Nx_padded)).astype(sim.np_dtype)
    sig = rng.standard_normal((N, 1)).astype(sim.np_dtype)

    def points(count):
        return np.stack([np.arange(count) % 3] + [rng.integers(2, m - 3, count) for m in n])

    sources = [wave.Source(points(3)[:, k % 3:k % 3 + 1], sig * (1 + k)) for k in range(shots)]
    osim = E.ElSim(sim.Nx, sim.dx, sim.N, sim.dt, sim.precision, sim.space_order, sim.stencil,
                   tuple(tuple(int(c == C) for c in pair) for pair in walls), sim.density,
                   sim.wavespeed_p, sim.wavespeed_s, "strain",
                   D.Pml(layer, 2.0, 1e-6, 2.0, faces) if layer else None)
    return sim, osim, gamma, sources, points(12)


CASES = [
    ((9, 12, 23), 2, 1, 30, "float32", OPEN, 0, ()),                   # one lane a thread
    ((15, 19, 18), 4, 2, 30, "float32", LINED, 4, (1, 2, 3, 4)),       # two, layers that meet walls
    ((13, 19, 17), 4, 4, 30, "float32", MIXED, 3, (0, 3, 4, 5)),       # four
    ((25, 27, 26), 8, 5, 30, "float32", LINED, 5, (1, 3, 4)),          # two threads a node
    ((23, 20, 21), 6, 3, 30, "float64", MIXED, 4, (0, 3, 5)),
]


@pytest.mark.parametrize("args", CASES, ids=lambda a: f"o{a[1]}-b{a[2]}-{a[4]}")
def test_a_3d_elastic_step_matches_the_oracle(args):
    from oracle import elastic as E

    print(f"case {args}", flush=True)
    sim, osim, gamma, sources, sensors = _case(*args)
    fields, records = wave.simulate_shots(sim, sources, gamma, sensors)
    for k, s in enumerate(sources):
        f, r = E.simulate(osim, s.position, s.signal, gamma, sensors)
        np.testing.assert_array_equal(host(records[k]), r, err_msg=f"shot {k}")
        np.testing.assert_array_equal(host(fields[k]), f, err_msg=f"shot {k}")
    observed = [host(r) * 0.9 for r in records]
    cost, gradient = utils.misfit_gradient(sim, sources, gamma, Receivers(sensors), observed)
    ocost, ograd = E.misfit_gradient(osim, [(s.position, s.signal) for s in sources], gamma,
                                     sensors, observed)
    assert abs(cost - ocost) <= 1e-5 * ocost
    assert rel_max(gradient, ograd) < (1e-4 if args[4] == "float32" else 1e-10)
