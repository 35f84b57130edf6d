"""Grids large enough that a 2D sweep runs its core kernels, against the oracle.

A 2D sweep launches two kernels a step: the core kernel streams the blocks
of the stream box, which hold no layer node and no node whose transposed
taps reach a layer; the general kernel takes every other node. The golden grids are too small to hold a core block, so these cases
build larger ones (sizes chosen so both kernels run, with points inside and
outside the core rectangle) and compare with the oracle on the same inputs:

- five shots (eight lanes: blocks 32 columns wide) on a 134 x 200 grid;
- one shot (one lane: blocks 256 columns wide) on a 100 x 560 grid.

Boxes this small hold fewer blocks than the library marches by default (it
leaves them to the general kernels), so the tests lower that threshold to 0.
"""

from __future__ import annotations

import importlib

import numpy as np
import pytest

from helpers import golden, host, oracle_sim, product_sim, rel_max

pytestmark = pytest.mark.gpu

S = importlib.import_module("cuwave_amd.sensitivity")
from cuwave_amd import utils, wave  # noqa: E402

F32_GRAD, F64 = 1e-4, 1e-10


@pytest.fixture(autouse=True)
def _march_every_box():
    # these grids are sized to hold core blocks; by default a box this small is
    # left to the general kernels, so have the stream kernels march it
    from cuwave_amd import _abi

    lib = _abi.load()
    previous = lib.cw_set_stream_threshold(0)
    yield
    lib.cw_set_stream_threshold(previous)


def _case(Nx, precision, N, seed):
    """An eighth-order acoustic CPML case (the physics of a golden case) on a larger grid."""
    base = golden("adj_pml_acoustic_o8_f32")
    z = {k: base[k] for k in ("kind", "dx", "dt", "space_order", "stencil", "boundary",
                              "materials", "pml", "pml_faces")}
    z.update(Nx=np.array(Nx), N=np.array(N), precision=np.array(precision))
    sim = product_sim(z)
    rng = np.random.default_rng(seed)
    shape = tuple(sim.Nx_padded)
    smooth = np.cumsum(np.cumsum(rng.standard_normal(shape), 0), 1)
    smooth = (smooth - smooth.min()) / (smooth.max() - smooth.min())
    z["indicator"] = (0.2 + 0.6 * smooth).astype(sim.np_dtype)
    return z, sim, rng


def _positions(rng, Nx, count, margin=3):
    return np.stack([rng.integers(margin, n - margin, count) for n in Nx]).astype(np.int32)


def test_a_batch_on_a_grid_with_core_blocks_steps_as_the_oracle():
    from oracle import driver

    z, sim, rng = _case((134, 200), "float32", 48, 11)
    osim = oracle_sim(z)
    print("case core forward f32 134x200 five shots", flush=True)
    sig = rng.standard_normal((sim.N, 1)).astype(sim.np_dtype)
    # shot 0 sits in a core block (rows 38..101, columns 32..159 of an eight-lane
    # sweep), shot 1 in the layer, the rest anywhere
    positions = [np.array([[60], [70]]), np.array([[5], [150]])]
    positions += [_positions(rng, sim.Nx, 1) for _ in range(3)]
    sensors = _positions(rng, sim.Nx, 12)
    sources = [wave.Source(p, sig * (1 + k)) for k, p in enumerate(positions)]
    fields, records = wave.simulate_shots(sim, sources, z["indicator"], sensors)
    for k, s in enumerate(sources):
        f, r = driver.simulate(osim, s.position, s.signal, z["indicator"], sensors)
        np.testing.assert_array_equal(host(fields[k]), f, err_msg=f"shot {k}")
        np.testing.assert_array_equal(host(records[k]), r, err_msg=f"shot {k}")


def test_one_shot_on_a_wide_grid_matches_the_oracle_adjoints():
    from oracle import driver

    z, sim, rng = _case((100, 560), "float64", 64, 12)
    osim = oracle_sim(z)
    print("case core adjoint f64 100x560 one shot", flush=True)
    sig = rng.standard_normal((sim.N, 1))
    # the source and three sensors in a core block (rows 38..69, columns
    # 256..511 of a one-lane sweep), close enough that the forward and adjoint
    # fields overlap within the run (else the gradient is round-off alone)
    src = wave.Source(np.array([[50], [300]]), sig)
    near = np.array([[46, 55, 60], [306, 294, 303]], dtype=np.int32)
    sensors = np.concatenate([near, _positions(rng, sim.Nx, 3)], axis=1)
    observed = 0.5 * rng.standard_normal((sim.N, sensors.shape[1]))
    ind = z["indicator"]
    cost, g, traces, _ = S.sensitivity(sim, src, ind, sensors, S.l2_misfit(observed))
    ocost, og, otraces, _ = driver.sensitivity(osim, src.position, src.signal, ind, sensors,
                                               driver.l2_misfit(observed))
    np.testing.assert_array_equal(host(traces), otraces)
    assert abs(cost - ocost) <= F64 * abs(ocost)
    assert rel_max(g["mass"], og["mass"]) < F64
    assert rel_max(g["stiff"], og["stiff"]) < F64
    _, g, _, _ = S.reconstruction_sensitivity(sim, src, ind, sensors, S.l2_misfit(observed))
    _, og, _, _ = driver.reconstruction_sensitivity(osim, src.position, src.signal, ind, sensors,
                                                    driver.l2_misfit(observed))
    assert rel_max(g["mass"], og["mass"]) < F64
    assert rel_max(g["stiff"], og["stiff"]) < F64


def test_a_batched_misfit_gradient_with_core_blocks_matches_the_oracle():
    from oracle import driver

    z, sim, rng = _case((134, 200), "float32", 48, 13)
    osim = oracle_sim(z)
    print("case core misfit f32 134x200 five shots", flush=True)
    sig = rng.standard_normal((sim.N, 1)).astype(sim.np_dtype)
    positions = [np.array([[60], [70]])] + [_positions(rng, sim.Nx, 1) for _ in range(4)]
    coords = np.stack([rng.uniform(3, n - 4, 9) * d for n, d in zip(sim.Nx, sim.dx)], axis=1)
    observed = [0.1 * rng.standard_normal((sim.N, len(coords))).astype(sim.np_dtype)
                for _ in positions]
    sources = [wave.Source(p, sig * (1 + k)) for k, p in enumerate(positions)]
    cost, gradient = utils.misfit_gradient(sim, sources, z["indicator"],
                                           utils.Sensors(sim, coords), observed)
    ocost, ogradient = driver.misfit_gradient(
        osim, [(s.position, s.signal) for s in sources], z["indicator"],
        driver.Sensors(osim, coords), observed)
    assert abs(cost - ocost) <= 1e-5 * abs(ocost)
    assert rel_max(gradient, ogradient) < F32_GRAD


@pytest.mark.parametrize("Nx, precision, shots", [((134, 200), "float32", 5),
                                                  ((100, 560), "float64", 1)])
def test_points_along_the_edges_of_core_blocks_match_the_oracle(Nx, precision, shots):
    from oracle import driver

    z, sim, rng = _case(Nx, precision, 32, 19)
    osim = oracle_sim(z)
    print(f"case core points {precision} {Nx} {shots} shots", flush=True)
    sig = rng.standard_normal((sim.N, 1)).astype(sim.np_dtype)
    # the rows beside the box's first (38) and second block row (70), the columns
    # beside a point tile (64, 128) and a one-lane block (256); several a node
    rows, cols = (36, 37, 38, 39, 69, 70), (31, 32, 63, 64, 127, 128)
    cols += (255, 256, 511, 512) if Nx[1] > 512 else ()
    sensors = np.array([(r, c) for r in rows for c in cols] + [(38, 64)] * 3,
                       dtype=np.int32).T
    sources = [wave.Source(np.array([[rows[k]], [cols[k]]]), sig * (1 + k))
               for k in range(shots)]
    fields, records = wave.simulate_shots(sim, sources, z["indicator"], sensors)
    for k, s in enumerate(sources):
        f, r = driver.simulate(osim, s.position, s.signal, z["indicator"], sensors)
        np.testing.assert_array_equal(host(fields[k]), f, err_msg=f"shot {k}")
        np.testing.assert_array_equal(host(records[k]), r, err_msg=f"shot {k}")
    # the adjoint, by the comparison and bounds of the batched gradient above
    coords = sensors.T * np.asarray(sim.dx)
    observed = [0.1 * rng.standard_normal((sim.N, len(coords))).astype(sim.np_dtype)
                for _ in sources]
    cost, gradient = utils.misfit_gradient(sim, sources, z["indicator"],
                                           utils.Sensors(sim, coords), observed)
    ocost, ogradient = driver.misfit_gradient(
        osim, [(s.position, s.signal) for s in sources], z["indicator"],
        driver.Sensors(osim, coords), observed)
    assert abs(cost - ocost) <= 1e-5 * abs(ocost)
    assert rel_max(gradient, ogradient) < (F32_GRAD if precision == "float32" else F64)


def test_the_illumination_map_with_core_blocks_matches_the_oracle():
    from oracle import driver

    z, sim, rng = _case((134, 200), "float32", 48, 14)
    osim = oracle_sim(z)
    print("case core illumination f32 134x200 five shots", flush=True)
    sig = rng.standard_normal((sim.N, 1)).astype(sim.np_dtype)
    positions = [np.array([[60], [70]])] + [_positions(rng, sim.Nx, 1) for _ in range(4)]
    sources = [wave.Source(p, sig * (1 + k)) for k, p in enumerate(positions)]
    illum = wave.illumination(sim, sources, z["indicator"])
    expect = driver.illumination(osim, [(s.position, s.signal) for s in sources],
                                 z["indicator"])
    assert rel_max(illum, expect) < 1e-5


def test_at_full_size_a_batch_of_32_steps_each_shot_as_alone():
    # the benchmark's grid (1090 x 1090, order 8, CPML), all 32 shots in one
    # launch: three of them bitwise as when run alone, fields and traces
    import sys

    from helpers import ROOT

    sys.path.insert(0, str(ROOT))
    import bench

    sim, true, _, sources, sensors = bench.workload(32, 120)
    print("case full size 1090x1090 32 shots 120 steps", flush=True)
    fields, records = wave.simulate_shots(sim, sources, true, sensors)
    for k in (0, 17, 31):
        f, r = wave.simulate(sim, sources[k], true, sensors)
        assert host(f).any()
        np.testing.assert_array_equal(host(fields[k]), host(f), err_msg=f"shot {k}")
        np.testing.assert_array_equal(host(records[k]), host(r), err_msg=f"shot {k}")


def test_at_full_size_the_batched_gradient_sums_the_shots_and_matches_the_oracle():
    # the benchmark's grid, 120 steps: the gradient of 8 shots in one batch is
    # the sum of the 8 run alone, and one shot's gradient is the oracle's
    import sys

    from oracle import driver

    from helpers import ROOT

    sys.path.insert(0, str(ROOT))
    import bench

    sim, true, start, sources, nodes = bench.workload(8, 120)
    print("case full size gradient 1090x1090 8 shots 120 steps", flush=True)
    coords = nodes.T * np.array(sim.dx)
    sensors = utils.Sensors(sim, coords)
    observed = utils.measure(sim, sources, true, sensors)
    cost, g = utils.misfit_gradient(sim, sources, start, sensors, observed)
    cost1, g1 = utils.misfit_gradient(sim, sources, start, sensors, observed, batch=1)
    assert abs(cost - cost1) <= 1e-5 * abs(cost1)
    assert rel_max(g, host(g1)) < F32_GRAD
    osim = driver.Sim("AcousticWave", sim.Nx, sim.dx, sim.N, sim.dt, "float32", 8,
                      materials=(1.0, 1.0, bench.C1**2, bench.C2**2),
                      pml=driver.Pml(sim.pml.width, sim.pml.wavespeed, sim.pml.reflection))
    s = sources[0]
    c0, g0 = utils.misfit_gradient(sim, [s], start, sensors, observed[:1])
    oc, og = driver.misfit_gradient(osim, [(s.position, s.signal)], start,
                                    driver.Sensors(osim, coords), [host(observed[0])])
    assert abs(c0 - oc) <= 1e-5 * abs(oc)
    assert rel_max(g0, og) < F32_GRAD


def test_on_a_caller_stream_the_frame_launches_join_it():
    # a 2D adjoint sweep runs its frame kernels on a stream of the library's
    # own: it must start after the caller stream's earlier work (the inputs it
    # fills) and end before that stream's next work (here a copy of the
    # outputs, enqueued with no synchronisation between). The forward half
    # runs on the caller's stream alone; it checks that a caller's stream
    # other than the null stream carries the fused steps unchanged.
    import sys

    import torch

    from helpers import ROOT

    sys.path.insert(0, str(ROOT))
    import bench

    sim, true, _, sources, sensors = bench.workload(32, 120)
    print("case caller stream 1090x1090 32 shots 120 steps", flush=True)
    fields, records = wave.simulate_shots(sim, sources, true, sensors)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        f2, r2 = wave.simulate_shots(sim, sources, true, sensors)
        f2c, r2c = f2.clone(), r2.clone()
    side.synchronize()
    for k in range(len(sources)):
        np.testing.assert_array_equal(host(f2c[k]), host(fields[k]), err_msg=f"shot {k}")
        np.testing.assert_array_equal(host(r2c[k]), host(records[k]), err_msg=f"shot {k}")
    # the adjoint sweep too: the gradient is the same bit for bit
    _, _, start, _, nodes = bench.workload(32, 120)
    sensors = utils.Sensors(sim, nodes.T * np.array(sim.dx))
    observed = utils.measure(sim, sources, true, sensors)
    cost, g = utils.misfit_gradient(sim, sources, start, sensors, observed)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        cost2, g2 = utils.misfit_gradient(sim, sources, start, sensors, observed)
        g2c = g2.clone()
    side.synchronize()
    assert cost2 == cost
    np.testing.assert_array_equal(host(g2c), host(g))


def test_side_by_side_adjoint_levels_equal_the_serialised_ones():
    # the core and frame launches of an adjoint level run on two streams; with
    # side streams off both run on the caller's stream, one after the other.
    # A race between them (a frame kernel reading a level the core has not
    # finished) would make the two gradients differ.
    import sys

    from helpers import ROOT

    from cuwave_amd import _abi

    sys.path.insert(0, str(ROOT))
    import bench

    sim, true, start, sources, nodes = bench.workload(32, 120)
    print("case side streams on/off 1090x1090 32 shots 120 steps", flush=True)
    sensors = utils.Sensors(sim, nodes.T * np.array(sim.dx))
    observed = utils.measure(sim, sources, true, sensors)
    lib = _abi.load()
    cost, g = utils.misfit_gradient(sim, sources, start, sensors, observed)
    previous = lib.cw_set_side_stream(0)
    try:
        cost_s, g_s = utils.misfit_gradient(sim, sources, start, sensors, observed)
    finally:
        lib.cw_set_side_stream(previous)
    assert previous == 1
    assert cost_s == cost
    np.testing.assert_array_equal(host(g_s), host(g))
