"""The unfused kernels that take four nodes of a z row per thread, against
the oracle, bit for bit: rows of every length modulo four and shorter than a
quad, single rows and planes, CPML layers on every face, on some, and so
thick that two ends of an axis meet in one quad or the layers are registered
in another order (corrected by launches of their own), in both curl orders
with lossy, magnetic and PEC blocks (pooled and dense coefficient lanes)."""
import math

import numpy as np
import pytest

import ems_amd as E
from oracle.bridge import OracleEngine

from test_gpu_parity import bits, same_fields

pytestmark = pytest.mark.gpu
F = E.Face
ALL = list(F)


def build(kind, cells, layers, curl, pool, graded):
    if graded:
        def lines(n, s):
            return np.array([s * (q + 0.25 * math.sin(1.3 * q)) for q in range(n + 1)])
        g = E.Grid([lines(cells[0], 1e-3), lines(cells[1], 1.1e-3), lines(cells[2], 0.9e-3)])
    else:
        g = E.Grid.uniform(cells, [1e-3] * 3)
    m = E.CellMaterials.vacuum(g)
    m.fill_box([(0, max(1, q // 2)) for q in cells],
               E.Material(eps_r=(3.1, 2.9, 3.3), mu_r=(1.4, 1.3, 1.5), kappa=(0.05, 0.04, 0.06),
                          sigma_m=(200.0, 0.0, 100.0)))
    if min(cells) > 4:
        m.fill_pec_box([(q // 2, q // 2 + 2) for q in cells])
    dt = E.TimeStep.courant(0.95).resolve(g)
    # (PMC walls where there is no layer: every edge of the smallest grids moves)
    wall = E.FaceCondition.Pec if layers else E.FaceCondition.Pmc
    lanes = E.coefficients(g, m, [wall] * 6, dt)
    if kind == "gpu":
        e = E.Engine(g, dt, lanes, curl_order=curl, pool=pool)
    else:
        e = OracleEngine(g, dt, lanes, curl_order=curl, threads=2, pool=pool)
    if layers:
        e.add_operator(E.CpmlBoundary.new(e, [(f, E.Cpml(cells=c, kappa_max=3.0, alpha_max=0.05))
                                              for f, c in layers]))
    rng = np.random.default_rng(5)
    n = g.nodes()
    for a in range(3):
        u = rng.standard_normal(n).astype(np.float32)
        u[lanes[3 + a] == 0.0] = 0.0  # (no voltage on PEC and padding edges)
        e.set_component(0, a, u)
    p = e.add_operator(E.Probe.voltage(E.Axis.Z, [q // 2 for q in (n[0], n[1], n[2] - 1)]))
    return e, p


CASES = [((6, 5, nz), [], False) for nz in range(1, 10)]
CASES += [((1, 7, 6), [], False), ((7, 1, 5), [], True), ((1, 1, 1), [], False)]
CASES += [((17, 13, nz), [(f, 3) for f in ALL], True) for nz in (9, 10, 11, 12, 64, 67)]
CASES += [((11, 14, 33), [(F.XMax, 4), (F.YMin, 2), (F.ZMax, 5)], False),
          ((12, 9, 20), [(F.ZMin, 3)], True), ((12, 9, 20), [(F.YMax, 3), (F.ZMin, 7)], False),
          ((10, 10, 8), [(F.ZMin, 3), (F.ZMax, 4)], False),      # both ends in one quad
          ((10, 11, 7), [(F.ZMax, 3), (F.YMin, 3), (F.XMin, 4)], False),  # z before y before x
          ((9, 10, 21), [(F.XMax, 4), (F.XMin, 4), (F.YMax, 5), (F.YMin, 5)], True),
          ((40, 300, 260), [(f, 8) for f in ALL], True)]         # several blocks per plane


@pytest.mark.parametrize("curl", (0, 1))
@pytest.mark.parametrize("cells,layers,graded", CASES)
def test_quad_kernels(cells, layers, graded, curl):
    pool = sum(cells) % 2 == 0 or bool(layers)
    big = cells[0] * cells[1] * cells[2] > 100000
    g, pg = build("gpu", cells, layers, curl, pool, graded)
    o, po = build("oracle", cells, layers, curl, pool, graded)
    for n in (1, 2) if big else (1, 6, 33):
        g.run(n)
        o.run(n)
        wg, wo = g.step_with_energy(), o.step_with_energy()
        assert np.float64(wg).tobytes() == np.float64(wo).tobytes(), (wg, wo)
    same_fields(g, o)
    assert np.array_equal(bits(pg.values()), bits(o.probe_values(po)))
    assert max(np.abs(g.u_component(a)).max() for a in range(3)) > 0.0


@pytest.mark.parametrize("which", (0, 1, 2, 3, 7, 11, 15))
def test_switches_agree(which):
    """Every choice of kernels, switched between runs, and the fused step
    after the unfused one (its H psi is read from the buffer the quads
    updated)."""
    cells, layers = (13, 12, 19), [(f, 3) for f in ALL]
    g, pg = build("gpu", cells, layers, 0, True, True)
    o, po = build("oracle", cells, layers, 0, True, True)
    g.run(3)
    g.set_unfused_prefetch(which)
    g.run(4)
    g.set_schedule(2, 3, 4)
    g.run(3)
    g.set_schedule(0)
    g.run(5)
    o.run(15)
    same_fields(g, o)
    assert np.array_equal(bits(pg.values()), bits(o.probe_values(po)))


def test_traffic_model_of_a_step():
    """The bytes of an unfused step do not depend on what ran before it."""
    cells, layers = (13, 12, 19), [(f, 3) for f in ALL]
    a, _ = build("gpu", cells, layers, 0, True, False)
    b, _ = build("gpu", cells, layers, 0, True, False)
    b.set_cpml_split(True)
    b.set_schedule(1, 7, 0)
    b.run(1)
    b.set_schedule(0)
    assert a.traffic_model() == b.traffic_model()
    a.close()
    b.close()
