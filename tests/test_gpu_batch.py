"""Batched stepping of uneven models: each model of a batch gives exactly
what its own engine gives alone (port traces, fields, run-until outcome),
for the lockstep run loop and for runs of a subset."""
import numpy as np
import pytest

import ems_amd as E
from ems_amd import workloads as W
from ems_amd.dispersive import Dispersive, Field, Pole

from test_gpu_parity import bits, same_fields
from test_gpu_quad import build as quad_build

pytestmark = pytest.mark.gpu

SIZES = [(8.0, 20.0, 1.0, 8), (10.0, 24.0, 2.5, 10), (9.0, 22.0, 0.0, 9), (12.0, 30.0, 3.0, 8)]


def models():
    return [W.patch_model(*s) for s in SIZES]


def engine(m):
    e = E.Engine(m.grid, m.dt, m.lanes)
    p = m.build_ops(e)
    return e, p


def limits():
    # -80 dB checked every 20 steps: these four models stop at three
    # different checks (3781, 3801 and 4501 steps on the oracle), so the
    # staggered stops of the batch run loop are exercised.
    return E.RunLimits(6000, E.EndCriteria(1e-8, check_interval=20),
                       excitation_end=E.Waveform.gaussian(2e9, 1e9).duration())


@pytest.mark.parametrize("prefetch", [False, True], ids=["noprefetch", "prefetch"])
@pytest.mark.parametrize("tile_rows", [3, 7, "packed"])
def test_batch_run_until_matches_single_runs(tile_rows, prefetch):
    ms = models()
    single = [engine(m) for m in ms]
    outs = []
    for e, p in single:
        e.set_schedule(1, 7 if tile_rows == "packed" else tile_rows, 0)
        outs.append(e.run_until(limits()))
    batch = [engine(m) for m in ms]
    b = E.EngineBatch([e for e, _ in batch])
    if tile_rows == "packed":
        b.set_schedule(7, 0, prefetch=prefetch, packed=True)
    else:
        b.set_schedule(tile_rows, 0, prefetch=prefetch)
    bouts = b.run_until(limits())
    for (e, p), (f, q), o, bo in zip(single, batch, outs, bouts):
        assert (o.reason, o.steps, o.timestep) == (bo.reason, bo.steps, bo.timestep)
        assert np.float64(o.energy).tobytes() == np.float64(bo.energy).tobytes()
        assert np.array_equal(bits(p.voltage()), bits(q.voltage()))
        assert np.array_equal(bits(p.current()), bits(q.current()))
        same_fields(e, f)
    assert len({o.steps for o in bouts}) > 1 and all(o.reason == E.StopReason.EnergyDecay
                                                     for o in bouts)
    b.close()


@pytest.mark.parametrize("packed", [False, True])
def test_batch_without_graphs_matches(packed):
    ms = models()
    runs = []
    for graphs in (True, False):
        batch = [engine(m) for m in ms]
        b = E.EngineBatch([e for e, _ in batch])
        b.set_schedule(7, 2 if packed else 0, packed=packed)
        b.set_graphs(graphs)
        b.run(37)  # K = 16 graphs twice, then single steps
        b.run(5, [True, False, True, False])
        runs.append((batch, b))
    for (e, p), (f, q) in zip(runs[0][0], runs[1][0]):
        same_fields(e, f)
        assert np.array_equal(bits(p.voltage()), bits(q.voltage()))
    for batch, b in runs:
        b.close()
        for e, _ in batch:
            e.close()


@pytest.mark.parametrize("packed", [False, True])
def test_batch_subset_runs(packed):
    ms = models()
    single = [engine(m) for m in ms]
    for e, _ in single:
        e.run(77)
    batch = [engine(m) for m in ms]
    b = E.EngineBatch([e for e, _ in batch])
    b.set_schedule(7, 2 if packed else 0, packed=packed)
    b.run(40)
    b.run(37)
    for (e, p), (f, q) in zip(single, batch):
        same_fields(e, f)
        assert np.array_equal(bits(p.voltage()), bits(q.voltage()))
    # Only models 1 and 3 advance; the others stay put.
    act = [False, True, False, True]
    b.run(25, act)
    for q, ((e, p), (f, _)) in enumerate(zip(single, batch)):
        if act[q]:
            e.run(25)
        same_fields(e, f)
    b.close()


def test_batch_refuses_models_out_of_step_and_duplicates():
    """Models of a batch step in lockstep: two models whose step parities
    differ (one has taken an odd number of steps more, as after a run loop
    with an odd check interval that stopped them at different checks) are
    refused, and so is one engine listed twice."""
    ms = models()[:2]
    (a, _), (b, _) = engine(ms[0]), engine(ms[1])
    a.run(1)
    batch = E.EngineBatch([a, b])
    with pytest.raises(E.EmsError, match="lockstep"):
        batch.run(2)
    batch.close()
    b.run(1)  # back in step: the same batch object works
    batch = E.EngineBatch([a, b])
    batch.run(2)
    batch.close()
    with pytest.raises(E.EmsError):
        E.EngineBatch([a, a])
    a.close()
    b.close()


@pytest.mark.parametrize("packed", [False, True])
def test_batch_after_single_runs(packed):
    """Models that stepped on their own first, one of them on another
    schedule (the same steps taken, the state in another buffer), step on
    together like engines of their own."""
    ms = models()[:2]
    (a, _), (b, _), (c, _), (d, _) = (engine(ms[q]) for q in (0, 1, 0, 1))
    b.set_schedule(1, 3, 2)
    a.run(3)
    b.run(3)
    batch = E.EngineBatch([a, b])
    batch.set_schedule(7, 2, packed=packed)
    for n in (2, 21):
        batch.run(n)
    a.run(2)  # (on the schedule it had before)
    c.run(28)
    d.run(26)
    for x, y in ((a, c), (b, d)):
        for f in (0, 1):
            for k in range(3):
                assert np.array_equal(x._read(f, k).view(np.uint32), y._read(f, k).view(np.uint32))


@pytest.mark.parametrize("packed", [False, True])
def test_batch_takes_models_of_equal_steps_on_any_schedule(packed):
    """Models that took the same steps, one of them unfused by choice (as the
    autotuner may leave it), are in step; so are models an odd number of
    unfused steps apart; models that are in step by neither count are not."""
    ms = models()[:2]
    (a, _), (b, _), (c, _), (d, _) = (engine(ms[q]) for q in (0, 1, 0, 1))
    a.set_schedule(0)
    batch = E.EngineBatch([a, b])
    batch.set_schedule(7, 2, packed=packed)
    a.run(3)
    batch.run(2)
    batch.run(2, [True, False])
    b.run(3)
    batch.run(18)
    c.run(25)
    d.run(23)
    for x, y in ((a, c), (b, d)):
        same_fields(x, y)
    x, y = engine(ms[0])[0], engine(ms[1])[0]
    x.set_schedule(0)
    x.run(2)
    y.run(1)
    out = E.EngineBatch([x, y])
    with pytest.raises(E.EmsError, match="lockstep"):
        out.run(2)
    out.close()
    batch.close()
    for e in (a, b, c, d, x, y):
        e.close()


def test_batch_leaves_the_models_their_schedules():
    """After a batch's run, and after a run it refuses, every model steps on
    its own schedule: the engine's choice (the unfused kernels), a fused
    tiling or the unfused one that were set; the same bits as alone."""
    ms = models()[:3]

    def three():
        es = [engine(m)[0] for m in ms]
        es[1].set_schedule(2, 3, 2)
        es[2].set_schedule(0)
        return es

    def own(es):  # (a fused step has no E kernel of its own)
        return [e.traffic_model()[1] > 0.0 for e in es]
    es, alone = three(), three()
    assert own(es) == [True, False, True]
    for packed in (False, True):
        b = E.EngineBatch(es)
        b.set_schedule(7, 2, packed=packed)
        b.run(5)
        assert own(es) == [True, False, True]
        b.close()
        for e in es:
            e.run(3)
    h_source, _ = engine(ms[0])
    h_source.add_operator(E.EdgeSource(E.Waveform.gaussian(2e9, 1e9)).kind(E.SourceKind.SoftH)
                          .edge(E.Axis.X, [6, 6, 3], 1.0))
    b = E.EngineBatch(es + [h_source])
    with pytest.raises(E.EmsError, match="unfused"):
        b.run(2)
    assert own(es) == [True, False, True]
    b.close()
    for e, f in zip(es, alone):
        e.run(18)
        f.run(34)
        same_fields(e, f)
        e.close()
        f.close()
    h_source.close()


def poles(e):
    """Lorentz poles in a block of a patch model's substrate."""
    d = Dispersive.new()
    w = 2.0 * np.pi * 4e9
    d.fill_cells(e.grid, [(10, 18), (9, 20), (1, 6)], Field.Electric, [Pole.lorentz(w, w, 1e9)])
    return e.add_operator(d)


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("packed", [False, True])
def test_batch_with_poles(packed, graphs):
    """A dispersive medium in one model of a batch, and one that another gets
    between two runs (a step has other launches then)."""
    ms = models()[:3]
    single, batch = [engine(m) for m in ms], [engine(m) for m in ms]
    b = E.EngineBatch([e for e, _ in batch])
    b.set_schedule(7, 2, packed=packed)
    b.set_graphs(graphs)
    media = [(poles(es[1][0])) for es in (single, batch)]
    late = []
    for n in (37, 24, 1, 16):
        b.run(n)
        for e, _ in single:
            e.run(n)
        if not late:
            late = [poles(es[2][0]) for es in (single, batch)]
    for (e, p), (f, q) in zip(single, batch):
        assert np.array_equal(bits(p.voltage()), bits(q.voltage()))
        same_fields(e, f)
    for x, y in (media, late):
        for s, t in zip(x.state(Field.Electric), y.state(Field.Electric)):
            assert np.array_equal(bits(np.asarray(s)), bits(np.asarray(t)))
            assert np.abs(np.asarray(s)).max() > 0.0
    b.close()
    for e, _ in single + batch:
        e.close()


# Slabs that the quad kernels leave to others: z registered before y before
# x, and two ends of z that meet in one quad. A batch of short rows with one
# such model steps with the packed fused kernel.
IRREGULAR = [((10, 11, 7), [(E.Face.ZMax, 3), (E.Face.YMin, 3), (E.Face.XMin, 4)]),
             ((10, 10, 8), [(E.Face.ZMin, 3), (E.Face.ZMax, 4)])]
REGULAR = ((13, 12, 19), [(f, 3) for f in E.Face])


@pytest.mark.parametrize("prefetch", [False, True], ids=["noprefetch", "prefetch"])
@pytest.mark.parametrize("curl", (0, 1))
@pytest.mark.parametrize("irregular", IRREGULAR, ids=["z_first", "one_quad"])
def test_batch_of_irregular_slabs(irregular, curl, prefetch):
    """The packed fused kernel's batch (the irregular model), and the quad
    kernels' between its runs (the others alone): models of both kinds as
    alone, with and without chunks of x."""
    shapes = [REGULAR, irregular, REGULAR]
    single = [quad_build("gpu", c, l, curl, True, False) for c, l in shapes]
    batch = [quad_build("gpu", c, l, curl, True, False) for c, l in shapes]
    b = E.EngineBatch([e for e, _ in batch])
    for chunks, n, act in ((0, 37, None), (3, 5, None), (3, 4, [True, False, True]), (3, 18, None)):
        b.set_schedule(7, chunks, prefetch=prefetch, packed=True)
        b.run(n, act)
        for q, (e, _) in enumerate(single):
            if act is None or act[q]:
                e.run(n)
    for (e, p), (f, r) in zip(single, batch):
        same_fields(e, f)
        assert np.array_equal(bits(p.values()), bits(r.values()))
    b.close()
    for e, _ in single + batch:
        e.close()
