"""GPU: several 2-D TM steps per launch (the default for lossless and
conductive 2-D runs) against the unfused kernels and O1.

A tile is 48 columns by 16 rows, or by 48 (FP32 from 1.18 M cells on 256
compute units on); a launch takes up to 8 steps.  Widths and heights sit at the
edges of the tiles, run lengths leave every remainder of the 8 steps and cross
the ends of the 128-row sample blocks.  The unfused kernels do the same
operations per cell: 1e-13 relative L2 in FP64, 1e-6 in FP32; O1 at 1e-10 /
1e-5, the bars of the other 2-D paths.
"""

import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

D = 20e-9
FREQS = [187e12, 193e12, 200e12]


def _sim(nx, ny, t, dtype, storage="auto", sigma=False, extra=False, seed=4):
    import prismo_amd as pa

    rng = np.random.default_rng(seed)
    eps = rng.choice([1.0, 2.085, 12.1], size=(nx, ny, 1))
    ma = {"eps_rel": eps}
    if sigma:
        ma["sigma_e"] = rng.choice([0.0, 300.0, 5e4], size=(nx, ny, 1))
    s = 1 - 1e-9
    px, py = (nx - 2 * t) * D, (ny - 2 * t) * D
    sim = pa.Simulation(size=(px * s, py * s, 0.0), resolution=1 / D, pml_layers=t,
                        courant_factor=0.99, scheme="yee", dtype=dtype,
                        pml=pa.PMLParams(t) if t else None, material_arrays=ma,
                        coefficient_storage=storage)
    sim.add_source(pa.PlaneWaveSource(center=(0.3 * px, 0.5 * py, 0.0), size=(0.0, 0.8 * py, 0.0),
                                      direction="+x", polarization="z", frequency=193e12,
                                      pulse_width=2e-15))
    if extra:
        # overlaps the line above in Ez; a per-cell profile on Ez and Hy
        sim.add_source(pa.ElectricDipole(position=(0.3 * px, 0.5 * py, 0.0), polarization="z",
                                         frequency=200e12, pulse_width=1e-15, amplitude=0.3))
        sim.add_source(pa.GaussianBeamSource(center=(0.5 * px, 0.5 * py, 0.0),
                                             size=(0.0, 0.6 * py, 0.0), direction="x",
                                             polarization="z", frequency=190e12,
                                             beam_waist=0.2 * py, pulse_width=2e-15))
    mon = pa.FieldMonitor(center=(0.6 * px, 0.5 * py, 0.0), size=(0.4 * px, 0.7 * py, 0.0),
                          components=["Ez", "Hx", "Hy"], time_domain=False,
                          frequencies=list(FREQS))
    sim.add_monitor(mon)
    return sim, mon


def _out(sim, mon):
    f = np.concatenate([sim.fields.to_numpy(c).ravel() for c in ("Ez", "Hx", "Hy")])
    s = np.concatenate([mon.frequency_stack(c).ravel() for c in mon.components])
    return f, s


def _both(nx, ny, t, dtype, runs, bar, start=False, **kw):
    import torch

    outs = []
    for fuse in (True, False):
        sim, mon = _sim(nx, ny, t, dtype, **kw)
        if start:      # fields everywhere from the first step on
            rng = np.random.default_rng(8)
            for c, amp in (("Ez", 1.0), ("Hx", 1 / 377), ("Hy", 1 / 377)):
                f = amp * rng.normal(size=tuple(sim.fields[c].shape))
                sim.fields[c] = torch.from_numpy(f.astype(np.float32).astype(np.float64))
        eng = sim.solver.updater.engine_for(sim.fields)
        if not fuse:
            eng.ctx.set_tuning(0, 4, 8, 0, 2)
        assert eng.ctx.fused_steps() == int(fuse)
        for n in runs:
            sim.run_steps(n)
        outs.append(_out(sim, mon))
    assert np.linalg.norm(outs[1][0]) > 0 and np.linalg.norm(outs[1][1]) > 0
    for a, b in zip(*outs):
        assert rel_l2(a, b) <= bar


@pytest.mark.parametrize("shape,t", [((40, 30), 6), ((56, 8), 0), ((57, 25), 3), ((113, 33), 8),
                                     ((9, 70), 0), ((120, 65), 20)])
@pytest.mark.parametrize("runs", [[61], [64], [3, 2, 1, 1, 5, 140]])
def test_fp64_equals_unfused(mi355x, shape, t, runs):
    _both(*shape, t, np.float64, runs, 1e-13)


@pytest.mark.parametrize("shape,t", [((47, 33), 5), ((48, 32), 0), ((49, 16), 3), ((96, 17), 4),
                                     ((97, 49), 0), ((95, 48), 9), ((40, 15), 0), ((144, 47), 8)])
@pytest.mark.parametrize("runs", [[9, 135], [6, 7, 131], [2, 12, 4, 5]])
@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-13), (np.float32, 1e-6)])
def test_tile_edges_equal_unfused(mi355x, shape, t, runs, dtype, bar):
    """One cell short of a tile's edge, on it and past it, in both directions,
    from fields everywhere."""
    _both(*shape, t, dtype, runs, bar, start=True)


@pytest.mark.parametrize("dtype,storage,bar", [(np.float64, "auto", 1e-13),
                                               (np.float32, "auto", 1e-6),
                                               (np.float32, "fp16", 1e-6)])
def test_sources_of_every_kind(mi355x, dtype, storage, bar):
    _both(90, 50, 8, dtype, [37, 100], bar, storage=storage, extra=True)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-13), (np.float32, 1e-6)])
def test_conductive_media(mi355x, dtype, bar):
    _both(75, 61, 7, dtype, [41], bar, sigma=True)


@pytest.mark.parametrize("shape,dtype,bar", [((1000, 800), np.float64, 1e-13),
                                             ((1000, 800), np.float32, 1e-6),
                                             ((1500, 1201), np.float32, 1e-6)])
def test_taller_tiles(mi355x, shape, dtype, bar):
    """Many 16-row tiles, and a grid large enough for 48-row ones."""
    _both(*shape, 10, dtype, [22], bar, start=True)


@pytest.mark.parametrize("shape", [(1152, 1152), (1153, 1103), (1199, 1057)])
@pytest.mark.parametrize("kw", [{}, {"storage": "fp16"}, {"sigma": True}, {"extra": True}],
                         ids=["cb", "fp16", "conductive", "sources"])
def test_48_row_tiles(mi355x, shape, kw):
    """FP32 grids of 1.18 M cells and more (24 tiles of 48 rows exactly, 23 less one
    row, 22 and one row), with every kind of coefficients and sources, past the end
    of a sample block."""
    _both(*shape, 10, np.float32, [133, 6, 15], 1e-6, start=True, **kw)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-10), (np.float32, 1e-5)])
def test_against_oracle(mi355x, dtype, bar):
    from oracle import compat as O0
    from oracle.yee import YeeOracle

    t, steps = 9, 150
    sim, mon = _sim(130, 59, t, dtype)
    sim.run_steps(steps)
    eps = sim.solver.updater.eps_rel[:, :, 0]
    one, zero = np.ones_like(eps), np.zeros_like(eps)
    _, Cb, _, Db = O0.coefficients(eps, one, zero, zero, sim.dt)
    from prismo_amd.core.coefficients import component_average

    o1 = YeeOracle(130, 59, 1, sim.grid.spacing, sim.dt,
                   {"Ez": component_average(Cb, "Ez", True)}, float(Db.flat[0]),
                   pml=(t, t, t, t, 0, 0))
    tt = 0.0
    for _ in range(steps):
        o1.step()
        tt += sim.dt
        for s in sim.sources:
            s.update_fields(o1.F, tt, sim.dt)
    got, _ = _out(sim, mon)
    ref = np.concatenate([o1.F[c].ravel() for c in ("Ez", "Hx", "Hy")])
    assert rel_l2(got, ref) <= bar


@pytest.mark.parametrize("start,n", [(0, 40), (1, 40), (5, 59), (8, 1)])
@pytest.mark.parametrize("stride", [1, 2, 4, 8, 10, 50])
def test_timing_stride(mi355x, start, n, stride):
    """Every launch that holds a step that is a multiple of the stride is timed:
    once in class 5, as its steps in class 2; a step taken by itself in place
    counts in class 2 alone."""
    sim, _ = _sim(60, 40, 5, np.float32)
    eng = sim.solver.updater.engine_for(sim.fields)
    eng.ctx.set_timing(True, stride=stride)
    eng.run(start, n)
    cuts, at = [], start                 # an even number of launches of up to 8
    while at < start + n:
        cuts.append(min(8, start + n - at))
        at += cuts[-1]
    alone = 0
    if len(cuts) % 2:
        if cuts[0] == 1:
            alone = 1
        else:
            cuts[:1] = [cuts[0] - 1, 1]
    at, launches, steps = start, 0, 0
    for k, m in enumerate(cuts):
        if any((at + i) % stride == 0 for i in range(m)):
            launches += not (alone and k == 0)
            steps += m
        at += m
    ms5, n5 = eng.ctx.timing(5)
    ms2, n2 = eng.ctx.timing(2)
    assert (n5, n2) == (launches, steps)
    assert (ms5 > 0) == (launches > 0) and (ms2 > 0) == (steps > 0)


def test_shape_of_one_step_launches_only(mi355x):
    sim, _ = _sim(60, 40, 5, np.float32)
    eng = sim.solver.updater.engine_for(sim.fields)
    assert eng.ctx.fused_shape() is None and eng.ctx.fused_steps() == 1
    eng.ctx.set_tuning(1, 4, 5, 0, 2)
    assert eng.ctx.fused_shape()[2] == 5
    eng.ctx.set_tuning(2, 4, 8, 0, 2)
    assert eng.ctx.fused_shape() is None and eng.ctx.fused_steps() == 2


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("t", [0, 6])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_a_diverged_run_leaves_nothing_behind(mi355x, dtype, t, bad):
    """Fields that are not finite leave the cells past each component's extent
    at zero, so a run after zeroing the fields is that of a new simulation (an
    odd count: its first step is taken in place)."""
    ny = 41
    outs = []
    for spoiled in (True, False):
        sim, _ = _sim(70, ny, t, dtype)
        eng = sim.solver.updater.engine_for(sim.fields)
        if spoiled:
            sim.fields["Ez"] = bad
            eng.run(0, 16)
            for c in ("Ez", "Hx", "Hy"):
                f = sim.fields[c]                      # a view [i, j] of rows of sy
                pad = f.as_strided((f.stride(1), ny), (1, f.stride(1))).clone()
                pad[:f.shape[0], :f.shape[1]] = 0
                assert bool((pad == 0).all()), c
            sim.fields.zero_fields()
            eng.reset_state()
        sim.fields["Ez"][20, 20] = 1.0
        eng.run(0, 25)
        outs.append(np.concatenate([sim.fields.to_numpy(c).ravel() for c in ("Ez", "Hx", "Hy")]))
    assert np.isfinite(outs[1]).all() and np.linalg.norm(outs[1]) > 0
    assert np.array_equal(*outs)
