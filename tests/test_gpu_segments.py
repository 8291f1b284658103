"""GPU: the fused 3-D step in 64-cell row segments (rows of any width, and
conductive media with Ca and Cb arrays) against O1 and the unfused kernels.

Widths put a segment boundary inside the high x CPML layer, in the last cell
of the row and nowhere (one segment); heights and depths leave
ragged tiles and chunks.  Tolerances: FP64 1e-10 relative L2 against O1 (the
bar of the whole-row kernel), FP32 1e-5; against the unfused kernels, which
do the same arithmetic, 1e-13 and 1e-6.
"""

import numpy as np
import pytest

from tests.conftest import rel_l2
from tests.test_gpu_fused import D, _all, _drive, _fields, _oracle, _sim

pytestmark = pytest.mark.gpu


def _seg(sim):
    """The engine, checked to step in 64-cell segments."""
    eng = sim.solver.updater.engine_for(sim.fields)
    shape = eng.ctx.fused_shape()
    assert shape[0] == 1 and shape[1] == 1 and shape[3] == eng.sy // 64, shape
    return eng


@pytest.mark.parametrize("shape,t", [((40, 20, 18), 4), ((64, 17, 9), 3), ((131, 13, 12), 5),
                                     ((192, 12, 11), 5), ((257, 23, 15), 4), ((320, 9, 8), 3),
                                     ((514, 12, 13), 5), ((190, 13, 12), 0)])
@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-10), (np.float32, 1e-5)])
def test_segments_match_oracle(mi355x, shape, t, dtype, bar):
    sim, eps = _sim(*shape, t=t, dtype=dtype, nsrc=2) if t else _sim_no_pml(shape, dtype)
    _seg(sim)
    steps = 41
    sim.run_steps(steps)
    o1 = _oracle(sim, eps, t)
    _drive(o1, sim, steps)
    assert rel_l2(_all(_fields(sim)), _all(o1.F)) <= bar


def _sim_no_pml(shape, dtype):
    import prismo_amd as pa

    rng = np.random.default_rng(5)
    eps = rng.choice([1.0, 2.085, 12.1], size=shape)
    s = 1 - 1e-9
    sim = pa.Simulation(size=tuple(n * D * s for n in shape), resolution=1 / D, pml_layers=0,
                        courant_factor=0.99, scheme="yee", material_arrays={"eps_rel": eps},
                        dtype=dtype)
    sim.add_source(pa.ElectricDipole(position=(10 * D, 7 * D, 6 * D), polarization="z",
                                     frequency=193e12, pulse_width=4e-15))
    return sim, eps


@pytest.mark.parametrize("ty,kchunk,order", [(3, 1, 0), (7, 2, 1), (3, 5, 2), (7, 30, 3)])
@pytest.mark.parametrize("dtype,storage,bar", [(np.float64, "auto", 1e-13),
                                               (np.float32, "fp16", 1e-6)])
def test_segments_equal_unfused(mi355x, dtype, storage, bar, ty, kchunk, order):
    """Every tile height, chunk and order, with boxes across the segment
    boundaries at 64 and 128, against the H and E launches."""
    import prismo_amd as pa

    out = []
    for fuse in (1, 0):
        sim, _ = _sim(150, 18, 14, t=4, dtype=dtype, storage=storage, nsrc=2)
        si = pa.LorentzMaterial(7.98, [pa.LorentzPole(omega_0=1.1e16, delta_epsilon=3.69,
                                                      gamma=1e13)])
        sim.add_dispersive_box(si, (50 * D, 2 * D, 2 * D), (130 * D, 9 * D, 5 * D))
        sim.add_dispersive_box(pa.DrudeMaterial(1.0, 1.37e16, 1.07e14), (40 * D, 0.0, 6 * D),
                               (70 * D, 10 * D, 8 * D))
        eng = sim.solver.updater.engine_for(sim.fields)
        eng.ctx.set_tuning(fuse, ty, kchunk, 0, order)
        assert eng.ctx.fused_steps() == fuse
        if fuse:
            _seg(sim)
        sim.run_steps(31)
        out.append(_all(_fields(sim)))
    assert rel_l2(out[0], out[1]) <= bar


@pytest.mark.parametrize("shape", [(100, 16, 13), (70, 15, 12), (250, 14, 13)])
@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-10), (np.float32, 1e-5)])
def test_conductive_media(mi355x, shape, dtype, bar):
    """sigma_e > 0 in blocks, mu = 1: Ca and Cb arrays only, in segments
    (whatever the row width), against O1 with the averaged Ca and Cb; an odd
    run, so its first step takes the unfused kernels."""
    import prismo_amd as pa
    from oracle import compat as O0
    from oracle.yee import YeeOracle

    t = 4
    rng = np.random.default_rng(9)
    eps = rng.choice([1.0, 2.085, 12.1], size=shape)
    sig = rng.choice([0.0, 300.0, 5e4], size=shape)
    s = 1 - 1e-9
    sim = pa.Simulation(size=tuple((n - 2 * t) * D * s for n in shape), resolution=1 / D,
                        pml_layers=t, courant_factor=0.99, scheme="yee", pml=pa.PMLParams(t),
                        material_arrays={"eps_rel": eps, "sigma_e": sig}, dtype=dtype)
    sim.add_source(pa.ElectricDipole(position=(10 * D, 5 * D, 3 * D), polarization="z",
                                     frequency=193e12, pulse_width=2e-15))
    eng = _seg(sim)
    assert eng.coeff_kind == 3
    steps = 45
    sim.run_steps(steps)
    Ca, Cb, _, Db = O0.coefficients(eps, np.ones(shape), sig, np.zeros(shape), sim.dt)
    at = {"Ex": O0._ex, "Ey": O0._ey, "Ez": O0._ez}
    o1 = YeeOracle(*shape, sim.grid.spacing, sim.dt, {c: f(Cb) for c, f in at.items()},
                   float(Db.flat[0]), ca={c: f(Ca) for c, f in at.items()}, pml=(t,) * 6)
    _drive(o1, sim, steps)
    assert rel_l2(_all(_fields(sim)), _all(o1.F)) <= bar
    with pytest.raises(NotImplementedError):
        eng.coefficient_at("Ez", ((0, 1), (0, 1), (0, 1)))


@pytest.mark.parametrize("shape", [(64, 8, 2), (65, 2, 40), (2, 30, 30), (300, 3, 3)])
def test_thin_grids(mi355x, shape):
    """One to three cells along an axis: chunks and tiles larger than the
    grid, no CPML, against the unfused kernels."""
    out = []
    for fuse in (1, 0):
        sim, _ = _sim_no_pml(shape, np.float64)
        eng = sim.solver.updater.engine_for(sim.fields)
        if not fuse:
            eng.ctx.set_tuning(0, 4, 8, 0, 2)
        assert eng.ctx.fused_steps() == fuse
        sim.run_steps(12)
        out.append(_all(_fields(sim)))
    assert rel_l2(out[0], out[1]) <= 1e-13
