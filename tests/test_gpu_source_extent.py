"""GPU: source boxes that reach past their component's extent (the C ABI takes
them; Simulation cuts its own).  The value is added to cells that no update
writes, where it accumulates: the curls next to E cells there read it, monitors
read any.  Whatever launch shape a plan could take and however a run is cut,
fields and samples are those of the unfused kernels.  A box inside the extent,
and an H box that no monitor sees, keep the fused ones.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = 20e-9
T = 32


class _Mon:
    """A monitor over one component box, samples only."""

    def __init__(self, comp, box):
        self.spec = {"boxes": [(comp, box, tuple(b - a for a, b in box))]}

    def device_spec(self):
        return self.spec


def _run(shape, dtype, comp, box, runs, tune=None, mon=True):
    import prismo_amd as pa
    from prismo_amd import _native as N
    from prismo_amd.sources.base import SourceTerm

    t, s, n = 3, 1 - 1e-9, sum(runs)
    sim = pa.Simulation(size=tuple((k - 2 * t) * D * s if k > 1 else 0.0 for k in shape),
                        resolution=1 / D, pml_layers=t, courant_factor=0.9, scheme="yee",
                        dtype=dtype, pml=pa.PMLParams(t),
                        material_arrays={"eps_rel": np.full(shape, 2.085)})
    eng = sim.solver.updater.engine_for(sim.fields)
    if tune:
        eng.ctx.set_tuning(*tune)
    table = np.sin(0.3 * np.arange(1, n + 1))
    eng.configure_io([SourceTerm(comp, box, table)], [_Mon(comp, box)] if mon else [],
                     times=np.arange(n) * sim.dt, sample_T=T)
    at = 0
    for m in runs:
        eng.run(at, m, N.RUN_SOURCES | (N.RUN_SAMPLE if mon else 0))
        at += m
    out = [sim.fields.to_numpy(c).ravel() for c in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")]
    if mon:
        out.append(eng.sample_rows(0, n).ravel())
    return eng, np.concatenate(out)


NX, NY, NZ = 70, 40, 12
# component, box past its extent, the same cut at it
BOXES = {
    "Ez x": ("Ez", ((NX - 3, NX), (9, 20), (0, 1)), ((NX - 3, NX - 1), (9, 20), (0, 1))),
    "Ez y": ("Ez", ((30, 50), (NY - 1, NY), (0, 1)), ((30, 50), (NY - 2, NY - 1), (0, 1))),
    "Hx x": ("Hx", ((NX - 2, NX), (9, 20), (0, 1)), ((NX - 2, NX - 1), (9, 20), (0, 1))),
    "Hy y": ("Hy", ((30, 50), (NY - 2, NY), (0, 1)), ((30, 50), (NY - 2, NY - 1), (0, 1))),
}
CUTS = ([25], [3, 9, 8, 5])


def _same_everywhere(shape, dtype, comp, past, inside, tunings):
    for mon in (False, True):
        unseen = comp[0] == "H" and not mon
        _, ref = _run(shape, dtype, comp, past, CUTS[0], (0, 4, 8, 0, 2), mon)
        assert np.linalg.norm(ref) > 0
        for tune in (None,) + tunings:
            for runs in CUTS:
                eng, got = _run(shape, dtype, comp, past, runs, tune, mon)
                off = np.linalg.norm(got - ref) / np.linalg.norm(ref)
                # (the fused kernels sum in another order: 1e-6 and 1e-13 as elsewhere)
                bar = 0 if not unseen else 1e-6 if dtype is np.float32 else 1e-13
                assert off <= bar, (mon, tune, runs, off)
                assert (eng.ctx.fused_steps() > 0) == unseen
    assert _run(shape, dtype, comp, inside, [8])[0].ctx.fused_steps() == 1


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("name", list(BOXES))
def test_2d(mi355x, name, dtype):
    _same_everywhere((NX, NY, 1), dtype, *BOXES[name], ((2, 4, 8, 0, 2), (1, 4, 3, 0, 2)))


@pytest.mark.parametrize("nx", [130, 100])    # 64-cell segments, whole rows of 128
@pytest.mark.parametrize("comp,axis", [("Ez", 0), ("Ey", 0), ("Ex", 1), ("Ex", 2), ("Hz", 2)])
def test_3d(mi355x, nx, comp, axis):
    n = (nx, NY, NZ)
    past = [(5, 9), (5, 9), (5, 9)]
    past[axis] = (n[axis] - 2, n[axis])
    inside = list(past)
    inside[axis] = (n[axis] - 2, n[axis] - 1)
    _same_everywhere(n, np.float32, comp, tuple(past), tuple(inside), ((1, 3, 4, 0, 3),))
