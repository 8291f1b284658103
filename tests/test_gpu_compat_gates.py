"""GPU: 2-D reference-arithmetic runs of many steps against the same steps one
at a time, bit for bit.

Within a run a step's gates come from flags that the kernels of the step before
left; a run of one step scans the fields.  Both must see the same: zero fields
until a source starts, TM and TE, a source that ends or brings in NaN, and
fields that are NaN or infinite from the start.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
D = 20e-9


def _sim(nx, ny, dipoles, sigma=False):
    import prismo_amd as pa

    rng = np.random.default_rng(5)
    ma = {"eps_rel": rng.choice([1.0, 2.085, 12.1], size=(nx, ny, 1))}
    if sigma:
        ma["sigma_e"] = rng.choice([0.0, 300.0, 5e4], size=(nx, ny, 1))
    s = 1 - 1e-9
    sim = pa.Simulation(size=(nx * D * s, ny * D * s, 0.0), resolution=1 / D, pml_layers=0,
                        courant_factor=0.9, dtype=np.float64, material_arrays=ma)
    for k, (x, y, pol, amp) in enumerate(dipoles):
        sim.add_source(pa.ElectricDipole(position=(x * nx * D, y * ny * D, 0.0),
                                         polarization=pol, frequency=(190 + 9 * k) * 1e12,
                                         pulse_width=1e-15, amplitude=amp))
    sim.add_monitor(pa.FieldMonitor(center=(0.5 * nx * D, 0.5 * ny * D, 0.0),
                                    size=(0.0, 0.4 * ny * D, 0.0), components=["Ez", "Hy"],
                                    time_domain=False, frequencies=[193e12]))
    return sim


CASES = {
    "tm": [(0.3, 0.5, "z", 1.0)],
    "te": [(0.3, 0.5, "x", 1.0)],
    "both": [(0.3, 0.5, "z", 1.0), (0.6, 0.4, "y", 0.5)],
    "overlap": [(0.3, 0.5, "z", 1.0), (0.3, 0.5, "z", -1.0)],
    "silent": [(0.3, 0.5, "z", 0.0)],
    "nan": [(0.3, 0.5, "z", float("nan"))],
    "none": [],
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("shape,sigma", [((64, 9), False), ((130, 67), True)])
@pytest.mark.parametrize("start", ["zero", "ez", "nan", "hz"])
def test_run_equals_single_steps(mi355x, name, shape, sigma, start):
    import torch

    got = []
    for runs in ([140], [1] * 140):
        sim = _sim(*shape, CASES[name], sigma)
        if start != "zero":
            c = "Hz" if start == "hz" else "Ez"
            f = torch.zeros_like(sim.fields[c])
            f[tuple(n // 3 for n in f.shape)] = float("nan") if start == "nan" else 1e-3
            sim.fields[c] = f
        for n in runs:
            sim.run_steps(n)
        got.append({c: sim.fields.to_numpy(c) for c in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")})
    for c in got[0]:
        assert np.array_equal(got[0][c], got[1][c], equal_nan=True), c


def test_a_call_that_fails_leaves_no_gates(mi355x):
    """A run that ends in an error after a step's E update (here: samples of steps
    outside the phasor tables are due first) has carried flags on without that
    step's sources; the next call scans the fields as they then are."""
    from prismo_amd import _native as N
    from prismo_amd.sources.base import SourceTerm

    nx, ny, i, j = 64, 30, 20, 11
    outs = []
    for failed in (True, False):
        sim = _sim(nx, ny, [])
        eng = sim.solver.updater.engine_for(sim.fields)
        if failed:
            box = ((i, i + 1), (j, j + 1), (0, 1))
            eng.configure_io([SourceTerm("Ez", box, np.ones(10))], sim.monitors,
                             times=np.arange(10) * sim.dt)
            eng.run(50, 2, N.RUN_SAMPLE)
            with pytest.raises(ValueError):
                eng.run(0, 5, N.RUN_SOURCES | N.RUN_SAMPLE | N.RUN_DFT)
        sim.fields["Ez"][i, j] = 1.0
        eng.run(0, 4)
        outs.append(np.concatenate([sim.fields.to_numpy(c).ravel() for c in ("Ez", "Hx", "Hy")]))
    assert np.count_nonzero(outs[1]) > 1
    assert np.array_equal(*outs)
