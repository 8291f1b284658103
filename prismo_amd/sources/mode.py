"""Mode source (src/prismo/sources/mode.py:19-360), rebuilt.

Same constructor as the reference (center, size, mode, direction, waveform,
amplitude, phase, name).  The reference never ran: it calls
``waveform.value`` (mode.py:219), which no waveform defines, then
multiplies the waveform (already carrying its carrier) by a second carrier
and adds the normal H component.  Here the waveform's own ``evaluate`` is
the time function, and the mode enters as a total-field / scattered-field
sheet.  The profile injected is the guided mode of the time-stepping grid
itself (prismo_amd.modes.yee) nearest the given mode (largest |E| overlap
on the plane, the given mode's x, y mapped as the reference maps them:
x-propagation (y, z), y: (x, z), z: (x, y)), solved on the source plane
with the simulation's own Cb (dispersive cells at eps_inf + Re chi(w0) of
the kernels' recursions).  With (a, b, c) cyclic, s the plane index along
the propagation axis a, and E, H that mode's transverse samples for
propagation along +a,

    E_b(s) += Cb/d_a H_c g(t_H)      H_b(s) -= sgn Db/d_a E_c g(t_E)
    E_c(s) -= Cb/d_a H_b g(t_H)      H_c(s) += sgn Db/d_a E_b g(t_E)

added after the E update of each step (E terms at t_H = t - dt/2 + sgn
d_a n_eff / (2 c), the time and place of the H samples; H terms at t_E = t,
for the next H update).  These make the update of every sample on the plane
see the incident mode on its other side, so the mode leaves the plane in
the chosen direction only.  ``phase`` shifts the carrier: the waveform is
read at t + phase / w0.
"""

from __future__ import annotations

from typing import Optional

import numpy as np
from scipy.interpolate import RegularGridInterpolator

from .. import _native as N
from .base import Source, SourceTerm

C0 = 299792458.0
EPS0 = 8.854187817e-12
_AX = {"x": 0, "y": 1, "z": 2}
_CYC = {0: (1, 2), 1: (2, 0), 2: (0, 1)}          # a -> (b, c), cyclic
_PLANE = {0: (1, 2), 1: (0, 2), 2: (0, 1)}        # a -> sim axes of mode (x, y)
_NAMES = "xyz"


class ModeSource(Source):
    def __init__(self, center, size, mode, direction: str, waveform, amplitude: float = 1.0,
                 phase: float = 0.0, name: Optional[str] = None):
        super().__init__(center, size, name)
        if direction not in ("+x", "-x", "+y", "-y", "+z", "-z"):
            raise ValueError(f"direction must be one of +x -x +y -y +z -z, got {direction!r}")
        self.mode = mode
        self.direction = direction
        self.waveform = waveform
        self.amplitude = amplitude
        self.phase = phase
        self.sign = +1 if direction[0] == "+" else -1
        self.axis = direction[-1].lower()
        self._sim = None
        self._sheets = None
        self.grid_neff = None

    def bind_simulation(self, sim) -> None:
        self._sim = sim

    def initialize(self, grid) -> None:
        super().initialize(grid)
        if grid.is_2d:
            raise NotImplementedError("mode sources are 3-D")
        self._sheets = None

    # --------------------------------------------------------------- grid mode
    def _plane_eps(self, eng, a):
        """Relative permittivity at the E samples of the source plane, on the
        (n_b - 1, n_c - 1) index window every component covers: from the
        simulation's own Cb (eps = dt / (eps0 Cb)); dispersive cells take
        eps_inf + Re chi(w0) of the recursions the kernels run."""
        b, c = _CYC[a]
        dims = self._grid.dimensions
        s = self._source_box["E" + _NAMES[b]][a][0]
        nb, nc = dims[b] - 1, dims[c] - 1
        w0 = 2 * np.pi * float(self.mode.frequency)
        dt = self._sim.dt
        out = {}
        for ax in (b, c, a):
            comp = "E" + _NAMES[ax]
            rng = [None, None, None]
            rng[a] = (s, s + 1)
            rng[b] = (0, nb)
            rng[c] = (0, nc)
            cb, _ = eng.coefficient_at(comp, tuple(rng))
            sel = [slice(None)] * 3
            sel[a] = 0
            cbp = cb[tuple(sel)]
            if b > c:
                cbp = cbp.T                        # -> (b, c) index order
            eps = dt / (EPS0 * cbp)
            zi = np.exp(1j * w0 * dt)
            for reg in getattr(self._sim, "_ade", []):
                if reg.comp != comp:
                    continue
                (i0, i1), (j0, j1), (k0, k1) = reg.box
                lo, hi = (i0, j0, k0), (i1, j1, k1)
                if not (lo[a] <= s < hi[a]):
                    continue
                c0, c1, c2, c3 = reg.c
                if reg.kind == 1:
                    chi = 0.5 * (c0 + c1 * zi) * (1 + zi) / (1 - c2 * zi - c3 * zi**2)
                else:
                    chi = 0.25 * dt * (1 + zi) ** 2 * c0 / ((1 - c1 * zi) * (1 - zi))
                ub, uc = slice(lo[b], min(hi[b], nb)), slice(lo[c], min(hi[c], nc))
                eps[ub, uc] = reg.eps_inf + np.real(chi)
            out[ax] = eps
        return out, s, nb, nc

    def _select(self, cands, a, nb, nc):
        """The grid mode closest to the given mode: largest overlap of |E_t|
        with the given profile on the plane (the reference's mapping of the
        mode's x, y to the plane), then nearest n_eff."""
        b, c = _CYC[a]
        u, v = _PLANE[a]
        g = self._grid
        nodes = lambda ax, n: g.origin[ax] + np.arange(n) * g.spacing[ax]
        m = self.mode
        mag = np.sqrt(np.abs(m.Ex) ** 2 + np.abs(m.Ey) ** 2)
        f = RegularGridInterpolator((m.x, m.y), mag, bounds_error=False, fill_value=0.0)
        cu, cv = nodes(u, {b: nb, c: nc}[u]), nodes(v, {b: nb, c: nc}[v])
        U, V = np.meshgrid(cu, cv, indexing="ij")
        ref = f(np.column_stack([U.ravel(), V.ravel()])).reshape(U.shape)
        if u != b:
            ref = ref.T                            # -> (b, c) index order
        best, key = None, None
        for n_eff, Eu, Ev, Hu, Hv in cands:
            t = np.sqrt(Eu**2 + Ev**2)
            ov = float(np.sum(t * ref) / np.sqrt(np.sum(t * t) * np.sum(ref * ref) + 1e-300))
            k = (round(ov, 3), -abs(n_eff - float(np.real(m.neff))))
            if key is None or k > key:
                best, key = (n_eff, Eu, Ev, Hu, Hv), k
        return best

    def _build(self):
        from ..modes.yee import yee_modes

        eng = self._sim.solver.updater.engine_for(self._sim.fields)
        if eng.coeff_kind in (N.COEFF_FULL, N.COEFF_CACB):
            raise NotImplementedError("mode sources in lossy or magnetic media")
        a = _AX[self.axis]
        b, c = _CYC[a]
        eps, s, nb, nc = self._plane_eps(eng, a)
        sp = self._grid.spacing
        cands = yee_modes(eps[b], eps[c], eps[a], sp[b], sp[c], sp[a],
                          2 * np.pi * float(self.mode.frequency), self._sim.dt, n_modes=4,
                          n_guess=float(np.real(self.mode.neff)))
        if not cands:
            raise RuntimeError("no guided mode of the grid near the given mode")
        n_eff, Eu, Ev, Hu, Hv = self._select(cands, a, nb, nc)
        self.grid_neff = n_eff
        self.grid_mode = (Eu, Ev, Hu, Hv)
        d = sp[a]
        db = float(eng.plan.db_const)
        A = self.amplitude
        # sheet: (component, profile on the (b, c) window, factor)
        want = {("E", b): (Hv, +1.0), ("E", c): (Hu, -1.0),
                ("H", b): (Ev, -self.sign), ("H", c): (Eu, +self.sign)}
        sheets = []
        for (kind, ax), (prof, sg) in want.items():
            comp = f"{kind}{_NAMES[ax]}"
            box = self._source_box[comp]
            lo = [r[0] for r in box]
            hi = [r[1] for r in box]
            lo[a], hi[a] = s, s + 1
            # the source window, clipped to the mode's (n_b, n_c) plane
            hi[b], hi[c] = min(hi[b], nb), min(hi[c], nc)
            if hi[b] <= lo[b] or hi[c] <= lo[c]:
                continue
            part = prof[lo[b]:hi[b], lo[c]:hi[c]]
            bx = tuple((lo[q], hi[q]) for q in range(3))
            if kind == "E":
                cb, _ = eng.coefficient_at(comp, bx)
                sel = [slice(None)] * 3
                sel[a] = 0
                cbp = cb[tuple(sel)]
                if b > c:
                    cbp = cbp.T
                val = A * sg * cbp / d * part
            else:
                val = A * sg * db / d * part
            full = np.zeros([bx[q][1] - bx[q][0] for q in range(3)])
            sel = [slice(None)] * 3
            sel[a] = 0
            full[tuple(sel)] = val.T if b > c else val
            sheets.append((kind, comp, bx, np.ascontiguousarray(full.transpose(2, 1, 0)).ravel()))
        self._sheets = sheets

    def _times(self, times):
        t = np.asarray(times, dtype=np.float64)
        if self.phase:
            t = t + self.phase / (2 * np.pi * float(self.mode.frequency))
        a = _AX[self.axis]
        shift = self.sign * self._grid.spacing[a] * self.grid_neff / (2 * C0)
        dt = self._sim.dt
        return t - dt / 2 + shift, t

    def device_terms(self, times):
        if not self.enabled or self._grid is None:
            return []
        if self._sim is None:
            raise RuntimeError("add the ModeSource to a Simulation first")
        if self._sheets is None:
            self._build()
        tH, tE = self._times(times)
        gH = self.waveform.table(tH)
        gE = self.waveform.table(tE)
        return [SourceTerm(comp, bx, gH if kind == "E" else gE, profile=p)
                for kind, comp, bx, p in self._sheets]

    def update_fields(self, fields, time: float, dt: float) -> None:
        if not self.enabled or self._grid is None:
            return
        if self._sheets is None:
            self._build()
        tH, tE = self._times([time])
        for kind, comp, bx, p in self._sheets:
            g = self.waveform.evaluate(float(tH[0] if kind == "E" else tE[0]))
            (i0, i1), (j0, j1), (k0, k1) = bx
            vals = p.reshape(k1 - k0, j1 - j0, i1 - i0).transpose(2, 1, 0) * g
            tgt = fields[comp][i0:i1, j0:j1, k0:k1]
            if isinstance(tgt, np.ndarray):
                tgt += vals
            else:
                import torch

                tgt += torch.from_numpy(np.ascontiguousarray(vals)).to(tgt)
