"""The C ABI: libpmfdtd loads (no GPU needed), exports every function the
header declares, and the ctypes mirror has the header's struct layout."""

import ctypes as C
import re
import subprocess
from pathlib import Path

import pytest

from prismo_amd import _native as N

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "pmfdtd.h"
HEADERS = sorted((ROOT / "include").glob("*.h"))


def declared_functions():
    names = set()
    for h in HEADERS:
        names |= set(re.findall(r"^\s*(?:const\s+)?\w+\*?\s+\**(pm_\w+)\s*\(", h.read_text(),
                                re.M))
    return sorted(names)


def test_header_declares_what_binding_binds():
    assert set(declared_functions()) == (set(N.SIGNATURES) | set(N.BATCH_SIGNATURES)
                                         | set(N.MLP_SIGNATURES) | set(N.GEOM_SIGNATURES))


def test_library_loads_and_exports_all_symbols():
    lib = N.load()
    for name in declared_functions():
        assert hasattr(lib, name), name
    assert lib.pm_abi_version() == N.ABI_VERSION


def test_errors_without_device_are_reported():
    lib = N.load()
    h = C.c_void_p()
    rc = lib.pm_create(10_000, None, C.byref(h))
    assert rc != 0 and not h.value


@pytest.mark.parametrize("off", [2, 4, 8, 12])
def test_net_train_refuses_an_unaligned_workspace(off):
    """Host check, before anything is launched."""
    lib = N.load()
    sizes = (C.c_int32 * 2)(4, 4)
    buf = (C.c_char * 8192)()
    base = (C.addressof(buf) + 15) // 16 * 16
    rc = lib.pm_mlp_net_train(None, 1, 1, sizes, base, base, base, base, 20, base, 512, base, base,
                              base, 1, None, 1, 1, base + off, base, 0.9, 0.999, 1e-8, 0.0, 0,
                              base)
    assert rc == -1


@pytest.mark.parametrize("precision,esz", [(N.FP32, 4), (N.FP64, 8)])
def test_batch_workspace_holds_layers_not_grids(precision, esz):
    """The second E-side CPML memory of a batch: what its layers take, beside the
    tables (under 2 % of one array of the grid)."""
    d = (N.pm_batch_design * 3)()
    layers = grid = 0
    for q, (nx, ny, t) in enumerate([(700, 500, 16), (701, 503, 0), (640, 900, 7)]):
        d[q].nx, d[q].ny, d[q].sy = nx, ny, (nx + 63) // 64 * 64
        for k in range(4):
            d[q].pml[k] = t
        layers += 2 * t * (ny + d[q].sy) * esz
        grid += ny * d[q].sy * esz
    p = N.pm_batch_plan()
    p.precision, p.coeff_kind, p.n_design, p.chunk = precision, N.COEFF_CB, 3, 8
    p.design = C.cast(d, C.POINTER(N.pm_batch_design))
    n = C.c_int64()
    assert N.load().pm_batch_workspace_bytes(C.byref(p), C.byref(n)) == 0
    assert layers <= n.value <= layers + 0.02 * grid


PROBE = r"""
#include <stddef.h>
#include <stdio.h>
#include "pmfdtd.h"
#include "pmbatch.h"
#include "pmgeom.h"
#define P(T, f) printf(#T "." #f " %zu\n", offsetof(T, f));
int main(void) {
  %FIELDS%
  return 0;
}
"""


STRUCTS = (N.pm_plan, N.pm_source, N.pm_sample_box, N.pm_dft_group, N.pm_ade_box,
           N.pm_batch_line, N.pm_batch_design, N.pm_batch_plan, N.pm_shape)


def test_struct_layout_matches_header(tmp_path):
    lines = []
    for cls in STRUCTS:
        lines.append(f'printf("{cls.__name__} %zu\\n", sizeof({cls.__name__}));')
        for fname, _ in cls._fields_:
            lines.append(f"P({cls.__name__}, {fname})")
    src = tmp_path / "probe.c"
    src.write_text(PROBE.replace("%FIELDS%", "\n  ".join(lines)))
    exe = tmp_path / "probe"
    subprocess.run(["gcc", "-std=c11", f"-I{HEADER.parent}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")
    got = dict(l.rsplit(" ", 1) for l in out if l.strip())
    for cls in STRUCTS:
        assert int(got[cls.__name__]) == C.sizeof(cls), cls.__name__
        for fname, _ in cls._fields_:
            assert int(got[f"{cls.__name__}.{fname}"]) == getattr(cls, fname).offset, (cls, fname)
