"""GPU: the batched step's passes of up to eight steps.

A cell's arithmetic depends neither on the tile it lies in nor on how a run is
cut into passes, so everything here is compared bit for bit.
"""

import numpy as np
import pytest

from tests.test_gpu_batch import _design

pytestmark = pytest.mark.gpu


def _run(sizes, dtype, storage, T, runs, graph):
    from prismo_amd.core.batch import BatchEngine

    built = [_design(nx, ny, 8, dtype, 100 + k) for k, (nx, ny) in enumerate(sizes)]
    eng = BatchEngine([b[0] for b in built], dtype=dtype, coefficient_storage=storage,
                      sample_T=T)
    eng._build(sum(runs))
    for n in runs:
        eng.ctx.run(n, graph=graph)
    eng.ctx.flush()
    eng._queued = sum(runs)
    eng.finish()
    m = built[0][0].monitors[0]
    return eng.fields(0), np.stack([m.frequency_stack(c) for c in m.components])


def _same(a, b):
    assert np.linalg.norm(a[1]) > 0
    assert np.array_equal(a[1], b[1])
    for c in ("Ez", "Hx", "Hy"):
        assert np.array_equal(a[0][c], b[0][c]), c


# sample blocks of 20 and 12 steps take three and two passes each
@pytest.mark.parametrize("dtype,storage", [(np.float64, "auto"), (np.float32, "auto"),
                                           (np.float32, "fp16")])
@pytest.mark.parametrize("T,runs,graph", [(20, [101], True), (12, [101], True),
                                          (20, [1, 3, 8, 60, 29], True),
                                          (20, [7, 1, 1, 92], False)])
def test_cuts_do_not_matter(mi355x, dtype, storage, T, runs, graph):
    sizes = [(32, 16), (33, 17), (81, 49)]   # 48 x 32, 49 x 33 and 97 x 65 cells
    # (the same blocks: a spectrum is summed block by block)
    _same(_run(sizes, dtype, storage, T, [101], False),
          _run(sizes, dtype, storage, T, runs, graph))


@pytest.mark.parametrize("storage", ["auto", "fp16"])
def test_tall_tiles(mi355x, storage):
    """With 1.2 M cells and more in the batch a tile has 48 rows."""
    _same(_run([(33, 81)], np.float32, storage, 32, [90], True),
          _run([(33, 81), (1100, 1100)], np.float32, storage, 32, [90], True))
