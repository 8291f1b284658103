"""GPU: the batched step's passes of up to eight steps.

A cell's arithmetic depends neither on the tile it lies in (48 columns by 16
rows, or by 48 in FP32 from 1.18 M cells in the batch on) nor on how a run is
cut into passes, so everything here is compared bit for bit, and at the tiles'
edges with the O1 oracle (1e-10 relative L2 in FP64, 1e-5 in FP32).
"""

import numpy as np
import pytest

from tests.conftest import rel_l2
from tests.test_gpu_batch import _design

pytestmark = pytest.mark.gpu


def _run(sizes, dtype, storage, T, runs, graph, xcd=1):
    from prismo_amd.core.batch import BatchEngine

    built = [_design(nx, ny, 8, dtype, 100 + k) for k, (nx, ny) in enumerate(sizes)]
    eng = BatchEngine([b[0] for b in built], dtype=dtype, coefficient_storage=storage,
                      sample_T=T)
    eng.ctx.set_tuning(4, xcd)
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


@pytest.mark.parametrize("dtype,storage", [(np.float64, "auto"), (np.float32, "auto"),
                                           (np.float32, "fp16")])
@pytest.mark.parametrize("runs,graph", [([1] * 101, False), ([1] * 7 + [9, 1, 20, 64], True),
                                        ([8, 1, 1, 8, 1, 82], True)])
def test_launches_of_one_step(mi355x, dtype, storage, runs, graph):
    """A step by itself takes tiles of 62 columns by 30 rows and updates the E-side
    memory in place; before and after passes of more, graphs from every pair of
    sets."""
    sizes = [(46, 44), (47, 45), (109, 17)]  # 62 x 60, 63 x 61 and 125 x 33 cells
    _same(_run(sizes, dtype, storage, 20, [101], False),
          _run(sizes, dtype, storage, 20, runs, graph))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("T", [1, 3, 9])
def test_sample_blocks_that_leave_one_step(mi355x, dtype, T):
    """Blocks of 1, 3 and 9 rows: passes of 1, 3, and 8 and 1 steps."""
    a = _run([(46, 44), (33, 17)], dtype, "auto", T, [37], False)
    b = _run([(46, 44), (33, 17)], dtype, "auto", 64, [37], False)
    for c in ("Ez", "Hx", "Hy"):
        assert np.linalg.norm(b[0][c]) > 0 and np.array_equal(a[0][c], b[0][c]), c
    # (a spectrum is summed block by block: the same samples in another order)
    assert rel_l2(a[1], b[1]) <= (1e-12 if dtype is np.float64 else 1e-5)


@pytest.mark.parametrize("tall", [False, True])
@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-10), (np.float32, 1e-5)])
def test_tile_edges_match_oracle(mi355x, dtype, bar, tall):
    """Designs one cell short of a tile's edge, on it and past it, alone and (tall)
    beside one that takes an FP32 batch to 48-row tiles."""
    from prismo_amd.core.batch import BatchEngine
    from tests.test_gpu_batch import _drive, _oracle

    t, steps = 8, 61
    cells = [(47, 33), (48, 32), (49, 47), (96, 48), (97, 49), (144, 65)]
    sizes = [(nx - 2 * t, ny - 2 * t) for nx, ny in cells] + ([(1100, 1100)] if tall else [])
    built = [_design(nx, ny, t, dtype, 100 + k) for k, (nx, ny) in enumerate(sizes)]
    eng = BatchEngine([b[0] for b in built], dtype=dtype, sample_T=20)
    eng.run_steps(steps)
    for d, (nx, ny) in enumerate(cells):
        sim, eps = built[d]
        assert tuple(sim.grid.dimensions[:2]) == (nx, ny)
        o1, ref = _oracle(sim, eps, t, eng.cb_host[d])
        _drive(o1, ref, sim, steps)
        got = eng.fields(d)
        a = np.concatenate([got[c].ravel() for c in ("Ez", "Hx", "Hy")])
        b = np.concatenate([o1.F[c].ravel() for c in ("Ez", "Hx", "Hy")])
        assert np.linalg.norm(b) > 0 and rel_l2(a, b) <= bar, d


@pytest.mark.parametrize("sizes", [[(33, 17), (81, 49)], [(33, 81), (1100, 1100)]])
def test_workgroup_order(mi355x, sizes):
    """Grouped by XCD or in launch order, 16- and 48-row tiles: the same bits."""
    _same(_run(sizes, np.float32, "fp16", 20, [45], True, xcd=0),
          _run(sizes, np.float32, "fp16", 20, [45], True, xcd=1))


def _engine(dtype, n):
    from prismo_amd.core.batch import BatchEngine

    sims = [_design(nx, ny, 8, dtype, 100 + k)[0] for k, (nx, ny) in enumerate([(33, 17), (60, 40)])]
    eng = BatchEngine(sims, dtype=dtype, sample_T=20)
    eng._build(n)
    return eng


def _replan(eng, at):
    """The plan again from the state a call left, at step `at`: the sets swapped
    where that is in set 1, CPML memory of Ez as it stands."""
    swap = eng.ctx.parity()
    eng.ctx.sync()
    for des in eng._arr:
        for name in eng._FIELD_ARRAYS if swap else ():
            a = getattr(des, name)
            a[0], a[1] = a[1], a[0]
    p = eng.plan
    p.src_e_table += 8 * at
    p.src_h_table += 8 * at
    p.table_step0, p.table_len, p.nfreq = at, p.table_len - at, 0
    eng.ctx.configure(p, keep=[eng._arr])
    return swap


def _state(eng, swap=0):
    eng.ctx.sync()
    q = eng.ctx.parity() ^ swap
    return [t.cpu().numpy() for b in eng._bufs
            for t in [b[n][q] for n in eng._FIELD_ARRAYS] + [b["psi_ex"], b["psi_ey"]]]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("cut", [1, 8, 11, 16, 29])
def test_state_between_calls(mi355x, dtype, cut):
    """After any call the design's arrays hold the whole state: fields and H-side
    memory in the set of pm_batch_parity, E-side memory in its one array.  A run
    goes on from them in a new plan, and from zeros put into them."""
    import torch

    n = 50
    ref = _engine(dtype, n)
    ref.ctx.run(n, graph=False)
    a = _engine(dtype, n)
    a.ctx.run(cut, graph=False)
    swap = _replan(a, cut)
    a.ctx.run(n - cut, graph=False)
    for x, y in zip(_state(a, swap), _state(ref)):
        assert np.array_equal(x, y)
    assert np.linalg.norm(_state(ref)[-2]) > 0

    z = _engine(dtype, n)
    z.ctx.run(cut, graph=False)
    z.ctx.sync()
    z._arena.zero_()
    z.stream.wait_stream(torch.cuda.current_stream())
    z.ctx.run(n - cut, graph=False)
    fresh = _engine(dtype, n)
    _replan(fresh, cut)
    fresh.ctx.run(n - cut, graph=False)
    for x, y in zip(_state(z), _state(fresh)):
        assert np.array_equal(x, y)
