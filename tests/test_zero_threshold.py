"""The exact form where the limiter's inputs are not finite: a sparsity threshold of 0 (or so small
that its reciprocal overflows), which scales every value to infinity or NaN, and infinite or NaN
values of f.  Results equal the oracle's bit for bit, NaN where it has NaN."""
import numpy as np
import pytest

import oracle as O
from tests import cases
from tests.test_recon_host import columns, lib   # noqa: F401  (lib: the host build of the reconstructions)
from vlasiator_amd import vacc as V
from vlasiator_amd import workloads as W


def _same(got, want):
    got, want = np.asarray(got), np.asarray(want)
    return np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~np.isnan(got)], want[~np.isnan(want)])


def _check_stream(lib, method, col, thr):
    n, nc = col.size - 8, O.ncoef(method)
    got = np.zeros(n * nc, np.float32)
    lib.recon_stream(method, col.ctypes.data, n, np.float32(thr), got.ctypes.data)
    st = np.stack([col[k:k + 9] for k in range(n)])
    want = O.coeff_batch(method, st, thr).reshape(-1)
    assert _same(got, want)
    return np.isfinite(want).sum()


@pytest.mark.parametrize("method", [O.PLM, O.PPM, O.PQM])
@pytest.mark.parametrize("thr", [0.0, 1e-40, -1e-15])
def test_reconstruction_without_a_threshold(lib, method, thr):   # noqa: F811
    finite = sum(_check_stream(lib, method, col, thr) for col in columns(7 + method))
    assert finite or (method == O.PLM and thr != -1e-15)   # a PLM cell without a threshold is NaN


@pytest.mark.parametrize("method", [O.PLM, O.PPM, O.PQM])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 3e38])
def test_reconstruction_of_values_that_are_not_finite(lib, method, bad):   # noqa: F811
    for i, col in enumerate(columns(11 + method)):
        n = col.size - 8
        for k in (0, n // 2, n - 1):
            c = col.copy()
            c[4 + k] = bad
            if i % 2:
                c[4 + max(k - 1, 0)] = bad
            _check_stream(lib, method, c, 1e-15)


@pytest.mark.gpu
@pytest.mark.parametrize("method", [O.PLM, O.PPM, O.PQM])
@pytest.mark.parametrize("dim", [0, 1, 2])
@pytest.mark.parametrize("kind", ["threshold 0", "infinite and NaN values"])
def test_exact_remap(method, dim, kind):
    w = W.config(0, ncells=3)
    cells = cases.build_cells(w)
    min_value = 0.0 if kind == "threshold 0" else w.min_value
    if min_value:
        rng = np.random.default_rng(dim)
        for _, f in cells:
            for bad in (np.nan, np.inf, -np.inf):
                f[rng.integers(f.shape[0]), rng.integers(64)] = bad
    isx = cases.oracle_intersections(w, dim)
    print(f"exact remap, {kind}, dim {dim}, method {method}", flush=True)
    ctx = V.Context(V.make_mesh(w.grid_length, w.vmin, w.vmax), V.make_species(w.mass, w.charge, min_value, w.add_width),
                    V.make_options(method))
    ctx.upload_cells(cells)
    ctx.set_intersections(isx)
    ctx.map_1d(dim)
    got = ctx.download_cells()
    ctx.close()
    m = cases.oracle_mesh(w)
    for i, (g, f) in enumerate(cells):
        g2, f2, _ = O.map_1d(m, g, f, isx[i, 4 * dim:4 * dim + 4], dim, method, min_value)
        g2, f2 = cases.sort_cell(g2, f2)
        assert np.array_equal(got[i][0], g2) and _same(got[i][1], f2), f"cell {i}"
