"""The limiter on the device, where its medians are v_med3_f32: exact remaps of values around and below
the smallest normal number, with equal, twofold, zero and opposite slopes, against the oracle bit
for bit.  tests/test_limiter_host.py compares the same expression in its host form."""
import numpy as np
import pytest

import oracle as O
from tests import cases
from vlasiator_amd import vacc as V

pytestmark = pytest.mark.gpu

LEN, VMIN, VMAX = (8, 6, 5), (-1e6,) * 3, (1e6,) * 3


def _cells(rng, scale):
    """Random walks along every axis whose steps have few distinct sizes, so that slopes tie, double,
    vanish and change sign; some values exactly zero or negative zero."""
    n = int(np.prod(LEN))
    out = []
    for _ in range(4):
        steps = rng.choice([0.0, 1.0, -1.0, 2.0, -2.0, 4.0, 0.5, 1e-3, 1e3], (n, 64)) * rng.choice([1.0, 1.0, 3.0, 1e-7], (n, 64))
        f = (np.abs(np.cumsum(steps, 1)) * scale).astype(np.float32)
        f[rng.random(f.shape) < 0.1] = 0.0
        f[rng.random(f.shape) < 0.02] = -0.0
        out.append((np.arange(n, dtype=np.uint32), f))
    return out


@pytest.mark.parametrize("method", [O.PLM, O.PPM, O.PQM])
@pytest.mark.parametrize("dim", [0, 1, 2])
@pytest.mark.parametrize("scale", [1e-45, 1e-42, 1e-38, 1e-30, 1e-22, 1.0])
def test_exact_remap_bits(method, dim, scale):
    """With a threshold of 1 the limiter sees the values as they are: subnormal differences and, up to
    1e-19, products of slopes that underflow."""
    rng = np.random.default_rng(100 * method + 10 * dim)
    cells = _cells(rng, scale)
    m = O.make_mesh(LEN, VMIN, VMAX)
    isx = np.zeros((len(cells), 12))
    dv = [2e6 / (4 * k) for k in LEN]
    a, b = [d for d in range(3) if d != dim]
    for i, dk in enumerate((1.0, 0.8, 1.3, 1.0)):
        isx[i, 4 * dim + 1 + dim] = dk * dv[dim]
        isx[i, 4 * dim + 1 + a], isx[i, 4 * dim + 1 + b] = 0.1 * dv[dim], -0.07 * dv[dim]
        isx[i, 4 * dim] = VMIN[dim] - 0.37 * dv[dim] * (i + 1)
    print(f"limiter bits, dim {dim}, method {method}, scale {scale}", flush=True)
    ctx = V.Context(V.make_mesh(LEN, VMIN, VMAX), V.make_species(1.67262158e-27, 1.60217653e-19, 1.0, 1),
                    V.make_options(method))
    ctx.upload_cells(cells)
    ctx.set_intersections(isx)
    ctx.map_1d(dim)
    got = ctx.download_cells()
    ctx.close()
    want = [O.map_1d(m, g, f, isx[i, 4 * dim:4 * dim + 4], dim, method, 1.0)[:2] for i, (g, f) in enumerate(cells)]
    cases.assert_cells_equal(got, want, f"scale {scale}")
    assert any((np.abs(f) > 0).any() for _, f in got)
