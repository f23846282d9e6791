"""The tolerance-form remap at the walls of the velocity mesh, on rows of one or several columns: cells
moved through either wall, some wholly outside, against the oracle."""
import numpy as np
import pytest

import oracle as O
from tests import cases
from vlasiator_amd import vacc as V


def _wall_cells(rng, method, dim, extent, side):
    """Mesh, cells and intersections of a pass along `dim` on a mesh of `extent` blocks: Maxwellians centred
    near the wall, with none or every second or third block along dim left out (rows of several
    columns), moved through the wall by part of a cell up to more than the whole mesh; dk at dv, at the
    span limit and at 2.5 dv, and the transverse shears that the span leaves room for."""
    n = np.array([6, 5, 7])
    n[dim] = extent
    dvs = np.array([1.0e4, 1.1e4, 0.9e4])
    vmin, vmax, dv = -2.0 * dvs * n, 2.0 * dvs * n, dvs[dim]
    blocks = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij"), -1).reshape(-1, 3)
    e = np.arange(64)
    c = np.stack([e & 3, (e >> 2) & 3, e >> 4], -1)
    centre = np.full(3, 0.5)
    centre[dim] = {"low": 0.05, "high": 0.95}[side]
    width = np.maximum(0.25, 3.0 / (4.0 * n))
    cells, isx = [], []
    for gaps in (0, 1, 2):
        b = blocks[blocks[:, dim] % (gaps + 1) != gaps] if gaps else blocks
        g = (b[:, 0] + n[0] * (b[:, 1] + n[1] * b[:, 2])).astype(np.uint32)
        o = np.argsort(g)
        x = (b[:, None, :] * 4 + c[None] + 0.5) / (4.0 * n)   # 0..1 over the mesh
        for shift in (0.3, 2.6, 5.0, 9.7, 4.0 * extent + 7.0):
            for dk in (dv, 0.7 * dv, 2.5 * dv):
                f = 1e-10 * np.exp(-(((x - centre) / width) ** 2).sum(-1)) * rng.uniform(0.9, 1.1)
                cells.append((g[o], f[o].astype(np.float32)))
                room = (6.0 * dk - 4.0 * dv) / 3.0 * 0.9 if dk < 2 * dv else 0.3 * dv
                slopes = dict(zip([a for a in range(3) if a != dim], (0.6 * room, -0.4 * room)))
                # (v - I) / dk is the target of v in the middle of the transverse plane
                base = vmin[dim] + shift * dv
                if side == "high":
                    base = min(vmin[dim] - shift * dv, vmax[dim] - (4 * extent + shift) * dk)
                row = np.zeros(12)
                row[4 * dim] = base - sum(2.0 * n[a] * s for a, s in slopes.items())
                for a in range(3):
                    row[4 * dim + 1 + a] = dk if a == dim else slopes[a]
                isx.append(row)
    return tuple(int(k) for k in n), tuple(vmin), tuple(vmax), cells, np.stack(isx)


def _check_walls(method, dim, extent, side):
    """Every value is the exact arithmetic's (units that it takes) or within the stated 5e-6 of the cell's
    maximum of the oracle's FP64 remap; the block lists are the oracle's."""
    rng = np.random.default_rng(1000 * method + 10 * dim + extent)
    length, vmin, vmax, cells, isx = _wall_cells(rng, method, dim, extent, side)
    min_value = 1e-16
    print(f"{side} wall, dim {dim}, {extent} blocks, method {method}, {len(cells)} cells", flush=True)
    ctx = V.Context(V.make_mesh(length, vmin, vmax), V.make_species(1.67262158e-27, 1.60217653e-19, min_value, 1),
                    V.make_options(method, fast_arith=True))
    ctx.upload_cells(cells)
    ctx.set_intersections(isx)
    st = ctx.map_1d(dim)
    got = ctx.download_cells()
    ctx.close()
    assert not st & V.STATUS_DK
    m = O.make_mesh(length, vmin, vmax)
    lean = 0
    for i, (g, f) in enumerate(cells):
        is4 = isx[i, 4 * dim:4 * dim + 4]
        g32, f32 = cases.sort_cell(*O.map_1d(m, g, f, is4, dim, method, min_value)[:2])
        g64, f64, _ = O.map_1d(m, g, f.astype(np.float64), is4, dim, method, min_value, fp64=True)
        assert np.array_equal(got[i][0], g32), i
        ref = np.zeros(f32.shape)
        common = np.isin(g64, g32)
        ref[np.searchsorted(g32, g64[common])] = f64[common]
        off = np.abs(got[i][1] - ref) > 5e-6 * f.max()
        assert np.array_equal(got[i][1][off], f32[off]), (i, int(off.sum()))
        lean += int((got[i][1] != f32).sum())
    return lean


@pytest.mark.gpu
@pytest.mark.parametrize("method", [O.PLM, O.PPM, O.PQM])
@pytest.mark.parametrize("dim", [0, 1, 2])
@pytest.mark.parametrize("extent", [1, 2, 4, 12])
def test_high_wall_matches_the_oracle(method, dim, extent):
    assert _check_walls(method, dim, extent, "high") > 0


@pytest.mark.gpu
@pytest.mark.parametrize("method", [O.PLM, O.PPM, O.PQM])
@pytest.mark.parametrize("dim", [0, 1, 2])
@pytest.mark.parametrize("extent", [1, 2, 4, 12])
def test_low_wall_matches_the_oracle(method, dim, extent):
    _check_walls(method, dim, extent, "low")


@pytest.mark.gpu
@pytest.mark.parametrize("store,ost", [(V.STORE_F32, O.ST_F32), (V.STORE_F16, O.ST_F16)])
@pytest.mark.parametrize("side", ["low", "high"])
def test_block_sums_at_the_walls(side, store, ost):
    """The pass that also stores block sums (the last of an acceleration), over the same cells: density
    and momentum from the sums equal those of the downloaded f to FP32 rounding."""
    rng = np.random.default_rng(5)
    length, vmin, vmax, cells, isx = _wall_cells(rng, O.PPM, 2, 4, side)
    for a in range(2):   # the x and y passes leave f where it is
        isx[:, 4 * a] = vmin[a]
        isx[:, 4 * a + 1 + a] = (vmax[a] - vmin[a]) / (4 * length[a])
    print(f"block sums, {side} wall, storage {store}", flush=True)
    ctx = V.Context(V.make_mesh(length, vmin, vmax), V.make_species(1.67262158e-27, 1.60217653e-19, 1e-16, 1),
                    V.make_options(V.PPM, storage=store, fast_arith=True))
    ctx.upload_cells(cells)
    ctx.set_intersections(isx)
    ctx.accelerate(0)
    mom = ctx.moments(len(cells))
    got = ctx.download_cells()
    ctx.close()
    m = O.make_mesh(length, vmin, vmax)
    for i, (g, f) in enumerate(got):
        want = np.asarray(O.moments(m, g, f))
        speed = max(np.abs(vmin).max(), np.abs(vmax).max())
        assert abs(mom[i, 0] - want[0]) <= 1e-6 * want[0]
        assert np.all(np.abs(mom[i, 1:] - want[1:]) <= 1e-6 * want[0] * speed)
