"""Loads and downloads around the size up to which they go through the pinned staging (1 MiB of
lists and f), in every storage form, and repeated calls on one context."""
import numpy as np
import pytest

from vlasiator_amd import vacc as V

pytestmark = pytest.mark.gpu

LEN = (40, 30, 20)


def _context(store=V.STORE_F32):
    return V.Context(V.make_mesh(LEN, (-1e6,) * 3, (1e6,) * 3), V.make_species(1.67262158e-27, 1.60217653e-19, 1e-12, 0),
                     V.make_options(V.PPM, storage=store))


def _cells(counts, seed):
    rng = np.random.default_rng(seed)
    return [(rng.choice(int(np.prod(LEN)), n, replace=False).astype(np.uint32),
             (10.0 ** rng.uniform(-14, -11, (n, 64))).astype(np.float32)) for n in counts]


# 4033 blocks of 260 bytes are the last total below 1 MiB; 4031 fit it with the rounding of the parts
SIZES = [[], [0], [1], [0, 3, 0], [600], [4000, 30], [4031], [4032], [4033], [4034], [9000], [1] * 2000]


@pytest.mark.parametrize("counts", SIZES, ids=lambda c: f"{len(c)}c{sum(c)}b")
def test_round_trip(counts):
    """The values come back bit for bit in ascending GID order, also on a context that held others."""
    ctx = _context()
    for seed in (1, 2):
        cells = _cells(counts, seed)
        ctx.upload_cells(cells)
        assert ctx.total_blocks() == sum(counts)
        got = ctx.download_cells()
        assert len(got) == len(cells)
        for (g, f), (g2, f2) in zip(cells, got):
            o = np.argsort(g)
            assert np.array_equal(g2, g[o]) and np.array_equal(f2, f[o])
    ctx.close()


@pytest.mark.parametrize("store", [V.STORE_BF16, V.STORE_F16])
@pytest.mark.parametrize("n", [1, 4000, 4100])
def test_16bit_download_is_the_same_by_either_path(store, n):
    """A block's code depends on its values alone, so the blocks of a small cell (staged download)
    equal the same blocks downloaded with 9000 others."""
    (g, f), rest = _cells([n], 3)[0], _cells([9000], 4)[0]
    small, large = _context(store), _context(store)
    small.upload_cells([(g, f)])
    large.upload_cells([(g, f), rest])
    a, b = small.download_cells()[0], large.download_cells()[0]
    small.close()
    large.close()
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_results_are_not_kept_from_one_call_to_the_next():
    """Moments, pressure and removed mass of two loads on one context equal those of fresh contexts."""
    ctx = _context()
    for seed in (5, 6):
        cells = _cells([300, 0, 41], seed)
        ctx.upload_cells(cells)
        other = _context()
        other.upload_cells(cells)
        for a, b in ((ctx.moments(3), other.moments(3)), (ctx.pressure(3), other.pressure(3)),
                     (ctx.moments(3), other.moments(3)), (ctx.adjust(3), other.adjust(3)),
                     (ctx.moments(3), other.moments(3))):
            assert np.array_equal(a, b)
        other.close()
    ctx.close()


def test_download_without_a_load_is_an_error():
    ctx = _context()
    off = np.zeros(1, np.uint64)
    assert V.lib().vacc_download_cells(ctx.h, off.ctypes.data, None, None) < 0
    ctx.close()
