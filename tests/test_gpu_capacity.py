"""A pass whose targets do not fit the block storage: the call returns VACC_E_STATE, the launches
behind that pass leave the unwritten list alone, calls that read it are refused, and the context
works again once cells are loaded.

20800 blocks that lie alone along x straddle two target blocks each when moved by half a block:
41600 targets, and the storage holds 1.5 times the blocks and 4160 more."""
import numpy as np
import pytest

from vlasiator_amd import vacc as V

pytestmark = pytest.mark.gpu

LEN, VMIN, VMAX = (40, 40, 40), (-1e6,) * 3, (1e6,) * 3
DV = 2e6 / 160


def context(method=V.PPM, store=V.STORE_F32, tolerance=False, graph=False, dynamic=0, conserve=False):
    sp = V.make_species(1.67262158e-27, 1.60217653e-19, 1e-15, 1, dynamic=dynamic, bulk=(1e3, 1e9), dyn_min=(1e-16, 1e-14),
                        conserve_mass=conserve)
    return V.Context(V.make_mesh(LEN, VMIN, VMAX), sp,
                     V.make_options(method, storage=store, fast_arith=tolerance, use_graph=graph))


def scattered_cell(seed=1):
    """Every third block along x, at every y and z."""
    x, y, z = np.meshgrid(np.arange(1, 40, 3), np.arange(40), np.arange(40), indexing="ij")
    g = np.sort((x + 40 * y + 1600 * z).reshape(-1)).astype(np.uint32)
    assert 2 * g.size > g.size + g.size // 2 + 64 + 4096
    rng = np.random.default_rng(seed)
    return g, (1e-12 * rng.uniform(1, 2, (g.size, 64))).astype(np.float32)


def compact_cell(seed=2, size=6):
    r = np.arange(17, 17 + size)
    x, y, z = np.meshgrid(r, r, r, indexing="ij")
    g = np.sort((x + 40 * y + 1600 * z).reshape(-1)).astype(np.uint32)
    rng = np.random.default_rng(seed)
    return g, (1e-12 * rng.uniform(1, 2, (g.size, 64))).astype(np.float32)


def half_block_shift():
    """Intersections that move f by two cells along x and leave y and z."""
    isx = np.zeros(12)
    for d in range(3):
        isx[4 * d], isx[4 * d + 1 + d] = VMIN[d], DV
    isx[0] -= 2 * DV
    return isx


def rotation():
    return [V.make_fields((0.0, 0.0, 5e-8), (0.0, 0.0, 0.0), 0.0364)]   # 10 degrees for protons


def refused(call):
    with pytest.raises(V.VaccError, match="error -4"):
        call()


CALLS = {
    "map_1d": lambda c: c.map_1d(0),
    "accelerate": lambda c: c.accelerate(0),
    "step": lambda c: c.step(0),
    "step, moments from the fields": lambda c: c.step(0, use_moments=False),
    "subcycled": lambda c: c.accelerate_subcycled(0.0364, 0),
}


@pytest.mark.parametrize("call", CALLS)
@pytest.mark.parametrize("form", ["exact f32", "tolerance f32", "tolerance bf16", "tolerance f32 graph",
                                  "exact f32 dynamic conserve"])
def test_overflow_is_an_error_and_a_load_clears_it(call, form):
    print(f"overflow in {call}, {form}", flush=True)
    kw = {"tolerance": "tolerance" in form, "store": V.STORE_BF16 if "bf16" in form else V.STORE_F32,
          "graph": "graph" in form, "dynamic": 1 if "dynamic" in form else 0, "conserve": "conserve" in form}
    ctx = context(**kw)
    for _ in range(2):
        ctx.upload_cells([scattered_cell()])
        ctx.set_intersections(half_block_shift())
        ctx.set_fields(rotation())
        refused(lambda: CALLS[call](ctx))
        nbr = (np.zeros(2, np.uint32), np.zeros(0, np.uint32))
        for later in (lambda: ctx.moments(1), lambda: ctx.pressure(1), lambda: ctx.download(), lambda: ctx.adjust(1),
                      lambda: ctx.adjust_spatial(1, *nbr), lambda: ctx.find_blocks([0], [5]),
                      lambda: ctx.find_blocks_noalloc([0], [5]), lambda: ctx.autotune(),
                      lambda: ctx.compute_intersections(rotation(), 0, use_moments=True), *(
                          (lambda f=f: f(ctx)) for f in CALLS.values() if f is not CALLS["subcycled"])):
            refused(later)
        # the same context after a load equals a fresh one
        fresh = context(**kw)
        got = []
        for c in (ctx, fresh):
            c.upload_cells([compact_cell()])
            c.set_fields(rotation())
            c.step(0)
            got.append((c.moments(1), *c.download_cells()[0]))
        for a, b in zip(*got):
            assert np.array_equal(a, b)
        fresh.close()
    ctx.close()


@pytest.mark.parametrize("use_moments", [False, True])
@pytest.mark.parametrize("bad", [0, 1, 2])
def test_populations_behind_one_that_overflows_are_finished(bad, use_moments):
    """Three populations of four cells, one of which overflows: the call is an error, and the others'
    counts, lists, f and removed mass are those of a step of their own, also through a translation."""
    from vlasiator_amd import trans as T
    print(f"population {bad} overflows, use_moments={use_moments}", flush=True)
    fields = rotation() * 4
    # the compact cells' content reaches their edges, so that the step changes their block counts
    cells = [[compact_cell(10 * p + i, 5 + i) for i in range(4)] for p in range(3)]
    cells[bad] = [scattered_cell(i) for i in range(4)]
    ctxs = [context(tolerance=True) for _ in range(3)]
    for ctx, cw in zip(ctxs, cells):
        ctx.upload_cells(cw)
        ctx.set_fields(fields)
    before = [ctx.total_blocks() for ctx in ctxs]
    loss = [np.full(4, -1.0) for _ in range(3)]
    refused(lambda: V.accelerate_populations(ctxs, 0, use_moments=use_moments, adjust=True, rho_loss=loss))
    pencils = T.build_pencils_uniform((4, 1, 1), (True, True, True), np.zeros(4, np.uint8), (1e7,) * 3, 0)
    for p in range(3):
        if p == bad:
            refused(lambda: ctxs[p].download())
            continue
        total = ctxs[p].total_blocks()
        assert total != before[p] and total == sum(ctxs[p].counts())
        T.set_pencils(ctxs[p], 0, pencils)
        got = [ctxs[p].download_cells()]
        T.trans_map_1d(ctxs[p], 0, 1.0)
        got.append(ctxs[p].download_cells())
        assert sum(g.size for g, _ in got[0]) == total
        if use_moments:   # a pivot of its own: only the counts compare
            continue
        alone, lost = context(tolerance=True), np.zeros(4)
        alone.upload_cells(cells[p])
        alone.set_fields(fields)
        alone.step(0, use_moments=False, rho_loss=lost)
        want = [alone.download_cells()]
        T.set_pencils(alone, 0, pencils)
        T.trans_map_1d(alone, 0, 1.0)
        want.append(alone.download_cells())
        for a, b in zip(got, want):
            for (g1, f1), (g2, f2) in zip(a, b):
                assert np.array_equal(g1, g2) and np.array_equal(f1, f2)
        assert np.array_equal(loss[p], lost)
        alone.close()
    for ctx in ctxs:
        ctx.close()
