"""The tolerance-form remap's target ring.

A deposit outside its column's target blocks has no row of its own: below the range it goes to
the row its target would have, above to the row behind the range.  On the CPU a model of the kernel's
ring (ring_host_check.hip) checks over random geometries, up to the deposit span that the
column build admits and with columns beyond both walls, that such a deposit never hits a row of a
block that is open, that a block stored to make room is finished, and that every block is stored
once with the values of a plain array."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle as O
from vlasiator_amd import vacc as V

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "ring_host_check.hip")
OUT = os.path.join(HERE, "_build", "libring_host_check.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    deps = [SRC] + [os.path.join(HERE, "..", "vlasiator_amd", "csrc", f) for f in ("vacc_lean.h", "vacc_common.h")]
    if not os.path.exists(OUT) or os.path.getmtime(OUT) < max(os.path.getmtime(d) for d in deps):
        subprocess.run([HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", SRC, "-o", OUT],
                       check=True, capture_output=True)
    L = C.CDLL(OUT)
    d, p = C.c_double, C.c_void_p
    L.ring_row.argtypes = [C.c_int, C.c_int, p, p, C.c_int, C.c_int, d, d, d, d, d, d, p, p, p, p]
    return L


def _geometry(rng, maxlen):
    """dk, di, dj within the span of the lean kernel, (4 dv + 3 |di| + 3 |dj|) / dk <= 6 and dk <= 3 dv,
    often at its limit; the row moved by up to 1.5 meshes either way."""
    dv = 1.0e4
    dk = dv * rng.choice([rng.uniform(2 / 3, 3.0), rng.uniform(2 / 3, 1.2), 2 / 3 + 1e-3, 1.0, 3.0])
    room = max(6.0 * dk - 4.0 * dv, 0.0) / 3.0 * rng.choice([0.0, rng.uniform(), 1.0 - 1e-6])
    share = rng.uniform()
    di, dj = share * room * rng.choice([-1, 1]), (1 - share) * room * rng.choice([-1, 1])
    b0, b1 = int(rng.integers(0, maxlen)), int(rng.integers(0, maxlen))
    vmin = -2.0 * dv * maxlen
    shift = rng.choice([0.0, rng.uniform(-1.5, 1.5)]) * 4 * dv * maxlen + rng.uniform(-8, 8) * dv
    # the pencil in the middle of the set starts at vmin + shift
    I = vmin + shift - (4 * b0 + 1.5) * di - (4 * b1 + 1.5) * dj
    return I, di, dj, dk, dv, vmin, b0, b1


@pytest.mark.parametrize("method", [O.PLM, O.PPM, O.PQM])
def test_ring_model(lib, method):
    rng = np.random.default_rng(100 + method)
    counts = np.zeros(5, np.int64)
    for it in range(6000):
        maxlen = int(rng.choice([1, 2, 3, 4, 5, 8, 13, 24]))
        occ = (rng.random(maxlen) < rng.choice([0.3, 0.6, 0.9, 1.0])).astype(np.uint8)
        src = np.where(np.repeat(occ, 4)[None, :], rng.uniform(0.5, 2.0, (16, 4 * maxlen)), 0.0).astype(np.float32)
        I, di, dj, dk, dv, vmin, b0, b1 = _geometry(rng, maxlen)
        stored, plain = np.zeros((4 * maxlen, 16), np.float32), np.zeros((4 * maxlen, 16), np.float32)
        seen = np.zeros(maxlen, np.int32)
        before = counts.copy()
        lib.ring_row(method, maxlen, occ.ctypes.data, src.ctypes.data, b0, b1, I, di, dj, dk, dv, vmin,
                     stored.ctypes.data, plain.ctypes.data, seen.ctypes.data, counts.ctypes.data)
        what = (it, maxlen, occ, I, di, dj, dk)
        assert counts[0] == before[0] and counts[1] == before[1], what
        assert seen.max() <= 1, what
        assert np.array_equal(stored, plain), what
    assert counts[2] > 10000 and counts[3] > 300   # deposits outside the range; units of several columns
    assert counts[4] > 50      # blocks stored to make room


@pytest.mark.gpu
@pytest.mark.parametrize("dim", [0, 1, 2])
@pytest.mark.parametrize("store", [V.STORE_F32, V.STORE_BF16])
def test_a_full_ring_is_no_error(dim, store):
    """Targets two thirds of a cell wide, where the ring is full while its oldest block, finished, waits
    for its store: the cells are remapped (their mass is kept) and not reported as passed through."""
    n = np.array([10, 9, 8])
    n[dim] = 40
    vmin, vmax = -2.0e4 * n, 2.0e4 * n
    dv, dk = 1.0e4, (2 / 3 + 1e-3) * 1.0e4
    row = np.arange(12, 24)
    blocks = np.stack(np.meshgrid(*[row if a == dim else np.arange(k) for a, k in enumerate(n)], indexing="ij"), -1)
    b = blocks.reshape(-1, 3)
    g = np.sort(b[:, 0] + n[0] * (b[:, 1] + n[1] * b[:, 2])).astype(np.uint32)
    f = (1e-12 * np.random.default_rng(dim).uniform(1, 2, (g.size, 64))).astype(np.float32)
    isx = np.zeros(12)
    # 48 source cells from cell 48 on take 72 targets from cell 40 on
    isx[4 * dim], isx[4 * dim + 1 + dim] = vmin[dim] + 48 * dv - 40.3 * dk, dk
    print(f"full ring, dim {dim}, storage {store}", flush=True)
    ctx = V.Context(V.make_mesh(n, vmin, vmax), V.make_species(1.67262158e-27, 1.60217653e-19, 1e-16, 1),
                    V.make_options(V.PPM, storage=store, fast_arith=True))
    ctx.upload_cells([(g, f)])
    ctx.set_intersections(isx)
    assert ctx.map_1d(dim) == 0
    assert ctx.status(1)[0] == 0
    got = ctx.download_cells()[0]
    ctx.close()
    assert got[0].size > 1.4 * g.size
    # the block sums that the 16-bit scales keep are trees of six roundings, taken twice; the deposits
    # round a few times more: some 20 roundings of 2^-24 at most in one direction
    assert abs(got[1].sum(dtype=np.float64) / f.sum(dtype=np.float64) - 1.0) < 2e-6
