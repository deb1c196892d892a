"""The tile sort with entries behind the live ones: entries that left through
the upper face and carriers that the shifted window crops take the key after
the last tile's, whose digits the live keys share in part (grids of 270 tiles,
two digits, and of 72250, three). Up to 2^18 entries (counted passes) and above
(scanned ones). Expected: the live entries in numpy's stable order of their
keys, exactly, and none of the others.
"""
import numpy as np
import pytest

import aprl_amd as A
from aprl_amd import bunch

pytestmark = pytest.mark.gpu

DZ = 1.0e-6
DX = 2.5 * DZ
CELLS = (4, 4, 0)


def entries(dims, n):
    """Interior entries, entries that cross the upper face in the first step and
    entries that turn into carriers beside it, in mixed order."""
    rng = np.random.default_rng(n)
    nx, ny, nz = dims
    third = n // 3
    inner = np.column_stack([rng.uniform(6, nx - 6, n - 2 * third), rng.uniform(6, ny - 6, n - 2 * third),
                             rng.uniform(2, nz - 4, n - 2 * third)])
    leave = np.column_stack([rng.uniform(6, nx - 6, third), rng.uniform(6, ny - 6, third),
                             rng.uniform(nz - 0.5, nz - 0.1, third)])
    carry = np.column_stack([rng.uniform(4.05, 4.3, third), rng.uniform(6, ny - 6, third),
                             rng.uniform(nz - 0.7, nz - 0.2, third)])
    x = np.concatenate([inner, leave, carry]) * [DX, DX, DZ]
    u = np.concatenate([rng.normal(0.0, 0.05, inner.shape), np.tile([0.0, 0.0, 8.0], (third, 1)),
                        np.tile([-6.0, 0.0, 0.1], (third, 1))])
    mixed = rng.permutation(n)
    return x[mixed], u[mixed]


@pytest.mark.parametrize("precision", ["fp64", "fp32-split"])
@pytest.mark.parametrize("dims,n", [((24, 24, 120), 3001), ((24, 24, 120), 2 ** 18), ((24, 24, 120), 2 ** 18 + 3),
                                    ((130, 130, 1000), 3001)])
def test_sort_behind(dims, n, precision):
    gpu = A.EBFieldGrid(A.EBGridGeometry(*dims, DX, DX, DZ, DZ / bunch.C_SI), precision=precision)
    win = A.MovingWindowFields(gpu, A.EBCPMLParameters(CELLS))
    cg = A.ConservativeSourceCoupling(gpu, "linear-binomial3")
    cg.setFrame(5.0)
    cg.setParticleBoundary(CELLS)
    x, u = entries(dims, n)
    store = A.ParticleStore(gpu, n)
    # a charge so small that the entries' own fields do not bend them
    store.upload(x, u, -1e-3 * bunch.QE / n, bunch.ME / n, np.ones(n))
    before = None
    for s in range(2):
        print(f"sort with entries behind, {dims} n={n} {precision} step {s}", flush=True)
        gpu.clearCurrent()
        win.beginStep(s, 50 - s)
        gpu.advanceMagnetic()
        win.setInlet()
        origin = np.array([0.0, 0.0, -s * DZ])
        if s:
            before = store.download(), store.states()
        cg.step(store, origin, s * DZ / bunch.C_SI)
        win.shift(s + 1, 49 - s)
    (x, _, _, _, _, ids), states = before
    cropped = (states == 1) & (x[:, 2] >= (dims[2] - 1) * DZ)
    assert len(ids) < n and np.count_nonzero(cropped) > 100
    cell = np.floor((x - [0.0, 0.0, -DZ]) / [DX, DX, DZ]).astype(np.int64)
    cell = np.clip(cell, 0, np.array(dims) - 1)
    ntx, nty = -(-dims[0] // 8), -(-dims[1] // 8)
    key = ((cell[:, 2] // 4) * nty + cell[:, 1] // 8) * ntx + cell[:, 0] // 8
    expected = ids[~cropped][np.argsort(key[~cropped], kind="stable")]
    got = store.download()[5]
    assert np.array_equal(got, expected[np.isin(expected, got)])
    assert len(got) > 0.3 * n and not np.isin(ids[cropped], got).any()
    assert cg.last_tiles == len(np.unique(key[~cropped]))
