"""The deposited current does not depend on how a tile's entries fall into
chunks: a tile's fixed-point sums are exact integers, and the shape's fixed
weights are applied to them without a rounding of each chunk's own. Bitwise:
the step of a bunch uploaded in another order, whose crowded tiles then hold
other entries in each of their chunks, and an FP32-split step whose chunks
hold 512 entries instead of 256 because of a few entries without charge in a
tile of their own.
"""
import numpy as np
import pytest

import aprl_amd as A
from aprl_amd import bunch

pytestmark = pytest.mark.gpu

DZ = 1.0e-6
DX = 2.0 * DZ
CELLS = (4, 4, 0)
DIMS = (21, 19, 34)


def step(shape, precision, x, u, q, ids):
    """Electric field, current and momenta (in id order) after one window step."""
    gpu = A.EBFieldGrid(A.EBGridGeometry(*DIMS, DX, DX, DZ, DZ / bunch.C_SI), precision=precision)
    win = A.MovingWindowFields(gpu, A.EBCPMLParameters(CELLS))
    rng = np.random.default_rng(1)
    for a in range(3):
        gpu.set_component(a, (1e3 * rng.standard_normal(gpu.component(a).shape)).astype(np.float32).astype(float))
    cg = A.ConservativeSourceCoupling(gpu, shape)
    cg.setParticleBoundary(CELLS)
    store = A.ParticleStore(gpu, len(q))
    store.upload(x, u, q, bunch.ME, np.ones(len(q)), ids)
    print(f"{shape} {precision} n={len(q)}", flush=True)
    gpu.clearCurrent()
    win.beginStep(0, 50)
    gpu.advanceMagnetic()
    win.setInlet()
    cg.step(store, np.zeros(3), 0.0)
    got = store.download()
    order = np.argsort(got[5])
    return [gpu.component(a) for a in (0, 1, 2, 6, 7, 8)], got[1][order], got[5][order]


def crowd(n):
    """Half of n entries in one cell column, so that tiles of one chunk and of
    several occur."""
    rng = np.random.default_rng(n)
    cell = np.stack([rng.integers(5, d - 5, n) for d in (*DIMS[:2], 26)], axis=1).astype(float)
    cell[: n // 2, :2] = 9.0
    x = ((cell + rng.uniform(0.01, 0.99, (n, 3))).astype(np.float32)).astype(float) * [DX, DX, DZ]
    u = (rng.normal(0.0, 0.1, (n, 3)) + [0.0, 0.0, 5.0]).astype(np.float32).astype(float)
    return x, u


def assert_equal(a, b):
    n = min(len(a[2]), len(b[2]))
    differing = [np.count_nonzero(p != q) for p, q in zip(a[0], b[0])]
    differing += [np.count_nonzero(a[k][:n] != b[k][:n]) for k in (1, 2)]
    assert not any(differing), differing
    assert all(np.any(p != 0.0) for p in a[0][3:])


@pytest.mark.parametrize("shape", ["linear-binomial3", "quintic-compensated"])
@pytest.mark.parametrize("precision,n", [("fp64", 12001), ("fp32-split", 12001), ("fp32-split", 2 ** 19 + 3)])
def test_upload_order(precision, n, shape):
    x, u = crowd(n)
    ids = np.arange(1, n + 1, dtype=np.uint64)
    q = np.full(n, -bunch.QE)
    p = np.random.default_rng(2).permutation(n)
    assert_equal(step(shape, precision, x, u, q, ids), step(shape, precision, x[p], u[p], q, ids[p]))


@pytest.mark.parametrize("shape", ["linear-binomial3", "quintic-compensated"])
def test_chunk_size(shape):
    n, more = 2 ** 19 - 1, 9
    x, u = crowd(n)
    ids = np.arange(1, n + more + 1, dtype=np.uint64)
    q = np.full(n + more, -bunch.QE)
    q[n:] = 0.0
    xm = np.concatenate([x, np.tile([9.5 * DX, 9.5 * DX, 30.5 * DZ], (more, 1))])
    um = np.concatenate([u, np.tile([0.0, 0.0, 5.0], (more, 1))])
    assert_equal(step(shape, "fp32-split", x, u, q[:n], ids[:n]), step(shape, "fp32-split", xm, um, q, ids))
