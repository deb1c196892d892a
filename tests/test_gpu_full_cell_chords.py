"""Particles at a tile's lower face that move one whole cell away from it in a
step (u / gamma rounds to -1 and c dt is the cell). The tile key and the chord
name the start's cell with the same arithmetic, so such a chord stays in the
tile box, which reaches one cell below the tile; z / h and z * (1 / h) do not
agree on the cell of these faces. Against the oracle within 1e-12."""
import numpy as np
import pytest

import harness as H
from aprl_amd import bunch

pytestmark = pytest.mark.gpu

DZ = 0.345e-6
DX = 2.0 * DZ
DIMS = (16, 16, 40)
CELLS = (3, 3, 0)
SHAPES = {"linear-binomial3": ("binomial3", True), "quintic-compensated": ("quintic", False)}


def faces():
    k = np.arange(8, DIMS[2] - 4, 4)
    z = k * DZ
    return z[(z / DZ == k) & (z * (1.0 / DZ) < k)]


@pytest.mark.parametrize("shape", list(SHAPES))
def test_full_cell_chords_match_oracle(shape):
    import aprl_amd as A
    oshape, smooth = SHAPES[shape]
    orc = H.CpuFields("orc", *DIMS, DX, DX, DZ, DZ / H.C_SI, 1)
    orc.install_window(CELLS)
    H.seeded_fields(orc, 4, scale=1e2)
    co = H.CpuCoupling(orc, oshape, smooth, cpml_cells=CELLS)
    gpu = A.EBFieldGrid(A.EBGridGeometry(*DIMS, DX, DX, DZ, DZ / H.C_SI))
    win = A.MovingWindowFields(gpu, A.EBCPMLParameters(CELLS))
    for a in range(9):
        gpu.set_component(a, orc.view(a))
    cg = A.ConservativeSourceCoupling(gpu, shape)
    cg.setParticleBoundary(CELLS)
    z = faces()
    n = len(z)
    assert n >= 4
    x = np.stack([np.full(n, 8.3 * DX), np.full(n, 7.6 * DX), z], axis=1)
    u = np.tile([0.0, 0.0, -1.0e9], (n, 1))
    q, m, ids = np.full(n, -bunch.QE * 50), np.full(n, bunch.ME * 50), np.arange(1, n + 1)
    co.set_particles(x, u, q, m, np.ones(n), ids)
    store = A.ParticleStore(gpu, n)
    store.upload(x, u, q, m, np.ones(n), ids)
    zero = [np.zeros(int(np.prod(H.component_shape(*DIMS, a)[1:]))) for a in range(6)]
    orc.clear_current(); gpu.clearCurrent()
    orc.window_begin(0, 50, zero[:3]); win.beginStep(0, 50)
    orc.window_advance_magnetic(); gpu.advanceMagnetic()
    orc.window_set_inlet(50, 1, *zero[:2]); win.setInlet()
    co.step(np.zeros(3), 0.0)
    cg.step(store, np.zeros(3), 0.0)
    for comps in ((0, 1, 2), (6, 7, 8)):
        e = np.concatenate([gpu.component(a).ravel() for a in comps])
        r = np.concatenate([orc.view(a).ravel() for a in comps])
        assert np.linalg.norm(r) > 0.0 and np.linalg.norm(e - r) <= 1e-12 * np.linalg.norm(r)
