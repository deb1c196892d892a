"""Device memory a first step takes for the tiles' current boxes: a tile of
one chunk needs one box, whatever the number of occupied tiles. A window whose
every inner tile holds one entry; the growth of the memory in use over the
step against one box per occupied tile (with the headroom of half) and the
step's other buffers, 2 MiB granules each.
"""
import gc

import numpy as np
import pytest
import torch

import aprl_amd as A
from aprl_amd import bunch

pytestmark = pytest.mark.gpu

DZ = 1.0e-6
DX = 2.0 * DZ
DIMS = (96, 96, 512)
BOX = {"linear-binomial3": 13 * 11 * 9, "quintic-compensated": 11 * 11 * 17}  # nodes of a tile's box


@pytest.mark.parametrize("precision", ["fp64", "fp32-split"])
@pytest.mark.parametrize("shape", list(BOX))
def test_first_step_memory(shape, precision):
    gpu = A.EBFieldGrid(A.EBGridGeometry(*DIMS, DX, DX, DZ, DZ / bunch.C_SI), precision=precision)
    win = A.MovingWindowFields(gpu, A.EBCPMLParameters((4, 4, 0)))
    cg = A.ConservativeSourceCoupling(gpu, shape)
    cg.setParticleBoundary((4, 4, 0))
    x = np.stack(np.meshgrid(np.arange(12.0, 84.0, 8.0) * DX, np.arange(12.0, 84.0, 8.0) * DX,
                             np.arange(6.5, 506.0, 4.0) * DZ, indexing="ij"), axis=-1).reshape(-1, 3)
    n = len(x)
    store = A.ParticleStore(gpu, n)
    store.upload(x, np.tile([0.0, 0.0, 5.0], (n, 1)), -bunch.QE, bunch.ME, np.ones(n))
    gpu.clearCurrent()
    win.beginStep(0, 50)
    gpu.advanceMagnetic()
    win.setInlet()
    gc.collect()  # stores and grids of other tests, if any are left
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    cg.step(store, np.zeros(3), 0.0)
    torch.cuda.synchronize()
    grown = before - torch.cuda.mem_get_info()[0]
    assert cg.last_tiles == n
    boxes = 1.5 * n * 3 * BOX[shape] * 8
    word = 8 if precision == "fp64" else 4
    sums = 6 * word * (DIMS[0] + 1) * (DIMS[1] + 1) * (DIMS[2] + 1)  # E* + E_old and E_cand + E_old
    print(f"{shape} {precision}: {n} tiles, {grown / 2**20:.0f} MiB, boxes {boxes / 2**20:.0f}, sums {sums / 2**20:.0f}")
    assert boxes <= grown <= boxes + sums + 64 * 2 ** 21
