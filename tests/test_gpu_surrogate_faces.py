"""Waves of the gated face kernel that hold no, a few, more than 16, more
than 32 and 64 rows for the network, on blocks of 8^3 and 16^3.

A face's flux depends on its own four cells only, never on which or how many
faces share its wave.  A periodic state moved by some cells puts each face
into another wave, with other neighbours and another row, so the step of the
moved state is the moved step bit for bit (same kernel, same operations per
face and cell, equal cell sizes).  A weak wave passes the gate on every face
(64 rows in each wave), a strong one on some (a wave's count then runs from
0 to above 32).

16^3 blocks are also compared with the CPU oracle, with the bounds of
test_gpu_surrogate_stage."""
import numpy as np
import pytest

import mlp_oracle as mo
from batsrus_amd.core import Mlp, Session
from batsrus_amd.grid import BlockGrid
from helpers import smooth_mhd_soa
from test_gpu_surrogate_stage import JUMP_TOL, SCHEME, _run

pytestmark = pytest.mark.gpu


def _shift(g, U, d):
    """The state moved by d = (i, j, k) cells over the periodic domain."""
    n = g.nI
    V = np.empty_like(U)
    full = np.empty((8, *[n * r for r in g.nRoot[::-1]]), U.dtype)
    box = [np.s_[:, k * n:(k + 1) * n, j * n:(j + 1) * n, i * n:(i + 1) * n]
           for i, j, k in g.iRoot_DB]
    for b, s in enumerate(box):
        full[s] = U[:, b]
    full = np.roll(full, d[::-1], axis=(1, 2, 3))
    for b, s in enumerate(box):
        V[:, b] = full[s]
    return V


def _step(g, U, params):
    with Session(g, precision="f32", **SCHEME) as s, Mlp(params) as m:
        s.set_surrogate(m, "network", BetaMin=0.0, JumpTol=JUMP_TOL)
        s.upload_soa(U)
        s.init_timestep()
        s.set_global_timestep()
        n0 = s.surrogate_counts()[1]   # the first time step's faces
        for stage in (1, 2):
            s.advance_stage(stage)
        return s.download_soa(), s.surrogate_counts()[1] - n0


@pytest.mark.parametrize("nRoot,nCell,amp", [
    ((1, 1, 1), 8, 0.02), ((4, 2, 1), 8, 0.6),
    ((1, 1, 1), 16, 0.02), ((2, 1, 1), 16, 0.6)])
def test_moved_state(nRoot, nCell, amp):
    print(f"case surrogate moved state {nRoot} {nCell} {amp}", flush=True)
    g = BlockGrid(nRoot=nRoot, nCell=(nCell,) * 3, order="morton")
    U = smooth_mhd_soa(g, seed=75, amp=amp)
    params = mo.init_params(seed=8)
    U1, n1 = _step(g, U, params)
    nFace = 2 * 3 * g.nBlock * (nCell + 1) * nCell ** 2
    assert (n1 == nFace) if amp < 0.1 else (0 < n1 < nFace)
    for d in ((1, 0, 0), (3, 5, 2)):
        V1, _ = _step(g, _shift(g, U, d), params)
        assert np.array_equal(_shift(g, U1, d), V1), d


@pytest.mark.parametrize("nRoot,amp", [((1, 1, 1), 0.2), ((2, 1, 1), 0.6)])
def test_blocks_of_16(nRoot, amp):
    print(f"case surrogate 16^3 {nRoot} {amp}", flush=True)
    g = BlockGrid(nRoot=nRoot, nCell=(16,) * 3, order="morton")
    _run(g, smooth_mhd_soa(g, seed=74, amp=amp), "network", seed=5)
