"""The gated faces of a periodic box and of the same box twice over: few faces
take workgroups of half size, many whole ones, and a face's flux is the same in
both, so the state of the doubled box is the box's state twice, bit for bit
(the rows counted are twice the box's).  76 blocks of 8^3 have 131,328 faces
and 152 have 262,656, on either side of the 262,144 where the sizes change; one
of the blocks alone and 151 (260,928) stay below."""
import numpy as np
import pytest

import mlp_oracle as mo
from batsrus_amd.grid import BlockGrid
from helpers import smooth_mhd_soa
from test_gpu_surrogate_faces import _step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,times", [(76, 2), (1, 151), (1, 152), (38, 4)])
@pytest.mark.parametrize("amp", [0.02, 0.6])
def test_a_box_repeated(n, times, amp):
    print(f"case surrogate repeated {n} {times} {amp}", flush=True)
    # side lengths that are exact in binary: equal cells in both boxes
    one = BlockGrid(nRoot=(1, 1, n), nCell=(8,) * 3, xyzMax=(8., 8., 8. * n))
    many = BlockGrid(nRoot=(times, 1, n), nCell=(8,) * 3,
                     xyzMax=(8. * times, 8., 8. * n))
    assert np.array_equal(np.unique(one.CellSize_DB), [1.0])
    assert np.array_equal(np.unique(many.CellSize_DB), [1.0])
    U = smooth_mhd_soa(BlockGrid(nRoot=(1, 1, n), nCell=(8,) * 3), seed=76,
                       amp=amp)
    first = {tuple(r): b for b, r in enumerate(one.iRoot_DB)}
    src = [first[(0, j, k)] for i, j, k in many.iRoot_DB]
    params = mo.init_params(seed=8)
    U1, n1 = _step(one, U, params)
    Um, nm = _step(many, np.ascontiguousarray(U[:, src]), params)
    assert nm == times * n1
    assert n1 > 0 or amp > 0.1   # eight cells of a strong wave: none smooth
    assert np.array_equal(Um, U1[:, src])
