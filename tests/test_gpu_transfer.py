"""States in and out of the device: FP64 states come back bit for bit, FP32
states as the nearest FP32 values, below and above the size at which host
threads share the copy, with a last chunk that is not full and with ghost
slabs behind each variable; a state that the stages wrote comes back the same
through both layouts."""
import numpy as np
import pytest

from batsrus_amd.amr import AmrGrid, sphere_refinement
from batsrus_amd.core import Session
from batsrus_amd.grid import BlockGrid
from helpers import smooth_mhd_soa

pytestmark = pytest.mark.gpu

GRIDS = {
    "one block": lambda: BlockGrid(nRoot=(1, 1, 1), nCell=(8, 8, 8)),
    "30 blocks": lambda: BlockGrid(nRoot=(5, 3, 2), nCell=(16, 16, 16)),
    "151 blocks": lambda: BlockGrid(nRoot=(151, 1, 1), nCell=(16, 16, 16)),
    "two levels, 148 blocks": lambda: AmrGrid(
        (5, 4, 4), sphere_refinement((5, 4, 4), 0.3)),
    "two levels, 1331 roots": lambda: AmrGrid(
        (11, 11, 11), sphere_refinement((11, 11, 11), 0.2)),
}


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("name", list(GRIDS))
def test_states_come_back(name, precision):
    print(f"case transfer {name} {precision}", flush=True)
    g = GRIDS[name]()
    rng = np.random.default_rng(3)
    U = smooth_mhd_soa(g, seed=4, amp=0.1)
    U[0] += rng.random(U[0].shape) * 1e-3
    want = U if precision == "f64" else U.astype(np.float32).astype(float)
    with Session(g, flux="rusanov", limiter="mc", precision=precision) as s:
        for scale in (1.0, 2.0):      # the slots are used again
            s.upload_soa(U * scale)
            assert np.array_equal(s.download_soa(), want * scale)
        s.upload_soa(U)
        s.init_timestep()
        s.advance(1)
        out = s.download_soa()
        assert np.isfinite(out).all() and not np.array_equal(out, want)
        assert np.array_equal(g.state_vgb_to_soa(s.download_state()), out)
