"""Fast speeds whose square's square is a subnormal number: the square root
keeps its accuracy there, so the time step of a field-free gas at rest with a
pressure of 1e-155 is the oracle's.  The argument of the root, 3e-310, is
known to 2^-1074 / 3e-310 = 2e-14 of itself; the speed then to half of that,
plus the rounding of the few operations behind it: 1e-13 in all."""
import numpy as np
import pytest

import pyoracle as po
from batsrus_amd.core import Session
from batsrus_amd.grid import BlockGrid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flux", ["rusanov", "linde", "hlld"])
@pytest.mark.parametrize("p", [1e-155, 3e-156, 0.7])
def test_time_step_of_tiny_sound_speeds(flux, p):
    print(f"case tiny speeds {flux} {p}", flush=True)
    g = BlockGrid(nRoot=(2, 1, 1), nCell=(8, 8, 8), order="morton")
    U0 = np.zeros((8, g.nBlock, 8, 8, 8))
    U0[0] = 1.0
    U0[7] = p
    scheme = dict(flux=flux, limiter="mc", beta=1.5, cfl=0.8)
    o = po.Session(g, po.config_from_dict(scheme, g), g.soa_to_state_vgb(U0))
    o.exchange()
    o.init_timestep()
    o.s.nStep += 1
    dto = o.set_global_timestep()
    with Session(g, **scheme) as s:
        s.upload_soa(U0)
        s.init_timestep()
        dtg = s.set_global_timestep()
    assert np.isfinite(dto) and abs(dtg - dto) <= 1e-13 * dto, (dtg, dto)
