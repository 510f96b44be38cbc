"""Blocks cut into parts by the launch: every part starts its z window with
the same code as a plane inside a block, so the state and the block time
steps are those of whole blocks bit for bit, whatever the number of parts the
launch rule takes for a grid of this size, over several steps (the parts'
minimum is taken anew each time) and with one- and three-stage schemes."""
import numpy as np
import pytest

from batsrus_amd.amr import AmrGrid, sphere_refinement
from batsrus_amd.core import Session
from batsrus_amd.grid import BlockGrid
from helpers import body_mask, smooth_mhd_soa

pytestmark = pytest.mark.gpu

HL = dict(flux="hlld", limiter="mc3", beta=1.5, cfl=0.8)
CASES = {
    # one block, a partly filled group, more items than workgroup places
    "8^3 one": ((1, 1, 1), 8, HL),
    "8^3 five": ((5, 1, 1), 8, HL),
    "8^3 powell": ((3, 2, 3), 8, dict(HL, UseDivbSource=True)),
    "8^3 2197": ((13, 13, 13), 8, dict(HL, flux="rusanov")),
    "16^3 one": ((1, 1, 1), 16, HL),
    "16^3 three, one stage": ((3, 1, 1), 16, dict(HL, nStage=1)),
    "16^3 rk3": ((2, 1, 2), 16, dict(HL, nStage=3, UseHalfStep=False)),
    "16^3 steady": ((3, 1, 2), 16, dict(HL, flux="linde",
                                        IsSteadyState=True)),
    "16^3 fp32": ((3, 2, 1), 16, dict(HL, precision="f32")),
    "16^3 540": ((9, 10, 6), 16, HL),
}


def _run(grid, U0, scheme, cells, steps=3, body=None):
    with Session(grid, **scheme) as s:
        if body is not None:
            s.set_body(*body, BodyRho=3.0, BodyP=2.0)
        if cells is not None:
            s.set_stage_shape(cells)
        s.upload_soa(U0)
        s.init_timestep()
        dt = [s.get_dtmax_b()]
        for _ in range(steps):
            s.advance(1)
            dt.append(s.get_dtmax_b())
        return s.download_soa(), np.array(dt)


@pytest.mark.parametrize("case", list(CASES))
def test_parts_give_the_bits_of_whole_blocks(case):
    print(f"case split {case}", flush=True)
    nRoot, nb, scheme = CASES[case]
    g = BlockGrid(nRoot=nRoot, nCell=(nb,) * 3, order="morton")
    U0 = smooth_mhd_soa(g, seed=21)
    ref = _run(g, U0, scheme, nb)
    assert ref[1].min() > 0 and np.isfinite(ref[1]).all()
    for cells in (None, nb // 2, nb // 4):
        got = _run(g, U0, scheme, cells)
        assert np.array_equal(got[0], ref[0]), cells
        assert np.array_equal(got[1], ref[1]), cells


def test_parts_across_levels_and_a_body():
    print("case split levels body", flush=True)
    g = AmrGrid((4, 4, 4), sphere_refinement((4, 4, 4), 0.3))
    U0 = smooth_mhd_soa(g, seed=22, amp=0.2)
    ref = _run(g, U0, HL, 8)
    for cells in (None, 4, 2):
        assert np.array_equal(_run(g, U0, HL, cells)[0], ref[0]), cells
    g = BlockGrid(nRoot=(3, 3, 3), nCell=(8, 8, 8), order="morton",
                  periodic=(False, False, False))
    U0 = smooth_mhd_soa(g, seed=23, amp=0.2)
    body = body_mask(g, 0.13)
    ref = _run(g, U0, HL, 8, body=body)
    got = _run(g, U0, HL, None, body=body)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
