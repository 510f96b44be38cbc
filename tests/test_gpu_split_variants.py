"""Parts of blocks in the kernel's variants, each an instantiation of its own:
low order faces, the resolution-change beta, two levels with the 8-wave source
and the TVD faces, B0, the body with B0 and the 8-wave source, steady state,
ensembles, FP32 states, every limiter.  State, block time steps and time are
those of whole blocks bit for bit in one-plane parts (what the library takes
for grids of this size), halves and quarters."""
import numpy as np
import pytest

from batsrus_amd.amr import AmrGrid
from batsrus_amd.core import Session
from batsrus_amd.ensemble import blast_ensemble
from batsrus_amd.grid import BlockGrid
from helpers import b0_dgb, body_mask, smooth_mhd_soa

pytestmark = pytest.mark.gpu

RC = dict(BetaLimiterResChange=1.2, nFaceLimiterResChange=2)
P = dict(UseDivbSource=True)
F32 = dict(precision="f32")
OPTIONS = {
    "low order": ("box", dict(UseAdaptiveLowOrder=True)),
    "low order f32": ("box", dict(F32, UseAdaptiveLowOrder=True)),
    "res beta": ("box", RC),
    "res beta f32 8-wave": ("levels", dict(F32, **RC, **P)),
    "f32": ("box", F32),
    "f32 8-wave steady": ("box", dict(F32, IsSteadyState=True, **P)),
    "levels 8-wave": ("levels", P),
    "levels res beta": ("levels", dict(RC, **P)),
    "tvd": ("levels", dict(UseTvdResChange=True)),
    "tvd 8-wave": ("levels", dict(UseTvdResChange=True, **P)),
    "tvd 8-wave f32": ("levels", dict(F32, UseTvdResChange=True, **P)),
    "tvd steady": ("levels", dict(UseTvdResChange=True, IsSteadyState=True)),
    "b0": ("box b0", {}),
    "b0 8-wave": ("box b0", P),
    "levels tvd b0 8-wave": ("levels b0", dict(UseTvdResChange=True, **P)),
    "body 8-wave": ("box body", P),
    "b0 body 8-wave": ("box b0 body", P),
    "b0 body 8-wave steady": ("box b0 body", dict(IsSteadyState=True, **P)),
    "levels b0 body 8-wave": ("levels b0 body", P),
    "levels tvd body": ("levels body", dict(UseTvdResChange=True)),
}
SCHEMES = [("rusanov", "minmod", 2), ("rusanov", "no", 2), ("linde", "mc", 2),
           ("linde", "mc", 1), ("hlld", "mc3", 2), ("hlld", "beta", 2)]


def _grid(what, nb):
    if "levels" in what:
        refine = np.zeros((2, 2, 2), bool)
        refine[0, 0, 0] = refine[1, 1, 0] = True
        return AmrGrid((2, 2, 2), refine, nCell=nb)
    return BlockGrid(nRoot=(3, 2, 3) if nb == 8 else (2, 1, 2),
                     nCell=(nb,) * 3, order="morton", periodic=(False,) * 3)


def _run(g, U0, scheme, cells, b0=None, body=None, runs=None):
    with Session(g, **scheme) as s:
        if b0 is not None:
            s.set_b0(b0, UseB0Source=True)
        if body is not None:
            s.set_body(*body, BodyRho=3.0, BodyP=2.0)
        if runs is not None:
            s.set_runs(runs)
        if cells is not None:
            s.set_stage_shape(cells)
        s.upload_soa(U0)
        s.init_timestep()
        dt = [s.get_dtmax_b()]
        for _ in range(3):
            s.advance(1)
            dt.append(s.get_dtmax_b())
        return s.download_soa(), np.array(dt), s.time()


def _same(g, U0, scheme, **kw):
    nb = g.nI
    ref = _run(g, U0, scheme, nb, **kw)
    assert np.isfinite(ref[0]).all()
    for cells in (None, nb // 2, nb // 4):
        got = _run(g, U0, scheme, cells, **kw)
        assert np.array_equal(got[0], ref[0]), cells
        assert np.array_equal(got[1], ref[1]), cells
        assert got[2] == ref[2], cells


@pytest.mark.parametrize("nb", [8, 16])
@pytest.mark.parametrize("option", list(OPTIONS))
def test_parts_of_every_variant(option, nb):
    what, extra = OPTIONS[option]
    g = _grid(what, nb)
    U0 = smooth_mhd_soa(g, seed=31, amp=0.2)
    kw = {}
    if "b0" in what:
        kw["b0"] = b0_dgb(g, lambda x, y, z: (0.1 * x, -0.1 * y, 0.2 + 0 * z))
    if "body" in what:
        kw["body"] = body_mask(g, 0.15, (0.25,) * 3) if "levels" in what \
            else body_mask(g, 0.2)
    for flux, lim, order in SCHEMES:
        if order == 1 and ("tvd" in option or "low" in option):
            continue
        if lim in ("minmod", "no") and "res beta" in option:
            continue
        print(f"case parts {option} {nb} {flux} {lim} {order}", flush=True)
        _same(g, U0, dict(flux=flux, limiter=lim, nOrder=order, beta=1.5,
                          cfl=0.6, **extra), **kw)


@pytest.mark.parametrize("wave8", [False, True])
def test_parts_of_an_ensemble(wave8):
    print(f"case parts ensemble {wave8}", flush=True)
    eg, U0 = blast_ensemble(nRun=5, nb_min=8, nb_max=120, seed=6)
    _same(eg, U0, dict(flux="hlld", limiter="mc", beta=1.5, cfl=0.6,
                       UseDivbSource=wave8), runs=eg.iBlockFirst_R)
