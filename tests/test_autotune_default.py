"""The autotuner and the shape that a session has by itself: it is among the
shapes that are timed, an empty choice leaves or sets it, and a table that was
measured without it is measured again."""
import json
import os

import numpy as np
import pytest

from batsrus_amd.autotune import (Autotuner, apply, candidates, domain_key,
                                  shapes, workload_key)
from batsrus_amd.core import Session
from batsrus_amd.grid import BlockGrid
from helpers import smooth_mhd_soa

SCHEME = dict(flux="hlld", limiter="mc", beta=1.5, cfl=0.8)
G = BlockGrid(nRoot=(4, 4, 4), nCell=(8, 8, 8), order="morton")


def test_the_default_is_among_the_shapes():
    s = shapes(G)
    own = [c for c in s if not c["cells_per_thread"]]
    assert {(c["xcd"], c["nWorkgroup"]) for c in own} == {(False, 0), (True, 0)}
    assert [c for c in s if c["cells_per_thread"]] == candidates(G)


def test_an_older_table_is_not_taken_for_measured(tmp_path):
    p = str(tmp_path / "t.json")
    old = dict(choice=dict(cells_per_thread=2, xcd=False, nWorkgroup=0,
                           graph=True), step_us=90.0, measured=[])
    keys = workload_key(G, SCHEME), domain_key(64 * 512, SCHEME)
    with open(p, "w") as f:
        json.dump({k: old for k in keys}, f)
    a = Autotuner(p)
    assert a.lookup(G, SCHEME) == old
    assert not any(a._measured(k) for k in keys)
    a.table[keys[0]] = dict(old, own_choice_measured=True)
    assert a._measured(keys[0])


@pytest.mark.gpu
def test_an_empty_choice_is_the_default(tmp_path):
    print("case autotune default", flush=True)
    U0 = smooth_mhd_soa(G, seed=9)
    out, ms = {}, {}
    with Session(G, **SCHEME) as s:
        for name, choice in (("untuned", None), ("whole", dict(
                cells_per_thread=8)), ("empty", {}), ("own, xcd", dict(
                cells_per_thread=0, xcd=True))):
            if choice is not None:
                apply(s, choice)
            s.upload_soa(U0)
            s.init_timestep()
            s.advance(3)
            out[name] = s.download_soa()
            t = []
            for _ in range(5):
                s.advance(2)
                t.append(s.last_stage_kernel_ms()[0])
            ms[name] = min(t)
    print(ms)
    for name in out:
        assert np.array_equal(out[name], out["untuned"]), name
    # 16 workgroups of whole blocks take four times as long as in the
    # library's one-plane parts (76 and 19 us per launch)
    for name in ("untuned", "empty", "own, xcd"):
        assert ms[name] < 0.5 * ms["whole"], name


@pytest.mark.gpu
def test_a_tuned_small_grid_is_not_behind_an_untuned_one(tmp_path):
    print("case autotune small grid", flush=True)
    at = Autotuner(os.path.join(str(tmp_path), "t.json"))
    e = at.tune(G, smooth_mhd_soa(G, seed=9), SCHEME)
    own = [m for m in e["measured"] if not m["cells_per_thread"]]
    assert len(own) == 4
    assert e["step_us"] <= min(m["step_us"] for m in own)
    assert at.tune(G, None, SCHEME) == e       # stored, not measured again
