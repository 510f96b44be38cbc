"""Opening a session makes no more runtime calls than its arrays need: a copy
or a clear for each that starts with something in it (a blocking copy takes
about 10 of the 130 us of a session of eight blocks)."""
import pytest

import hooked

pytestmark = pytest.mark.gpu

CODE = """
from batsrus_amd.core import Session
from batsrus_amd.grid import BlockGrid
g = BlockGrid(nRoot=(2, 2, 2), nCell=(8, 8, 8), order="morton")
Session(g, flux="hlld", limiter="mc").close()
n0 = [hooks.hook_count(k) for k in (MALLOC, MEMCPY, MEMSET)]
Session(g, flux="hlld", limiter="mc").close()
print([hooks.hook_count(k) - n for k, n in zip((MALLOC, MEMCPY, MEMSET), n0)])
"""


def test_opening_a_session():
    print("case opening a session", flush=True)
    malloc, memcpy, memset = eval(hooked.run(CODE))
    print(malloc, memcpy, memset)
    # two state buffers, neighbours, cell sizes, time steps, scalars, the runs'
    # first blocks, each block's run, error word, partial sums, side states
    assert malloc <= 11
    # scalars, the runs' first blocks, neighbours and cell sizes of the
    # default grid (the session's own are ordered on its stream)
    assert memcpy <= 4
    # each block's run, error word, time steps, side states
    assert memset <= 4
