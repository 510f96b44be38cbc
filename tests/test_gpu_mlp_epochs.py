"""Training over several epochs does not depend on when the runtime reads the
permutation it was given to copy: with copies that read their source in stream
order, while the host is at the next epochs' shuffles, the weights and errors
are those of copies that read it at once."""
import pytest

import hooked

pytestmark = pytest.mark.gpu

CODE = """
import hashlib
import numpy as np
import mlp_oracle as mo
from batsrus_amd.core import Mlp
rng = np.random.default_rng(4)
n = 400003
X = rng.standard_normal((n, 16)).astype(np.float32)
T = (X[:, :8] * X[:, 8:] + 0.1).astype(np.float32)
with Mlp(mo.init_params(seed=3)) as m:
    m.set_data(X, T)
    loss, err = m.train(6, batch=4096, seed=11)
    w = m.params()[0]
print(hashlib.sha256(w.tobytes() + err.tobytes()).hexdigest(), loss)
"""


def test_permutations_are_copied_as_they_were():
    print("case epochs", flush=True)
    want = hooked.run(CODE)
    assert hooked.run(CODE, HOOK_DEFER="1") == want
    assert hooked.run(CODE, HOOK_DEFER="1", HOOK_NO_PINNED="1") == want
