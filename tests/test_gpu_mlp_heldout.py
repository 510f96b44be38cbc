"""The held-out errors of a training call, summed on the device, against the
same sums in numpy over the same samples (the seeded split restated here):
one sample, a workgroup's 32 rows and a few more, and more rows than one
round of the grid's workgroups takes (8192).  The network's outputs are the
same bits on both sides; what differs is the order of at most n FP64
additions, so sqrt(num / den) agrees within n 2^-53 < 2e-12."""
import numpy as np
import pytest

import mlp_oracle as mo
from batsrus_amd.core import Mlp

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def _held(n, n_hold, seed):
    """The last n_hold samples of the seeded permutation (splitmix64)."""
    perm, s = list(range(n)), seed
    for i in range(n, 1, -1):
        s = (s + 0x9E3779B97F4A7C15) & M64
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & M64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
        j = (z ^ (z >> 31)) % i
        perm[i - 1], perm[j] = perm[j], perm[i - 1]
    return np.array(perm[n - n_hold:])


@pytest.mark.parametrize("n,hold", [(2, 0.5), (64, 0.5), (70, 0.5),
                                    (20001, 0.45)])
def test_heldout_errors(n, hold):
    print(f"case held-out {n} {hold}", flush=True)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 16)).astype(np.float32)
    T = (rng.standard_normal((n, 8)) * np.arange(1, 9)).astype(np.float32)
    h = _held(n, int(hold * n), 7)
    with Mlp(mo.init_params(seed=3)) as m:
        Y = m.forward(X[h]).astype(np.float64)
        m.set_data(X, T)
        _, e = m.train(0, batch=64, hold=hold, seed=7)
    t = T[h].astype(np.float64)
    num, den = ((Y - t) ** 2).sum(0), (t ** 2).sum(0)
    want = np.sqrt(np.concatenate([[num.sum() / den.sum()], num / den]))
    np.testing.assert_allclose(e[:9], want, rtol=2e-12, atol=0)
    np.testing.assert_allclose(e[9:], want, rtol=2e-12, atol=0)
