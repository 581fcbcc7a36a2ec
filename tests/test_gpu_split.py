"""The NTT split's getter and setter: a new handle reports the default (0), and
setting what was read restores the handle, also after the autotuner."""
import numpy as np
import pytest

from orc import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,others", [(2048, [2048]), (4096, [64, 4096]), (16384, [64, 128, 256]), (65536, [256])])
def test_split_round_trip(gpu, N, others):
    from aoa_amd import FORWARD, Params
    P, O = Params(N, 2, 2, 48), Oracle(N, 2, 2, 48)
    x = O.random_poly(np.random.default_rng(N), 4)
    ref = x.copy()
    O.ntt(ref, 0, 4, FORWARD)

    def check():
        d = P.to_device(x)
        P.ntt(d, 0, 4, FORWARD)
        assert np.array_equal(P.to_host(d), ref)

    assert P.ntt_split() == 0
    for tuned in (False, True):
        if tuned:
            print("autotune", N, flush=True)
            assert set(P.autotune_ntt(reps=2)) == set(others)
            assert P.ntt_split() in others
        old = P.ntt_split()
        for n1 in others + [0]:
            P.set_ntt_split(n1)
            assert P.ntt_split() == n1
            check()
            P.set_ntt_split(old)
            assert P.ntt_split() == old
            check()
