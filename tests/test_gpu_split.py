"""The NTT split's getter and setter: a new handle reports the default (0), and
setting what was read restores the handle, also after the autotuner.  A split's
tables are built on its first use, by whoever comes first."""
import ctypes
import threading

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


def test_tables_on_first_use(gpu):
    """A parameter set of N = 2^16 and 61 primes holds its 122 MiB of twiddles once
    (and as much again for its other tables at most) until a split is used."""
    import torch
    from aoa_amd import Params
    Params(65536, 30, 0, 48)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    P = Params(65536, 30, 0, 48)
    held = (free - torch.cuda.mem_get_info()[0]) / 2**20
    assert held < 250, held
    P.set_ntt_split(256)
    assert (free - torch.cuda.mem_get_info()[0]) / 2**20 > held + 122


def test_batches_share_the_tables(gpu):
    """Batches on one handle in two threads, each with its split from the start."""
    import torch
    from aoa_amd import FORWARD, Batch, Params, check
    from aoa_amd._lib import NttItem
    P, O = Params(16384, 3, 2, 48), Oracle(16384, 3, 2, 48)
    x = [O.random_poly(np.random.default_rng(i), 3) for i in range(2)]
    got = {}

    def run(n1):
        d = [P.to_device(v) for v in x]
        torch.cuda.synchronize()
        s, B = torch.cuda.Stream(), Batch()
        item = NttItem()
        item.poly[0], item.poly[1] = d[0].data_ptr(), d[1].data_ptr()
        item.level, item.dir = 2, FORWARD
        check(B.lib.aoa_batch_add_ntt(B.h, P.h, ctypes.byref(item), 1))
        B.set_options(ntt_split=n1)
        with torch.cuda.stream(s):
            B.launch(stream=s)
        s.synchronize()
        got[n1] = [P.to_host(v) for v in d]

    ts = [threading.Thread(target=run, args=(n1,)) for n1 in (64, 256)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for n1 in (64, 256):
        for v, g in zip(x, got[n1]):
            ref = v.copy()
            O.ntt(ref, 0, 3, FORWARD)
            assert np.array_equal(g, ref), n1
