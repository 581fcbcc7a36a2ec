"""The batch autotuner's NTT splits: timed where the batch has transforms, equal
programs' results otherwise, of which the first is kept."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PROGRAM = ("prime_major", "xcd_chunks", "strict_split")


def _batch(P, rng, transforms):
    from aoa_amd import FORWARD, Batch, check
    from aoa_amd._lib import NttItem

    def poly(nlimbs):
        return P.to_device(np.concatenate([rng.integers(0, P.primes[r], P.N, dtype=np.uint64) for r in range(nlimbs)]))

    key = [poly(P.k + P.kl) for _ in range(2)]
    B = Batch()
    B.add_mul(P, key, [([poly(P.k), poly(P.k)], [poly(P.k), poly(P.k)], [P.zeros(P.k), P.zeros(P.k)], P.k - 1)])
    if transforms:
        B.barrier()
        d = [poly(P.k) for _ in range(2)]
        item = NttItem()
        item.poly[0], item.poly[1] = d[0].data_ptr(), d[1].data_ptr()
        item.level, item.dir = P.k - 1, FORWARD
        check(B.lib.aoa_batch_add_ntt(B.h, P.h, ctypes.byref(item), 1))
        B._keep.append(d)
    return B


def test_splits_without_transforms_repeat_one_result(gpu):
    from aoa_amd import Params
    P = Params(16384, 4, 0, 48)
    B = _batch(P, np.random.default_rng(1), False)
    cands = B.autotune(reps=2)
    by_program = {}
    for c in cands:
        by_program.setdefault(tuple(c[f] for f in PROGRAM), []).append(c)
    assert len(by_program) == 8 and all(len(v) == len(cands) // 8 for v in by_program.values())
    for same in by_program.values():
        assert len({(c["ms"], c["checksum"]) for c in same}) == 1
    best = min(cands, key=lambda c: c["ms"])
    assert best["ntt_split"] == 0 and B.options() == {f: best[f] for f in B.OPTION_FIELDS}


def test_splits_with_transforms_are_timed(gpu):
    from aoa_amd import Params
    P = Params(16384, 4, 0, 48)
    B = _batch(P, np.random.default_rng(2), True)
    cands = B.autotune(reps=2)
    assert {c["ntt_split"] for c in cands} == {0, 64, 128, 256}
    assert len({c["ms"] for c in cands}) > len(cands) // 2
