"""Transforms, products and rotations of residues at the ends and the middle of
their range (0, 1, (p-1)/2, (p+1)/2, p-1), mixed, in runs and constant: the
residues that carry the signed FP64 forms furthest.  Equal to the oracle's."""
import numpy as np
import pytest

from orc import Oracle

pytestmark = pytest.mark.gpu

SHAPES = [(2048, 3, 4, 48), (4096, 3, 4, 45), (16384, 3, 3, 48), (32768, 2, 3, 45), (65536, 3, 4, 48), (65536, 2, 2, 45),
          (65536, 10, 9, 48)]


def _poly(O, rng, nlimbs, kind):
    out = np.empty((nlimbs, O.N), dtype=np.uint64)
    for r in range(nlimbs):
        p = O.primes[r]
        v = np.array([0, 1, (p - 1) // 2, (p + 1) // 2, p - 1], dtype=np.uint64)
        if kind == "mixed":
            out[r] = v[rng.integers(0, 5, O.N)]
        elif kind == "runs":
            out[r] = np.repeat(v[rng.integers(0, 5, O.N // 128)], 128)
        else:
            out[r] = v[{"half": 2, "top": 4}[kind]]
    return out.reshape(-1)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "N%d_k%d_K%d_p%d" % s)
def test_extreme_residues(gpu, shape):
    from aoa_amd import FORWARD, INVERSE, Params
    N, k, kl, prec = shape
    P, O = Params(N, k, kl, prec), Oracle(N, k, kl, prec)
    rng = np.random.default_rng(sum(shape))
    level, n = k - 1, (k - 1) * N
    for kind in ("mixed", "runs", "half", "top"):
        print("extremes", shape, kind, flush=True)
        c = [_poly(O, rng, k, kind) for _ in range(4)]
        key = [_poly(O, rng, k + kl, "mixed" if kind == "runs" else kind) for _ in range(2)]
        for dirn in (FORWARD, INVERSE):
            d, ref = P.to_device(key[0]), key[0].copy()
            P.ntt(d, 0, k + kl, dirn)
            O.ntt(ref, 0, k + kl, dirn)
            assert np.array_equal(P.to_host(d), ref), (kind, dirn)
        dc, dk = [P.to_device(x) for x in c], [P.to_device(x) for x in key]
        out, ws = [P.zeros(k), P.zeros(k)], P.workspace(level)
        ref = O.hommul(c[:2], c[2:], key, level)
        P.hommul(out, dc[:2], dc[2:], dk, level, ws)
        for y in range(2):
            assert np.array_equal(P.to_host(out[y])[:n], ref[y][:n]), (kind, "product", y)
        ref = O.rotate_left(c[:2], key, 5, level)
        P.rotate_left(out, dc[:2], dk, 5, level, ws)
        for y in range(2):
            assert np.array_equal(P.to_host(out[y]), ref[y]), (kind, "rotation", y)
