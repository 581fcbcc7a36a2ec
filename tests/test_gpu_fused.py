"""The fused key-switching kernels at the edges of their tiles: limb counts
around the matrix step of 8 inputs and blocks of 16 outputs, the smallest and
largest rings and limb counts, every level that changes a tail, special bases
of other sizes than k + 1, and both ModDown modes.  Residues are compared with
the oracle's, which restates the reference's integer arithmetic: equal."""
import numpy as np
import pytest

from orc import Oracle

pytestmark = pytest.mark.gpu

# (N, k, kl, prec, levels)
SHAPES = [
    (2048, 2, 1, 55, [0, 1]),
    (2048, 64, 64, 55, [63]),
    (2048, 48, 52, 45, [31, 32, 47]),
    (4096, 9, 7, 52, [6, 7, 8]),
    (4096, 18, 16, 48, [15, 16, 17]),
    (8192, 16, 17, 45, [7, 15]),
    (16384, 10, 15, 48, [1, 9]),
    (32768, 8, 8, 52, [5]),
    (65536, 7, 9, 55, [4]),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "N%d_k%d_K%d_p%d" % s[:4])
@pytest.mark.parametrize("exact", [False, True])
def test_fused_parity(gpu, shape, exact):
    from aoa_amd import Params
    N, k, kl, prec, levels = shape
    P, O = Params(N, k, kl, prec), Oracle(N, k, kl, prec)
    P.set_moddown_exact(exact)
    O.set_moddown_exact(exact)
    rng = np.random.default_rng(N + k + kl)
    key = [O.random_poly(rng, k + kl) for _ in range(2)]
    dk = [P.to_device(x) for x in key]
    for level in levels:
        print("fused N=%d k=%d K=%d prec=%d level=%d exact=%d" % (N, k, kl, prec, level, exact), flush=True)
        c1 = [O.random_poly(rng, k) for _ in range(2)]
        c2 = [O.random_poly(rng, k) for _ in range(2)]
        d1, d2 = [P.to_device(x) for x in c1], [P.to_device(x) for x in c2]
        ws = P.workspace(level)
        out = [P.zeros(k), P.zeros(k)]
        ref = O.rotate_left(c1, key, 3, level)
        P.rotate_left(out, d1, dk, 3, level, ws)
        n = (level + 1) * N
        for y in range(2):
            assert np.array_equal(P.to_host(out[y])[:n], ref[y][:n]), "rotation c%d level %d" % (y, level)
        if level == 0:
            continue
        ref = O.hommul(c1, c2, key, level)
        P.hommul(out, d1, d2, dk, level, ws)
        n = level * N
        for y in range(2):
            assert np.array_equal(P.to_host(out[y])[:n], ref[y][:n]), "product c%d level %d" % (y, level)
