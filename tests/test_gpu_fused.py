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


def _ref_barrett(x, p):
    """The reference's reduction of x < 2^128 (aoa-ntt/src/cuda/htrans/common.cu:257-291)."""
    nb = p.bit_length()
    mu = (1 << 2 * nb) // p
    A = x - ((x >> (2 * nb - 64)) * mu >> 64) * p
    r = ((A & ((1 << nb) - 1)) - (A >> nb) * p) & ((1 << nb) - 1)
    return r - p if r >= p else r


def test_many_deviating_products(gpu):
    """Every coefficient of every special limb in the deviation window of one
    limb's product, so that every coefficient is corrected in place several
    times: the key's special limbs are made for it from the ModUp of the
    polynomial 1."""
    from aoa_amd import FORWARD, Params
    N, k, kl, prec = 2048, 4, 5, 48
    P, O = Params(N, k, kl, prec), Oracle(N, k, kl, prec)
    q, b = [int(p) for p in P.primes[:k]], [int(p) for p in P.primes[k:]]
    B, Q = 1, 1
    for x in b:
        B *= x
    for x in q:
        Q *= x
    rng = np.random.default_rng(5)
    key = [O.random_poly(rng, k + kl) for _ in range(2)]
    special = np.zeros((k + kl, N), dtype=np.uint64)
    for j in range(kl):
        i = 1 + j % (k - 1)
        c = (B // b[j]) % q[i]
        inv, eps = pow(c, -1, q[i]), (1 << q[i].bit_length()) - q[i]
        tries = ((eps + r) * inv % q[i] + n * q[i] for r in range(20000) for n in range(b[j] // q[i]))
        a = next(x for x in tries if _ref_barrett(x * c, q[i]) != x * c % q[i])
        v = sum(pow(Q // x, -1, x) * (Q // x) for x in q) % b[j]
        special[k + j, :] = a * (B // b[j]) * pow(v, -1, b[j]) % b[j]
    d = P.to_device(special.reshape(-1))
    P.ntt(d, 0, k + kl, FORWARD)
    key[0].reshape(k + kl, N)[k:] = P.to_host(d).reshape(k + kl, N)[k:]
    one = np.zeros((k, N), dtype=np.uint64)
    one[:, 0] = 1
    c1 = [O.random_poly(rng, k), one.reshape(-1)]
    ref = O.rotate_left(c1, key, 0, k - 1)
    O.set_moddown_exact(True)
    plain = O.rotate_left(c1, key, 0, k - 1)
    assert (ref[0] != plain[0]).sum() > 2 * N  # three limbs deviate
    out, dk = [P.zeros(k), P.zeros(k)], [P.to_device(x) for x in key]
    P.rotate_left(out, [P.to_device(x) for x in c1], dk, 0, k - 1, P.workspace(k - 1))
    for y in range(2):
        assert np.array_equal(P.to_host(out[y]), ref[y]), y
