"""Residues that aoa_eltwise_scalar leaves outside [0, p): it uses its 64-bit
scalar as given, so that adding a constant above a prime raises residues past
it and subtracting one wraps those below the difference to just under 2^64.
Products, transforms and the rotation after an inverse transform give what they
give for the same residues reduced first.  The constants are those of adding
and subtracting 1 to 200 at a scale of 2^prec; residues 0 and 1 are
planted, which every subtraction wraps."""
import numpy as np
import pytest

from orc import Oracle

pytestmark = pytest.mark.gpu

SHAPES = [(2048, 4, 5, 45), (4096, 4, 5, 48), (4096, 3, 4, 52), (8192, 3, 4, 45), (65536, 3, 2, 48), (32768, 2, 3, 55),
          (65536, 10, 9, 48), (32768, 10, 9, 52)]  # the last two: both key halves in a workgroup


def _cases(O, rng, nlimbs):
    """(op, constant, residues, the same with the constant applied mod each prime)"""
    from aoa_amd import ADD, SUB
    N = O.N
    for op, v in ((ADD, 3), (ADD, 20), (ADD, 200), (SUB, 1), (SUB, 17)):
        c = v << O.prec
        x = O.random_poly(rng, nlimbs)
        for r in range(nlimbs):
            at = rng.choice(N, 40, replace=False)
            x[r * N + at] = np.arange(40, dtype=np.uint64) % np.uint64(2)
        want = x.copy()
        for r in range(nlimbs):
            p = O.primes[r]
            k = (c if op == ADD else -c) % p
            want[r * N:(r + 1) * N] = (x[r * N:(r + 1) * N] + np.uint64(k)) % np.uint64(p)
        yield op, c, x, want


def _setup(shape):
    from aoa_amd import Params
    N, k, kl, prec = shape
    P, O = Params(N, k, kl, prec), Oracle(N, k, kl, prec)
    O.prec = prec
    return P, O, np.random.default_rng(sum(shape))


def _raise(P, O, op, c, x):
    """x with the constant applied by aoa_eltwise_scalar; q0's stay canonical."""
    n = x.size // P.N
    d = P.to_device(x)
    P.eltwise_scalar(op, d, d, c, 0, n)
    got = P.to_host(d)
    assert (got[:P.N] < O.primes[0]).all()
    assert (got[P.N:2 * P.N] >= np.uint64(O.primes[1])).any()
    return d


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "N%d_k%d_K%d_p%d" % s)
def test_products(gpu, shape):
    from aoa_amd import Batch
    import torch
    P, O, rng = _setup(shape)
    k, N, level = P.k, P.N, P.k - 1
    evk = [O.random_poly(rng, k + P.kl) for _ in range(2)]
    dk = [P.to_device(x) for x in evk]
    for op, c, x, want in _cases(O, rng, k):
        c2 = [O.random_poly(rng, k) for _ in range(2)]
        c1 = O.random_poly(rng, k)
        raised = _raise(P, O, op, c, x)
        rest = [P.to_device(a) for a in [c1] + c2]
        # the raised component in each place of the product
        for host, dev in (([want, c1] + c2, [raised, rest[0]] + rest[1:]), (c2 + [c1, want], rest[1:] + [rest[0], raised]),
                          ([want, want] * 2, [raised] * 4)):
            print("product", shape, op, c, flush=True)
            ref = O.hommul(host[:2], host[2:], evk, level)
            out = [P.zeros(k), P.zeros(k)]
            P.hommul(out, dev[:2], dev[2:], dk, level, P.workspace(level))
            outs = {"plain": out}
            # one launch for all forms of arithmetic, and one for each
            for ss in (-1, 1):
                two = [[P.zeros(k), P.zeros(k)] for _ in range(2)]
                B = Batch()
                B.add_mul(P, dk, [(dev[:2], dev[2:], o, level) for o in two])
                B.set_options(strict_split=ss)
                B.launch()
                torch.cuda.synchronize()
                B.close()
                outs.update({("batch", ss, i): o for i, o in enumerate(two)})
            for name, o in outs.items():
                for y in range(2):
                    assert np.array_equal(P.to_host(o[y])[:level * N], ref[y][:level * N]), (name, y, op, c)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "N%d_k%d_K%d_p%d" % s)
def test_transforms_rotation_and_client_side(gpu, shape):
    import torch
    from aoa_amd import FORWARD, INVERSE, Batch
    P, O, rng = _setup(shape)
    k, N, level = P.k, P.N, P.k - 1
    rtk = [O.random_poly(rng, k + P.kl) for _ in range(2)]
    dk = [P.to_device(x) for x in rtk]
    for op, c, x, want in _cases(O, rng, k):
        print("transform", shape, op, c, flush=True)
        back = None
        for dirn in (FORWARD, INVERSE):
            d, ref = _raise(P, O, op, c, x), want.copy()
            P.ntt(d, 0, k, dirn)
            O.ntt(ref, 0, k, dirn)
            assert np.array_equal(P.to_host(d), ref), (dirn, op, c)
            back = d
        # a rotation of the transformed component, and a key switch of the residues themselves
        other = O.random_poly(rng, k)
        got = [P.zeros(k), P.zeros(k)]
        P.rotate_left(got, [back, P.to_device(other)], dk, 3, level, P.workspace(level))
        exp = O.rotate_left([ref, other], rtk, 3, level)
        for y in range(2):
            assert np.array_equal(P.to_host(got[y]), exp[y]), ("rotation", y, op, c)
        P.keyswitch(got[0], got[1], _raise(P, O, op, c, x), dk[0], dk[1], level, P.workspace(level),
                    add0=_raise(P, O, op, c, x))
        canon = [P.zeros(k), P.zeros(k)]
        P.keyswitch(canon[0], canon[1], P.to_device(want), dk[0], dk[1], level, P.workspace(level), add0=P.to_device(want))
        for y in range(2):
            assert (got[y] == canon[y]).all(), ("key switch", y, op, c)
        # rotations of the residues themselves, plain and accumulated in a batch
        exp = O.rotate_left([want, want], rtk, 3, level)
        raised = [_raise(P, O, op, c, x) for _ in range(2)]
        P.rotate_left(got, raised, dk, 3, level, P.workspace(level))
        B, bout = Batch(), [P.zeros(k), P.zeros(k)]
        B.add_rotate(P, [(raised, bout, dk, 3, level, True)])
        B.launch()
        torch.cuda.synchronize()
        B.close()
        p = np.repeat(np.array(O.primes[:k], dtype=np.uint64), N)
        for y in range(2):
            assert np.array_equal(P.to_host(got[y]), exp[y]), ("rotation of residues", y, op, c)
            assert np.array_equal(P.to_host(bout[y]), (exp[y] + want) % p), ("rotate and add", y, op, c)
        # encryption of the message and under the key, decryption of the component and under the key
        outs = []
        for v in (P.to_device(want), _raise(P, O, op, c, x)):
            enc = [P.zeros(k), P.zeros(k), v.clone()]
            P.encrypt(enc[0], enc[1], enc[2], v, v, 5, 1, P.zeros(3 * k))
            dec = [P.zeros(k), v.clone(), P.to_device(other)]
            P.decrypt(dec[0], dec[1], dec[2], v, level)
            outs.append(enc + dec)
        for name, a, b in zip(("c0", "c1", "m", "plain", "c0 after", "c1 after"), *outs):
            assert (a == b).all(), (name, op, c)
