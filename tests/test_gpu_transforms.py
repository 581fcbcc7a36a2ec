"""The transforms' default kernels, encryption and decryption built on them
against the explicit splits (which the oracle covers), over every ring
dimension and form of arithmetic: residues are equal.  With overlapping buffers
encryption takes its general path, with the same results as before."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (N, k, kl, prec): every N, both forms below the 63-bit prime, one limb of each kind at least
SHAPES = [(2048, 3, 2, 55), (2048, 17, 3, 45), (4096, 4, 5, 52), (4096, 2, 1, 48), (8192, 5, 3, 48), (16384, 3, 4, 55),
          (32768, 4, 2, 45), (65536, 2, 3, 55), (65536, 3, 1, 48)]


def _split(N):
    return N if N <= 4096 else 64 if N <= 16384 else 256


def _uniform(P, rng, nlimbs):
    return P.to_device(np.concatenate([rng.integers(0, P.primes[r], P.N, dtype=np.uint64) for r in range(nlimbs)]))


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "N%d_k%d_K%d_p%d" % s)
def test_transforms_match_splits(gpu, shape):
    from aoa_amd import FORWARD, INVERSE, Params
    P, Q = Params(*shape), Params(*shape)
    Q.set_ntt_split(_split(P.N))
    R = P.k + P.kl
    rng = np.random.default_rng(sum(shape))
    x = _uniform(P, rng, R)
    for res0, nres in ((0, R), (0, 1), (1, R - 1), (P.k, P.kl)):
        print("transform", shape, res0, nres, flush=True)
        a, b = x.clone(), x.clone()
        for dirn in (FORWARD, INVERSE, INVERSE):
            P.ntt(a, res0, nres, dirn)
            Q.ntt(b, res0, nres, dirn)
            assert (a == b).all(), (dirn, res0, nres)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "N%d_k%d_K%d_p%d" % s)
@pytest.mark.parametrize("alias", [None, "c0", "c1"])
def test_encrypt_decrypt_match_splits(gpu, shape, alias):
    from aoa_amd import Params
    P, Q = Params(*shape), Params(*shape)
    Q.set_ntt_split(_split(P.N))
    k = P.k
    rng = np.random.default_rng(sum(shape) + 1)
    pk, s, m = [_uniform(P, rng, k) for _ in range(2)], _uniform(P, rng, k), _uniform(P, rng, k)
    got = []
    for H in (P, Q):
        print("encrypt", shape, alias, H is P, flush=True)
        c, mm, ws = [P.zeros(k), P.zeros(k)], m.clone(), P.zeros(3 * k)
        if alias:
            c[int(alias[1])] = mm
        H.encrypt(c[0], c[1], mm, pk[0], pk[1], 7, 3, ws)
        enc = [t.clone() for t in (c[0], c[1], mm)]
        lv = k - 1 if alias is None else k - 2
        d, t = [m.clone(), pk[0].clone()], P.zeros(k)
        if alias:
            t = d[int(alias[1])]
        H.decrypt(t, d[0], d[1], s, lv)
        got.append(enc + d + [t])
    for name, a, b in zip(("c0", "c1", "m", "d0", "d1", "plain"), *got):
        assert (a == b).all(), name


@pytest.mark.parametrize("logn", range(16))
def test_encoder_sizes_bitexact(gpu, logn):
    """Both directions of the special FFT, encode and decode at every slot
    count of N = 2^16: equal to the oracle's bit for bit."""
    import ctypes
    import torch
    import orc
    from aoa_amd import FORWARD, INVERSE, Params
    N, n, scale = 65536, 1 << logn, 1 << 48
    P, O = Params(N, 2, 0, 48), orc.Oracle(N, 2, 0, 48)
    rng = np.random.default_rng(logn)
    z = rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.complex128).view(np.float64).copy()).cuda()
    bits = lambda a: np.ascontiguousarray(a).view(np.uint64)
    print("encoder n=%d" % n, flush=True)
    for dirn in (FORWARD, INVERSE):
        t, ref = dev(z), np.ascontiguousarray(z).view(np.float64).copy()
        P.special_fft(t, n, dirn)
        orc.load().orc_fft_special(ref.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), n, N, int(dirn == INVERSE))
        assert np.array_equal(bits(t.cpu().numpy()), bits(ref)), dirn
    out, vals = P.zeros(2), dev(z)
    P.encode(out, vals, n, scale)
    assert np.array_equal(bits(vals.cpu().numpy()), bits(ref))  # left in place
    want = O.encode(z, scale).reshape(2, N)
    got = P.to_host(out).reshape(2, N)
    for r in range(2):
        assert np.array_equal(got[r], want[r] % np.uint64(O.primes[r])), r
    back = dev(np.zeros(n))
    P.decode(back, out, n, scale)
    assert np.array_equal(bits(back.cpu().numpy()), bits(O.decode(want[0], n, scale)))
