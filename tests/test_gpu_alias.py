"""Decryption with a key that overlaps the ciphertext (the ciphertext's own
transformed limbs, or those a limb further on): as with a split set, where the
key is read after both components are transformed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2048, 6, 2, 48), (16384, 5, 2, 55), (65536, 4, 2, 45)], ids=lambda s: "N%d_k%d_K%d_p%d" % s)
@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("ahead", [0, 1])
def test_decrypt_key_overlaps(gpu, shape, which, ahead):
    from aoa_amd import Params
    P, Q = Params(*shape), Params(*shape)
    N, L = P.N, P.k - 1
    Q.set_ntt_split(N if N <= 4096 else 64 if N <= 16384 else 256)
    rng = np.random.default_rng(sum(shape))
    c = [np.concatenate([rng.integers(0, min(P.primes[:P.k]), N, dtype=np.uint64) for _ in range(L + 1)]) for _ in range(2)]
    got = []
    for H in (P, Q):
        print("decrypt", shape, which, ahead, H is P, flush=True)
        d, m = [H.to_device(x) for x in c], H.zeros(L)
        H.decrypt(m, d[0], d[1], d[which][ahead * N:], L - 1)
        got.append([m] + d)
    for a, b in zip(*got):
        assert (a == b).all()
