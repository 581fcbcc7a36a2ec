"""The serving loop's step budget: an operation is charged the workspace that a
batch uses for it, so a product (or rotation) runs in a budget of just that, one
a step, and is refused by one byte less."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["mul", "rot"])
def test_step_budget_is_what_a_batch_uses(gpu, kind):
    import torch
    from aoa_amd import AoaError, Batch, Params, Server
    P = Params(4096, 5, 0, 48)
    rng = np.random.default_rng(3)
    level, n = P.k - 1, P.k * P.N

    def poly(nlimbs):
        return P.to_device(np.concatenate([rng.integers(0, P.primes[r], P.N, dtype=np.uint64) for r in range(nlimbs)]))

    key = [poly(P.k + P.kl) for _ in range(2)]
    c, m = [[poly(P.k) for _ in range(2)] for _ in range(2)]
    ref, batch_out = [P.zeros(P.k), P.zeros(P.k)], [P.zeros(P.k), P.zeros(P.k)]
    B = Batch()
    if kind == "mul":
        P.hommul(ref, c, m, key, level, P.workspace(level))
        B.add_mul(P, key, [(c, m, batch_out, level)])
        ops, n = [("mul",)], level * P.N
    else:
        P.rotate_left(ref, c, key, 2, level, P.workspace(level))
        B.add_rotate(P, [(c, batch_out, key, 2, level, False)])
        ops = [("rot", 2)]
    used = B.build()
    for short in (0, 1):
        srv = Server(pool_bytes=1 << 26, step_ws_bytes=used + 256 - short, max_active=4)
        ks = srv.register(P, key, {2: key})
        outs = [[P.zeros(P.k), P.zeros(P.k)] for _ in range(2)]
        args = [(ks, c, level, kind == "mul", m if kind == "mul" else None, ops, o) for o in outs]
        if short:
            with pytest.raises(AoaError):
                srv.submit(*args[0])
        else:
            ids = [srv.submit(*a) for a in args]
            for _ in range(8):
                srv.step()
            torch.cuda.synchronize()
            assert all(srv.result(i)[0] == Server.DONE for i in ids)
            for o in outs:
                for y in range(2):
                    assert (o[y][:n] == ref[y][:n]).all()
        srv.close()
