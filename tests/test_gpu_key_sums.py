"""GPU parity of the key inner product's 64-bit sums at the edges: one to
five key groups (an even and an odd number of products between folds), with
and without the P fold, on random residues and on the largest ones. Whole
numbers: every word equals the oracle's."""
import numpy as np
import pytest

from conftest import SEED_BASE
from gpu_util import assert_same, dev_key, full_key, uniform

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("main,aux", [(3, 3), (7, 4), (9, 3), (8, 2), (10, 2)])
@pytest.mark.parametrize("largest", [False, True])
def test_key_products(rns24, main, aux, largest):
    import cheddar_amd as ck
    import ckks_oracle as O
    primes = rns24["main_primes"] + rns24["auxiliary_primes"]
    args = (16, primes[:main], primes[main:main + aux])
    ctx, P = ck.Context(*args), O.Param(*args)
    level = main - 1
    pidx = list(P.level_primes(level))
    top = np.array([P.prime(i) - 1 for i in range(P.num_primes)], np.uint32)[:, None]

    def poly(seed):
        v = uniform(P, pidx, SEED_BASE + seed)
        return np.broadcast_to(top[pidx], v.shape).copy() if largest else v

    x, add_b, add_a, b2 = (poly(5400 + i) for i in range(4))
    kb, ka = full_key(P, SEED_BASE + 5410)
    if largest:
        kb[:] = top[None]
        ka[:] = top[None]
    dx, db, da, d2 = (ck.to_device(v) for v in (x, add_b, add_a, b2))
    key = dev_key(kb, ka)
    out = [torch.empty((main + aux, P.n), dtype=torch.int32, device="cuda") for _ in range(2)]
    for ab, aa, hb, ha in ((None, None, None, None), (db, da, add_b, add_a),
                           (db, None, add_b, None)):
        ctx.mult_key_no_moddown(out[0], out[1], dx, key, level, ab, aa)
        torch.cuda.synchronize()
        want = P.mult_key_no_moddown(level, x, kb, ka, hb, ha)
        for j in range(2):
            assert_same(ck.to_host(out[j]), want[j], f"key product poly {j}")
    res = [torch.empty((main - 1, P.n), dtype=torch.int32, device="cuda") for _ in range(2)]
    ctx.hmult(res, [db, dx], [d2, da], key, level)
    torch.cuda.synchronize()
    want = P.hmult(level, [add_b, x], [b2, add_a], (kb, ka), rescale=True)
    for j in range(2):
        assert_same(ck.to_host(res[j]), want[j], f"hmult poly {j}")
