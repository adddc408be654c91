"""GPU parity of the hoisted baby steps (one pass per row of 256 words,
products summed in 64 bits) at the edges: 1 to 8 key groups, a number of limbs that is no multiple of the
launch's window of eight, one rotation, eight and nine (two launches), the
smallest and largest rotation, single calls and a batched plan.
Whole numbers: every word equals the oracle's."""
import numpy as np
import pytest

from conftest import SEED_BASE
from gpu_util import assert_same, dev_key, full_key, uniform

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("main,aux,rots", [(3, 3, [1]), (7, 4, [32767, 2]), (9, 3, [5]),
                                           (8, 2, [1, 32767, 16384]), (10, 2, [9, 77]),
                                           (4, 2, [1, 2, 3, 5, 8, 13, 21, 34, 55]),
                                           (6, 1, [32767, 12]), (13, 2, [3]),
                                           (8, 1, [1, 16384, 30])])
def test_baby_steps(rns24, main, aux, rots):
    import cheddar_amd as ck
    import ckks_oracle as O
    primes = rns24["main_primes"] + rns24["auxiliary_primes"]
    args = (16, primes[:main], primes[main:main + aux])
    ctx, P = ck.Context(*args), O.Param(*args)
    level = main - 1
    ct = [uniform(P, P.level_primes(level), SEED_BASE + 5200 + j) for j in range(2)]
    # keys of the largest residues too: the 64-bit sums at their bounds
    keys = [full_key(P, SEED_BASE + 5300 + 50 * i) for i in range(len(rots))]
    top = np.array([P.prime(i) - 1 for i in range(P.num_primes)], np.uint32)[:, None]
    keys[0][0][:, :, :4096] = top[None]
    ct[1][:, :4096] = top[[int(p) for p in P.level_primes(level)]]
    outs = [[torch.empty((main + aux, P.n), dtype=torch.int32, device="cuda")
             for _ in range(2)] for _ in rots]
    ctx.hrot_hoisted(outs, [ck.to_device(v) for v in ct], [dev_key(*k) for k in keys], rots,
                     level, moddown=False)
    torch.cuda.synchronize()
    for i, r in enumerate(rots):
        want = P.hoisted_baby_step(level, ct, keys[i], r)
        for j in range(2):
            assert_same(ck.to_host(outs[i][j]), want[j], f"baby step {r} poly {j}")
    # the same rotations as a batched plan of two items
    items = [[[torch.full_like(o, -1) for o in pair] for pair in outs] for _ in range(2)]
    d_ct = [ck.to_device(v) for v in ct]
    ck.Plan.hrot_hoisted(ctx, [level, level], [d_ct, d_ct], [dev_key(*k) for k in keys], rots,
                         items, moddown=False).run()
    torch.cuda.synchronize()
    for item in items:
        for i in range(len(rots)):
            for j in range(2):
                assert torch.equal(item[i][j], outs[i][j]), (i, j)
