"""GPU parity of the BaseConv fused with the forward column stages at the
edges of its forms: 1 to 24 sources (every count of sources per lane group
and k-step), destination counts with every remainder of four, launches of
few and of many quads. Whole numbers: every word equals the oracle's."""
import pytest

from conftest import SEED_BASE
from gpu_util import assert_same, uniform

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("main,aux", [(5, 1), (6, 4), (7, 5), (9, 8), (10, 9), (13, 12),
                                      (15, 13), (16, 16), (15, 17), (9, 23), (23, 9)])
def test_modup_and_moddown(rns24, main, aux):
    import cheddar_amd as ck
    import ckks_oracle as O
    primes = rns24["main_primes"] + rns24["auxiliary_primes"]
    args = (16, primes[:main], primes[main:main + aux])
    ctx, P = ck.Context(*args), O.Param(*args)
    level = main - 1
    for lv in (level, 2):
        x = uniform(P, P.level_primes(lv), SEED_BASE + 5000 + main)
        beta, tot = ctx.modup_beta(lv), ctx.num_q(lv) + aux
        out = torch.zeros((beta * tot, P.n), dtype=torch.int32, device="cuda")
        ctx.modup(out, ck.to_device(x), lv)
        torch.cuda.synchronize()
        assert_same(ck.to_host(out).reshape(beta, tot, P.n), P.modup(x, lv), f"modup {lv}")
    for kind, drop in ((ck.CK_MODDOWN, 0), (ck.CK_MODDOWN_RESCALE, 1)):
        y = uniform(P, P.level_primes(level, with_aux=True), SEED_BASE + 5100 + main)
        out = torch.empty((ctx.num_q(level - drop), P.n), dtype=torch.int32, device="cuda")
        ctx.moddown([out], [ck.to_device(y)], level, kind)
        torch.cuda.synchronize()
        assert_same(ck.to_host(out), P.moddown(y, level, kind), f"moddown kind {kind}")
