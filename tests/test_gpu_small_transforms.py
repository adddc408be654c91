"""GPU parity of the two-pass transforms at the edges of the column kernels'
rule: four columns a workgroup (to 4 limbs), eight (to 64, inverse to 40), 16
values a thread above; single calls and plans, both directions, both Montgomery
options, in place and not, primes of 20 to 31 bits, the residues 0, q - 1, (q - 1) / 2 and (q + 1) / 2
in every limb. Whole numbers: every word equals the oracle's."""
import pytest

from conftest import SEED_BASE, load_params
from gpu_util import assert_same, uniform

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _inputs(P, pidx, count):
    xs = []
    for k in range(count):
        x = uniform(P, pidx, SEED_BASE + 6100 + k)
        for i, p in enumerate(pidx):
            q = P.prime(p)
            x[i, :4] = x[i, -4:] = (0, q - 1, (q - 1) // 2, (q + 1) // 2)
            x[i, 256:512] = q - 1
        xs.append(x)
    return xs


@pytest.mark.parametrize("inverse,mont", [(False, False), (False, True), (True, False),
                                          (True, True)])
@pytest.mark.parametrize("params,np3,polys",
                         [("rns24_aux8.json", (1, 0, 0), 1),
                          ("bootparam_40.json", (1, 1, 2), 1),
                          ("bootparam_30.json", (3, 0, 2), 1),
                          ("rns24_aux8.json", (24, 0, 8), 1),
                          ("bootparam_40.json", (43, 4, 12), 1),
                          ("rns24_aux8.json", (1, 0, 0), 4),
                          ("bootparam_30.json", (5, 0, 0), 1),
                          ("rns24_aux8.json", (24, 0, 8), 2),
                          ("bootparam_30.json", (40, 0, 0), 1),
                          ("bootparam_30.json", (41, 0, 0), 1),
                          ("rns24_aux8.json", (5, 0, 8), 5)])
def test_small_transform(params, np3, polys, inverse, mont):
    import cheddar_amd as ck
    import ckks_oracle as O
    d = load_params(params)
    ctx, P = ck.Context.from_json(d), O.Param.from_json(d)
    O.set_threads(8)
    xs = _inputs(P, P.np_primes(*np3), polys)
    fn = P.intt_np if inverse else P.ntt_np
    want = [fn(x, *np3, mont_conv=mont) for x in xs]
    src = [ck.to_device(x) for x in xs]
    dst = [torch.full_like(s, -1) for s in src]
    ctx.set_plan_forms(ntt="valu")
    plan = ck.Plan.ntt(ctx, src, dst, np3, inverse=inverse, mont_conv=mont)
    assert plan.info()["form"] == 0 and plan.info()["launches"] == 2
    plan.run()
    torch.cuda.synchronize()
    for k in range(polys):
        assert_same(ck.to_host(dst[k]), want[k], f"plan, poly {k}")
    call = ctx.intt if inverse else ctx.ntt
    for k in range(polys):
        call(dst[k], src[k], *np3, mont_conv=mont)
        call(src[k], src[k], *np3, mont_conv=mont)
    torch.cuda.synchronize()
    for k in range(polys):
        assert_same(ck.to_host(dst[k]), want[k], f"call, poly {k}")
        assert_same(ck.to_host(src[k]), want[k], f"call in place, poly {k}")


@pytest.mark.parametrize("inverse,mont", [(False, False), (False, True), (True, False),
                                          (True, True)])
@pytest.mark.parametrize("params,np3,polys",
                         [("rns24_aux8.json", (1, 0, 0), 88), ("rns24_aux8.json", (1, 0, 0), 89),
                          ("rns24_aux8.json", (24, 0, 8), 11), ("bootparam_40.json", (43, 4, 12), 6),
                          ("rns24_aux8.json", (1, 0, 0), 353)])
def test_many_limbs(params, np3, polys, inverse, mont):
    """both sides of the row kernels' lines (88 limbs inverse, 352 forward), in
    place and not: 16 values a thread above, 16 rows a workgroup"""
    import cheddar_amd as ck
    import ckks_oracle as O
    d = load_params(params)
    ctx, P = ck.Context.from_json(d), O.Param.from_json(d)
    O.set_threads(8)
    ctx.set_plan_forms(ntt="valu")
    kinds = min(polys, 5)
    xs = _inputs(P, P.np_primes(*np3), kinds)
    fn = P.intt_np if inverse else P.ntt_np
    want = [fn(x, *np3, mont_conv=mont) for x in xs]
    src = [ck.to_device(xs[k % kinds]) for k in range(polys)]
    dst = [torch.full_like(s, -1) for s in src]
    for out in (dst, src):
        plan = ck.Plan.ntt(ctx, src, out, np3, inverse=inverse, mont_conv=mont)
        assert plan.info()["form"] == 0
        plan.run()
        torch.cuda.synchronize()
        for k in range(polys):
            assert_same(ck.to_host(out[k]), want[k % kinds], f"poly {k}")
