"""GPU parity of the one-pass int8 transforms at the edges of their rule:
the smallest batch that takes them, whole rounds of 256 limbs, a short last
round (two vector passes: 1, 5, 64, 65 and 127 limbs, both sides of the column
kernels' lines) and a long one (128), both directions, both Montgomery
options, primes of 20 to 31 bits, the residues 0, q - 1, (q - 1) / 2 and
(q + 1) / 2 in every limb. Whole numbers: every word equals the oracle's."""
import numpy as np
import pytest

from conftest import SEED_BASE, load_params
from gpu_util import assert_same, uniform

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("params,np3,polys,launches",
                         [("rns24_aux8.json", (24, 0, 8), 6, 1),
                          ("rns24_aux8.json", (16, 0, 0), 16, 1),
                          ("rns24_aux8.json", (1, 0, 0), 257, 3),
                          ("rns24_aux8.json", (9, 0, 0), 29, 3),
                          ("rns24_aux8.json", (24, 0, 8), 10, 3),
                          ("rns24_aux8.json", (3, 0, 0), 107, 3),
                          ("rns24_aux8.json", (1, 0, 0), 383, 3),
                          ("rns24_aux8.json", (24, 0, 8), 12, 1),
                          ("rns24_aux8.json", (17, 0, 0), 11, 2),
                          ("bootparam_40.json", (43, 4, 12), 4, 1),
                          ("bootparam_30.json", (48, 0, 12), 4, 1)])
@pytest.mark.parametrize("inverse,mont", [(False, False), (False, True), (True, True),
                                          (True, False)])
def test_one_pass(params, np3, polys, launches, inverse, mont):
    import cheddar_amd as ck
    import ckks_oracle as O
    d = load_params(params)
    ctx, P = ck.Context.from_json(d), O.Param.from_json(d)
    O.set_threads(8)
    pidx = P.np_primes(*np3)
    kinds = min(polys, 5)  # distinct polynomials, repeated over the batch
    xs = []
    for k in range(kinds):
        x = uniform(P, pidx, SEED_BASE + 5500 + k)
        for i, p in enumerate(pidx):
            q = P.prime(p)
            x[i, :4] = x[i, -4:] = (0, q - 1, (q - 1) // 2, (q + 1) // 2)
        xs.append(x)
    xs[-1][:] = np.array([P.prime(p) - 1 for p in pidx], np.uint32)[:, None]
    fn = P.intt_np if inverse else P.ntt_np
    want = [fn(x, *np3, mont_conv=mont) for x in xs]
    src = [ck.to_device(xs[k % kinds]) for k in range(polys)]
    dst = [torch.full_like(s, -1) for s in src]
    plan = ck.Plan.ntt(ctx, src, dst, np3, inverse=inverse, mont_conv=mont)
    limbs = polys * sum(np3)
    # 187 limbs: below the rule, two vector passes
    assert plan.info()["launches"] == launches, limbs
    plan.run()
    torch.cuda.synchronize()
    for k in range(polys):
        assert_same(ck.to_host(dst[k]), want[k % kinds], f"poly {k}")


@pytest.mark.parametrize("options,launches", [({}, 1), ({"ntt8_blocks": 16}, 2),
                                              ({"ntt8_blocks": 4}, 2),
                                              ({"ntt8_chunk": 512}, 4), ({"ntt8_chunk": 0}, 1)])
def test_two_pass_form_by_option(rns24, oracle_rns24, options, launches):
    """1024 limbs (several workgroup rounds): every explicit shape, 16 blocks
    too, takes the two-pass int8 form"""
    import cheddar_amd as ck
    P, np3, polys = oracle_rns24, (24, 0, 8), 32
    ctx = ck.Context.from_json(rns24)
    ctx.set_plan_forms(ntt="int8", **options)
    xs = [uniform(P, P.np_primes(*np3), SEED_BASE + 5700 + k) for k in range(3)]
    want = [P.ntt_np(x, *np3, mont_conv=True) for x in xs]
    src = [ck.to_device(xs[k % 3]) for k in range(polys)]
    dst = [torch.full_like(s, -1) for s in src]
    plan = ck.Plan.ntt(ctx, src, dst, np3, inverse=False, mont_conv=True)
    assert plan.info()["launches"] == launches and plan.info()["form"] == 1
    plan.run()
    torch.cuda.synchronize()
    for k in range(polys):
        assert_same(ck.to_host(dst[k]), want[k % 3], f"poly {k}")


@pytest.mark.parametrize("np3,polys,form", [((2, 0, 0), 1, 0), ((24, 0, 0), 1, 0),
                                            ((13, 0, 8), 9, 0), ((1, 0, 0), 191, 0),
                                            ((24, 0, 8), 6, 1)])
def test_forward_form_by_size(rns24, oracle_rns24, np3, polys, form):
    """nothing set: two vector passes below 192 limbs, one int8 pass from
    there; the form asked for at every size"""
    import cheddar_amd as ck
    P = oracle_rns24
    xs = [uniform(P, P.np_primes(*np3), SEED_BASE + 5800 + k) for k in range(min(polys, 3))]
    want = [P.ntt_np(x, *np3, mont_conv=True) for x in xs]
    src = [ck.to_device(xs[k % 3]) for k in range(polys)]
    for asked, got in ((None, form), ("int8", 1), ("valu", 0)):
        ctx = ck.Context.from_json(rns24)
        ctx.set_plan_forms(ntt=asked)
        dst = [torch.full_like(s, -1) for s in src]
        plan = ck.Plan.ntt(ctx, src, dst, np3, inverse=False, mont_conv=True)
        assert plan.info()["form"] == got and plan.info()["launches"] == (1 if got and form else 2)
        plan.run()
        torch.cuda.synchronize()
        for k in range(polys):
            assert_same(ck.to_host(dst[k]), want[k % 3], f"{asked}, poly {k}")


def test_plans_created_by_several_threads(rns24, oracle_rns24):
    """a fresh context's first plans, forward and inverse, from four threads at
    once: the tables they share are built once"""
    import threading

    import cheddar_amd as ck
    P, np3, polys = oracle_rns24, (24, 0, 8), 6
    ctx = ck.Context.from_json(rns24)
    x = uniform(P, P.np_primes(*np3), SEED_BASE + 5900)
    src = [ck.to_device(x) for _ in range(polys)]
    dst = [[torch.full_like(s, -1) for s in src] for _ in range(4)]
    plans, errors, start = [None] * 4, [], threading.Barrier(4)

    def build(i):
        try:
            start.wait()
            plans[i] = ck.Plan.ntt(ctx, src, dst[i], np3, inverse=bool(i & 1), mont_conv=True)
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=build, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for p in plans:
        assert p.info()["launches"] == 1
        p.run()
    torch.cuda.synchronize()
    for i in range(4):
        want = (P.intt_np if i & 1 else P.ntt_np)(x, *np3, mont_conv=True)
        for k in range(polys):
            assert_same(ck.to_host(dst[i][k]), want, f"thread {i} poly {k}")
