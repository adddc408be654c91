"""The work that a user of the CKKS key-switching core has it do, as cases to time.

An encrypted program spends its time in a few operations: products of two
ciphertexts (tensor, relinearization, rescale), rotations, products with
plaintexts, linear transforms (many rotations of one ciphertext against
plaintext diagonals), and the transforms of encoding and decoding. They run
from the level of a fresh ciphertext down to the last levels before a
bootstrap, one ciphertext at a time in a dependent chain (latency counts) or
many at once in a batched plan (throughput counts). The parameter sets are
the repository's: rns24_aux8 (24 primes, one per level, 8 auxiliary primes)
and bootparam_40 (levels of main and terminal primes, 12 auxiliary primes),
N = 2^16. Ciphertexts and evaluation keys are uniform residues, which is what
they are under encryption. All outputs are whole numbers.
"""
import functools
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cheddar-fhe_amd"))
import cheddar_amd as ck  # noqa: E402

N = 65536
PARAMS = {
    "rns24_aux8": os.path.join(ROOT, "cheddar-fhe_amd", "params", "rns24_aux8.json"),
    "bootparam_40": os.path.join(ROOT, "tests", "golden", "params", "bootparam_40.json"),
}


def listed():
    return [
        # the last product before a bootstrap: three limbs, launches and latency
        {"name": "hmult_low", "op": "hmult", "params": "rns24_aux8", "level": 2,
         "rescale": True},
        # a product of two fresh ciphertexts at 24 limbs
        {"name": "hmult_top", "op": "hmult", "params": "rns24_aux8", "level": 23,
         "rescale": True},
        # a product in a bootstrappable set, at a level whose rescale swaps
        # terminal primes for main ones (22 limbs -> 21)
        {"name": "hmult_boot40", "op": "hmult", "params": "bootparam_40", "level": 15,
         "rescale": True},
        # one rotation in the middle of a program, an odd number of limbs
        {"name": "hrot_mid", "op": "hrot", "params": "rns24_aux8", "level": 12},
        # a plaintext product, a plaintext sum and the rescale: a dense layer's step
        {"name": "ptmult", "op": "ptmult", "params": "rns24_aux8", "level": 18},
        # all rotations of one ciphertext that a convolution or a matrix
        # product with few diagonals takes
        {"name": "hoisted", "op": "hoisted", "params": "bootparam_40", "level": 12, "rots": 9},
        # one stage of the homomorphic DFT of a bootstrap at the top level:
        # baby steps, giant steps, one rescale
        {"name": "transform_boot40", "op": "transform", "params": "bootparam_40", "level": 28,
         "baby": 8, "giant": 4},
        # a server's batch of products at mixed levels
        {"name": "hmult_batch", "op": "hmult_plan", "params": "rns24_aux8", "items": 64, "low": 7,
         "high": 23},
        # a server's batch of hoisted rotations at mixed levels
        {"name": "hoisted_batch", "op": "hoisted_plan", "params": "rns24_aux8", "items": 8,
         "low": 7, "high": 23, "rots": 16},
        # encoding: one polynomial into the NTT domain in Montgomery form
        {"name": "ntt_single", "op": "ntt", "params": "rns24_aux8", "polys": 1, "main": 13,
         "aux": 0, "inverse": False},
        # encoding a batch of plaintexts for key-switched sums (all 32 primes)
        {"name": "ntt_batch", "op": "ntt", "params": "rns24_aux8", "polys": 64, "main": 24,
         "aux": 8, "inverse": False},
        # decoding a batch: back to coefficients, an odd number of limbs
        {"name": "intt_batch", "op": "ntt", "params": "rns24_aux8", "polys": 21, "main": 19,
         "aux": 0, "inverse": True},
    ]


def _log_int(rng, low, high):
    return min(high, int(low * math.exp(rng.random() * math.log((high + 1) / low))))


def draw(rng):
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = _draw(rng)
        if case not in known:
            return case


def _draw(rng):
    op = rng.choice(["hmult", "hmult", "hrot", "ptmult", "hoisted", "transform", "hmult_plan",
                     "hoisted_plan", "ntt", "ntt"])
    params = rng.choice(["rns24_aux8", "bootparam_40"])
    top = {"rns24_aux8": 23, "bootparam_40": 28}[params]
    if op in ("hmult", "hrot", "ptmult"):
        case = {"op": op, "params": params, "level": rng.randint(1, top)}
        if op == "hmult":
            case["rescale"] = rng.random() < 0.7
        return case
    if op == "hoisted":
        return {"op": op, "params": params, "level": rng.randint(1, top),
                "rots": rng.randint(2, 12)}
    if op == "transform":
        return {"op": op, "params": "bootparam_40", "level": rng.randint(4, 28),
                "baby": rng.randint(3, 8), "giant": rng.randint(2, 4)}
    if op in ("hmult_plan", "hoisted_plan"):
        low = rng.randint(2, 12)
        case = {"op": op, "params": "rns24_aux8", "items": _log_int(rng, 3, 60), "low": low,
                "high": rng.randint(low + 3, 23)}
        if op == "hoisted_plan":
            case["items"] = _log_int(rng, 1, 8)
            case["rots"] = rng.randint(2, 16)
        return case
    return {"op": "ntt", "params": "rns24_aux8", "polys": _log_int(rng, 1, 60),
            "main": rng.randint(2, 24), "aux": rng.choice([0, 8]),
            "inverse": rng.random() < 0.5}


# ---- what a program holds ----------------------------------------------------


@functools.lru_cache(maxsize=None)
def _context(params):
    """A program makes one context per parameter set and keeps it."""
    return ck.Context.from_json(PARAMS[params])


@functools.lru_cache(maxsize=None)
def _primes(params):
    """All primes in the library's order: terminal reversed, main, auxiliary."""
    d = ck.load_param_json(PARAMS[params])
    return tuple(d.get("terminal_primes", [])[::-1] + d["main_primes"] + d["auxiliary_primes"])


class _Draws:
    """Uniform residues from one seed."""

    def __init__(self, params, seed):
        self.params = params
        self.primes = _primes(params)
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def poly(self, pidx):
        t = torch.empty((len(pidx), N), dtype=torch.int32, device="cuda")
        for i, p in enumerate(pidx):
            t[i].random_(0, self.primes[p], generator=self.gen)
        return t

    def key(self, ctx):
        every = range(len(self.primes))
        return tuple([self.poly(every) for _ in range(ctx.dnum)] for _ in range(2))


def _level_primes(ctx, level):
    m, t = ctx.level_np(level)
    return list(range(ctx.max_ter - t, ctx.max_ter + m))


def _up_primes(ctx, level):
    return _level_primes(ctx, level) + list(range(ctx.L, ctx.L + ctx.alpha))


def _levels(case):
    """Mixed levels of a batch, the same for every seed."""
    rng = random.Random(case["items"] * 1000 + case["low"] * 50 + case["high"])
    return [rng.randint(case["low"], case["high"]) for _ in range(case["items"])]


def _rotations(case, seed):
    return sorted(random.Random(seed).sample(range(1, N // 2), case["rots"]))


def _empty(limbs):
    return torch.empty((limbs, N), dtype=torch.int32, device="cuda")


def _outputs(sizes):
    """One buffer for many output polynomials, and the polynomials in it."""
    whole = _empty(sum(sizes))
    return whole, list(torch.split(whole, sizes))


def prepare(case, seed):
    op = case["op"]
    ctx = _context(case["params"])
    d = _Draws(case["params"], seed)
    s = {"op": op, "ctx": ctx, "case": case, "seed": seed}
    if op in ("hmult", "hrot", "ptmult", "hoisted", "transform"):
        level = s["level"] = case["level"]
        q = _level_primes(ctx, level)
        s["np"] = ctx.level_np(level) + (0,)
        s["ct"] = [d.poly(q) for _ in range(2)]
    if op == "hmult":
        s["ct2"] = [d.poly(q) for _ in range(2)]
        s["key"] = d.key(ctx)
        s["to"] = level - 1 if case["rescale"] else level
        s["out"] = [_empty(ctx.num_q(s["to"])) for _ in range(2)]
    elif op == "hrot":
        s["rot"] = random.Random(seed).randrange(1, N // 2)
        s["key"] = d.key(ctx)
        s["out"] = [_empty(len(q)) for _ in range(2)]
    elif op == "ptmult":
        s["mul"], s["add"] = d.poly(q), d.poly(q)
        s["prod"] = [_empty(len(q)) for _ in range(2)]
        s["out"] = [_empty(ctx.num_q(level - 1)) for _ in range(2)]
    elif op == "hoisted":
        s["rots"] = _rotations(case, seed)
        s["keys"] = [d.key(ctx) for _ in s["rots"]]
        s["out"] = [[_empty(len(q)) for _ in range(2)] for _ in s["rots"]]
    elif op == "transform":
        nb, ng = case["baby"], case["giant"]
        up = _up_primes(ctx, level)
        rng = random.Random(seed)
        stride = rng.randrange(1, N // 2 // (nb * ng))
        s["baby_rots"] = [stride * b for b in range(1, nb)]
        s["giant_rots"] = [stride * nb * g for g in range(1, ng)]
        s["baby_keys"] = [d.key(ctx) for _ in s["baby_rots"]]
        s["giant_keys"] = [d.key(ctx) for _ in s["giant_rots"]]
        s["pts"] = [[d.poly(up) for _ in range(nb)] for _ in range(ng)]
        primes = _primes(case["params"])
        big_p = math.prod(primes[ctx.L:])
        s["p_const"] = torch.tensor([big_p * 2**32 % primes[p] for p in q], dtype=torch.int32,
                                    device="cuda")
        s["up"] = ctx.level_np(level) + (ctx.alpha,)
        s["baby"] = [[torch.zeros((len(up), N), dtype=torch.int32, device="cuda")
                      for _ in range(2)] for _ in range(nb)]
        s["accum"] = [[_empty(len(up)) for _ in range(2)] for _ in range(ng)]
        s["down"] = [_empty(len(q)) for _ in s["giant_rots"]]
        s["switched"] = [[_empty(len(up)) for _ in range(2)] for _ in s["giant_rots"]]
        s["out"] = [_empty(ctx.num_q(level - 1)) for _ in range(2)]
    elif op == "hmult_plan":
        levels = _levels(case)
        s["levels"] = levels
        s["cts"], s["ct2s"] = ([[d.poly(_level_primes(ctx, v)) for _ in range(2)]
                                for v in levels] for _ in range(2))
        s["key"] = d.key(ctx)
        sizes = [ctx.num_q(v - 1) for v in levels for _ in range(2)]
        s["out"], parts = _outputs(sizes)
        s["plan"] = ck.Plan.hmult(ctx, levels, list(zip(parts[::2], parts[1::2])), s["cts"],
                                  s["ct2s"], s["key"])
    elif op == "hoisted_plan":
        levels = _levels(case)
        s["levels"], s["rots"] = levels, _rotations(case, seed)
        s["cts"] = [[d.poly(_level_primes(ctx, v)) for _ in range(2)] for v in levels]
        s["keys"] = [d.key(ctx) for _ in s["rots"]]
        sizes = [ctx.num_q(v) for v in levels for _ in range(2 * len(s["rots"]))]
        s["out"], parts = _outputs(sizes)
        pairs = list(zip(parts[::2], parts[1::2]))
        k = len(s["rots"])
        s["plan"] = ck.Plan.hrot_hoisted(ctx, levels, s["cts"], s["keys"], s["rots"],
                                         [pairs[k * i:k * (i + 1)] for i in range(len(levels))])
    else:
        pidx = [ctx.max_ter + i for i in range(case["main"])]
        pidx += [ctx.L + i for i in range(case["aux"])]
        s["np"] = (case["main"], 0, case["aux"])
        s["src"] = [d.poly(pidx) for _ in range(case["polys"])]
        s["out"], parts = _outputs([len(pidx)] * case["polys"])
        if case["polys"] > 1:
            s["plan"] = ck.Plan.ntt(ctx, s["src"], parts, s["np"], inverse=case["inverse"],
                                    mont_conv=True)
    return s


def run(s):
    op, ctx = s["op"], s["ctx"]
    if "plan" in s:
        s["plan"].run()
    elif op == "hmult":
        ctx.hmult(s["out"], s["ct"], s["ct2"], s["key"], s["level"],
                  rescale=s["case"]["rescale"])
    elif op == "hrot":
        ctx.hrot(s["out"], s["ct"], s["key"], s["rot"], s["level"])
    elif op == "ptmult":
        ctx.mult(s["prod"], s["ct"], [s["mul"], s["mul"]], s["np"])
        ctx.add(s["prod"][:1], s["prod"][:1], [s["add"]], s["np"])
        ctx.rescale(s["out"], s["prod"], s["level"])
    elif op == "hoisted":
        ctx.hrot_hoisted(s["out"], s["ct"], s["keys"], s["rots"], s["level"])
    elif op == "transform":
        level, nq = s["level"], len(s["ct"][0])
        # baby steps in the raised basis; the unrotated one is P * ct
        ctx.hrot_hoisted(s["baby"][1:], s["ct"], s["baby_keys"], s["baby_rots"], level,
                         moddown=False)
        ctx.mult_const([v[:nq] for v in s["baby"][0]], s["ct"], s["p_const"], s["np"])
        ctx.gs_accum(s["accum"], s["baby"], s["pts"], s["up"])
        # each other giant step: its a part down, key switched and rotated
        ctx.moddown(s["down"], [v[1] for v in s["accum"][1:]], level, ck.CK_MODDOWN)
        for k, out in enumerate(s["switched"]):
            ctx.mult_key_no_moddown(out[0], out[1], s["down"][k], s["giant_keys"][k], level)
        srcs, rots = [], []
        for k, r in enumerate(s["giant_rots"]):
            srcs += [s["switched"][k], [s["accum"][k + 1][0], None]]
            rots += [r, r]
        ctx.permute_accum(s["accum"][0], srcs, rots, s["up"], accumulate=True)
        ctx.moddown(s["out"], s["accum"][0], level, ck.CK_MODDOWN_RESCALE)
    elif s["case"]["inverse"]:
        ctx.intt(s["out"], s["src"][0], *s["np"])
    else:
        ctx.ntt(s["out"], s["src"][0], *s["np"], mont_conv=True)
    return s["out"]


# ---- what a pass cannot do without -------------------------------------------


def work(case):
    """Inputs, keys and plaintexts read once and outputs written once; one
    operation per modular product or sum of the transforms, base conversions
    and products on the way."""
    op = case["op"]
    ctx = _context(case["params"])
    limb = 4 * N
    ntt = 3 * 16 * N // 2  # one transform of one limb

    def switch(level, polys=2):
        """ModUp, key products, and the ModDown of `polys` polynomials."""
        q, tot = ctx.num_q(level), ctx.num_q(level) + ctx.alpha
        beta = ctx.modup_beta(level)
        up = q * ntt + (beta * tot - q) * (ntt + 2 * ctx.alpha * N) + 4 * beta * tot * N
        return up + polys * (ctx.alpha * ntt + q * (ntt + 2 * ctx.alpha * N))

    def key_limbs(level):
        """the key limbs of the level's groups and primes, both halves"""
        return 2 * ctx.modup_beta(level) * (ctx.num_q(level) + ctx.alpha)

    limbs = ops = 0
    if op in ("hmult", "hrot", "ptmult", "hoisted", "transform"):
        q = ctx.num_q(case["level"])
        below = ctx.num_q(case["level"] - 1)
        tot = q + ctx.alpha
    if op == "hmult":
        limbs = 4 * q + key_limbs(case["level"]) + 2 * (below if case["rescale"] else q)
        ops = switch(case["level"]) + 5 * q * N
    elif op == "hrot":
        limbs, ops = 4 * q + key_limbs(case["level"]), switch(case["level"])
    elif op == "ptmult":
        limbs, ops = 4 * q + 2 * below, 3 * q * N + 2 * q * ntt
    elif op == "hoisted":
        r = case["rots"]
        limbs = 2 * q + r * (key_limbs(case["level"]) + 2 * q)
        ops = switch(case["level"], 0) + r * (switch(case["level"]) - switch(case["level"], 0))
    elif op == "transform":
        nb, ng = case["baby"], case["giant"]
        limbs = 2 * q + (nb + ng - 2) * key_limbs(case["level"]) + nb * ng * tot + 2 * below
        ops = switch(case["level"], 0) * ng + switch(case["level"], ng + 1) + 4 * nb * ng * tot * N
    elif op == "hmult_plan":
        levels = _levels(case)
        limbs = key_limbs(max(levels))
        for v in levels:
            limbs += 4 * ctx.num_q(v) + 2 * ctx.num_q(v - 1)
            ops += switch(v) + 5 * ctx.num_q(v) * N
    elif op == "hoisted_plan":
        levels, r = _levels(case), case["rots"]
        limbs = r * key_limbs(max(levels))
        for v in levels:
            limbs += 2 * ctx.num_q(v) * (1 + r)
            ops += switch(v, 0) + r * (switch(v) - switch(v, 0))
    else:
        count = case["polys"] * (case["main"] + case["aux"])
        limbs, ops = 2 * count, count * ntt
    return {"bytes": limbs * limb, "flops": ops}


# ---- the same results in 64-bit integers ---------------------------------------
# Stored NTT-domain values are x 2^32 mod q; output position k of a transform
# holds the value at psi^(2 brv(k) + 1), psi = g^((q - 1) / 2N) with g the
# smallest generator of the prime.


def _brv(bits):
    i = torch.arange(1 << bits)
    r = torch.zeros_like(i)
    for b in range(bits):
        r |= ((i >> b) & 1) << (bits - 1 - b)
    return r


@functools.lru_cache(maxsize=None)
def _psi(q):
    m, factors, f = q - 1, [], 2
    while f * f <= m:
        if m % f == 0:
            factors.append(f)
            while m % f == 0:
                m //= f
        f += 1
    factors += [m] if m > 1 else []
    g = next(g for g in range(2, q) if all(pow(g, (q - 1) // f, q) != 1 for f in factors))
    return pow(g, (q - 1) // (2 * N), q)


@functools.lru_cache(maxsize=None)
def _powers(q, inverse):
    """psi^brv(j) (or its inverse), j < N, on the GPU."""
    base = pow(_psi(q), -1, q) if inverse else _psi(q)
    p = torch.ones(1, dtype=torch.int64, device="cuda")
    step = base
    for _ in range(16):
        p = torch.cat([p, p * step % q])
        step = step * step % q
    return p[_brv(16).to("cuda")]


class _Exact:
    """Polynomials as int64 [limbs, N] over the primes `pidx` of a context."""

    def __init__(self, case):
        self.ctx = _context(case["params"])
        self.primes = _primes(case["params"])

    def mod(self, pidx):
        return torch.tensor([self.primes[p] for p in pidx], device="cuda")[:, None]

    def consts(self, pidx, f):
        """f(q) mod q for each prime"""
        return torch.tensor([f(self.primes[p]) % self.primes[p] for p in pidx],
                            device="cuda")[:, None]

    def mont(self, x, y, pidx):
        """x y 2^-32"""
        m = self.mod(pidx)
        return x * y % m * self.consts(pidx, lambda q: pow(2**32, -1, q)) % m

    def ntt(self, x, pidx):
        w = torch.stack([_powers(self.primes[p], False) for p in pidx])
        m, k = self.mod(pidx)[:, :, None, None], 1
        x = x.reshape(len(pidx), 1, 1, N)
        while k < N:
            x = x.reshape(len(pidx), k, 2, N // k // 2)
            a, b = x[:, :, :1], x[:, :, 1:] * w[:, k:2 * k, None, None] % m
            x = torch.cat([(a + b) % m, (a - b) % m], 2)
            k *= 2
        return x.reshape(len(pidx), N)

    def intt(self, x, pidx):
        w = torch.stack([_powers(self.primes[p], True) for p in pidx])
        m, k = self.mod(pidx)[:, :, None, None], N // 2
        while k:
            x = x.reshape(len(pidx), k, 2, N // k // 2)
            a, b = x[:, :, :1], x[:, :, 1:]
            x = torch.cat([(a + b) % m, (a - b) % m * w[:, k:2 * k, None, None] % m], 2)
            k //= 2
        inv = self.consts(pidx, lambda q: pow(N, -1, q))
        return x.reshape(len(pidx), N) * inv % self.mod(pidx)

    def base_conv(self, x, src, dst, scale=1):
        """NTT-domain limbs x of `src` to NTT-domain limbs of `dst`: the sum of
        centred [x_i scale (S / s_i)^-1]_{s_i} (S / s_i), not reduced mod S."""
        big = math.prod(self.primes[p] for p in src)
        r = 2**32
        c = self.consts(src, lambda q: scale * pow(big // q * r, -1, q))
        v = self.intt(x, src) * c % self.mod(src)
        v = torch.where(v > self.mod(src) // 2, v - self.mod(src), v)
        m = self.mod(dst)
        out = torch.zeros((len(dst), N), dtype=torch.int64, device="cuda")
        for i, p in enumerate(src):
            out = (out + v[i] * self.consts(dst, lambda q: big // self.primes[p] * r) % m) % m
        return self.ntt(out, dst)

    def switch(self, x, level, key, rows=None):
        """sum over the ModUp groups of x of their raised limbs times the key"""
        raised = self.raise_groups(x, level) if rows is None else rows
        up = _up_primes(self.ctx, level)
        out = []
        for half in key:
            acc = 0
            for g, limbs in raised:
                acc = acc + self.mont(limbs, half[g].long()[up], up)
            out.append(acc % self.mod(up))
        return out

    def raise_groups(self, x, level):
        q, up = _level_primes(self.ctx, level), _up_primes(self.ctx, level)
        a, first = self.ctx.alpha, self.ctx.max_ter - self.ctx.level_np(level)[1]
        raised = []
        for g in range(self.ctx.modup_beta(level)):
            own = [p for p in q if g * a <= p < (g + 1) * a]
            if not own:
                continue
            rest = [p for p in up if p not in own]
            conv = self.base_conv(x[[p - first for p in own]], own, rest)
            limbs = torch.empty((len(up), N), dtype=torch.int64, device="cuda")
            limbs[[up.index(p) for p in own]] = x[[p - first for p in own]]
            limbs[[up.index(p) for p in rest]] = conv
            raised.append((g, limbs))
        return raised

    def times_p(self, x, level):
        """P x in the raised basis: zero on the auxiliary limbs"""
        q = _level_primes(self.ctx, level)
        big = math.prod(self.primes[self.ctx.L:])
        up = x * self.consts(q, lambda m: big) % self.mod(q)
        return torch.cat([up, torch.zeros_like(up[:1]).expand(self.ctx.alpha, N)])

    def down(self, x, level, to, aux=True):
        """x over the level's primes (and the auxiliary ones) divided by the
        primes that level `to` does not have; primes that only `to` has are
        multiplied in first."""
        have = _up_primes(self.ctx, level) if aux else _level_primes(self.ctx, level)
        want = _level_primes(self.ctx, to)
        gone = [p for p in have if p not in want]
        new = math.prod(self.primes[p] for p in want if p not in have)
        conv = self.base_conv(x[[have.index(p) for p in gone]], gone, want, new)
        kept = torch.zeros_like(conv)
        for i, p in enumerate(want):
            if p in have:
                kept[i] = x[have.index(p)] * (new % self.primes[p]) % self.primes[p]
        big = math.prod(self.primes[p] for p in gone)
        m = self.mod(want)
        return (kept - conv) % m * self.consts(want, lambda q: pow(big, -1, q)) % m

    def rotate(self, x, rot):
        k = _brv(16)
        at = ((2 * k + 1) * pow(5, rot, 2 * N) % (2 * N) - 1) // 2
        return x[:, k[at].to("cuda")]


def exact(case, seed):
    def whole(v):
        return [whole(x) for x in v] if isinstance(v, list) else v.int()

    return whole(_exact_of(_Exact(case), prepare(case, seed)))


def _exact_hmult(e, ct, ct2, key, level, to):
    q, up = _level_primes(e.ctx, level), _up_primes(e.ctx, level)
    (b1, a1), (b2, a2) = [v.long() for v in ct], [v.long() for v in ct2]
    d = [e.mont(b1, b2, q), (e.mont(b1, a2, q) + e.mont(a1, b2, q)) % e.mod(q),
         e.mont(a1, a2, q)]
    acc = e.switch(d[2], level, key)
    return [e.down((acc[j] + e.times_p(d[j], level)) % e.mod(up), level, to)
            for j in range(2)]


def _exact_rotated(e, ct, rots, keys, level, down=True):
    up = _up_primes(e.ctx, level)
    b, a = (v.long() for v in ct)
    rows = e.raise_groups(a, level)
    for rot, key in zip(rots, keys):
        kb, ka = e.switch(a, level, key, rows)
        pair = [(kb + e.times_p(b, level)) % e.mod(up), ka]
        yield [e.rotate(e.down(v, level, level) if down else v, rot) for v in pair]


def _exact_of(e, s):
    op = s["op"]
    if op == "hmult":
        return _exact_hmult(e, s["ct"], s["ct2"], s["key"], s["level"], s["to"])
    if op == "hrot":
        return next(_exact_rotated(e, s["ct"], [s["rot"]], [s["key"]], s["level"]))
    if op == "ptmult":
        level, q = s["level"], _level_primes(e.ctx, s["level"])
        b, a = (e.mont(v.long(), s["mul"].long(), q) for v in s["ct"])
        return [e.down(v, level, level - 1, False) for v in ((b + s["add"].long()) % e.mod(q), a)]
    if op == "hoisted":
        return list(_exact_rotated(e, s["ct"], s["rots"], s["keys"], s["level"]))
    if op == "transform":
        level, up = s["level"], _up_primes(e.ctx, s["level"])
        baby = [[e.times_p(v.long(), level) for v in s["ct"]]]
        baby += _exact_rotated(e, s["ct"], s["baby_rots"], s["baby_keys"], level, False)
        total = None
        for g, rot in enumerate([0] + s["giant_rots"]):
            acc = [sum(e.mont(x[j], pt.long(), up) for x, pt in zip(baby, s["pts"][g])) % e.mod(up)
                   for j in range(2)]
            if g:
                kb, ka = e.switch(e.down(acc[1], level, level), level, s["giant_keys"][g - 1])
                acc = [e.rotate(acc[0] + kb, rot), e.rotate(ka, rot)]
            total = acc if total is None else [(t + v) % e.mod(up) for t, v in zip(total, acc)]
        return [e.down(v, level, level - 1) for v in total]
    if op == "hmult_plan":
        rows = [_exact_hmult(e, s["cts"][i], s["ct2s"][i], s["key"], v, v - 1)
                for i, v in enumerate(s["levels"])]
        return torch.cat([v for pair in rows for v in pair])
    if op == "hoisted_plan":
        return torch.cat([v for i, level in enumerate(s["levels"])
                          for pair in _exact_rotated(e, s["cts"][i], s["rots"], s["keys"], level)
                          for v in pair])
    pidx = [e.ctx.max_ter + i for i in range(s["np"][0])]
    pidx += [e.ctx.L + i for i in range(s["np"][2])]
    r = e.consts(pidx, lambda q: 2**32)
    outs = []
    for x in s["src"]:
        if s["case"]["inverse"]:
            plain = x.long() * e.consts(pidx, lambda q: pow(2**32, -1, q)) % e.mod(pidx)
            outs.append(e.intt(plain, pidx))
        else:
            outs.append(e.ntt(x.long() * r % e.mod(pidx), pidx))
    return torch.cat(outs)
