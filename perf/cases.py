"""Performance cases of the photon walk through its public entry points.

Each case is one call a program makes: a single run (heat and heat2, or the
raw integer tallies), a batch of parameter sets, or a burst of requests to a
server.  ``listed()`` names the fixed cases, ``draw(rng)`` gives others of the
same ranges, ``prepare`` makes what the program holds before the call,
``run`` makes the call, ``work`` counts what it cannot do without and
``exact`` walks the same photons in binary64 with numpy.
"""
import math

import numpy as np

import tiny_mc_amd as tmc
from tiny_mc_amd import serve_load

# Physics the tests, the benchmark and the precision study use.
PHYSICS = {
    "default": dict(mu_a=2.0, mu_s=20.0, shells=101, microns_per_shell=50.0),  # params.h
    "lowalb": dict(mu_a=10.0, mu_s=10.0, shells=51, microns_per_shell=100.0),  # albedo 0.5
    "highalb": dict(mu_a=0.5, mu_s=50.0, shells=201, microns_per_shell=20.0),  # albedo 0.99
    "stress": dict(mu_a=0.01, mu_s=100.0, shells=401, microns_per_shell=10.0),  # albedo 0.9999
}

FLOP_PER_ABSORPTION = 40.5  # binary32 operations of one pass of photon()'s loop

# Absorptions of the largest drawn case (the largest listed ones have more).
DRAWN_MAX = 2.0e10
# The variants that walk slower get a smaller share of it.
DRAWN_MAX_FP64 = 4.0e9

_server = None  # a program keeps one server open for all its requests


def _case(name, kind, physics="default", photons=0, **kw):
    c = {"name": name, "kind": kind}
    if physics:
        c.update(PHYSICS[physics])
    if photons:
        c["photons"] = photons
    c.update(kw)
    return c


def listed():
    return [
        # one frame of the viewer: 20 photons continuing a stream (cg_mc.c)
        _case("viewer_frame", "raw", photons=20, frames=True),
        # the reference program as shipped: 32,768 photons, heat and heat2
        _case("reference_32768", "run", photons=32768),
        # a small high-albedo run, as the statistical tests make by the hundred
        _case("highalb_4096", "run", "highalb", photons=4096),
        # an ordinary run of an odd size
        _case("ordinary_3000017", "raw", photons=3000017),
        # the benchmark's step
        _case("large_2e30", "raw", photons=1 << 30),
        # short walks: photons end every ten absorptions or so
        _case("albedo05_2e27", "raw", "lowalb", photons=1 << 27),
        # the reference's own direction sampler, ragged size
        _case("rejection_2e24", "raw", photons=(1 << 24) + 3, sampler=tmc.SAMPLER_REJECTION),
        # the precision study's physics in binary32: walks of 70,000 absorptions
        _case("stress_2e17", "raw", "stress", photons=1 << 17),
        # the study's reference arithmetic
        _case("fp64_2e20", "raw", photons=1 << 20, precision=tmc.PRECISION_FP64),
        # a one-off batch of small sets: plan, run and release in one call
        _case("batch_once_64", "batch", None, sets=64, mix=1, scale=0.02, plan=False),
        # a sweep whose plan is kept and replayed
        _case("sweep_512", "batch", None, sets=512, mix=0, scale=0.125, plan=True),
        # a burst of requests to a resident server
        _case("serve_burst_384", "serve", None, requests=384, mix=3),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_physics(rng):
    r = rng.random()
    if r < 0.35:
        return dict(PHYSICS["default"])
    if r < 0.6:
        return dict(PHYSICS[rng.choice(["lowalb", "highalb", "stress"])])
    # the sweep's ranges
    return dict(mu_a=round(math.exp(rng.uniform(math.log(0.05), math.log(10.0))), 4),
                mu_s=round(math.exp(rng.uniform(math.log(10.0), math.log(200.0))), 3),
                shells=rng.choice([51, 101, 201, 401]),
                microns_per_shell=round(rng.uniform(10.0, 100.0), 2))


def draw(rng):
    kind = rng.choice(["run", "raw", "raw", "raw", "raw", "batch", "batch", "serve"])
    if kind == "serve":
        return {"kind": kind, "requests": _log_int(rng, 16, 256), "mix": rng.randrange(1000)}
    if kind == "batch":
        c = {"kind": kind, "sets": _log_int(rng, 8, 256), "mix": rng.randrange(1000),
             "scale": round(math.exp(rng.uniform(math.log(0.003), math.log(0.1))), 4), "plan": rng.random() < 0.7}
        while _absorptions(c) > DRAWN_MAX:
            c["scale"] = round(c["scale"] / 2, 5)
        return c
    c = {"kind": kind, **_draw_physics(rng)}
    if kind == "raw":
        r = rng.random()
        if r < 0.25:
            c["sampler"] = tmc.SAMPLER_REJECTION
        elif r < 0.4:
            c["precision"] = rng.choice([tmc.PRECISION_FP32_WEIGHT, tmc.PRECISION_FP32_COMPENSATED,
                                         tmc.PRECISION_FP64])
        if r < 0.1 or 0.4 <= r < 0.55:
            c["math"] = tmc.MATH_OWN
        if rng.random() < 0.25:
            c["wide_seed"] = True  # a seed beyond 32 bits
    most = (DRAWN_MAX_FP64 if c.get("precision") else DRAWN_MAX) / _per_photon(c)
    c["photons"] = _log_int(rng, 20, max(64, min(1 << 28, int(most))))
    return c


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------


def _seed(case, seed):
    s = 7919 * seed + 12345
    return s + ((2 * (seed % 1000) + 1) << 40) if case.get("wide_seed") else s


def _params(case):
    return tmc.Params(case["mu_a"], case["mu_s"], case["shells"], case["microns_per_shell"], case["photons"])


def _sets(case, seed):
    """The sets of a batch: the case's physics and budgets, seeds of `seed`."""
    sets = tmc.sweep_sets(case["sets"], seed=case["mix"], photon_scale=case["scale"])
    return [(p, _seed(case, seed) + i) for i, (p, _) in enumerate(sets)]


def _requests(case, seed):
    reqs = serve_load.draw_requests(case["requests"], seed=case["mix"])
    return [(p, _seed(case, seed) + i) for i, (p, _) in enumerate(reqs)]


def _open_server():
    global _server
    if _server is None:
        # idle_ms: the resident kernel leaves the GPU soon after a burst
        _server = tmc.Server(idle_ms=2)
    return _server


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "seed": _seed(case, seed)}
    if kind == "batch":
        s["sets"] = _sets(case, seed)
        if case["plan"]:
            s["plan"] = tmc.BatchPlan(s["sets"], tmc.BatchOptions(use_graph=True))
    elif kind == "serve":
        s["requests"] = _requests(case, seed)
        s["server"] = _open_server()
    else:
        s["params"] = _params(case)
        if kind == "raw":
            s["options"] = dict(sampler=case.get("sampler", tmc.SAMPLER_ANALYTIC),
                                precision=case.get("precision", tmc.PRECISION_FP32),
                                math=case.get("math", tmc.MATH_HARDWARE),
                                first_photon=case["photons"] * (seed % 3000) if case.get("frames") else 0)
    return s


def run(state):
    kind = state["kind"]
    if kind == "run":
        heat, heat2 = tmc.run(state["params"], state["seed"])
        return {"heat": heat, "heat2": heat2}
    if kind == "raw":
        tally, stats = tmc.run_raw(state["params"], state["seed"], **state["options"])
        return {"tally": tally.view(np.int64), "absorptions": stats.interactions}
    if kind == "batch":
        tally, stats = state["plan"].run() if "plan" in state else tmc.batch_run(state["sets"])
        return {"tally": tally.view(np.int64), "absorptions": stats.interactions}
    server = state["server"]
    ids = [server.submit(p, seed) for p, seed in state["requests"]]
    done = [server.wait(i, timeout=60.0) for i in ids]
    if any(d is None for d in done):
        raise TimeoutError("a request was not served within 60 s")
    return {"tally": np.concatenate([t for t, _ in done]).view(np.int64),
            "absorptions": np.array([st.interactions for _, st in done], dtype=np.int64)}


# ---------------------------------------------------------------------------
# what the call cannot do without
# ---------------------------------------------------------------------------


def _per_photon(c):
    """Mean absorptions per photon: the first cycle to the cutoff, then a
    ninth of a cycle more (one survivor in ten goes on)."""
    a = np.float32(np.float32(c["mu_s"]) / (np.float32(c["mu_s"]) + np.float32(c["mu_a"])))
    k1 = math.ceil(math.log(0.001) / math.log(float(a)))
    k2 = math.ceil(math.log(0.1) / math.log(float(a)))
    return k1 + k2 / 9.0


def _of(p):
    return {"mu_a": p.mu_a, "mu_s": p.mu_s}


def _absorptions(case):
    kind = case["kind"]
    if kind in ("run", "raw"):
        return case["photons"] * _per_photon(case)
    pairs = _sets(case, 0) if kind == "batch" else _requests(case, 0)
    return sum(p.photons * _per_photon(_of(p)) for p, _ in pairs)


def work(case):
    kind = case["kind"]
    if kind in ("run", "raw"):
        shells = case["shells"]
    else:
        pairs = _sets(case, 0) if kind == "batch" else _requests(case, 0)
        shells = sum(p.shells for p, _ in pairs)
    out = 16 if kind == "run" else 32  # two doubles, or two 128-bit sums, per shell
    return {"bytes": float(out * shells), "flops": FLOP_PER_ABSORPTION * _absorptions(case)}


# ---------------------------------------------------------------------------
# the same photons in binary64
# ---------------------------------------------------------------------------


def _philox(k, photon, key):
    """Philox4x32-10 of counter (k, 0, photon low, photon high)."""
    m = np.uint64(0xFFFFFFFF)
    s32 = np.uint64(32)
    c0, c1 = k.astype(np.uint64), np.zeros(len(k), np.uint64)
    c2, c3 = photon & m, photon >> s32
    k0, k1 = key & 0xFFFFFFFF, key >> 32
    for _ in range(10):
        p0 = c0 * np.uint64(0xD2511F53)
        p1 = c2 * np.uint64(0xCD9E8D57)
        c0, c1, c2, c3 = (p1 >> s32) ^ c1 ^ np.uint64(k0), p1 & m, (p0 >> s32) ^ c3 ^ np.uint64(k1), p0 & m
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return [((w >> np.uint64(8)) + np.uint64(1)).astype(np.float64) * 2.0**-24 for w in (c0, c1, c2, c3)]


def exact(case, seed):
    """heat and heat2 of a small run, walked in binary64; None for raw
    tallies (whole numbers) and for runs of over four million absorptions."""
    if case["kind"] != "run" or _absorptions(case) > 4.0e6:
        return None
    key = _seed(case, seed)
    mu_a, mu_s = float(np.float32(case["mu_a"])), float(np.float32(case["mu_s"]))
    albedo = mu_s / (mu_s + mu_a)
    spm = 1e4 / float(np.float32(case["microns_per_shell"])) / (mu_a + mu_s)
    shells = case["shells"]
    photon = np.arange(case["photons"], dtype=np.uint64)
    n = len(photon)
    k = np.zeros(n, np.int64)
    x, y, z = np.zeros(n), np.zeros(n), np.zeros(n)
    u, v, w = np.zeros(n), np.zeros(n), np.ones(n)
    weight = np.ones(n)
    heat, heat2 = np.zeros(shells), np.zeros(shells)
    while len(photon):
        u0, u1, u2, u3 = _philox(k, photon, key)
        t = -np.log(u0)
        x, y, z = x + t * u, y + t * v, z + t * w
        shell = np.minimum(np.sqrt(x * x + y * y + z * z) * spm, shells - 1).astype(np.int64)
        d = (1.0 - albedo) * weight
        heat += np.bincount(shell, d, shells)
        heat2 += np.bincount(shell, d * d, shells)
        weight = weight * albedo
        u = 2.0 * u1 - 1.0
        s = np.sqrt(1.0 - u * u)
        v, w = s * np.cos(2.0 * np.pi * u2), s * np.sin(2.0 * np.pi * u2)
        k = k + 1
        low = weight < float(np.float32(0.001))
        keep = ~(low & (u3 > float(np.float32(0.1))))
        weight = np.where(low, weight / float(np.float32(0.1)), weight)
        photon, k, weight = photon[keep], k[keep], weight[keep]
        x, y, z, u, v, w = x[keep], y[keep], z[keep], u[keep], v[keep], w[keep]
    return {"heat": heat, "heat2": heat2}
