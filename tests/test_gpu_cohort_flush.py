"""A run of one workgroup that moves its sums out of LDS on the way (a word
takes 2^20 deposits) and still ends as the lone workgroup it is, against the
lane-per-photon walk (GPU tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MU = dict(mu_a=0.0014, mu_s=100.0)  # albedo 1 - 1.4e-5
FLUSH = (1 << 20) - 64 * 32  # deposits from which on a workgroup moves its sums out


def _cadence():
    """Absorptions to the first roulette, and from there to the second."""
    a = np.float32(MU["mu_s"]) / (np.float32(MU["mu_s"]) + np.float32(MU["mu_a"]))
    w, k, cuts = np.float32(1.0), 0, []
    while len(cuts) < 2:
        w, k = w * a, k + 1
        if w < np.float32(0.001):
            w = w / np.float32(0.1)
            cuts.append(k)
    return cuts[0], cuts[1] - cuts[0]


def _roulette_word(seed, photon, k):
    m = 0xFFFFFFFF
    c, k0, k1 = [k, 0, photon & m, photon >> 32], seed & m, seed >> 32
    for _ in range(10):
        a, b = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [(b >> 32) ^ c[1] ^ k0, b & m, (a >> 32) ^ c[3] ^ k1, a & m]
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    return c[3]


@pytest.mark.parametrize("shells", [101, 2000])
@pytest.mark.parametrize("capped", [False, True])
def test_lone_workgroup_that_flushed(tmc, shells, capped):
    k1, k2 = _cadence()
    kmax = k1 + k2 - 1000 if capped else 0
    assert 2 * k1 + (k2 - 1000) > FLUSH
    seed = next(s for s in range(1000) if sum(_roulette_word(s, p, k1 - 1) < 0x19999900 for p in (0, 1)) == 1)
    print(f"cohort flush: shells={shells} seed={seed} k1={k1} k2={k2} kmax={kmax}", flush=True)
    p = tmc.Params(photons=2, shells=shells, microns_per_shell=50.0, **MU)
    got, st = tmc.run_raw(p, seed, max_interactions=kmax)
    want, ws = tmc.run_raw(p, seed, max_interactions=kmax, block=256)
    assert (st.interactions, st.truncated) == (ws.interactions, ws.truncated)
    assert st.interactions > FLUSH and st.truncated == int(capped)
    np.testing.assert_array_equal(got, want)
