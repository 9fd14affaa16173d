"""Capped runs of the cohort and lockstep walks, whose weight table ends with
the cap, against the lane-per-photon walk: caps within the first cycle, at its
roulette and beside it, albedos whose whole table does and does not fit (GPU
tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GEOMETRY = dict(shells=101, microns_per_shell=50.0)


def first_roulette(mu_a, mu_s):
    a = np.float32(mu_s) / (np.float32(mu_s) + np.float32(mu_a))
    w, k = np.float32(1.0), 0
    while not w < np.float32(0.001):
        w, k = w * a, k + 1
    return k


@pytest.mark.parametrize("mu_a", [20.0, 0.5, 0.002, 2e-5])  # albedo 0.5, 0.976, 0.9999, 1 - 1e-6
@pytest.mark.parametrize("photons", [20, 3000, 40000, 300000])
@pytest.mark.parametrize("sampler", [0, 1])
def test_caps(tmc, mu_a, photons, sampler):
    k1 = first_roulette(mu_a, 20.0) if mu_a > 1e-3 else 0
    beside = [k1 - 1, k1, k1 + 1] if 2 < k1 < 2000 else []
    for kmax in [1, 2, 65, 300, 513] + beside:
        print(f"caps: mu_a={mu_a} photons={photons} sampler={sampler} kmax={kmax}", flush=True)
        p = tmc.Params(mu_a=mu_a, mu_s=20.0, photons=photons, **GEOMETRY)
        kw = dict(sampler=sampler, max_interactions=kmax, first_photon=(1 << 32) - 11)
        got, st = tmc.run_raw(p, 77, **kw)
        want, ws = tmc.run_raw(p, 77, block=256, **kw)
        assert (st.interactions, st.truncated) == (ws.interactions, ws.truncated)
        np.testing.assert_array_equal(got, want)
