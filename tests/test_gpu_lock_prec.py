"""Lockstep runs of the precision variants (no launch shape given) against the
lane-per-photon walk of the same photons (block given): ragged sizes on either
side of the packing of survivors, indices across a multiple of 2^32, the
smallest and largest shell counts, photons past the weight table, and a cap,
which keeps to the lane-per-photon walk (GPU tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEFAULT = dict(mu_a=2.0, mu_s=20.0, shells=101, microns_per_shell=50.0)
HIGHALB = dict(mu_a=0.05, mu_s=50.0, shells=201, microns_per_shell=20.0)
LOWALB = dict(mu_a=10.0, mu_s=10.0, shells=51, microns_per_shell=100.0)


def check(tmc, phys, photons, precision, sampler=0, first=0, kmax=0):
    print(f"lock prec: {phys} photons={photons} precision={precision} sampler={sampler} first={first}", flush=True)
    p = tmc.Params(photons=photons, **phys)
    kw = dict(sampler=sampler, precision=precision, first_photon=first, max_interactions=kmax)
    got, st = tmc.run_raw(p, (9 << 40) + photons, **kw)
    want, ws = tmc.run_raw(p, (9 << 40) + photons, block=256, **kw)
    np.testing.assert_array_equal(got, want)
    assert (st.interactions, st.truncated) == (ws.interactions, ws.truncated)


@pytest.mark.parametrize("precision", [1, 2, 3])
@pytest.mark.parametrize("sampler", [0, 1])
@pytest.mark.parametrize("phys,photons,first", [
    (DEFAULT, 1, 0), (DEFAULT, 63, 5), (DEFAULT, 65, (1 << 32) - 7), (DEFAULT, 65537, 0), (LOWALB, 700001, 3 << 32),
    (HIGHALB, 1500, 0), (dict(DEFAULT, shells=1), 300, 0), (dict(DEFAULT, shells=450), 70000, (1 << 33) - 69999),
    (dict(DEFAULT, shells=451), 3000, 0), (dict(mu_a=100.0, mu_s=1e-30, shells=3, microns_per_shell=50.0), 200, 0)])
def test_sizes(tmc, phys, photons, first, precision, sampler):
    check(tmc, phys, photons, precision, sampler, first)


@pytest.mark.parametrize("precision", [1, 2, 3])
def test_two_packings_and_a_cap(tmc, precision):
    check(tmc, DEFAULT, 1000003, precision)
    check(tmc, DEFAULT, 5000, precision, kmax=74)
    check(tmc, DEFAULT, 5000, precision, sampler=1, kmax=1)


@pytest.mark.parametrize("precision", [1, 3])
def test_past_the_table(tmc, precision):
    """A photon outlives the table of a one-photon run (four roulettes, the last
    after 20 absorptions) with a
    chance of 10^-4 and more: found by the binary32 walk among 2^15."""
    p = tmc.Params(photons=1, **LOWALB)
    long = [i for i in range(1 << 15)
            if tmc.run_raw(p, 77, first_photon=i, max_interactions=21)[1].truncated]
    assert long
    for i in long:
        want, ws = tmc.run_raw(p, 77, first_photon=i, precision=precision, block=64)
        got, st = tmc.run_raw(p, 77, first_photon=i, precision=precision)
        np.testing.assert_array_equal(got, want)
        assert st.interactions == ws.interactions
