"""The lockstep walk of large binary32 runs (more than 32,768 photons with the
analytic sampler, 49,152 with the other) against the oracle's mirror: ragged sizes on either side of its
levels, photon indices across a multiple of 2^32, caps at and beside a
roulette, several slices, and the walk of the same photons in two runs (GPU
tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEFAULT = dict(mu_a=2.0, mu_s=20.0, shells=101, microns_per_shell=50.0)
HIGHALB = dict(mu_a=0.5, mu_s=50.0, shells=201, microns_per_shell=20.0)
LOWALB = dict(mu_a=10.0, mu_s=10.0, shells=51, microns_per_shell=100.0)


def check(tmc, orc, hw_tables, phys, photons, seed, first=0, math=0, kmax=0):
    print(f"lock: {phys} photons={photons} seed={seed} first={first} math={math} kmax={kmax}", flush=True)
    tally, st = tmc.run_raw(tmc.Params(photons=photons, **phys), seed, first_photon=first, math=math,
                            max_interactions=kmax)
    kw = dict(max_k=kmax) if kmax else {}
    want, n = orc.mirror32(orc.params(**phys), seed, photons, first=first, sampler=0,
                           tables=hw_tables if math == 0 else None, **kw)
    assert st.interactions == n
    np.testing.assert_array_equal(tally, want)
    return st


@pytest.mark.parametrize("math", [0, 1])
@pytest.mark.parametrize("phys,photons", [(DEFAULT, 49153), (DEFAULT, 65535), (DEFAULT, 400001), (DEFAULT, 4000037),
                                          (LOWALB, 524289), (LOWALB, 9000001), (HIGHALB, 60000),
                                          (dict(DEFAULT, shells=450, microns_per_shell=9.0), 70000),
                                          (dict(DEFAULT, shells=1), 50000),
                                          (dict(mu_a=100.0, mu_s=1e-30, shells=3, microns_per_shell=50.0), 60000)])
def test_sizes(tmc, orc, hw_tables, phys, photons, math):
    check(tmc, orc, hw_tables, phys, photons, 71 + photons, math=math)


@pytest.mark.parametrize("first", [(1 << 32) - 100000, (1 << 32) - 1, 5 << 32, (1 << 33) - 199990])
def test_index_crossings(tmc, orc, hw_tables, first):
    check(tmc, orc, hw_tables, DEFAULT, 200000, (7 << 40) + 3, first=first)


@pytest.mark.parametrize("kmax", [1, 72, 73, 74, 96, 97, 98, 121, 122, 200])
def test_caps_beside_the_roulettes(tmc, orc, hw_tables, kmax):
    st = check(tmc, orc, hw_tables, DEFAULT, 600000, 5, kmax=kmax)
    assert st.truncated > 0 or kmax == 200  # past six roulettes 0.6 photons are expected


def test_more_than_one_slice(tmc):
    """2^26 + 12,345 photons (two slices of 2^26) equal the sum of the two
    parts of the range run alone, which other sizes of launch walk."""
    n, a = (1 << 26) + 12345, 41000003
    whole, st = tmc.run_raw(tmc.Params(photons=n, **DEFAULT), 99)
    lo, s1 = tmc.run_raw(tmc.Params(photons=a, **DEFAULT), 99)
    hi, s2 = tmc.run_raw(tmc.Params(photons=n - a, **DEFAULT), 99, first_photon=a)
    other, s3 = tmc.run_raw(tmc.Params(photons=n, **DEFAULT), 99, weight_table=649)  # lane per photon
    assert st.interactions == s1.interactions + s2.interactions == s3.interactions
    np.testing.assert_array_equal(whole, other)

    def big(t):
        return [int(t[2 * i]) + (int(t[2 * i + 1]) << 64) for i in range(2 * 101)]

    assert big(whole) == [x + y for x, y in zip(big(lo), big(hi))]


def test_alternating_runs(tmc, orc, hw_tables):
    """Large and small runs of different physics and sizes, one after the
    other: each finds its words clear and its lists large enough."""
    for i, (phys, photons) in enumerate([(DEFAULT, 70000), (HIGHALB, 300), (LOWALB, 3000000), (DEFAULT, 50000),
                                         (DEFAULT, 20), (HIGHALB, 70000)]):
        check(tmc, orc, hw_tables, phys, photons, 160 + i)


@pytest.mark.parametrize("math", [0, 1])
@pytest.mark.parametrize("phys,photons,first,kmax", [
    (DEFAULT, 49153, 0, 0), (DEFAULT, 400001, (1 << 32) - 1000, 0), (LOWALB, 524289, 0, 0), (HIGHALB, 60000, 7 << 33, 0),
    (dict(DEFAULT, shells=450, microns_per_shell=9.0), 70000, 0, 0), (dict(DEFAULT, shells=451), 60000, 0, 0),
    (dict(DEFAULT, shells=1), 50000, 3, 0), (dict(mu_a=100.0, mu_s=1e-30, shells=3, microns_per_shell=50.0), 60000, 0, 0),
    (DEFAULT, 100003, 0, 1), (DEFAULT, 100003, 0, 74), (DEFAULT, 100003, 0, 99)])
def test_rejection_sampler(tmc, phys, photons, first, kmax, math):
    """The rejection sampler's groups of absorptions, whose later attempts are
    gathered over the wave, against the lane-per-photon walk (block given)."""
    print(f"lock rejection: {phys} photons={photons} first={first} kmax={kmax} math={math}", flush=True)
    p = tmc.Params(photons=photons, **phys)
    kw = dict(sampler=1, first_photon=first, math=math, max_interactions=kmax)
    got, st = tmc.run_raw(p, (5 << 40) + photons, **kw)
    want, ws = tmc.run_raw(p, (5 << 40) + photons, block=256, **kw)
    np.testing.assert_array_equal(got, want)
    assert (st.interactions, st.truncated) == (ws.interactions, ws.truncated)


def test_rejection_sampler_against_the_oracle(tmc, orc, hw_tables):
    tally, st = tmc.run_raw(tmc.Params(photons=50007, **DEFAULT), 12, sampler=1)
    want, n = orc.mirror32(orc.params(**DEFAULT), 12, 50007, sampler=1, tables=hw_tables)
    assert st.interactions == n
    np.testing.assert_array_equal(tally, want)


@pytest.mark.parametrize("math", [0, 1])
@pytest.mark.parametrize("phys,photons,first,kmax", [
    (DEFAULT, (1 << 22) + 1001, (1 << 32) - (1 << 21), 0), (LOWALB, (1 << 25) + 77, 0, 0),
    (DEFAULT, (1 << 23) + 5, 0, 50), (DEFAULT, (1 << 22) + 3, 0, 73), (dict(DEFAULT, shells=133), 5000001, 0, 0),
    (dict(DEFAULT, shells=134), 5000001, 0, 0), (dict(DEFAULT, shells=1), 5000001, 0, 0)])
def test_counted_first_cycles(tmc, phys, photons, first, kmax, math):
    """First cycles of 3e8 absorptions and more, counted by absorption and shell
    where the counts fit (at 73 absorptions up to 133 shells)."""
    print(f"lock counted: {phys} photons={photons} first={first} kmax={kmax} math={math}", flush=True)
    p = tmc.Params(photons=photons, **phys)
    kw = dict(first_photon=first, math=math, max_interactions=kmax)
    got, st = tmc.run_raw(p, 31, **kw)
    want, ws = tmc.run_raw(p, 31, block=256, **kw)
    np.testing.assert_array_equal(got, want)
    assert (st.interactions, st.truncated) == (ws.interactions, ws.truncated)


@pytest.mark.parametrize("photons,first,kw", [
    ((1 << 27) + 12345, 0, {}), ((1 << 27) + 99, (1 << 32) - (1 << 26) - 5, {}), ((1 << 27) + 1, 0, dict(sampler=1)),
    ((1 << 27) + 77, 0, dict(precision=1))])
def test_slices(tmc, photons, first, kw):
    """Runs of more than one slice (2^27 photons), against the lane-per-photon
    walk (block given); the precision variants' slices are the same."""
    print(f"lock slices: photons={photons} first={first} {kw}", flush=True)
    p = tmc.Params(photons=photons, **LOWALB)
    got, st = tmc.run_raw(p, 8, first_photon=first, **kw)
    want, ws = tmc.run_raw(p, 8, first_photon=first, block=256, **kw)
    np.testing.assert_array_equal(got, want)
    assert st.interactions == ws.interactions


@pytest.mark.parametrize("sampler,photons", [(0, 32768), (0, 32769), (0, 49152), (1, 49152), (1, 49153)])
def test_line_to_the_cohort_walk(tmc, orc, hw_tables, sampler, photons):
    tally, st = tmc.run_raw(tmc.Params(photons=photons, **DEFAULT), 3, sampler=sampler)
    want, n = orc.mirror32(orc.params(**DEFAULT), 3, photons, sampler=sampler, tables=hw_tables)
    assert st.interactions == n
    np.testing.assert_array_equal(tally, want)
