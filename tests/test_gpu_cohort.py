"""The cohort walk (runs of up to 2^17 photons) against the oracle's mirror:
sizes on either side of its cohort shapes, caps at and beside a roulette,
photons that outlive its weight table, tables in LDS and in device memory,
and runs that alternate with the other walk (GPU tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEFAULT = dict(mu_a=2.0, mu_s=20.0, shells=101, microns_per_shell=50.0)
HIGHALB = dict(mu_a=0.5, mu_s=50.0, shells=201, microns_per_shell=20.0)
LOWALB = dict(mu_a=10.0, mu_s=10.0, shells=51, microns_per_shell=100.0)


def check(tmc, orc, hw_tables, phys, photons, seed, first=0, sampler=0, math=0, kmax=0):
    print(f"cohort: {phys} photons={photons} seed={seed} first={first} sampler={sampler} math={math} kmax={kmax}",
          flush=True)
    tally, st = tmc.run_raw(tmc.Params(photons=photons, **phys), seed, first_photon=first, sampler=sampler, math=math,
                            max_interactions=kmax)
    kw = dict(max_k=kmax) if kmax else {}
    want, n = orc.mirror32(orc.params(**phys), seed, photons, first=first, sampler=sampler,
                           tables=hw_tables if math == 0 else None, **kw)
    assert st.interactions == n
    np.testing.assert_array_equal(tally, want)
    return st


@pytest.mark.parametrize("photons", [1, 2, 63, 64, 65, 1000, 4097, 8193, 16385, 1 << 17, (1 << 17) + 1])
@pytest.mark.parametrize("sampler", [0, 1])
def test_sizes(tmc, orc, hw_tables, sampler, photons):
    check(tmc, orc, hw_tables, DEFAULT, photons, 1000 + photons, sampler=sampler)


@pytest.mark.parametrize("phys,photons", [(HIGHALB, 1), (HIGHALB, 513), (HIGHALB, 5000), (LOWALB, 70000),
                                          (dict(DEFAULT, shells=6500, microns_per_shell=1.0), 3000),
                                          (dict(mu_a=100.0, mu_s=1e-30, shells=3, microns_per_shell=50.0), 500)])
@pytest.mark.parametrize("math", [0, 1])
def test_physics(tmc, orc, hw_tables, phys, photons, math):
    check(tmc, orc, hw_tables, phys, photons, (5 << 33) + 1, first=(1 << 32) - 40, math=math)


@pytest.mark.parametrize("kmax", [1, 72, 73, 74, 96, 97, 98])
def test_caps_beside_the_roulettes(tmc, orc, hw_tables, kmax):
    """Default physics ends its cycles at absorptions 73, 97, ...: a cap just
    before, at and after one."""
    st = check(tmc, orc, hw_tables, DEFAULT, 20000, 5, kmax=kmax)
    assert st.truncated == (20000 if kmax < 73 else st.truncated) and st.truncated > 0


def _survivors(seed, n, cuts):
    """Photons of [0, n) that survive the roulettes after `cuts` absorptions
    each (Philox word 3 of block (cut - 1, 0) below the kill threshold)."""
    m = np.uint64(0xFFFFFFFF)
    p = np.arange(n, dtype=np.uint64)
    for cut in cuts:
        c0, c1 = np.full(len(p), cut - 1, np.uint64), np.zeros(len(p), np.uint64)
        c2, c3 = p & m, p >> np.uint64(32)
        k0, k1 = seed & 0xFFFFFFFF, seed >> 32
        for _ in range(10):
            a, b = c0 * np.uint64(0xD2511F53), c2 * np.uint64(0xCD9E8D57)
            c0, c1, c2, c3 = ((b >> np.uint64(32)) ^ c1 ^ np.uint64(k0), b & m,
                              (a >> np.uint64(32)) ^ c3 ^ np.uint64(k1), a & m)
            k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
        p = p[c3 < 0x19999900]
    return p


def test_photons_that_outlive_the_table(tmc, orc, hw_tables):
    """A run of one photon has a table of four roulettes: photons that survive
    all of them walk on without it."""
    a = np.float32(20.0) / np.float32(22.0)
    w, k, cuts = np.float32(1.0), 0, []
    while len(cuts) < 4:
        w, k = np.float32(w * a), k + 1
        if w < np.float32(0.001):
            w = np.float32(w / np.float32(0.1))
            cuts.append(k)
    lucky = _survivors(77, 1 << 17, cuts)
    assert len(lucky) >= 3
    for p in lucky[:3]:
        for sampler in (0, 1):
            st = check(tmc, orc, hw_tables, DEFAULT, 1, 77, first=int(p), sampler=sampler)
            assert st.interactions > cuts[-1]
        st = check(tmc, orc, hw_tables, DEFAULT, 1, 77, first=int(p), kmax=cuts[-1] + 2)
        assert st.interactions == cuts[-1] + 2 and st.truncated == 1


def test_alternating_runs(tmc, orc, hw_tables):
    """Runs of this walk leave their device words clear for the next one,
    also where the other walk or another shell count came between."""
    for i, (phys, photons) in enumerate([(DEFAULT, 3000), (HIGHALB, 700), (DEFAULT, 1 << 18), (LOWALB, 5000),
                                         (DEFAULT, 20), (DEFAULT, 0), (DEFAULT, 40000)]):
        check(tmc, orc, hw_tables, phys, photons, 60 + i)
