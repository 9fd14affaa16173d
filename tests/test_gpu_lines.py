"""Runs at the lines between the walks that the other files leave out, against
the lane-per-photon walk: more shells than the lockstep waves hold, four-wave
workgroups of the rejection sampler, and long cycles in more than one slice (GPU
tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEFAULT = dict(mu_a=2.0, mu_s=20.0, shells=101, microns_per_shell=50.0)
HIGHALB = dict(mu_a=0.5, mu_s=50.0, shells=201, microns_per_shell=20.0)


@pytest.mark.parametrize("phys,photons,sampler", [
    *[(dict(DEFAULT, shells=s, microns_per_shell=9.0), n, r) for s in (451, 2000) for n in (1 << 17, (1 << 17) + 1)
      for r in (0, 1)],  # many cohorts to a workgroup, and past the line
    *[(p, n, 1) for p in (DEFAULT, HIGHALB) for n in (262144, 262145, 300007, 327681)],
    (DEFAULT, (1 << 27) + 12345, 0)])
def test_lines(tmc, phys, photons, sampler):
    print(f"lines: {phys} photons={photons} sampler={sampler}", flush=True)
    p = tmc.Params(photons=photons, **phys)
    got, st = tmc.run_raw(p, 99, sampler=sampler, first_photon=5)
    want, ws = tmc.run_raw(p, 99, sampler=sampler, first_photon=5, block=256)
    assert st.interactions == ws.interactions
    np.testing.assert_array_equal(got, want)
