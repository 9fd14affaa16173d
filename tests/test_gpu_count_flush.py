"""Counted first cycles of few shells, whose pairs' absorptions go to one, four
and more threads when the counts are added up, against the lane-per-photon walk
(GPU tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mu_a,mu_s,photons", [(2.0, 20.0, (1 << 22) + 77), (10.0, 10.0, (1 << 25) + 5),
                                               (0.5, 50.0, (1 << 19) + 3)])  # 73, 10 and 690 absorptions
@pytest.mark.parametrize("shells", [1, 2, 7, 8, 24, 56, 57, 121])
def test_few_shells(tmc, mu_a, mu_s, photons, shells):
    print(f"count flush: mu_a={mu_a} mu_s={mu_s} photons={photons} shells={shells}", flush=True)
    p = tmc.Params(mu_a=mu_a, mu_s=mu_s, shells=shells, microns_per_shell=3000.0 / shells, photons=photons)
    got, st = tmc.run_raw(p, 13, first_photon=1 << 32)
    want, ws = tmc.run_raw(p, 13, first_photon=1 << 32, block=256)
    assert st.interactions == ws.interactions
    np.testing.assert_array_equal(got, want)
