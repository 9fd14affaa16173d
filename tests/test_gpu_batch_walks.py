"""Batches on either side of the line between the lockstep and the lane-per-
photon walk, and sets of several parts and slices in lockstep, against the
lane-per-photon walk of each set alone (GPU tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(tmc, sets, keep):
    if keep:
        with tmc.BatchPlan(sets) as plan:
            runs = [plan.run(), plan.run()]
    else:
        runs = [tmc.batch_run(sets)]
    want = [tmc.run_raw(p, seed, first_photon=first, block=256) for p, seed, first in sets]
    for flat, st in runs:
        assert st.interactions == sum(w.interactions for _, w in want)
        for i, (t, (w, _)) in enumerate(zip(tmc.split_tallies(sets, flat), want)):
            np.testing.assert_array_equal(t, w, err_msg=f"set {i}")


@pytest.mark.parametrize("mu_s,nsets,photons", [(1.0, 3, 70001), (7.0, 40, 3001), (20.0, 64, 16384), (20.0, 65, 65537),
                                                (220.0, 300, 65), (220.0, 5, 1 << 20), (220.0, 2, (1 << 22) + 1)])
@pytest.mark.parametrize("keep", [False, True])
def test_either_side(tmc, mu_s, nsets, photons, keep):
    print(f"batch walks: mu_s={mu_s} nsets={nsets} photons={photons} keep={keep}", flush=True)
    phys = dict(mu_a=20.0, mu_s=mu_s, shells=31, microns_per_shell=50.0)
    sets = [(tmc.Params(photons=photons + i % 3, **phys), 11 + i, (1 << 32) - 5 * i) for i in range(nsets)]
    check(tmc, sets, keep)


def test_parts_and_slices_of_long_cycles(tmc):
    """Sets of more than 2^26 photons, and more survivors than one slice holds."""
    phys = dict(mu_a=1.0, mu_s=20.0, shells=51, microns_per_shell=100.0)  # 142 absorptions to the first roulette
    sets = [(tmc.Params(photons=(1 << 27) + 5, **phys), 3, 0),
            (tmc.Params(photons=(1 << 27) + 77, **phys), 4, (1 << 32) - (1 << 26) - 9)]
    print("batch walks: parts and slices", flush=True)
    check(tmc, sets, False)
