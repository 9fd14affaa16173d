"""The lockstep walk of a batch (automatic options, analytic sampler) against
the lane-per-photon walk of the same sets: ragged photon counts on either side
of a wave's batch, indices across multiples of 2^32, wide seeds, one and two
lockstep cycles, sets of several parts and slices, graph replays, and beside a
resident serving kernel (GPU tests, bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PHYS = [dict(mu_a=2.0, mu_s=20.0, shells=101, microns_per_shell=50.0),
        dict(mu_a=0.5, mu_s=50.0, shells=201, microns_per_shell=20.0),
        dict(mu_a=10.0, mu_s=10.0, shells=51, microns_per_shell=100.0),
        dict(mu_a=0.01, mu_s=30.0, shells=450, microns_per_shell=9.0),
        dict(mu_a=100.0, mu_s=1e-30, shells=1, microns_per_shell=50.0)]


def ragged(tmc, counts):
    sets = []
    for i, n in enumerate(counts):
        first = (0, 5, (1 << 32) - 40, (1 << 63) - n, (3 << 32) - 1)[i % 5]
        sets.append((tmc.Params(photons=n, **PHYS[(i * 3) % 5]), (0x9E3779B97F4A7C15 * (i + 1)) % 2**64, first))
    return sets


def check(tmc, sets, math=0, flat=None, st=None):
    """Every set equals the same photons walked a lane each, alone."""
    if flat is None:
        flat, st = tmc.batch_run(sets, tmc.BatchOptions(math=math))
    total = 0
    for i, ((p, seed, first), t) in enumerate(zip(sets, tmc.split_tallies(sets, flat))):
        want, ws = tmc.run_raw(p, seed, first_photon=first, math=math, block=256)
        np.testing.assert_array_equal(t, want, err_msg=f"set {i}: {p} first={first}")
        total += ws.interactions
    assert st.interactions == total
    assert (st.interactions + st.idle_lane_steps) % 64 == 0


@pytest.mark.parametrize("math", [0, 1])
@pytest.mark.parametrize("counts", [[1], [0, 63, 64, 65, 0, 1, 127], [4097] * 10, [100000, 3, 40001, 700, 64, 20011],
                                    [1500007, 1, 600001, 64]])  # the last: two lockstep cycles
def test_ragged_sets(tmc, counts, math):
    print(f"batch lock: {counts} math={math}", flush=True)
    check(tmc, ragged(tmc, counts), math)


def test_graph_replays(tmc):
    sets = ragged(tmc, [1200011, 900001, 5, 30000])
    with tmc.BatchPlan(sets, tmc.BatchOptions(use_graph=True)) as plan:
        for r in range(3):
            flat, st = plan.run()
            check(tmc, sets, flat=flat, st=st)  # (eager runs between the replays)


def test_parts_and_slices(tmc):
    """Sets of more than 2^26 photons, and more survivors than one slice holds."""
    short = PHYS[2]
    sets = [(tmc.Params(photons=(1 << 27) + 5, **short), 3, 0),
            (tmc.Params(photons=(1 << 27) + 77, **short), 4, (1 << 32) - (1 << 26) - 9)]
    check(tmc, sets)


def test_beside_a_server(tmc):
    """Plans made before and beside a resident serving kernel (two workgroup
    slots per compute unit reserved)."""
    sets = ragged(tmc, [5000, 70001, 64])
    long_req = (tmc.Params(mu_a=0.01, mu_s=100.0, shells=101, photons=1 << 10), 77)
    with tmc.BatchPlan(sets) as before:
        with tmc.Server(max_shells=101, reserve_per_cu=2) as server:
            rid = server.submit(*long_req)
            flat, st = before.run()
            beside, bs = tmc.batch_run(sets)
            server.wait(rid, 60.0)
        check(tmc, sets, flat=flat, st=st)
        check(tmc, sets, flat=beside, st=bs)
        flat, st = before.run()
        check(tmc, sets, flat=flat, st=st)
