"""A server whose requests arrive while a run or a batch in lockstep is on the
device: the call ends, the requests are served, and all results are those of
the same work alone (GPU tests, bit-exact)."""
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HIGHALB = dict(mu_a=0.5, mu_s=50.0, shells=201, microns_per_shell=20.0)
SMALL = dict(mu_a=2.0, mu_s=20.0, shells=101, microns_per_shell=50.0)


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("reserve", [0, 2])
def test_requests_during_a_call(tmc, batch, reserve):
    print(f"serve during a run: batch={batch} reserve={reserve}", flush=True)
    p = tmc.Params(photons=1 << 24, **HIGHALB)
    sets = [(tmc.Params(photons=1 << 22, **HIGHALB), 40 + i) for i in range(6)]

    def work():
        return tmc.batch_run(sets)[0] if batch else tmc.run_raw(p, 9)[0]

    alone = work()
    small = [(tmc.Params(photons=1000 + i, **SMALL), 500 + i) for i in range(40)]
    want = [tmc.run_raw(q, s, block=256)[0] for q, s in small]
    got = []
    with tmc.Server(max_shells=201, reserve_per_cu=reserve, idle_ms=2) as server:
        caller = threading.Thread(target=lambda: got.extend([work(), work()]))
        caller.start()
        time.sleep(0.005)  # (the first call takes 20 ms and more)
        served = []
        for q, s in small:
            served.append(server.submit(q, s))
            time.sleep(0.002)
        tallies = [server.wait(i, 60.0) for i in served]
        caller.join(60.0)
        assert not caller.is_alive()
    assert all(t is not None for t in tallies)
    for t, w in zip(tallies, want):
        np.testing.assert_array_equal(t[0], w)
    assert len(got) == 2
    for t in got:
        np.testing.assert_array_equal(t, alone)
