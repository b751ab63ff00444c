"""A queue that cannot hold a run's recoils: the run ends in queue-full, soon, and the
context runs the next one as if nothing had been."""
import time

import numpy as np
import pytest

from mytrim_amd import configs, gpu

pytestmark = pytest.mark.gpu


# 64 slots and stacks of two entries: the first collisions of 512 cascades overflow
# them.  Waves that had claimed entries which were then never published once ran what
# lay in their stacks again, and its recoils kept the queue full
@pytest.mark.parametrize("make,n_hist", [(configs.c2_cu_cu, 2000), (lambda n: configs.vacancy_case("cu", 1e3, n), 70000)],
                         ids=["cu_500keV", "cu_1keV"])
@pytest.mark.parametrize("feeders", [0, 20])
def test_overflow_ends_the_run(make, n_hist, feeders):
    prob = make(n_hist)
    e = gpu.Engine(0)
    try:
        ref = e.run(prob)
        e.tune(queue_cap=64, stack_cap=2, primary_waves64=feeders)
        t0 = time.time()
        for _ in range(3):
            with pytest.raises(gpu.MtError, match="queue-full"):
                e.run(prob)
        assert time.time() - t0 < 30.0  # full runs take 11 and 3 ms
        e.tune()
        r = e.run(prob)
        assert r["n_flight"] == ref["n_flight"] and np.array_equal(r["vac_hist"], ref["vac_hist"])
    finally:
        e.close()
