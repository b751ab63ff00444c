"""Admission of primaries: the estimate of a cascade's flights that sizes the
queue and its budget (CPU), and runs at the edges of the small-batch rule and
of queues too small for the batch (GPU)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle_lib as O
from mytrim_amd import configs

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


# full cascades in an infinite or large target; the estimate's own claim is 0.64
# to 1.0 times its value, and a few dozen histories scatter by up to a third
@pytest.mark.parametrize("prob", [configs.c1_he_fe(60), configs.c5_c_w(40), configs.c2_cu_cu(3),
                                  configs.vacancy_case("cu", 1e4, 60), configs.vacancy_case("xe", 1e5, 10)],
                         ids=["he_fe", "c_w", "cu_cu", "cu_cu_10keV", "xe_u"])
def test_flights_estimate(prob, tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "flights_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "mytrim_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), "-o", exe,
                    os.path.join(HERE, "native", "flights_check.cpp")], check=True, capture_output=True)
    p, el = prob.primaries, prob.materials[0].elements[0]
    line = "%r %r %r %r %r %r" % (float(p.Z[0]), float(p.m[0]), float(p.E[0]), float(el.Z), el.m, el.Edisp)
    est = float(subprocess.run([exe], input=line, check=True, capture_output=True, text=True).stdout)
    flights = O.run(prob, rng=1, nthreads=4)["n_flight"] / prob.n_hist
    assert 0.64 / 1.34 < flights / est < 1.0 * 1.34


INTS = ["n_coll", "n_flight", "vac", "repl", "subst", "inter", "lost", "newton", "range_n"]
HISTS = ["range_hist", "lat_y_hist", "vac_hist", "repl_hist"]


def assert_same(a, b):
    for k in INTS:
        assert a[k] == b[k], k
    for k in HISTS:
        assert np.array_equal(a[k], b[k]), k
    for k in ("Eel", "Enuc", "Elost", "Eunf"):
        assert a[k] == pytest.approx(b[k], rel=1e-11), k


# one primary; one more than a wave, than one per SIMD, than two per SIMD; the
# last size of the small-batch rule (64 per SIMD) and the next
@pytest.mark.gpu
@pytest.mark.parametrize("n_hist", [1, 65, 1025, 2049, 65536, 65537])
def test_small_batch_shapes_agree(n_hist):
    from mytrim_amd import gpu
    prob = configs.vacancy_case("cu", 1e3, n_hist, seed=13)
    e = gpu.Engine(0)
    try:
        ref = e.run(prob)
        assert ref["n_flight"] == n_hist + ref["vac"] + ref["repl"] + ref["subst"]
        for kw in ({"block": 64, "blocks_per_cu": 1}, {"block": 128, "blocks_per_cu": 5}, {"blocks_per_cu": 3},
                   {"primary_waves64": 20}):
            e.tune(**kw)
            assert_same(ref, e.run(prob))
    finally:
        e.close()


# queues that hold a fraction of the batch's flights: the budget is kept, and
# the run does not overflow them
@pytest.mark.gpu
@pytest.mark.parametrize("make,n_hist", [(configs.c1_he_fe, 20000), (configs.c5_c_w, 2000), (configs.c2_cu_cu, 600)],
                         ids=["he_fe", "c_w", "cu_cu"])
def test_small_queue_keeps_its_budget(make, n_hist):
    from mytrim_amd import gpu
    prob = make(n_hist, seed=19)
    e = gpu.Engine(0)
    try:
        ref = e.run(prob)
        e.tune(queue_cap=1 << 16)
        assert_same(ref, e.run(prob))
        e.tune()
        assert_same(ref, e.run(prob, noalloc=True))
    finally:
        e.close()


# ions leave through the faces and the rare sums (lost, unfollowed) add up
@pytest.mark.gpu
def test_rare_energy_sums():
    from mytrim_amd import gpu
    e = gpu.Engine(0)
    try:
        for prob in (configs.wire_b_si(3000, seed=3), configs.c2_cu_cu(500, seed=3).with_(follow_max_gen=1)):
            r = e.run(prob)
            out = r["Eel"] + r["Enuc"] + r["Eunf"] + r["Elost"] + r["Edrop"] + r["Evac"]
            assert out == pytest.approx(r["E0"], rel=1e-9)
            o = O.run(prob, rng=1, nthreads=4)
            for k in ("Eunf", "Elost", "Edrop"):
                assert r[k] == pytest.approx(o[k], rel=0.01), k
            assert r["range_sum"] == pytest.approx(o["range_sum"], rel=0.01)
    finally:
        e.close()
