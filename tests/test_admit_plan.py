"""Which primaries of a batch may be live at once: the estimate of a primary's
direct recoils and the admission rules (mt_tune.h) on the CPU, and batches whose
recoils fill a queue too small for them on the GPU."""
import dataclasses
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle_lib as O
from mytrim_amd import configs
from mytrim_amd.problem import Element, Material, Primaries
from test_admission import assert_same

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
FE, CU, W, U, C = ((26, 55.845, 40.0, 7.87), (29, 63.546, 30.0, 8.96), (74, 183.84, 90.0, 19.3), (92, 238.03, 40.0, 19.0),
                   (6, 12.011, 25.0, 2.2))
IONS = {"H": (1, 1.008), "He": (2, 4.0026), "C": (6, 12.011), "Cu": (29, 63.546), "Xe": (54, 131.29), "U": (92, 238.03)}
STATIC_SLOTS, MAX_SLOTS = 1 << 21, 1 << 27


def infinite(ion, E, target, n_hist, seed=5):
    Z, m, Ed, rho = target
    base, w = configs.c2_cu_cu(n_hist, seed=seed), 1.0e7
    return base.with_(materials=[Material(rho, [Element(Z, m, 1.0, Ed, 3.0)])],
                      geometry=dataclasses.replace(base.geometry, w=(w, w, w)),
                      primaries=Primaries.single(*IONS[ion], E, (w / 2, w / 2, w / 2)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("admit") / "admit_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "mytrim_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), "-o", exe, os.path.join(HERE, "native", "admit_check.cpp")],
                   check=True, capture_output=True)
    return lambda line: [float(x) for x in subprocess.run([exe], input=line, check=True, capture_output=True,
                                                          text=True).stdout.split()]


def direct(check, ion, E, target):
    return check("direct %r %r %r %r %r %r" % (*map(float, IONS[ion]), E, float(target[0]), target[1], target[2]))[0]


# the estimate's own claim is 0.9 to 1.9 of the truth; a few hundred recoils
# scatter by a tenth
@pytest.mark.parametrize("ion,E,target,n", [("H", 1e5, FE, 400), ("He", 1e4, FE, 200), ("He", 1e5, FE, 100),
                                            ("He", 2e6, FE, 60), ("C", 1e5, W, 60), ("C", 2e6, W, 40), ("Cu", 1e3, CU, 200),
                                            ("Cu", 1e4, CU, 100), ("Cu", 5e5, CU, 20), ("Xe", 1e5, U, 40),
                                            ("Xe", 3e7, U, 4), ("U", 1e6, C, 10), ("Cu", 1e9, CU, 2)])
def test_direct_estimate(check, ion, E, target, n):
    prob = infinite(ion, E, target, n).with_(follow_max_gen=2)
    truth = O.run(prob, rng=1, nthreads=4)["n_flight"] / n - 1.0
    assert 0.9 / 1.1 < direct(check, ion, E, target) / truth < 1.9 * 1.1
    assert direct(check, ion, target[2], target) == 0.0  # no transfer reaches the threshold


def plan(check, n, flights, d, qcap, waves=2048, block=256, stack=128, feeders=0, d_all=None):
    v = check("plan %d %r %r %r %d %d 1024 %d %d %d" % (n, flights, n * d if d_all is None else d_all, d, qcap, waves,
                                                        block, stack, feeders))
    return dict(zip(("strict", "share", "late", "budget", "floor", "cap", "stagger", "first"), v))


# measured per live cascade: flights, direct recoils, the part of the direct ones
# that waits while the lanes hold primaries
@pytest.mark.parametrize("n", [65536, 131072, 1 << 22])
@pytest.mark.parametrize("ion,E,target,flights,d,waits", [("He", 1e5, FE, 98.0, 30.0, 0.93), ("C", 2e6, W, 485.0, 79.3, 0.76)])
def test_light_ions_fit_the_static_queue(check, n, ion, E, target, flights, d, waits):
    p = plan(check, n, 1.05 * flights, direct(check, ion, E, target), STATIC_SLOTS)
    live = min(n, max(p["floor"], min(p["budget"] / flights, p["cap"])))
    assert p["strict"] and live * d * waits < 0.85 * STATIC_SLOTS + 0.5 * 128 * 2048
    assert live > 10000  # and lanes enough are busy


# measured: 3.55 times the direct recoils wait of 65 536 histories of 2 MeV Xe in UO2
# that start at once, 4.05 of 8192 of 30 MeV, 1.0 of 65 536 of 1 MeV U in C
def test_large_queue_is_not_filled_at_once(check):
    xe2, xe30 = (13240.0, 373.0), (44500.0, 1446.0)  # flights, estimate of the direct recoils
    assert plan(check, 65536, 3.7 * xe2[0], xe2[1], MAX_SLOTS)["share"] == 64
    assert plan(check, 8192, 4.0 * xe30[0], xe30[1], MAX_SLOTS)["share"] == 8
    assert plan(check, 65536, 27524.0, 565.0, MAX_SLOTS)["share"] == 64
    for n in (40000, 65536, 131072, 10 ** 6):
        p = plan(check, n, 4.0 * xe30[0], xe30[1], MAX_SLOTS)
        live = min(n, max(p["floor"], min(p["budget"] / xe30[0], p["cap"])))
        assert p["strict"] and not p["share"] and 0.1 * live * xe30[0] < MAX_SLOTS
    # what starts at once in a large batch is one primary a lane
    assert not plan(check, 10 ** 6, 8010.0, 184.0, MAX_SLOTS, waves=3072)["strict"]
    assert not plan(check, 10 ** 6, 48618.0, 373.0, MAX_SLOTS, waves=3072, d_all=4e7)["strict"]


def test_rules_at_their_edges(check):
    for n in (1, 64 * 1024, 64 * 1024 + 1):  # small: at most 64 primaries per SIMD, a queue of its size
        p = plan(check, n, 20.0, 0.0, 1 << 21)
        assert p["share"] == (0 if n > 65536 else -(-n // 1024)) and not p["strict"]
    assert plan(check, 4096, 1024.0, 30.0, STATIC_SLOTS)["strict"] == 0  # twice the slots
    assert plan(check, 4097, 1024.0, 30.0, STATIC_SLOTS)["strict"] == 1
    # what may start at first may stay live: 512 at least, a wave each at most
    assert plan(check, 10 ** 6, 8010.0, 184.0, STATIC_SLOTS)["floor"] == 2048
    assert plan(check, 10 ** 6, 48618.0, 373.0, STATIC_SLOTS)["floor"] == int((12 * STATIC_SLOTS + 1024 * 2048) / 48618.0)
    p = plan(check, 1000, 1e6, 1e5, 1 << 16)
    assert p["strict"] and p["floor"] == 512 and p["cap"] < 512
    assert plan(check, 1000, 1e6, 1e5, 1 << 16, waves=256)["floor"] == 256
    assert plan(check, 1000, 10.0, 3.0, 1 << 16, feeders=20)["share"] == 0


# the blocks start one after another only where there is a primary for each lane
@pytest.mark.parametrize("waves", [2048, 3072])
@pytest.mark.parametrize("feeders", [0, 62])
def test_few_primaries_are_not_left_to_the_first_blocks(check, waves, feeders):
    for n in (65537, 64 * waves - 1):
        p = plan(check, n, 104.0, 30.0, 1 << 27, waves=waves, feeders=feeders)
        # 64 primaries per wave: the waves that start before the last is taken
        # are not a small part of the launch (a nap is 1.07 us, an admission some 10)
        assert p["stagger"] <= 48 and not p["share"] and not p["strict"]
    if feeders == 0:
        assert plan(check, 64 * waves, 104.0, 30.0, 1 << 27, waves=waves)["stagger"] == 256


# with wave roles: the feeders' first admission takes the batch (64 a feeder, half as
# many again) and nothing is held back, or the first cascades are few
def test_feeders_take_a_batch_or_start_slowly(check):
    he = lambda n, **kw: plan(check, n, 104.0, 30.0, 1 << 27, waves=3072, feeders=62, **kw)
    feeder_waves = 3072 * 62 // 64
    for n in (100, 2 * 10 ** 5, 96 * feeder_waves):
        assert he(n)["first"] > n and he(n)["budget"] >= 104.0 * n and he(n)["stagger"] <= 16
    for n in (96 * feeder_waves + 1, 4 * 10 ** 5, 10 ** 6):
        p = he(n)
        assert p["first"] == 16 * 3072 and p["stagger"] <= 16 and not p["strict"]
        # never more flights, nor direct recoils, than the queue bears
        assert p["budget"] <= 7.5 * (1 << 27) + 6144 * 3072
        assert p["budget"] / 104.0 * 30.0 < 1 << 27
    # long cascades: the queue's share, not 224 cascades per wave
    p = plan(check, 10 ** 6, 48618.0, 373.0, 1 << 27, waves=3072, feeders=10, d_all=4e7)
    assert p["budget"] == 7.5 * (1 << 27) + 6144 * 3072 and p["cap"] * 80.0 < 1.01 * (1 << 27)
    # without roles, and where the cascades are reserved, nothing of this
    assert plan(check, 10 ** 6, 104.0, 30.0, 1 << 27, waves=3072)["first"] > 1e17
    assert plan(check, 10 ** 6, 104.0, 30.0, 1 << 21, waves=3072, feeders=62)["first"] > 1e17


# batches on both sides of what the feeders take at once: the same results
@pytest.mark.gpu
@pytest.mark.parametrize("n_hist", [61440, 61441, 150000])
def test_batches_around_the_feeders_first_admission(n_hist):
    from mytrim_amd import gpu
    prob = configs.vacancy_case("cu", 1e3, n_hist, seed=13)
    e = gpu.Engine(0)
    try:
        ref = e.run(prob)
        for k in (1, 20, 62):
            e.tune(primary_waves64=k)
            assert_same(ref, e.run(prob))
    finally:
        e.close()


# light ions whose direct recoils overflowed 2^21 slots, or nearly did
@pytest.mark.gpu
@pytest.mark.parametrize("ion,E,target,n", [("C", 2e6, W, 70000), ("He", 1e5, FE, 200000)])
def test_light_ions_through_the_static_queue(ion, E, target, n):
    from mytrim_amd import gpu
    prob = infinite(ion, E, target, n)
    e = gpu.Engine(0)
    try:
        ref, r = e.run(prob), e.run(prob, noalloc=True)
        assert_same(ref, r)
        assert r["queue_peak"] < 0.9 * STATIC_SLOTS / 16
    finally:
        e.close()


# mixed ions, as drawn and with the largest cascades first
@pytest.mark.gpu
@pytest.mark.parametrize("heaviest_first", [False, True])
def test_mixed_ions_through_the_static_queue(heaviest_first):
    from mytrim_amd import gpu
    prob = configs.c4_mixed_uo2(100000, seed=3, w=4000.0, geometry_seed=2345)
    if heaviest_first:
        q = prob.primaries
        o = np.lexsort((-q.E, -q.Z))
        prob = prob.with_(primaries=dataclasses.replace(q, Z=q.Z[o], m=q.m[o], E=q.E[o], pos=q.pos[o], dir=q.dir[o]))
    e = gpu.Engine(0)
    try:
        assert_same(e.run(prob), e.run(prob, noalloc=True))
    finally:
        e.close()


# a queue that keeps its budget, with and without wave roles
@pytest.mark.gpu
@pytest.mark.parametrize("feeders", [1, 20, 63])
def test_small_queue_with_roles(feeders):
    from mytrim_amd import gpu
    e = gpu.Engine(0)
    try:
        for prob in (configs.c1_he_fe(20000, seed=19), configs.c2_cu_cu(300, seed=19)):
            e.tune()
            ref = e.run(prob)
            e.tune(queue_cap=1 << 16, primary_waves64=feeders)
            assert_same(ref, e.run(prob))
            e.tune(primary_waves64=feeders)
            assert_same(ref, e.run(prob, noalloc=True))
    finally:
        e.close()
