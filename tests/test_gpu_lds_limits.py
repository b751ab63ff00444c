"""Targets at the limit of a workgroup's LDS (160 KiB): tables, recoil stacks and
what else a kernel keeps there."""
import dataclasses

import numpy as np
import pytest

import oracle_lib as O
from mytrim_amd import configs, gpu
from mytrim_amd.problem import Element, Material

pytestmark = pytest.mark.gpu


def compound(n, n_hist):
    """n elements in one material, the primary another species: the tables take
    544 + (n + 1) (64 + 392 n) bytes: 72 784 for 13, 150 784 for 19."""
    els = [Element(Z, 2.0 * Z + 1.0, 1.0, 25.0, 3.0) for Z in range(20, 20 + n)]
    return configs.vacancy_case("cu", 1e3, n_hist, seed=7).with_(materials=[Material(7.0, els)])


# one wave per block, 76 B a stack entry (rounded up to 16): 150 784 + 7600 of
# 163 840; all but 48 B; half of the LDS but for 16 B, which takes two blocks
@pytest.mark.parametrize("n_el,blocks,stack_cap", [(19, 1, 100), (19, 1, 171), (13, 2, 120)])
def test_cascades_in_a_full_lds(n_el, blocks, stack_cap):
    prob = compound(n_el, 200)
    e = gpu.Engine(0)
    try:
        e.tune(block=64, blocks_per_cu=blocks, stack_cap=stack_cap, lds_hist=-1)
        r = e.run(prob)
        e.tune(block=64, blocks_per_cu=1, stack_cap=64, lds_hist=-1)
        s = e.run(prob)
        assert r["grid"] == blocks * s["grid"]
        for k in ("n_coll", "n_flight", "vac", "repl", "subst", "inter"):
            assert r[k] == s[k] > 0, k
        assert np.array_equal(r["vac_hist"], s["vac_hist"])
        o = O.run(prob, rng=1, nthreads=4)
        assert r["n_flight"] == pytest.approx(o["n_flight"], rel=0.01)
    finally:
        e.close()


def test_flight_in_a_full_lds():
    """20 elements in 5 materials, the ion one of them: 163 744 of 163 840 bytes."""
    Zs = list(range(20, 40))
    mats = [Material(7.0, [Element(Z, 2.0 * Z + 1.0, 1.0, 25.0, 3.0) for Z in Zs[4 * k:4 * k + 4]]) for k in range(5)]
    base = configs.vacancy_case("cu", 1e3, 1)
    prob = base.with_(materials=mats, geometry=dataclasses.replace(base.geometry, layers=(2.0e4,) * 5))
    u = 1.0 - np.random.default_rng(5).random(40000)
    ion = lambda: gpu.Ion(20, 41.0, 1.0e5, (5.0, 50.0, 50.0), (1.0, 0.0, 0.0), 0, -1, 0, 3.0)
    e = gpu.Engine(0)
    try:
        e.set_target(prob)
        used, ev = e.trim_flight(ion(), u)
        # the layers behind the first one are never reached: the same flight in
        # the first material alone
        e.set_target(prob.with_(materials=mats[:1], geometry=dataclasses.replace(base.geometry, layers=(1.0e5,))))
        used1, ev1 = e.trim_flight(ion(), u)
        assert len(ev) > 10 and max(x.pka_pos[0] for x in ev) < 2.0e4
        assert used == used1 and len(ev) == len(ev1)
        assert all(bytes(a) == bytes(b) for a, b in zip(ev, ev1))
    finally:
        e.close()
