"""Function batches through the mapped chunks (2^16 elements each): sizes at the
edges of a chunk and of the second, against the same elements in other chunks,
and tables too large for a block's LDS."""
import numpy as np
import pytest

import oracle_lib as O
from mytrim_amd import configs, gpu
from mytrim_amd.problem import Element, Material

pytestmark = pytest.mark.gpu
CHUNK = 1 << 16


@pytest.mark.parametrize("n", [1, 97, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK, 3 * CHUNK + 5])
def test_batches_by_chunk(n):
    rng = np.random.default_rng(n)
    e = gpu.Engine(0)
    try:
        e.set_target(configs.c2_cu_cu(1))
        E = np.exp(rng.uniform(np.log(10.0), np.log(1e7), n))
        eps, b = np.exp(rng.uniform(np.log(1e-4), np.log(30.0), n)), 8.0 * np.sqrt(1.0 - rng.random(n))
        se, sc = e.stopping(6, 12.011, 0, E), e.scatter(eps, b)
        for i in {0, n // 2, n - 1, min(n - 1, CHUNK - 1), min(n - 1, CHUNK)}:
            assert se[i] == e.stopping(6, 12.011, 0, E[i:i + 1])[0]
            assert [x[i] for x in sc] == [x[0] for x in e.scatter(eps[i:i + 1], b[i:i + 1])]
        m = min(n, 200)
        ref = np.array([O.getrstop(6, 12.011, x, 8.96, [(29, 63.546, 1.0)]) for x in E[-m:]])
        assert np.max(np.abs(se[-m:] - ref) / ref) < 1e-12
        assert np.all(np.isfinite(sc[0])) and np.all(sc[3] >= 0)
    finally:
        e.close()


def test_tables_past_lds():
    """16 elements of one compound: 17 species x 16 elements of constants."""
    els = [Element(Z, 2.0 * Z + 1.0, 1.0, 25.0, 3.0) for Z in range(20, 36)]
    prob = configs.c2_cu_cu(1).with_(materials=[Material(7.0, els)])
    E = np.geomspace(10.0, 1e7, 300)
    e = gpu.Engine(0)
    try:
        e.set_target(prob)
        se = e.stopping(54, 131.29, 0, E)
        ref = np.array([O.getrstop(54, 131.29, x, 7.0, [(el.Z, el.m, el.t) for el in els]) for x in E])
        assert np.max(np.abs(se - ref) / ref) < 1e-12
    finally:
        e.close()


@pytest.mark.parametrize("n_el", [2, 16])
def test_repeated_calls_agree(n_el):
    """A context's first small batches, its later ones and large ones take other
    ways to the kernel; tables of 16 elements do not go to LDS."""
    els = [Element(Z, 2.0 * Z + 1.0, 1.0, 25.0, 3.0) for Z in range(20, 20 + n_el)]
    prob = configs.c2_cu_cu(1).with_(materials=[Material(7.0, els)])
    E = np.geomspace(10.0, 1e7, 2 * CHUNK + 3)
    e, whole = gpu.Engine(0), gpu.Engine(0)
    try:
        e.set_target(prob)
        whole.set_target(prob)
        ref = whole.stopping(54, 131.29, 0, E)
        for n in (1, 2048, 2049, 2047, 97, CHUNK + 1, 5):
            assert np.array_equal(e.stopping(54, 131.29, 0, E[:n]), ref[:n]), n
            assert np.array_equal(e.stopping(54, 131.29, 0, E[-n:]), ref[-n:]), n
        m = ref[::CHUNK]
        exact = np.array([O.getrstop(54, 131.29, x, 7.0, [(el.Z, el.m, el.t) for el in els]) for x in E[::CHUNK]])
        assert np.max(np.abs(m - exact) / exact) < 1e-12
    finally:
        e.close()
        whole.close()


def test_outputs_over_later_inputs():
    """Results written over inputs that a later chunk reads, or over their own."""
    n, shift = 3 * CHUNK + 5, CHUNK + 4321
    rng = np.random.default_rng(3)
    E = np.exp(rng.uniform(np.log(10.0), np.log(1e7), n))
    eps, b = np.exp(rng.uniform(np.log(1e-4), np.log(30.0), n)), 8.0 * np.sqrt(1.0 - rng.random(n))
    L, p = gpu.lib(), lambda a: a.ctypes.data_as(gpu.dp)
    e = gpu.Engine(0)
    try:
        e.set_target(configs.c2_cu_cu(1))
        se, sc = e.stopping(6, 12.011, 0, E), e.scatter(eps, b)
        for s in (0, shift):
            buf = np.concatenate([E, np.zeros(s)])
            assert L.mt_stopping_batch(e.h, 6, 12.011, 0, p(buf), n, p(buf[s:])) == 0
            assert np.array_equal(buf[s:s + n], se)
            buf, bb = np.concatenate([eps, np.zeros(s)]), b.copy()
            ct, st, it = np.zeros(n), np.zeros(n), np.zeros(n, np.int32)
            assert L.mt_scatter_batch(e.h, 0, p(buf), p(bb), n, p(buf[s:]), p(ct), p(st), it.ctypes.data_as(gpu.ip)) == 0
            for got, want in zip((buf[s:s + n], ct, st, it), sc):
                assert np.array_equal(got, want)
    finally:
        e.close()
