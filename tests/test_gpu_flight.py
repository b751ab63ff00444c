"""The single-flight kernel at the edges of its draws and buffers: exactly as many
uniforms or events as the flight needs, one fewer, and draws that give a zero
normal (the reference draws again, trim.C:322-333)."""
import ctypes as C

import numpy as np
import pytest

from mytrim_amd import configs, gpu

pytestmark = pytest.mark.gpu

CASES = {"solid": (configs.c2_cu_cu(1), (29, 63.546, 2.0e4)), "layers": (configs.c3_ag_layers(1), (2, 4.0026, 3.0e4)),
         "wire": (configs.wire_b_si(1), (5, 11.0, 5.0e4)), "moliere": (configs.c2_cu_cu(1).with_(potential=1), (54, 131.29, 1.0e4)),
         "ckr": (configs.c5_c_w(1).with_(potential=2), (6, 12.011, 1.0e4))}


def fly(e, prob, ion, u, max_events=4096):
    Z, m, E = ion
    p = prob.primaries
    io = gpu.Ion(Z, m, E, tuple(float(v) for v in p.pos[0]), tuple(float(v) for v in p.dir[0]), 0, -1, 0, 3.0)
    u = np.ascontiguousarray(u)
    used, n, ev = C.c_longlong(), C.c_int(), (gpu.Event * max_events)()
    rc = gpu.lib().mt_trim_flight(e.h, C.byref(io), u.ctypes.data_as(gpu.dp), len(u), C.byref(used), ev, max_events,
                                  C.byref(n))
    return rc, used.value, n.value, bytes(ev)[:n.value * C.sizeof(gpu.Event)], bytes(io)


@pytest.mark.parametrize("case", sorted(CASES))
def test_flight_edges(case):
    prob, ion = CASES[case]
    u = 1.0 - np.random.default_rng(5).random(40000)
    e = gpu.Engine(0)
    try:
        e.set_target(prob)
        full = fly(e, prob, ion, u)
        rc, used, n, _, _ = full
        assert rc == 0 and n > 1
        assert fly(e, prob, ion, u[:used], n) == full
        assert fly(e, prob, ion, u[:used - 1])[:3] == (-7, used - 1, n - 1)
        assert fly(e, prob, ion, u[:used - 4])[0] == -7
        assert fly(e, prob, ion, u[:1])[:3] == (-7, 1, 0)
        rc, _, got, _, _ = fly(e, prob, ion, u, n - 1)
        assert rc == -7 and got == n - 1
        # a triple at the centre of the ball has no normal: drawn again, the
        # flight is the same; first collision, last collision, both, twice in a row
        zero = np.full(3, 0.5)
        for at in ([3], [used - 3], [3, used - 3], [3, 3]):
            v = np.insert(u, [i for i in at for _ in range(3)], np.tile(zero, len(at)))
            rc, used2, n2, ev2, io2 = fly(e, prob, ion, v)
            assert (rc, used2, n2) == (0, used + 3 * len(at), n)
            assert (ev2, io2) == (full[3], full[4])
        v = np.concatenate([u[:used - 3], zero])
        assert fly(e, prob, ion, v)[:3] == (-7, used, n - 1)
    finally:
        e.close()
