"""ogsx_pattern_footprint is what a system takes from the device: a server admits
systems by it."""
import ctypes as C

import pytest

import ogs5_amd as ox
from ogs5_amd import workloads as W
from devbuf import hip

pytestmark = pytest.mark.gpu


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert hip().hipDeviceSynchronize() == 0
    assert hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _stream_bytes(count=16):
    """What the driver takes for a stream (every system has one)."""
    before = _free_bytes()
    streams = [C.c_void_p() for _ in range(count)]
    for st in streams:
        assert hip().hipStreamCreateWithFlags(C.byref(st), 1) == 0
    taken = before - _free_bytes()
    for st in streams:
        assert hip().hipStreamDestroy(st) == 0
    return taken / count


# one block (with arrays of 1 MiB and more in it, and without), and several
@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("make", [lambda: W.hex_flow(12, n_transient=1, steady=False),
                                  lambda: W.quad_flow(90, 71, n_steps=1),
                                  lambda: W.quad_flow(31, 30, n_steps=1),
                                  lambda: W.hex_flow(17, n_transient=1, steady=False),
                                  lambda: W.hex_flow(40, n_transient=1, steady=False)])
def test_footprint_is_what_systems_take(make, prec):
    sc = make()
    m = sc.mesh
    pat = ox.Pattern(m.n_nodes, m.etype, m.conn)
    each = pat.footprint(prec)
    stream = min(_stream_bytes() for _ in range(2))  # (the first warms up)
    systems = []

    def create(count):
        for _ in range(count):
            s = ox.System(pat, prec)
            s.set_elements(**sc.element_kwargs())
            assert s.device_bytes() == each
            systems.append(s)

    create(4)
    before = _free_bytes()
    create(32)
    taken = (before - _free_bytes()) / 32
    print(f"footprint {each}, taken {taken:.0f}, of it a stream {stream:.0f}")
    # the driver rounds allocations past 1 MiB up to pages of 2 MiB: one of them,
    # or a dozen and more of a system of tens of MB
    assert taken <= (1.0 if each <= (8 << 20) else 1.25) * each + (2 << 20) + max(stream, 4.4e6)
    for s in systems:
        s.close()
