"""The parts of a device-gated context's close that run without a device: the service thread ends wherever it is stopped
(idle, with a token no step began, with a layer that never exports), and a step of the close that does not end is named."""
import ctypes as C

import pytest

from test_dgcore_parity import OurCore, _lib


@pytest.mark.timeout(60)
@pytest.mark.parametrize("where", range(5))
def test_service_ends_when_stopped(where):
    _, L = _lib()
    halted = C.c_uint32()
    for _ in range(40):
        core = OurCore([8] * 4, 12 + 4, 2, 26, 4, [65536] * 3, list(range(32)), wb_defer=1, inclusive=0)
        try:
            core.tsa.check(L.tsa_test_dgcore_service_stop(core.h, where, C.byref(halted)))
            assert halted.value == 3
        finally:
            core.close()


@pytest.mark.parametrize("slow_ms,want", [(0, ""), (400, "second;")])
def test_a_step_that_lasts_is_named(slow_ms, want):
    tsa, L = _lib()
    out = C.create_string_buffer(256)
    tsa.check(L.tsa_test_close_watch(100, slow_ms, out, 256))
    assert out.value.decode() == want
