"""The launches a call makes, by the names the context marks them with."""
import ctypes as C

from phoebus_amd.device import synchronize


def launch_names(phx, call):
    """The names of the launches that call() marks in the context."""
    L, n, ms, name = phx.L, C.c_int(), C.c_float(), C.create_string_buffer(64)
    L.phx_rt_profile_start(phx.h)
    L.phx_rt_profile_reset(phx.h)
    call()
    synchronize()
    L.phx_rt_profile_count(phx.h, C.byref(n))
    out = []
    for i in range(n.value):
        assert L.phx_rt_profile_get(phx.h, i, name, 64, C.byref(ms)) == 0
        out.append(name.value.decode())
    L.phx_rt_profile_stop(phx.h)
    return out
