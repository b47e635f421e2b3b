"""The C++ task mirror (phoebus_amd/host/phx_host.hpp), called through its exported symbols:
update::UpdateFillDerived, which the one-block driver runs, equals the three tasks that it
stands for, fluid::FluxCT, update::FluxDivergenceUpdate and fluid::ConservedToPrimitive."""
import ctypes as C
import sys

import numpy as np
import pytest

import _physics as PH
from phoebus_amd import _abi as A
from phoebus_amd.api import Phx, block, block_shape, fluid_params, mgr
from phoebus_amd.device import synchronize

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def phx():
    ctx = Phx(0)
    yield ctx
    ctx.close()


class MeshBlockData:
    """A phx::host::MeshBlockData with two containers, its primitives set on the entire block."""

    def __init__(self, phx, p, b, prim):
        self.L, self.mem = phx.L, C.create_string_buffer(8192)  # room for the object
        self.this = C.c_void_p((C.addressof(self.mem) + 63) // 64 * 64)
        self._call("13MeshBlockDataC1EP7phx_ctxRK16phx_fluid_paramsRK9phx_blocki", None,
                   C.c_void_p(phx.h), C.byref(p), C.byref(b), C.c_int(2))
        self.sh, self.nc, self.np_ = block_shape(b), 8 if p.mhd else 5, 10 if p.mhd else 7
        f = self.fields(0)
        assert f.prim
        q = np.ascontiguousarray(prim)
        assert self.L.phx_rt_memcpy_htod(f.prim, q.ctypes.data, q.nbytes) == 0

    def _call(self, name, res, *args, const=False):
        fn = self.L["_ZN" + ("K" if const else "") + "3phx4host" + name]
        fn.restype, fn.argtypes = res, [C.c_void_p] + [type(a) if not hasattr(a, "_obj") else
                                                       C.c_void_p for a in args]
        return fn(self.this, *args)

    def task(self, name, *args):
        assert self._call(name, C.c_int, *args) == 0, name  # TaskStatus::complete

    def fields(self, container):
        return self._call("13MeshBlockData6fieldsEi", A.BlockFields, C.c_int(container),
                          const=True)

    def close(self):
        self._call("13MeshBlockDataD1Ev", None)

    def snapshot(self):
        synchronize()
        f, out = self.fields(0), {}
        for name, ptr, n in (("prim", f.prim, self.np_), ("cons0", f.cons, self.nc),
                             ("cons1", self.fields(1).cons, self.nc), ("temp", f.temp, 1),
                             ("mu", f.c2p_mu, 1), ("fail", f.fail, 1),
                             ("cell_sig", f.cell_sig, 3)):
            out[name] = np.empty((n,) + self.sh)
            assert self.L.phx_rt_memcpy_dtoh(out[name].ctypes.data, ptr, out[name].nbytes) == 0
        return out


DATA = "EPNS0_13MeshBlockDataE"
CASES = [(A.GEOM_MINKOWSKI, False, (37,)), (A.GEOM_MINKOWSKI, False, (9, 8, 7)),
         (A.GEOM_MINKOWSKI, True, (19,)), (A.GEOM_MINKOWSKI, True, (17, 9)),
         (A.GEOM_MINKOWSKI, True, (10, 9, 8)), (A.GEOM_SPHERICAL_KS, False, (11, 9)),
         (A.GEOM_SPHERICAL_KS, True, (12, 10)), (A.GEOM_FMKS, True, (9, 8, 10))]


@pytest.mark.parametrize("geom,mhd,nx", CASES)
def test_update_fill_derived_is_its_three_tasks(phx, geom, mhd, nx):
    say(f"[gpu] UpdateFillDerived vs its tasks, geom {geom} mhd {mhd} {nx}")
    xmin, dx = {A.GEOM_MINKOWSKI: ((0.0,) * 3, (0.1, 0.2, 0.3)),
                A.GEOM_SPHERICAL_KS: ((4.0, 0.6, 0.0), (0.25, 0.05, 0.05)),
                A.GEOM_FMKS: ((1.4, 0.3, 0.0), (0.05, 0.02, 0.05))}[geom]
    b = block(len(nx), nx, 4, xmin=xmin, dx=dx)
    p = fluid_params(gamma=13.0 / 9.0, mhd=mhd, geom=geom, a=0.9375,
                     floors=dict(rho0=1e-6, sie0=1e-6), ceilings=(50.0, 100.0),
                     mgr_params=mgr(derefine_poles=False, h=0.3))
    sh = block_shape(b)
    prim = PH.random_prims(np.random.default_rng(sum(nx)), int(np.prod(sh)), mhd, 13.0 / 9.0,
                           wmax=2.0)
    if geom != A.GEOM_MINKOWSKI:
        prim[1:4] *= 0.1
        prim[5:8] *= 0.1 if mhd else 1.0
    prim = prim.reshape((-1,) + sh)
    one, many = (MeshBlockData(phx, p, b, prim) for _ in range(2))
    dt = C.c_double(1e-4)
    for m in (one, many):
        for c in (0, 1):
            m.task("5fluid20PrimitiveToConservedEPNS0_13MeshBlockDataEi", C.c_int(c))
    # the two stages of a step: U^n (0) to U_1 (1), then U_1 and U^n to U^{n+1} (0)
    for s_in, beta, s_out in ((0, 1.0, 1), (1, 0.5, 0)):
        for m in (one, many):
            m.task("5fluid15CalculateFluxes" + DATA)
            if geom != A.GEOM_MINKOWSKI:
                m.task("5fluid25CalculateFluidSourceTerms" + DATA)
        upd = (C.c_int(s_in), C.c_int(0), C.c_double(beta), dt, C.c_int(s_out))
        one.task("6update17UpdateFillDerivedEPNS0_13MeshBlockDataEiiddi", *upd)
        many.task("5fluid6FluxCT" + DATA)
        many.task("6update20FluxDivergenceUpdateEPNS0_13MeshBlockDataEiiddi", *upd)
        many.task("5fluid20ConservedToPrimitiveEPNS0_13MeshBlockDataEi", C.c_int(s_out))
        a, w = one.snapshot(), many.snapshot()
        for name in w:
            assert np.array_equal(a[name], w[name], equal_nan=True), (beta, name)
    assert np.any(a["cons0"] != 0.0) and np.mean(a["fail"]) > 0.5
    one.close()
    many.close()
