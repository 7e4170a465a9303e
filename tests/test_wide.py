"""GPU: fields of 4 GiB and more, past the shared bricks' 32-bit byte offsets.

520 x 1024 x 1024 points (2^29 + 2^23), flat but for the last 12 planes, which lie on both sides of
a field's byte 2^32: the RHS, the constraints and the derivative maxima there against those of the
last 20 planes taken as a grid of their own, whose fields are 168 MB. Both sum the same terms in the
same order; 1e-12 normwise as for the grids of usual size.
"""
from __future__ import annotations

import pytest
import torch

from conftest import gpu_available

from bssn3d_hip import _lib
from bssn3d_hip.rhs import rhs_into, stream_handle
from bssn3d_hip.state import PhysicsParams, scalars

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a HIP device")]

DEV = "cuda:0"
H3 = (0.1, 0.11, 0.09)
NX, NY, NZ = 520, 1024, 1024
CUT, FLAT = 500, 508               # first plane of the small grid; first plane that is not flat
TOL = 1e-12


def close(big, small):
    """Planes from FLAT to the end, normwise per array, an array at a time (the whole is GBs)."""
    for a, b in zip(big, small):
        x, y = a[FLAT:], b[FLAT - CUT:]
        assert (x - y).abs().max() <= TOL * y.abs().max()


def test_fields_past_4_gib():
    torch.cuda.empty_cache()
    need = (2 * 24 + 8) * NX * NY * NZ * 8
    free = torch.cuda.mem_get_info()[0]
    if free < need:
        pytest.skip(f"needs {need / 1e9:.0f} GB of device memory, {free / 1e9:.0f} GB free")
    print(f"[case] {NX} x {NY} x {NZ}", flush=True)
    F = torch.zeros((24, NX, NY, NZ), dtype=torch.float64, device=DEV)
    for f in (0, 1, 3, 6, 8):
        F[f] = 1.0
    g = torch.Generator(device=DEV).manual_seed(1)
    for f in range(24):
        F[f, FLAT:] += 1e-3 * torch.rand((NX - FLAT, NY, NZ), dtype=torch.float64, device=DEV,
                                         generator=g)
    S = F[:, CUT:].contiguous()
    lib, st, h3 = _lib.load(), stream_handle(F.device), _lib.dbl(H3)
    for order in (4, 6, 8):
        print(f"[case] order {order}", flush=True)
        HM = [torch.empty((4,) + tuple(u.shape[1:]), dtype=torch.float64, device=DEV)
              for u in (F, S)]
        am = [torch.empty(138, dtype=torch.float64, device=DEV) for _ in (F, S)]
        for u, hm, a in zip((F, S), HM, am):
            _lib.check(lib.bssn_constraints_f64(u.data_ptr(), hm.data_ptr(), *u.shape[1:], order,
                                                h3, st))
            _lib.check(lib.bssn_deriv_bundle_absmax_f64(u.data_ptr(), a.data_ptr(), *u.shape[1:],
                                                        order, h3, st))
        close(*HM)
        assert bool((am[0] > 0).all()) and torch.equal(am[0], am[1])
        del HM
    out = [torch.empty_like(u) for u in (F, S)]
    for u, o in zip((F, S), out):
        rhs_into(u, o, scalars(PhysicsParams(), *H3, 0.02, 0.4), 4)
    close(*out)
    del F, S, out
    torch.cuda.empty_cache()
