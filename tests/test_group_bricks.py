"""GPU: the fused kernels on bricks shared by four waves (grids of more than 1024 wave-private
bricks), against the oracle and against the wave-private kernels of the batched form, at extents
one short of, on and one past the 4 x 4 x 16 brick, thin axes, and on both sides of the rule that
picks the kernel.

Tolerance 1e-12 normwise per field. The states are sinusoids of 12 to 24 points per wave and
amplitude 0.05 at h ~ 0.1, so second derivatives are ~1 and their rounding error, eps times the
sum of the stencil's weights over h^2 (order 8: 2.2e-16 x 6.5 / 0.0081), is below 2e-13 of the
rates they enter; every other term is smaller.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from conftest import gpu_available, normwise

from bssn3d_hip import _lib
from bssn3d_hip.batch import Block, BlockBatch
from bssn3d_hip.constraints import ConstraintSolver
from bssn3d_hip.evolve import BSSNEvolution
from bssn3d_hip.grid import Grid
from bssn3d_hip.rhs import bfp_buffers, rhs_into, stream_handle
from bssn3d_hip.state import PhysicsParams, scalars

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a HIP device")]

TOL = 1e-12
DEV = "cuda:0"
H3 = (0.1, 0.11, 0.09)
P = PhysicsParams()


def waves(shape, seed, periodic=False, ng=0):
    """24 sinusoids, a whole number of waves per interior axis where periodic."""
    rng = np.random.default_rng(seed)
    F = np.zeros((24,) + tuple(shape))
    for f in range(24):
        arg = rng.uniform(0, 6)
        for a, n in enumerate(shape):
            m = n - 2 * ng
            cycles = max(1, m // 16) if periodic else m / rng.uniform(12, 24)
            x = 2 * np.pi * cycles * (np.arange(n) - ng) / m
            arg = arg + rng.choice([-1, 1]) * x.reshape([-1 if b == a else 1 for b in range(3)])
        F[f] = 0.05 * np.sin(arg)
    for f in (0, 1, 3, 6, 8):
        F[f] += 1.0
    return F


def waves_of(n, ng, seed):
    return waves([v + 2 * ng for v in n], seed, True, ng)


def bricks(shape):
    return int(np.prod([(n + 3) // 4 for n in shape]))


@pytest.mark.parametrize("shape", [(40, 40, 40), (36, 44, 47), (37, 45, 48), (35, 43, 49),
                                   (2, 70, 260), (41, 3, 433), (85, 90, 9)])
@pytest.mark.parametrize("order", [4, 6, 8])
@pytest.mark.parametrize("ko", [0.0, 0.1])
def test_rhs(shape, order, ko):
    print(f"[case] rhs {shape} order {order} ko {ko}", flush=True)
    assert (bricks(shape) > 1024) == (shape != (40, 40, 40))
    F = waves(shape, seed=sum(shape) + order)
    S16 = scalars(P, *H3, 0.02, 0.4)
    Fd = torch.from_numpy(F).to(DEV)
    out = torch.empty_like(Fd)
    rhs_into(Fd, out, S16, order, ko)
    err = normwise(out.cpu().numpy(), O.rhs(F, S16, order, ko_sigma=ko))
    assert err.max() < TOL, err


@pytest.mark.parametrize("interior,order,integrator,bc",
                         [((41, 45, 48), 4, "rk4", "periodic"),
                          ((40, 43, 49), 4, "rk4_2_2", "periodic"),
                          ((44, 42, 47), 6, "rk4", "none"),
                          ((42, 41, 65), 6, "rk4_2_2", "periodic"),
                          ((45, 44, 47), 8, "rk4", "periodic"),
                          ((41, 42, 47), 4, "rk4", "carried"),
                          ((40, 43, 48), 6, "rk4_2_2", "carried")])
def test_steps(interior, order, integrator, bc):
    print(f"[case] {integrator} {interior} order {order} {bc}", flush=True)
    ng = 3 if order == 4 else 4
    grid = Grid(*interior, *H3, ng=ng)
    F = waves(grid.shape, seed=order, periodic=True, ng=ng)
    dt = 0.02
    evo = BSSNEvolution(grid, P, order=order, ko_sigma=0.1, integrator=integrator,
                        bc="none" if bc == "none" else "periodic",
                        ghosts="carried" if bc == "carried" else "synced")
    got = evo.evolve(torch.from_numpy(F).to(DEV), dt, 2, t0=0.1).data.cpu().numpy()
    S16 = scalars(P, *H3, dt, 0.1)
    ref = O.evolve(F, S16, dt, 2, t0=0.1, integrator=integrator, order=order, ko_sigma=0.1,
                   ng=ng, periodic=bc != "none")    # periodic: with the ghosts it carries
    if bc == "periodic":
        ref = O.periodic_sync(ref, ng)
    err = normwise(got, ref)
    assert err.max() < TOL, err


@pytest.mark.parametrize("sizes,order", [([(42, 39, 50)], 4), ([(34, 61, 64)], 6),
                                         ([(16, 17, 15), (12, 20, 33), (9, 16, 16)] * 8, 4),
                                         ([(20, 8, 31), (33, 12, 48)] * 4, 8)])
@pytest.mark.parametrize("waves", [0, 64])
def test_batched_form_equals_single_grid(sizes, order, waves):
    """Blocks through the batched kernels (shared bricks; persistent waves: wave-private bricks)
    and one by one through the single-grid ones: the same bits."""
    print(f"[case] batch {sizes[:3]} order {order} waves {waves}", flush=True)
    ng = 3 if order == 4 else 4
    h = [tuple(v * (1 + 0.1 * (b % 3)) for v in H3) for b in range(len(sizes))]
    batch = BlockBatch([Block(n=n, h=q) for n, q in zip(sizes, h)], ng=ng, device=DEV)
    assert sum(bricks(n) for n in sizes) > 1024
    batch.set_launch(waves)
    U = batch.empty_pool()
    for b, n in enumerate(sizes):
        batch.view(U, b).copy_(torch.from_numpy(waves_of(n, ng, b)))
    start, out = U.clone(), torch.empty_like(U)
    batch.rhs_into(U, out, P, 0.02, order=order, ko_sigma=0.1)
    batch.step_(U, 0.0, 0.02, P, order=order, ko_sigma=0.1, bc="periodic")
    for b, (n, q) in enumerate(zip(sizes, h)):
        F = batch.view(start, b).clone()
        one = torch.empty_like(F)
        rhs_into(F, one, scalars(P, *q, 0.02, 0.0), order, 0.1)
        assert torch.equal(batch.view(out, b), one), b
        BSSNEvolution(Grid(*n, *q, ng=ng), P, order=order, ko_sigma=0.1).step_(F, 0.0, 0.02)
        assert torch.equal(batch.view(U, b), F), b


@pytest.mark.parametrize("n", [(64, 66, 8), (48, 47, 56), (63, 64, 20)])
@pytest.mark.parametrize("order", [4, 6, 8])
@pytest.mark.parametrize("ko", [0.0, 0.1])
def test_grids_of_either_form(n, order, ko):
    """More wave-private bricks than the chip holds, but thin along z or with a last round of
    shared bricks nearly empty, so that the rule keeps some orders and kinds wave-private: the same
    bits as persistent waves on wave-private bricks."""
    print(f"[case] either form {n} order {order} ko {ko}", flush=True)
    ng = 3 if order == 4 else 4
    batch = BlockBatch([Block(n=n, h=H3)], ng=ng, device=DEV)
    batch.set_launch(64)
    U = batch.empty_pool()
    batch.view(U, 0).copy_(torch.from_numpy(waves_of(n, ng, order)))
    F, out = batch.view(U, 0).clone(), torch.empty_like(U)
    one = torch.empty_like(F)
    batch.rhs_into(U, out, P, 0.02, order=order, ko_sigma=ko)
    rhs_into(F, one, scalars(P, *H3, 0.02, 0.0), order, ko)
    assert torch.equal(batch.view(out, 0), one)
    batch.step_(U, 0.0, 0.02, P, order=order, ko_sigma=ko, bc="periodic")
    BSSNEvolution(Grid(*n, *H3, ng=ng), P, order=order, ko_sigma=ko).step_(F, 0.0, 0.02)
    assert torch.equal(batch.view(U, 0), F)


@pytest.mark.parametrize("sizes", [[(16, 16, 8)] * 80, [(9, 9, 13)] * 60,
                                   [(12, 12, 20), (8, 16, 6), (16, 7, 24)] * 14])
@pytest.mark.parametrize("order", [4, 6, 8])
def test_batches_of_either_form(sizes, order):
    """Batches whose blocks leave much of a brick empty, along z (where the rule keeps some orders
    wave-private) or along x and y: the same bits as persistent waves on wave-private bricks."""
    print(f"[case] batch form {sizes[:3]} x {len(sizes)} order {order}", flush=True)
    ng = 3 if order == 4 else 4
    assert sum(bricks(n) for n in sizes) > 1024
    batch = BlockBatch([Block(n=n, h=H3) for n in sizes], ng=ng, device=DEV)
    A = batch.empty_pool()
    for b, n in enumerate(sizes):
        batch.view(A, b).copy_(torch.from_numpy(waves_of(n, ng, b % 5)))
    B, outs = A.clone(), []
    for U, launch in ((A, 0), (B, 64)):
        batch.set_launch(launch)
        outs.append(torch.zeros_like(U))
        batch.rhs_into(U, outs[-1], P, 0.02, order=order, ko_sigma=0.1)
        batch.step_(U, 0.0, 0.02, P, order=order, ko_sigma=0.1, bc="periodic")
    for b in range(len(sizes)):
        assert torch.equal(batch.view(outs[0], b), batch.view(outs[1], b)), b
        assert torch.equal(batch.view(A, b), batch.view(B, b)), b


@pytest.mark.parametrize("shape", [(5, 6, 7), (9, 4, 17), (20, 23, 31), (12, 13, 48)])
@pytest.mark.parametrize("order", [4, 6, 8])
def test_bundle_maxima_and_constraints(shape, order):
    """The derivative bundle, its per-array maxima and the constraints. A derivative's rounding
    error is bounded by eps times the number of roundings (under 64) times the sum of its
    stencil's weights times max|u|; the maxima are those of the stored bundle exactly."""
    print(f"[case] bundle {shape} order {order}", flush=True)
    F = waves(shape, seed=order)
    Fd = torch.from_numpy(F).to(DEV)
    D = torch.empty((138,) + tuple(shape), dtype=torch.float64, device=DEV)
    amax = torch.empty(138, dtype=torch.float64, device=DEV)
    lib, st, h3 = _lib.load(), stream_handle(Fd.device), _lib.dbl(H3)
    _lib.check(lib.bssn_deriv_bundle_f64(Fd.data_ptr(), D.data_ptr(), *shape, order, h3, st))
    _lib.check(lib.bssn_deriv_bundle_absmax_f64(Fd.data_ptr(), amax.data_ptr(), *shape, order,
                                                h3, st))
    assert torch.equal(amax, D.abs().flatten(1).max(dim=1).values)
    got, ref = D.cpu().numpy(), O.deriv_bundle(F, list(H3), order)
    c1, c2 = (np.abs(O.stencil(k, order)).sum() for k in (0, 1))
    for d in range(138):
        if d < 72:
            f, a = divmod(d, 3)
            mag = c1 / H3[a]
        else:
            s, q = divmod(d - 72, 6)
            f = O.IDX[O.S2_FIELDS[s]]
            i, j = O.PAIRS[q]
            mag = c2 / H3[i] ** 2 if i == j else c1 * c1 / (H3[i] * H3[j])
        assert np.abs(got[d] - ref[d]).max() <= 64 * 2.2e-16 * mag * np.abs(F[f]).max(), d
    grid = Grid(*[max(n - 2 * 2, 1) for n in shape], *H3, ng=(order // 2))
    C = ConstraintSolver(grid, order=order).constraints(Fd)
    err = normwise(torch.stack([C[k] for k in ("H", "M0", "M1", "M2")]).cpu().numpy(),
                   O.constraints(F, list(H3), order))
    assert err.max() < TOL, err


@pytest.mark.parametrize("shape", [(24, 23, 25), (40, 40, 40), (41, 45, 49), (48, 47, 56),
                                   (70, 72, 8), (33, 130, 16)])
@pytest.mark.parametrize("order", [4, 6, 8])
def test_constraints_of_either_form(shape, order):
    """The constraints on both sides of the rule that picks their form."""
    print(f"[case] constraints {shape} order {order}", flush=True)
    F = waves(shape, seed=order)
    grid = Grid(*[n - 4 for n in shape], *H3, ng=order // 2)
    C = ConstraintSolver(grid, order=order).constraints(torch.from_numpy(F).to(DEV))
    err = normwise(torch.stack([C[k] for k in ("H", "M0", "M1", "M2")]).cpu().numpy(),
                   O.constraints(F, list(H3), order))
    assert err.max() < TOL, err


@pytest.mark.parametrize("shape", [(150, 90, 7), (290, 130, 4), (41, 45, 49)])
@pytest.mark.parametrize("order", [4, 6, 8])
def test_bundle_of_either_form(shape, order):
    """The bundle thin along z (wave-private bricks) and not, in each storage, against the oracle's
    with the bound of a derivative's rounding error above. The maxima, which have one form, are
    those of the stored bundle exactly, over more bricks than they have workgroups; BFP storage
    holds the fp64 bundle's values at 2^-e."""
    print(f"[case] bundle {shape} order {order}", flush=True)
    F = waves(shape, seed=order)
    Fd = torch.from_numpy(F).to(DEV)
    D = torch.empty((138,) + tuple(shape), dtype=torch.float64, device=DEV)
    amax = torch.empty(138, dtype=torch.float64, device=DEV)
    lib, st, h3 = _lib.load(), stream_handle(Fd.device), _lib.dbl(H3)
    _lib.check(lib.bssn_deriv_bundle_f64(Fd.data_ptr(), D.data_ptr(), *shape, order, h3, st))
    _lib.check(lib.bssn_deriv_bundle_absmax_f64(Fd.data_ptr(), amax.data_ptr(), *shape, order,
                                                h3, st))
    assert torch.equal(amax, D.abs().flatten(1).max(dim=1).values)
    got, ref = D.cpu().numpy(), O.deriv_bundle(F, list(H3), order)
    c1, c2 = (np.abs(O.stencil(k, order)).sum() for k in (0, 1))
    for d in range(138):
        if d < 72:
            f, a = divmod(d, 3)
            mag = c1 / H3[a]
        else:
            s, q = divmod(d - 72, 6)
            f = O.IDX[O.S2_FIELDS[s]]
            i, j = O.PAIRS[q]
            mag = c2 / H3[i] ** 2 if i == j else c1 * c1 / (H3[i] * H3[j])
        assert np.abs(got[d] - ref[d]).max() <= 64 * 2.2e-16 * mag * np.abs(F[f]).max(), d
    e = [int(v) for v in 24 - np.frexp(amax.cpu().numpy())[1]]
    Q, _ = bfp_buffers(Fd, 32)
    _lib.check(lib.bssn_deriv_bundle_bfp(Fd.data_ptr(), Q.data_ptr(), (ctypes.c_int * 138)(*e), 32,
                                         *shape, order, h3, st))
    scale = torch.tensor([2.0 ** v for v in e], dtype=torch.float64, device=DEV)
    stored = Q[Q.numel() - 4 * D.numel():].view(torch.int32).view(D.shape)   # after the header
    assert torch.equal(stored.double(), torch.round(D * scale.view(-1, 1, 1, 1)))
