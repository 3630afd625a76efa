"""Meshes that keep each distinct geometry record once (boxes: row numbers per face and cell slot) and meshes past
that table's limit (every face and slot keeps its own record), both against the CPU oracle: FP64 to 1e-12 and mixed
to 1e-6 per field, as the parity tests."""
import dataclasses

import numpy as np
import pytest

from ablate_amd.mesh import ArrayMesh, BoxMesh
from tests.fvcases import Case, inflow_x, rel_err_per_field

pytestmark = pytest.mark.gpu


def stretched(cells, periodic):
    """A box whose coordinates are stretched smoothly per direction, so that nearly every face has its own record."""
    box = BoxMesh(cells, [0.0] * len(cells), [1.0] * len(cells), periodic)
    a, dim = box.arrays, len(cells)
    warp = lambda x: x + 0.05 * np.sin(2.0 * np.pi * x)  # noqa: E731  (keeps the period and the end points)
    n, xf, xc = np.array(a.face_normal), np.array(a.face_centroid), np.array(a.cell_centroid)
    axis = np.argmax(np.abs(n[:, :dim]), axis=1)
    area, vol = np.ones(len(n)), np.ones(len(xc))
    for d, m in enumerate(cells):
        h = 1.0 / m
        width = lambda x: warp(x + 0.5 * h) - warp(x - 0.5 * h)  # noqa: E731
        area *= np.where(axis == d, 1.0, width(xf[:, d]))
        vol *= width(xc[:, d])
        mid = lambda x: 0.5 * (warp(x + 0.5 * h) + warp(x - 0.5 * h))  # noqa: E731
        xf[:, d] = np.where(axis == d, warp(xf[:, d]), mid(xf[:, d]))
        xc[:, d] = mid(xc[:, d])
    normal = np.sign(n) * area[:, None] * (np.abs(n) > 0)
    mesh = ArrayMesh(dataclasses.replace(a, face_normal=normal, face_centroid=xf, cell_centroid=xc, cell_volume=vol),
                     source=box.source_cells())
    mesh.lower, mesh.upper, mesh.parent = box.lower, box.upper, box  # (box owns the arrays not replaced)
    return mesh


NS = dict(recon="leastsquares", limiter="barthjespersen", mu=0.3, k=2.0)
MESHES = {
    "odd": lambda: BoxMesh([13, 11, 9], [0, 0, 0], [1, 1, 1], [False, True, True]),
    "one_block_and_a_cell": lambda: BoxMesh([5, 13, 4], [0, 0, 0], [1, 2, 0.7], [False, True, True]),
    "quads": lambda: BoxMesh([23, 17], [0, 0], [1.3, 0.9], [False, True]),
    "stretched": lambda: stretched([21, 13, 11], [False, True, True]),
    "stretched_quads": lambda: stretched([70, 50], [False, True]),
}


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("limiter", ["barthjespersen", "vanleer"])
@pytest.mark.parametrize("mesh", MESHES)
def test_rhs_with_and_without_geometry_rows(mesh, limiter, form, torch_cuda):
    torch = torch_cuda
    print(f"[rows] {mesh} {limiter} {form}", flush=True)
    case = Case(mesh, MESHES[mesh](), **dict(NS, limiter=limiter), n_species=2, diff=0.1, bcs=inflow_x(2),
                phase=(0.3, 0.2, 0.1))
    U0 = case.initial_state()
    Rref, _ = case.oracle_rhs(U0.copy())
    solver = case.solver(form)
    U = torch.tensor(U0, device="cuda")
    R = torch.zeros_like(U)
    solver.compute_rhs(0.0, U, R)
    err = rel_err_per_field(R.cpu().numpy(), Rref, case.mesh.n_interior)
    assert err.max() <= (1e-12 if form == "fp64" else 1e-6), err


@pytest.mark.parametrize("mesh", ["odd", "stretched"])
def test_adjoint_dot_product(mesh, torch_cuda):
    """<Rbar, R(U + h V) - R(U - h V)> / 2h = <Ubar, V> along V = U, on which R is affine (see the scale check of the
    benchmark's adjoint): the adjoint kernels read the same rows as the forward ones."""
    torch = torch_cuda
    case = Case(mesh, MESHES[mesh](), **NS, bcs={0: {"kind": "outflow"}, 1: {"kind": "outflow"}}, phase=(0.3, 0.2, 0.1))
    solver = case.solver()
    U = torch.tensor(case.initial_state(), device="cuda")
    NI = case.mesh.n_interior
    V = U.clone()
    V[:, NI:] = 0.0
    Rb = torch.zeros_like(U)
    Rb[:, :NI] = torch.randn(U.shape[0], NI, dtype=torch.float64, device="cuda",
                             generator=torch.Generator(device="cuda").manual_seed(3))
    Ub = torch.zeros_like(U)
    solver.rhs_vjp(0.0, U.clone(), Rb, Ub)
    Rp, Rm = torch.zeros_like(U), torch.zeros_like(U)
    h = 1e-3
    solver.compute_rhs(0.0, U + h * V, Rp)
    solver.compute_rhs(0.0, U - h * V, Rm)
    fd = float((Rb * (Rp - Rm)).sum()) / (2 * h)
    assert abs(fd - float((Ub * V).sum())) <= 1e-8 * abs(fd)
