"""A state value that is not finite, one cell away from a boundary cell: the cell's species gradient is not finite, but the
boundary's ghost has no gradient, and its adjoint (inflow parameters, caller-filled ghost rows) stays finite where the face
takes the ghost's side."""
import numpy as np
import pytest

from ablate_amd import synthetic
from ablate_amd.mesh import BoxMesh
from tests.fvcases import Case, ghost_and_at_face, inflow_x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("bcs", [inflow_x, ghost_and_at_face])
def test_ghost_side_adjoint_next_to_a_bad_cell(bcs, value, torch_cuda):
    torch = torch_cuda
    print(f"[nonfinite] {bcs.__name__} {value}", flush=True)
    mesh = BoxMesh([6, 5, 4], [0, 0, 0], [1, 1, 1], [False, True, True], ordering="natural")
    case = Case("c", mesh, recon="leastsquares", limiter="barthjespersen", n_species=2, bcs=bcs(2), phase=(0.3, 0.2, 0.1))
    solver = case.solver()
    cells = np.asarray(mesh.arrays.face_cells)
    boundary = cells[np.asarray(mesh.arrays.face_bc) == 0]
    L, ghost = boundary[7]
    beside = [q for q in np.unique(cells[(cells == L).any(axis=1)]) if q != L and q in boundary[:, 0]]
    U0 = case.initial_state()
    U0[5, beside[0]] = value
    U = torch.tensor(U0, device="cuda")
    Rb = synthetic.adjoint_seed(U0.shape[0], mesh.n_cells, mesh.n_interior, cells=mesh.source_cells())
    Ub = torch.zeros_like(U)
    theta = solver.rhs_vjp(0.0, U, torch.tensor(Rb, device="cuda"), Ub)
    assert not bool(torch.isfinite(Ub[:, int(L)]).all())  # the bad gradient reaches the cell itself
    assert np.isfinite(theta).all()
    assert bool(torch.isfinite(Ub[:, int(ghost)]).all())
