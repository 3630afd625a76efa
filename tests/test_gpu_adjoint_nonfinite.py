"""Adjoints of states that are not finite in one cell beside a boundary cell: they spread as far as the terms read the value,
not through ghosts and left-out slots that stand in for each other in the kernels' loads."""
import numpy as np
import pytest

from ablate_amd import synthetic
from ablate_amd.mesh import BoxMesh
from tests.fvcases import Case, all_outflow, ghost_and_at_face, inflow_x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("bcs", [inflow_x, ghost_and_at_face])
def test_ghost_side_adjoint_next_to_a_bad_cell(bcs, value, torch_cuda):
    """The bad cell's neighbour has no finite species gradient, but the ghost behind it has none at all: its adjoint (inflow
    parameters, caller-filled ghost rows) stays finite where the face takes the ghost's side."""
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


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("mesh", ["quads", "hexes"])
def test_bad_energy_reaches_its_own_density_adjoint(mesh, value, torch_cuda):
    """Without an advection flux the temperature gradients alone read the energy, linearly: of all adjoints only the density's
    at the same cell holds its value."""
    torch = torch_cuda
    print(f"[nonfinite] {mesh} {value}", flush=True)
    box = BoxMesh([7, 5], [0, 0], [1, 1], [False, True]) if mesh == "quads" else BoxMesh([4, 5, 3], [0, 0, 0], [1, 1, 1],
                                                                                       [False, True, True])
    case = Case("c", box, flux="off", mu=0.5, k=5.0, bcs=all_outflow(2))
    solver = case.solver()
    U0 = case.initial_state()
    Rb = synthetic.adjoint_seed(U0.shape[0], box.n_cells, box.n_interior, cells=box.source_cells())
    for cell in range(box.n_interior):
        U1 = U0.copy()
        U1[1, cell] = value
        Ub = torch.zeros(U0.shape, dtype=torch.float64, device="cuda")
        solver.rhs_vjp(0.0, torch.tensor(U1, device="cuda"), torch.tensor(Rb, device="cuda"), Ub)
        bad = np.argwhere(~np.isfinite(Ub.cpu().numpy()[:, : box.n_interior])).tolist()
        assert bad == [[0, cell]], (cell, bad)
