"""Calls whose output takes the place of an input (R = U, Ubar = Rbar, Ubar = U) against the same call with a buffer of its
own: the results are the same bit for bit, ghost rows included."""
import numpy as np
import pytest

from ablate_amd import synthetic
from ablate_amd.mesh import BoxMesh, TetBoxMesh
from tests.fvcases import Case, all_outflow, ghost_and_at_face, inflow_x

pytestmark = pytest.mark.gpu

NS = dict(recon="leastsquares", limiter="barthjespersen", mu=0.3, k=2.0, phase=(0.3, 0.2, 0.1))
box = lambda n: BoxMesh([n, n - 2, n - 1], [0, 0, 0], [1, 1, 1], [False, True, True])  # noqa: E731
CASES = {
    # several workgroups each, so that one's writes can meet another's reads
    "species_first_order": lambda: Case("a", box(31), n_species=10, bcs=inflow_x(10), phase=(0.3, 0.2, 0.1)),
    "euler_first_order": lambda: Case("b", box(31), bcs=ghost_and_at_face(), phase=(0.3, 0.2, 0.1)),
    "ns_caller_ghosts": lambda: Case("c", box(23), bcs=ghost_and_at_face(), **NS),
    "ns_species": lambda: Case("d", box(19), n_species=3, diff=0.1, bcs=ghost_and_at_face(3), **NS),
    "tets_outflow": lambda: Case("e", TetBoxMesh(8, 0.2), flux="rusanov", n_species=2, diff=0.1, bcs=all_outflow(6), **NS),
}


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("name", CASES)
def test_rhs_in_place(name, form, torch_cuda):
    torch = torch_cuda
    print(f"[in place] rhs {name} {form}", flush=True)
    case = CASES[name]()
    solver = case.solver(form)
    NI = case.mesh.n_interior
    U0 = torch.tensor(case.initial_state(), device="cuda")
    for strategy in ["tile", "face_flux"]:
        solver.set_strategy(strategy)
        for accumulate in [False, True]:
            U = U0.clone()
            R = U0.clone()
            solver.compute_rhs(0.0, U, R, accumulate=accumulate)
            V = U0.clone()
            solver.compute_rhs(0.0, V, V, accumulate=accumulate)
            assert torch.equal(V[:, :NI], R[:, :NI]), (strategy, accumulate)
            # accumulated in place, the ghost rows are the state's
            assert torch.equal(V[:, NI:], U[:, NI:] if accumulate else R[:, NI:]), (strategy, accumulate)


@pytest.mark.parametrize("onto", ["Rbar", "U"])
@pytest.mark.parametrize("name", CASES)
def test_vjp_in_place(name, onto, torch_cuda):
    torch = torch_cuda
    print(f"[in place] vjp {name} onto {onto}", flush=True)
    case = CASES[name]()
    solver = case.solver()
    U0 = torch.tensor(case.initial_state(), device="cuda")
    Rb0 = torch.tensor(synthetic.adjoint_seed(U0.shape[0], case.mesh.n_cells, case.mesh.n_interior,
                                              cells=case.mesh.source_cells()), device="cuda")
    want = torch.full_like(U0, np.nan)
    theta = solver.rhs_vjp(0.0, U0.clone(), Rb0, want)
    U, Rb = U0.clone(), Rb0.clone()
    out = Rb if onto == "Rbar" else U
    theta2 = solver.rhs_vjp(0.0, U, Rb, out)
    assert torch.equal(out, want)
    np.testing.assert_array_equal(theta, theta2)
