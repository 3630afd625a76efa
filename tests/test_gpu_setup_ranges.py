"""Meshes beyond 65536 cells and faces, whose layout (face geometry, least-squares weights) is built in several ranges at
once: the right-hand side by the strategies that read it against the CPU oracle, to the parity tests' 1e-12."""
import pytest

from ablate_amd.mesh import BoxMesh, TetBoxMesh
from tests.fvcases import Case, all_outflow, inflow_x, rel_err_per_field

pytestmark = pytest.mark.gpu

NS = dict(recon="leastsquares", limiter="barthjespersen", mu=0.3, k=2.0, phase=(0.3, 0.2, 0.1))
CASES = {
    "open_hexes": lambda: Case("a", BoxMesh([71, 43, 23], [0, 0, 0], [1, 1, 1], [False, True, True]), bcs=inflow_x(), **NS),
    "tets": lambda: Case("b", TetBoxMesh(23, 0.2), flux="rusanov", bcs=all_outflow(6), **NS),
}


@pytest.mark.parametrize("name", CASES)
def test_rhs_of_a_layout_built_in_ranges(name, torch_cuda):
    torch = torch_cuda
    print(f"[ranges] {name}", flush=True)
    case = CASES[name]()
    assert case.mesh.n_interior > 1 << 16
    U0 = case.initial_state()
    Rref, _ = case.oracle_rhs(U0.copy())
    solver = case.solver()
    U = torch.tensor(U0, device="cuda")
    for strategy in ["tile", "face_flux", "fused", "march"]:
        if not solver.has_strategy(strategy):
            continue
        solver.set_strategy(strategy)
        R = torch.zeros_like(U)
        solver.compute_rhs(0.0, U, R)
        err = rel_err_per_field(R.cpu().numpy(), Rref, case.mesh.n_interior)
        assert err.max() <= 1e-12, (strategy, err)
