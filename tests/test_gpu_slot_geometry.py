"""Hexes and quads whose cell slots all have their own geometry (jittered centroids), past the limit of the geometry tables in
either precision: the kernels that read the slot-major arrays, periodic (one weight set) and open, against the CPU oracle (FP64
1e-12 per field, as the parity tests; mixed to a rounding bound) and, for the adjoint, against torch.autograd of the independent
restatement (1e-10, as the adjoint tests)."""
import dataclasses

import numpy as np
import pytest
import torch as _torch

from ablate_amd import synthetic
from ablate_amd.mesh import ArrayMesh, BoxMesh
from tests.fvcases import Case, all_outflow, ghost_and_at_face, inflow_x, rel_err_per_field
from tests.test_torch_restatement import PHASE, thetas_of, torch_model2

pytestmark = pytest.mark.gpu

TABLE_LIMIT = 4096  # distinct records of a geometry table (kMaxDistinctRows)


def jittered(cells, periodic):
    """A box with every centroid moved by up to 5 % of a cell (areas, normals and volumes as they were)."""
    box = BoxMesh(cells, [0.0] * len(cells), [1.0] * len(cells), periodic)
    a, dim = box.arrays, len(cells)
    rng = np.random.default_rng(11)
    move = lambda x: x + np.pad(rng.uniform(-0.05, 0.05, (len(x), dim)) / np.array(cells), ((0, 0), (0, 3 - dim)))  # noqa: E731
    mesh = ArrayMesh(dataclasses.replace(a, face_centroid=move(np.array(a.face_centroid)),
                                         cell_centroid=move(np.array(a.cell_centroid))), source=box.source_cells())
    mesh.lower, mesh.upper, mesh.parent = box.lower, box.upper, box  # (box owns the arrays not replaced)
    a = mesh.arrays
    offsets = [a.face_centroid - a.cell_centroid[a.face_cells[:, 0]]]
    inner = a.face_cells[:, 1] < a.n_interior
    shift = a.face_shift if a.face_shift is not None else np.zeros_like(a.face_centroid)
    offsets.append((a.face_centroid - a.cell_centroid[a.face_cells[:, 1]] - shift)[inner])
    assert len(np.unique(np.concatenate(offsets).astype(np.float32)[:, :dim], axis=0)) > TABLE_LIMIT
    return mesh


def halved(cells, periodic, directions):
    """A box whose faces across the given directions come as two halves side by side: cells of more faces."""
    box = BoxMesh(cells, [0.0] * len(cells), [1.0] * len(cells), periodic)
    a, dim = box.arrays, len(cells)
    axis = np.argmax(np.abs(np.asarray(a.face_normal)), axis=1)
    # (a boundary face stays whole: a ghost cell has one face)
    two = np.isin(axis, directions) & (np.asarray(a.face_cells)[:, 1] < a.n_interior)
    of = np.repeat(np.arange(a.n_faces), 1 + two)
    half, second = two[of], np.r_[False, of[1:] == of[:-1]]
    take = lambda x: None if x is None else np.array(x)[of]  # noqa: E731
    normal, centroid = take(a.face_normal), take(a.face_centroid)
    normal[half] *= 0.5
    along = (axis[of] + 1) % dim
    centroid[np.arange(len(of)), along] += np.where(half, np.where(second, 0.25, -0.25) / np.array(cells)[along], 0.0)
    mesh = ArrayMesh(dataclasses.replace(a, n_faces=len(of), face_cells=take(a.face_cells), face_normal=normal,
                                         face_centroid=centroid, face_shift=take(a.face_shift), face_bc=take(a.face_bc)),
                     source=box.source_cells())
    mesh.lower, mesh.upper, mesh.parent = box.lower, box.upper, box  # (box owns the arrays not replaced)
    return mesh


MESHES = {
    "hexes_periodic": lambda: jittered([12, 11, 10], [True] * 3),
    "hexes_open": lambda: jittered([13, 11, 9], [False, True, True]),
    "quads_periodic": lambda: jittered([37, 41], [True, True]),
    "quads_open": lambda: jittered([41, 31], [False, True]),
}
OPEN = {True: inflow_x, False: lambda ns: {}}
NS = dict(recon="leastsquares", mu=0.3, k=2.0, phase=PHASE)


def rounding_bound(case, U0):
    """Per field: what rounding the geometry alone to single precision does to the residual, times the roundings that the
    mixed form puts between a state difference and a flux (differences and weighted sums of up to six slots 8, limiter 4,
    projection 3, flux perturbation 8)."""
    exact, rounded = torch_model2(case), torch_model2(case)
    for name in ["w", "wa", "wg", "dxf", "dxL", "dxR"]:
        t = getattr(rounded, name)
        setattr(rounded, name, t.to(_torch.float32).to(_torch.float64))
    U, thetas = _torch.tensor(U0), thetas_of(case)
    return 23.0 * rel_err_per_field(rounded(U, thetas).numpy(), exact(U, thetas).numpy(), case.mesh.n_interior)


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("limiter", ["barthjespersen", "vanleer", "none"])
@pytest.mark.parametrize("mesh", MESHES)
def test_rhs_with_slot_major_geometry(mesh, limiter, form, torch_cuda):
    torch = torch_cuda
    print(f"[slots] {mesh} {limiter} {form}", flush=True)
    case = Case(mesh, MESHES[mesh](), **NS, limiter=limiter, n_species=2, diff=0.1, bcs=OPEN[mesh.endswith("open")](2))
    U0 = case.initial_state()
    Rref, _ = case.oracle_rhs(U0.copy())
    solver = case.solver(form)
    U = torch.tensor(U0, device="cuda")
    R = torch.zeros_like(U)
    solver.compute_rhs(0.0, U, R)
    err = rel_err_per_field(R.cpu().numpy(), Rref, case.mesh.n_interior)
    bound = 1e-12
    if form == "mixed":  # the restatement knows Barth-Jespersen and no limiter; others round alike
        alike = dataclasses.replace(case, limiter="barthjespersen" if limiter == "vanleer" else limiter)
        bound = rounding_bound(alike, U0)
        print(f"[slots] bound {bound} error {err}", flush=True)
    assert np.all(err <= bound), err


ADJOINT = {
    "hexes_periodic": lambda: Case("a", MESHES["hexes_periodic"](), **NS, limiter="barthjespersen"),
    "hexes_open_species": lambda: Case("b", MESHES["hexes_open"](), **NS, limiter="barthjespersen", n_species=3, diff=0.1,
                                       bcs=inflow_x(3)),
    "hexes_open_unlimited": lambda: Case("c", MESHES["hexes_open"](), **NS, limiter="none",
                                         bcs={0: {"kind": "outflow"}, 1: {"kind": "outflow"}}),
    "hexes_open_ghosts": lambda: Case("d", MESHES["hexes_open"](), **NS, limiter="barthjespersen", n_species=2, diff=0.1,
                                      bcs=ghost_and_at_face(2)),
    "hexes_open_inviscid": lambda: Case("e", MESHES["hexes_open"](), recon="leastsquares", limiter="barthjespersen",
                                        phase=PHASE, bcs=inflow_x()),
    "hexes_viscous_first_order": lambda: Case("f", MESHES["hexes_open"](), mu=0.3, k=2.0, phase=PHASE, bcs=inflow_x()),
    "quads_periodic": lambda: Case("g", MESHES["quads_periodic"](), **NS, limiter="barthjespersen", n_species=1, diff=0.1),
    "quads_open_species": lambda: Case("h", MESHES["quads_open"](), **NS, limiter="barthjespersen", n_species=2, diff=0.1,
                                       bcs=all_outflow(2)),
    # cells of eight and six faces (never in tables)
    "eight_faces": lambda: Case("i", halved([7, 6, 5], [True] * 3, [0]), **NS, limiter="barthjespersen"),
    "eight_faces_open": lambda: Case("j", halved([7, 6, 5], [False, True, True], [0]), **NS, limiter="barthjespersen",
                                     n_species=2, diff=0.1, bcs=ghost_and_at_face(2)),
    "eight_sides": lambda: Case("k", halved([9, 8], [True, True], [0, 1]), **NS, limiter="barthjespersen", n_species=2,
                                diff=0.1),
    "six_sides_open": lambda: Case("l", halved([9, 8], [False, True], [1]), **NS, limiter="none", bcs=inflow_x()),
}


@pytest.mark.parametrize("name", ADJOINT)
def test_adjoint_with_slot_major_geometry(name, torch_cuda):
    torch = torch_cuda
    print(f"[slots] adjoint {name}", flush=True)
    case = ADJOINT[name]()
    U0 = case.initial_state()
    NI = case.mesh.n_interior
    Rb = synthetic.adjoint_seed(U0.shape[0], case.mesh.n_cells, NI, cells=case.mesh.source_cells())
    solver = case.solver()
    U = torch.tensor(U0, device="cuda")
    Ub = torch.full_like(U, np.nan)
    theta_bar = solver.rhs_vjp(0.0, U, torch.tensor(Rb, device="cuda"), Ub)
    Ug = Ub.cpu().numpy()
    Ut = _torch.tensor(U0, requires_grad=True)
    thetas = {s: t.clone().requires_grad_(True) for s, t in thetas_of(case).items()}
    out = torch_model2(case)(Ut, thetas)
    grads = _torch.autograd.grad((out * _torch.tensor(Rb)).sum(), [Ut] + list(thetas.values()))
    ref = grads[0].numpy()
    err = np.linalg.norm(Ug[:, :NI] - ref[:, :NI]) / np.linalg.norm(ref[:, :NI])
    print(f"[slots] adjoint {name} rel err {err:.3e}", flush=True)
    assert err <= 1e-10, err
    np.testing.assert_allclose(Ug[:, NI:], ref[:, NI:], rtol=1e-9, atol=1e-11 * np.abs(ref).max())
    for (slot, _), g in zip(thetas.items(), grads[1:]):
        np.testing.assert_allclose(theta_bar[slot], g.numpy(), rtol=1e-9, atol=1e-12 * np.abs(g.numpy()).max())
