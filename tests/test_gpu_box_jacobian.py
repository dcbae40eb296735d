"""Row-tile Jacobian of Kuhn-split uniform boxes against the general chunk kernel on the same
mesh: lattices smaller and longer than a tile, Hilbert, line by line and random numbering (the
last one falls back to the general lattice kernels), tiles cut short by their box."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# both sides sum at most six terms a block (24 on the diagonal), each a few FP64 roundings;
# the parity tests' own tolerance
RTOL = 1e-12


def _numbered(mesh, dims, order):
    from platoanalyze_amd.mesh import TetMesh

    n = mesh.num_nodes
    if order == "hilbert":
        return mesh
    if order == "lines":
        ijk = np.rint(mesh.coords / (np.array([2.0, 1.5, 1.0]) / np.array(dims))).astype(int)
        old = np.lexsort((ijk[:, 0], ijk[:, 1], ijk[:, 2]))
    elif order == "runs":  # runs of 21 consecutive nodes in random order
        cut = np.random.default_rng(2).permutation((n + 20) // 21)
        old = np.concatenate([np.arange(21 * c, min(n, 21 * c + 21)) for c in cut])
    else:
        old = np.random.default_rng(3).permutation(n)
    new = np.empty(n, np.int64)
    new[old] = np.arange(n)
    return TetMesh(np.ascontiguousarray(mesh.coords[old]), np.ascontiguousarray(new[mesh.conn].astype(np.int32)))


def _close(a, b, what):
    err = float((a - b).abs().max() / b.abs().max())
    assert err <= RTOL, (what, err)


@pytest.mark.parametrize("dims,order", [((1, 1, 1), "hilbert"), ((3, 3, 3), "hilbert"), ((13, 9, 6), "hilbert"),
                                        ((90, 1, 1), "lines"), ((1, 1, 47), "lines"), ((33, 7, 5), "lines"),
                                        ((20, 10, 10), "hilbert"), ((11, 12, 9), "runs"), ((6, 5, 7), "random")])
@pytest.mark.parametrize("model,p", [("SIMP", 3.0), ("SIMP", 2.6), ("Heaviside", 2.0)])
def test_gpu_box_jacobian_tiles(monkeypatch, dims, order, model, p):
    from platoanalyze_amd.elliptic import ElasticModel, EssentialBC, Traction, VectorFunction
    from platoanalyze_amd.mesh import build_box, faces_on_plane, nodes_on_plane

    print(f"case: row tiles {dims} {order} {model} {p}", flush=True)
    mesh = _numbered(build_box(*dims, 2.0, 1.5, 1.0), dims, order)
    fv, fe = faces_on_plane(mesh, 0, 2.0, 1e-9)

    def make():
        return ElasticModel(mesh, 1.7, 0.31, essential_bcs=[EssentialBC(nodes_on_plane(mesh, 0, 0.0), d, 0.0) for d in range(3)],
                            tractions=[Traction(fv, fe, (0.3, -0.2, -1.0))], box=dims, penalty_model=model,
                            penalty_exponent=p, penalty_minimum=1e-3, regularization_length=0.8)

    tiles = make()
    monkeypatch.setenv("PA_BOX_ASSEMBLY", "0")
    general = make()
    assert tiles.box_assembly and not general.box_assembly
    rng = np.random.default_rng(sum(dims))
    u = torch.as_tensor(rng.normal(size=tiles.num_dofs), device="cuda")
    z = torch.as_tensor(rng.uniform(0.05, 0.95, tiles.num_nodes), device="cuda")
    Ra, Rb = torch.full_like(u, np.nan), torch.empty_like(u)
    Ka = VectorFunction(tiles).gradient_u(u, z, residual_out=Ra).entries
    Kb = VectorFunction(general).gradient_u(u, z, residual_out=Rb).entries
    _close(Ka, Kb, "K")
    _close(Ra, Rb, "R")
    assert torch.equal(VectorFunction(tiles).gradient_u(None, z).entries, Ka)
