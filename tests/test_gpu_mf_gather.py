"""FP32 matrix-free operator of general meshes by row sums of element forces kept in LDS,
through the mixed-precision solves that use it: chunks smaller than a work-group, several
chunks, shuffled node numbers (full node tables), and a fan of tets around an axis whose
chunk has too many elements for LDS and takes the atomic sums; and the FP64 element kernels
of general meshes with long element lists."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _graded(dims, shuffle):
    from platoanalyze_amd.mesh import TetMesh, build_box

    m = build_box(*dims, 2.0, 1.0, 1.0)
    x = m.coords * (1.0 + 0.2 * np.sin(m.coords))
    if not shuffle:
        return TetMesh(np.ascontiguousarray(x), m.conn)
    new = np.random.default_rng(4).permutation(m.num_nodes)
    y = np.empty_like(x)
    y[new] = x
    return TetMesh(y, np.ascontiguousarray(new[m.conn].astype(np.int32)))


def _fan(n):
    """n wedges around the z axis, three layers of tets each."""
    from platoanalyze_amd.mesh import TetMesh

    layers = 3
    a = 2 * np.pi * np.arange(n) / n
    ring = np.stack([np.cos(a), np.sin(a)], 1)
    nodes, conn = [], []
    for k in range(layers + 1):
        nodes += [[0.0, 0.0, k]] + [[p[0], p[1], k] for p in ring]
    w = n + 1
    for k in range(layers):
        for i in range(n):
            p = [k * w, k * w + 1 + i, k * w + 1 + (i + 1) % n]
            q = [v + w for v in p]
            conn += [[p[0], p[1], p[2], q[2]], [p[0], p[1], q[2], q[1]], [p[0], q[1], q[2], q[0]]]
    x = np.array(nodes, float)
    c = np.array(conn, np.int32)
    d = np.linalg.det(x[c[:, 1:]] - x[c[:, :1]])
    c[d < 0] = c[d < 0][:, [0, 2, 1, 3]]
    return TetMesh(x, c)


@pytest.mark.parametrize("mesh", ["one", "small", "chunks", "shuffled", "fan"])
def test_gpu_mf_gather_solutions(mesh):
    """Against the FP64 solve.  Both stop at 1e-10 of the load; the condition numbers of
    these meshes are below 1e4, so the solutions agree to 1e-6."""
    from platoanalyze_amd.elliptic import ElasticModel, EssentialBC, Problem, Traction
    from platoanalyze_amd.mesh import faces_on_plane, nodes_on_plane

    print(f"case: matrix-free rows {mesh}", flush=True)
    m = {"one": lambda: _graded((1, 1, 1), False), "small": lambda: _graded((3, 2, 2), False),
         "chunks": lambda: _graded((17, 9, 8), False), "shuffled": lambda: _graded((9, 8, 7), True),
         "fan": lambda: _fan(50)}[mesh]()
    x = m.coords
    fv, fe = faces_on_plane(m, 2, float(x[:, 2].max()), 1e-9)
    model = ElasticModel(m, 1.0, 0.3, essential_bcs=[EssentialBC(nodes_on_plane(m, 2, 0.0), d, 0.0) for d in range(3)],
                         tractions=[Traction(fv, fe, (0.3, -0.2, -1.0))])
    z = torch.as_tensor(np.random.default_rng(1).uniform(0.3, 1.0, m.num_nodes), device="cuda")
    u = {p: Problem(model, tolerance=1e-10, precision=p).solution(z) for p in ("fp64", "mixed")}
    assert float((u["mixed"] - u["fp64"]).norm() / u["fp64"].norm()) < 1e-6


@pytest.mark.parametrize("times", [3, 12])
@pytest.mark.parametrize("penalty", [("SIMP", 3.0), ("SIMP", 1.0), ("RAMP", 3.0)])
def test_gpu_element_kernels_long_lists(times, penalty):
    """A mesh whose elements are listed several times is several meshes: the density
    gradients gather from LDS (3 times: up to 2400 entries a chunk) or add with atomics (12
    times).  Both sides are FP64 sums of at most a few hundred terms a node."""
    from platoanalyze_amd.criteria import StressPNorm, dRdz_T_apply
    from platoanalyze_amd.elliptic import ElasticModel, EssentialBC, PhysicsScalarFunction, VectorFunction
    from platoanalyze_amd.mesh import TetMesh, nodes_on_plane

    print(f"case: long element lists x{times} {penalty}", flush=True)
    m = _graded((9, 8, 7), False)
    many = TetMesh(m.coords, np.ascontiguousarray(np.repeat(m.conn, times, axis=0)))
    one, more = (ElasticModel(x, 1.0, 0.3, essential_bcs=[EssentialBC(nodes_on_plane(x, 2, 0.0), 0, 0.0)],
                              penalty_model=penalty[0], penalty_exponent=penalty[1]) for x in (m, many))
    rng = np.random.default_rng(6)
    u, lam = (torch.as_tensor(rng.normal(size=one.num_dofs), device="cuda") for _ in range(2))
    z = torch.as_tensor(rng.uniform(0.2, 0.9, one.num_nodes), device="cuda")

    def close(a, b):
        assert float((a - times * b).abs().max() / (times * b).abs().max()) < 1e-12

    close(PhysicsScalarFunction(more).gradient_z(u, z), PhysicsScalarFunction(one).gradient_z(u, z))
    close(dRdz_T_apply(more, u, lam, z), dRdz_T_apply(one, u, lam, z))
    close(VectorFunction(more).value(u, z), VectorFunction(one).value(u, z))
    close(VectorFunction(more).gradient_u(u, z).entries, VectorFunction(one).gradient_u(u, z).entries)
    a, b = StressPNorm(more, 1.0, "von_mises", 0.5), StressPNorm(one, 1.0, "von_mises", 0.5)
    close(a.gradient_u(u, z), b.gradient_u(u, z))
    close(a.gradient_z(u, z), b.gradient_z(u, z))
