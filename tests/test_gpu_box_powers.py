"""Uniform Kuhn-split boxes with a power or a sine per tet (non-integer SIMP, Heaviside,
non-integer p-norms), on both sides of the box sizes where they change kernels, against the
general chunk kernels on the same mesh."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# both sides sum at most 24 tets a node, each to a few dozen FP64 roundings; the parity
# tests' own tolerance
RTOL = 1e-12

SIZES = [(37, 35, 35), (38, 35, 35), (76, 35, 35), (79, 35, 35)]  # 49248, 50544, 99792, 103680 nodes
PENALTIES = [("SIMP", 2.6), ("Heaviside", 2.0)]


def _close(got, ref, what):
    err = float((got - ref).abs().max() / ref.abs().max())
    assert err <= RTOL, (what, err)


def _models(monkeypatch, dims, penalty):
    from platoanalyze_amd.elliptic import ElasticModel, EssentialBC, Traction
    from platoanalyze_amd.mesh import build_box, faces_on_plane, nodes_on_plane

    print(f"case: powers on boxes {dims} {penalty}", flush=True)
    mesh = build_box(*dims, 2.0, 1.5, 1.0)
    fv, fe = faces_on_plane(mesh, 0, 2.0, 1e-9)

    def make():
        return ElasticModel(mesh, 1.7, 0.31, penalty[1], 1e-3,
                            [EssentialBC(nodes_on_plane(mesh, 0, 0.0), d, 0.0) for d in range(3)],
                            [Traction(fv, fe, (0.3, -0.2, -1.0))], box=dims, penalty_model=penalty[0],
                            regularization_length=0.8)

    box = make()
    monkeypatch.setenv("PA_BOX_ASSEMBLY", "0")
    general = make()
    assert box.box_assembly and not general.box_assembly
    rng = np.random.default_rng(sum(dims))
    dev = lambda a: torch.as_tensor(a, device="cuda")  # noqa: E731
    return box, general, dev(rng.normal(size=box.num_dofs)), dev(rng.normal(size=box.num_dofs)), dev(
        rng.uniform(0.05, 0.95, box.num_nodes))


@pytest.mark.parametrize("dims", SIZES)
@pytest.mark.parametrize("penalty", PENALTIES)
def test_gpu_box_powers_functions(monkeypatch, dims, penalty):
    from platoanalyze_amd.criteria import StressPNorm, dRdz_T_apply
    from platoanalyze_amd.elliptic import PhysicsScalarFunction, Problem

    a, b, u, lam, z = _models(monkeypatch, dims, penalty)
    fa, fb = PhysicsScalarFunction(a).value(u, z), PhysicsScalarFunction(b).value(u, z)
    assert abs(fa - fb) <= RTOL * fb
    (ga, ca), (gb, cb) = Problem(a).criterionGradient(z, u), Problem(b).criterionGradient(z, u)
    _close(ga, gb, "dC/dz")
    assert abs(ca - cb) <= RTOL * cb
    _close(dRdz_T_apply(a, u, lam, z), dRdz_T_apply(b, u, lam, z), "adjoint product")
    for measure, p, q in (("voigt", 6.0, 0.5), ("von_mises", 3.5, 0.7)):
        pa, pb = StressPNorm(a, p, measure, q), StressPNorm(b, p, measure, q)
        assert abs(pa.value(u, z) - pb.value(u, z)) <= RTOL * pb.value(u, z)
        _close(pa.gradient_u(u, z), pb.gradient_u(u, z), f"{measure} dF/du")
        _close(pa.gradient_z(u, z), pb.gradient_z(u, z), f"{measure} dF/dz")


@pytest.mark.parametrize("dims", SIZES[2:])
@pytest.mark.parametrize("penalty", PENALTIES)
def test_gpu_box_powers_residual(monkeypatch, dims, penalty):
    from platoanalyze_amd.elliptic import PhysicsScalarFunction, VectorFunction

    a, b, u, _, z = _models(monkeypatch, dims, penalty)
    _close(VectorFunction(a).value(u, z), VectorFunction(b).value(u, z), "residual")
    _close(PhysicsScalarFunction(a).gradient_u(u, z), PhysicsScalarFunction(b).gradient_u(u, z), "K u")


@pytest.mark.parametrize("dims", SIZES[2:])
@pytest.mark.parametrize("penalty", PENALTIES)
def test_gpu_box_powers_jacobian(monkeypatch, dims, penalty):
    from platoanalyze_amd.elliptic import VectorFunction

    a, b, u, _, z = _models(monkeypatch, dims, penalty)
    Ra, Rb = torch.full_like(u, np.nan), torch.empty_like(u)
    _close(VectorFunction(a).gradient_u(u, z, residual_out=Ra).entries,
           VectorFunction(b).gradient_u(u, z, residual_out=Rb).entries, "K")
    _close(Ra, Rb, "R")
