"""Dirichlet elimination on a caller's graph that lists columns more than once: every block of
the constrained rows and columns is cleared, against the oracle's loops."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("repeats", [1, 2, 3])
def test_gpu_constraints_repeated_columns(repeats):
    from platoanalyze_amd.elliptic import ElasticModel, EssentialBC, apply_constraints
    from platoanalyze_amd.mesh import build_box

    print(f"case: constraints with columns listed {repeats} times", flush=True)
    mesh = build_box(5, 3, 3, 2.0, 1.0, 1.0)
    rm, ci = orc.graph(mesh.conn, mesh.num_nodes)
    rng = np.random.default_rng(repeats)
    cols = [rng.permutation(np.repeat(ci[rm[r]:rm[r + 1]], repeats)) for r in range(mesh.num_nodes)]
    rm = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    ci = np.concatenate(cols).astype(np.int32)
    fixed = np.flatnonzero(mesh.coords[:, 0] == 0.0).astype(np.int32)
    bcs = [EssentialBC(fixed, 0, 0.0), EssentialBC(fixed, 1, 0.01), EssentialBC(fixed[::2], 2, -0.02)]
    m = ElasticModel(mesh, 1.0, 0.3, 3.0, 1e-3, bcs, graph=(rm, ci))
    dofs = np.concatenate([3 * fixed, 3 * fixed + 1, 3 * fixed[::2] + 2])
    vals = np.concatenate([np.zeros(len(fixed)), np.full(len(fixed), 0.01), np.full(len(fixed[::2]), -0.02)])
    K, b = rng.normal(size=9 * len(ci)), rng.normal(size=3 * mesh.num_nodes)
    Kc, bc = orc.apply_constraints(rm, ci, K, b, dofs, vals, 0.5)
    dK, db = torch.from_numpy(K.copy()).cuda(), torch.from_numpy(b.copy()).cuda()
    apply_constraints(m, dK, db, 0.5)
    assert np.array_equal(dK.cpu().numpy(), Kc)
    # at most 3 x 45 products of normal values with 0.01 a component
    assert np.abs(db.cpu().numpy() - bc).max() <= 1e-13
