"""Device memory of calls that allocate a handle's vectors on first use."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def _used(fn):
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    fn()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0]


def _pages(*doubles):
    page = 2 << 20
    return sum((8 * n + page - 1) // page * page for n in doubles)


def test_gpu_pnorm_gradient_workspace():
    """A large mesh's p-norm gradient takes four node vectors and the block diagonal, and no
    second direction: that belongs to solves of meshes up to 100000 nodes (here 5.6 MB)."""
    from platoanalyze_amd import _capi
    from platoanalyze_amd.elliptic import ElasticModel
    from platoanalyze_amd.mesh import build_box

    def call(dims):
        m = ElasticModel(build_box(*dims, 2.0, 1.0, 1.0), box=dims)
        n = m.num_nodes
        u, z, g = (torch.ones(k, dtype=torch.float64, device="cuda") for k in (3 * n, n, n))

        def gradient():
            m._stream()
            _capi.call("pa_stress_pnorm", m.handle, *(C.c_void_p(t.data_ptr()) for t in (u, z)), 1, 8.0, 0.5, None, None,
                       C.c_void_p(g.data_ptr()))

        return n, gradient

    call((4, 3, 3))[1]()  # the kernels' code is loaded
    n, gradient = call((96, 48, 48))
    used = _used(gradient)
    print(f"workspace of {n} nodes: {used / 2**20:.1f} MB", flush=True)
    assert used <= _pages(3 * n, 3 * n, 3 * n, 3 * n, 9 * n) + (2 << 20)
    assert _used(gradient) <= 0
