"""Calls that return with work queued on the handle's scratch, followed by calls on other
streams: the later call waits for that work, whatever handle value its stream has."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DIMS = (48, 24, 24)


def _model(box=True):
    from platoanalyze_amd.elliptic import ElasticModel, EssentialBC
    from platoanalyze_amd.mesh import build_box, nodes_on_plane

    mesh = build_box(*DIMS, 2.0, 1.0, 1.0)
    fixed = nodes_on_plane(mesh, 0, 0.0)
    m = ElasticModel(mesh, 1.0, 0.3, essential_bcs=[EssentialBC(fixed, d, 0.0) for d in range(3)], box=DIMS if box else None)
    rng = np.random.default_rng(11)
    u = torch.as_tensor(rng.normal(size=m.num_dofs), device="cuda")
    z = torch.as_tensor(rng.uniform(0.2, 0.9, m.num_nodes), device="cuda")
    return m, u, z


def test_gpu_stream_created_after_a_destroyed_one():
    from platoanalyze_amd import _capi
    from platoanalyze_amd.criteria import StressPNorm

    m, u, z = _model()
    f = StressPNorm(m, 8.0, "von_mises", 0.5)
    v = 2.0 * u
    want = f.gradient_u(u, z), f.value(v, z)
    torch.cuda.synchronize()
    hip = _capi.lib()  # symbols of the runtime it is linked to
    hip.hipStreamCreate.argtypes, hip.hipStreamDestroy.argtypes = [C.c_void_p], [C.c_void_p]
    seen, got = set(), []
    for k in range(6):
        s = C.c_void_p()
        assert hip.hipStreamCreate(C.byref(s)) == 0
        seen.add(s.value)
        _capi.call("pa_set_stream", m.handle, s)
        if k % 2 == 0:
            g = torch.empty_like(u)
            torch.cuda.synchronize()
            _capi.call("pa_stress_pnorm", m.handle, C.c_void_p(u.data_ptr()), C.c_void_p(z.data_ptr()), 1, 8.0, 0.5,
                       None, C.c_void_p(g.data_ptr()), None)
            got.append(g)
        else:
            value = C.c_double()
            _capi.call("pa_stress_pnorm", m.handle, C.c_void_p(v.data_ptr()), C.c_void_p(z.data_ptr()), 1, 8.0, 0.5,
                       C.byref(value), None, None)
            assert value.value == want[1]
        assert hip.hipStreamDestroy(s) == 0
    print("stream handles:", len(seen), "of 6", flush=True)
    torch.cuda.synchronize()
    for g in got:
        assert float((g - want[0]).abs().max()) <= 1e-12 * float(want[0].abs().max())
