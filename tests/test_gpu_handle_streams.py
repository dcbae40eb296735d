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


def _volume_gradient(m, z):
    """Volume's dV/dz without the value, which leaves partial sums queued."""
    from platoanalyze_amd import _capi

    g = torch.empty_like(z)
    m._stream()
    _capi.call("pa_volume", m.handle, C.c_void_p(z.data_ptr()), 0, 3.0, 1e-3, 1.0, None, C.c_void_p(g.data_ptr()), None)
    return g


@pytest.mark.parametrize("path", ["bricks", "lattice", "chunks"])
def test_gpu_gradients_then_values_on_another_stream(monkeypatch, path):
    from platoanalyze_amd.elliptic import PhysicsScalarFunction, VectorFunction, Volume

    print(f"case: queued gradients, then values on another stream, {path}", flush=True)
    if path == "lattice":
        monkeypatch.setenv("PA_BOX_RES_KUHN", "0")
        monkeypatch.setenv("PA_BOX_JAC_KUHN", "0")
    m, u, z = _model(path != "chunks")
    f, vf, vol = PhysicsScalarFunction(m), VectorFunction(m), Volume(m, "SIMP", 3.0, 1e-3)
    v, w = 2.0 * u, 0.5 * z
    want = [f.gradient_z(v, z), f.value(u, z), _volume_gradient(m, w), vol.value(z), vf.value(v, z), vf.value(u, w)]
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(6):
        with torch.cuda.stream(a):
            gz = f.gradient_z(v, z)
        with torch.cuda.stream(b):
            energy = f.value(u, z)
        with torch.cuda.stream(a):
            gv = _volume_gradient(m, w)
        with torch.cuda.stream(b):
            volume = vol.value(z)
        with torch.cuda.stream(a):
            r0 = vf.value(v, z)
        with torch.cuda.stream(b):
            r1 = vf.value(u, w)
        torch.cuda.synchronize()
        assert energy == want[1] and volume == want[3]
        # the chunk kernels' gradient sums may differ in their order from run to run
        for got, ref in ((gz, want[0]), (gv, want[2]), (r0, want[4]), (r1, want[5])):
            assert float((got - ref).abs().max()) <= 1e-12 * float(ref.abs().max())
