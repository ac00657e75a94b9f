"""What a call that waits has done is there for every stream when it returns: the
context's stream is idle, and a read on a stream that does not wait for it
(a torch side stream) finds the new values."""
import ctypes as ct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def solver(m, n, prec, **kw):
    import fwcases
    import fwgpu
    import fwsetup
    c = fwcases.beach_1d(mglob=m, nglob=n, xslp=0.4 * m, xc_wk=0.2 * m, sponge_west=min(10.0, 0.1 * m))
    c.params.update({"PERIODIC": False, "WAVEMAKER": "NONE", "DIRECT_SPONGE": False})
    g = fwgpu.Solver(fwsetup.build_state(c, prec), prec, **kw)
    g.lib.fw_get_stream.argtypes = [ct.c_void_p, ct.POINTER(ct.c_void_p)]
    g.lib.fw_field_device.argtypes = [ct.c_void_p, ct.c_int, ct.POINTER(ct.c_void_p), ct.POINTER(ct.c_int)]
    g.lib.hipStreamQuery.argtypes = [ct.c_void_p]
    return g


def idle(g):
    s = ct.c_void_p()
    assert g.lib.fw_get_stream(g.ctx, ct.byref(s)) == 0
    return g.lib.hipStreamQuery(s) == 0


def on_side_stream(g, name):
    """The field as a torch side stream reads it now."""
    import torch
    p, pitch = ct.c_void_p(), ct.c_int()
    assert g.lib.fw_field_device(g.ctx, g.lib.fw_field_id(name.encode()), ct.byref(p), ct.byref(pitch)) == 0

    class Plane:
        __cuda_array_interface__ = {"shape": g.shape_of(name), "strides": (pitch.value * g.rb, g.rb),
                                    "typestr": "<f%d" % g.rb, "data": (p.value, False), "version": 2}
    view = torch.as_tensor(Plane(), device="cuda")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        a = view.clone()
    s.synchronize()
    return a.cpu().numpy()


# less than one slot of the ring, several of them, many
@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("m,n", [(57, 44), (700, 500), (1700, 1300)])
def test_upload(m, n, prec, gpu_available):
    print(f"\n[visibility] upload {m} x {n} {prec}", flush=True)
    g = solver(m, n, prec)
    rng = np.random.default_rng(m)
    for rep in range(8):
        a = rng.standard_normal(g.shape_of("Eta")).astype(g.rdt)
        g.upload("Eta", a)
        assert idle(g)
        assert on_side_stream(g, "Eta").tobytes() == a.tobytes(), rep
    g.close()
