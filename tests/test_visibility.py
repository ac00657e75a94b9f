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


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("m,n,prec", [(60, 40, "sp"), (1500, 1000, "sp"), (700, 500, "dp")])
def test_breaking(m, n, prec, full, gpu_available):
    """Ages and viscosities, and with every intermediate kept the roller flux,
    whose kernel is the last of WAVE_BREAKING."""
    print(f"\n[visibility] breaking {m} x {n} {prec} full={full}", flush=True)
    g = solver(m, n, prec, full_state=full)
    rng = np.random.default_rng(m)
    shape = g.shape_of("Eta")
    g.set_clock(0.1, 0.0)
    g.upload("H", np.full(shape, 2.0))
    names = ["AGE_BREAKING", "nu_break"] + (["ROLLER_FLUX"] if full else [])
    for rep in range(8):
        for k in ("ETAT", "ETAx", "ETAy", "U", "V", "Eta"):  # (the roller flux is proportional to Eta - ETAmean)
            g.upload(k, 6.0 * rng.standard_normal(shape))
        g.breaking()
        if full:
            assert idle(g)
        seen = {k: on_side_stream(g, k) for k in names}
        g.synchronize()
        for k, v in seen.items():
            assert v.tobytes() == g.download(k).tobytes(), (k, rep)
    assert all(np.count_nonzero(v) > 0 for v in seen.values())
    g.close()
