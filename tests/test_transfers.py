"""Field transfers through the ring of pinned slots (512 KB, four of them):
less than one slot, exactly one and two, one row more, more than the ring
holds, odd counts of elements and the face arrays' extra row or column, in
both widths.  They are copies, so what comes back is what went up, bit for
bit, and the neighbours of the field's rows are not touched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# interior sizes; arrays are (n + 6) x (m + 6): 512 x 256 FP32 and 256 x 256
# FP64 elements are one slot
SIZES = [(3, 3), (57, 44), (506, 250), (506, 251), (250, 250), (506, 506), (1201, 331), (1023, 777)]


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("m,n", SIZES)
def test_round_trip(m, n, prec, gpu_available):
    import fwcases
    import fwgpu
    import fwsetup
    print(f"\n[transfers] {prec} {m} x {n}", flush=True)
    c = fwcases.beach_1d(mglob=m, nglob=n, xslp=0.4 * m, xc_wk=0.2 * m, sponge_west=min(10.0, 0.1 * m))
    c.params.update({"PERIODIC": False, "WAVEMAKER": "NONE", "DIRECT_SPONGE": False})
    g = fwgpu.Solver(fwsetup.build_state(c, prec), prec)
    rng = np.random.default_rng(m * 1000 + n)
    sent = {}
    for k in ("Eta", "P", "Q", "MASK", "U"):
        shape, dt = g.shape_of(k), np.int32 if k == "MASK" else g.rdt
        sent[k] = rng.integers(-2 ** 31, 2 ** 31, shape).astype(np.int32) if k == "MASK" else \
            rng.standard_normal(shape).astype(dt)
        g.upload(k, sent[k])
    for rep in range(2):
        for k, v in sent.items():
            assert g.download(k).tobytes() == v.tobytes(), (k, rep)
    g.close()


@pytest.mark.parametrize("h,w,b", [(1, 1, 1), (17, 9, 3), (64, 64, 16), (331, 401, 2), (512, 700, 1)])
def test_network_arrays(h, w, b, gpu_available):
    """A batch gives what its samples give alone (copies of other lengths)."""
    import fwcnn
    print(f"\n[transfers] network {b} x {h} x {w}", flush=True)
    x = np.random.default_rng(h * w).standard_normal((b, 5, h, w)).astype(np.float32)
    net = fwcnn.Net(h, w, b, fwcnn.init_params(3, last_scale=1.0))
    whole = net.forward(x)
    for k in range(b):
        assert net.forward(x[k:k + 1]).tobytes() == whole[k].tobytes(), k
    net.close()
