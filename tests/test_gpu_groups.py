"""Workgroup caps (set_tuning(max_groups=...)) on the tiled engine with the
automatic halo and shape, bit for bit against the oracle: caps below, between
and above the tiles of the shallowest halo, of the planned depth and of the
16-row windows, for 2D rows, 3D planes, batches and the stepper."""
import numpy as np
import pytest
import torch

import fastgeodis_amd as FG
import oracle

pytestmark = pytest.mark.gpu

CAPS = [1, 3, 10, 20, 40, 64, 100, 300]


@pytest.fixture(params=CAPS)
def cap(request, device):
    old = FG.get_tuning()
    FG.set_tuning(max_groups=request.param)
    yield request.param
    FG.set_tuning(**old)


def equal(got, want):
    return np.array_equal(np.asarray(got, np.float32).view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


def make(seed, C, shape):
    rng = np.random.default_rng(seed)
    img = rng.random((1, C, *shape), dtype=np.float32)
    m = (rng.random((1, 1, *shape)) > 0.3).astype(np.float32)
    return img, m, torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda()


@pytest.mark.parametrize("lamb", [1.0, 0.5])
def test_rows(cap, lamb):
    # rows of 512: 10 tiles at K = 6, 128 at K = 30; columns of 150: 3 and 38
    img, m, ti, tm = make(cap, 2, (150, 512))
    print(f"rows cap={cap} lamb={lamb}", flush=True)
    assert equal(FG.generalised_geodesic2d(ti, tm, 1e10, lamb, 2).cpu(), oracle.py_geodesic2d(img, m, 1e10, lamb, 2))
    assert equal(FG.GSF2d(ti, tm, 0.1, 1e3, lamb, 1).cpu(), oracle.py_gsf2d(img, m, 0.1, 1e3, lamb, 1))


@pytest.mark.parametrize("lamb", [1.0, 0.5])
def test_planes(cap, lamb):
    # D pass planes of 100 x 130: 15 tiles of 32 rows at K = 5, 27 at K = 10, 51 of 16 rows
    sp = [2.0, 1.0, 0.8]
    img, m, ti, tm = make(cap, 1, (30, 100, 130))
    print(f"planes cap={cap} lamb={lamb}", flush=True)
    assert equal(FG.generalised_geodesic3d(ti, tm, sp, 1e10, lamb, 2).cpu(),
                 oracle.py_geodesic3d(img, m, sp, 1e10, lamb, 2))
    assert equal(FG.signed_generalised_geodesic3d(ti, tm, sp, 1e10, lamb, 1).cpu(),
                 oracle.py_signed_geodesic3d(img, m, sp, 1e10, lamb, 1))


def test_batch_and_stepper(cap):
    specs = [((33, 40, 70), [1.0, 1.5, 0.7]), ((90, 200), [1.0, 1.0, 1.0]), ((20, 64, 90), [1.0, 1.0, 1.0])]
    insts, wants = [], []
    for k, (shape, sp) in enumerate(specs):
        img, m, ti, tm = make(10 * cap + k, 1, shape)
        insts.append(FG.Instance(ti, tm, 1e10, 1.0, iter=1, spacing=sp if len(shape) == 3 else None))
        wants.append(oracle.py_geodesic3d(img, m, sp, 1e10, 1.0, 1) if len(shape) == 3
                     else oracle.py_geodesic2d(img, m, 1e10, 1.0, 1))
    print(f"batch cap={cap}", flush=True)
    for got, want in zip(FG.geodesic_batch(insts), wants):
        assert equal(got.cpu(), want)
    if cap < 10:
        return  # the stepper refuses planes whose first sweep is not tiled
    st = FG.FastGeodisCpp.Stepper(16 << 20, 8, torch.cuda.current_device())
    outs = {}
    for k, (shape, sp) in enumerate(specs):
        ticket, out = st.add(insts[k].image, insts[k].softmask, sp, 0, 1e10, 1.0, 0.0, 1)
        outs[ticket] = (out, wants[k])
    while st.active():
        for ticket in st.step():
            out, want = outs[ticket]
            assert equal(out.cpu(), want)
