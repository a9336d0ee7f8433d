"""3D sweeps on planes whose windows end in waves without rows (trailing waves
leave, others compute only the steps that can reach the tile's own rows), bit
for bit against the oracle: rows around one window, around tile edges and
multiples of the own rows at each halo depth, NaN and infinite values."""
import numpy as np
import pytest
import torch

import fastgeodis_amd as FG
import oracle

pytestmark = pytest.mark.gpu

ROWS = [2, 3, 15, 16, 17, 20, 31, 32, 33, 45]


def equal(got, want):
    got, want = np.asarray(got, np.float32), np.asarray(want, np.float32)
    return bool(np.all((got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))))


@pytest.mark.parametrize("halo,shape", [(0, 0), (5, 0), (10, 0), (15, 0), (5, 7), (3, 3), (10, 4), (10, 6), (4, 1)])
@pytest.mark.parametrize("lamb,C", [(1.0, 1), (0.5, 2), (1.25, 1), (1.0, 3)])
def test_rows(device, halo, shape, lamb, C):
    rng = np.random.default_rng(halo * 16 + shape)
    old = FG.get_tuning()
    FG.set_tuning(halo=halo, shape=shape)
    try:
        for k, rows in enumerate(ROWS):
            dims = [rows, 12 + 5 * k, 40 + 7 * k]
            dims = tuple(dims[(i + k) % 3] for i in range(3))  # the short side along each axis in turn
            img = rng.random((1, C, *dims), dtype=np.float32)
            m = np.ones((1, 1, *dims), np.float32)
            for value in (0, 0, np.nan, np.inf):
                m[(0, 0) + tuple(rng.integers(0, s) for s in dims)] = value
            img[(0, 0) + tuple(rng.integers(0, s) for s in dims)] = np.nan
            sp = [1.5, 1.0, 0.7]
            print(f"planes halo={halo} shape={shape} lamb={lamb} C={C} {dims}", flush=True)
            with np.errstate(all="ignore"):
                want = oracle.py_geodesic3d(img, m, sp, 1e10, lamb, 1)
            got = FG.generalised_geodesic3d(torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda(), sp, 1e10, lamb, 1)
            assert equal(got.cpu().numpy(), want)
    finally:
        FG.set_tuning(**old)


@pytest.mark.parametrize("shape,C,dims", [(2, 4, (2, 700, 800)), (1, 2, (2, 900, 1200))])
def test_wide_planes_in_the_reference_order(device, shape, C, dims):
    """Planes of 350 and 660 tiles with lamb > 1 (candidates kept for the
    reference's order): two and three workgroups a compute unit are resident, so
    the sweeps are tiled and the stepper takes them."""
    rng = np.random.default_rng(shape)
    img = rng.random((1, C, *dims), dtype=np.float32)
    m = (rng.random((1, 1, *dims)) > 0.01).astype(np.float32)
    m[0, 0, 0, 100, 100] = np.nan
    sp = [1.5, 1.0, 0.7]
    ti, tm = torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda()
    with np.errstate(all="ignore"):
        want = oracle.py_geodesic3d(img, m, sp, 1e10, 1.25, 1)
    old = FG.get_tuning()
    FG.set_tuning(shape=shape)
    try:
        assert equal(FG.generalised_geodesic3d(ti, tm, sp, 1e10, 1.25, 1).cpu().numpy(), want)
        st = FG.FastGeodisCpp.Stepper(64 << 20, 4, torch.cuda.current_device())
        _, out = st.add(ti, tm, sp, 0, 1e10, 1.25, 1.0 - 1.25, 1)
        while st.active():
            st.step()
        assert equal(out.cpu().numpy(), want)
    finally:
        FG.set_tuning(**old)
