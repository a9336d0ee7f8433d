"""One-row sweeps (2D rows and columns) at the sizes where their tiling can go
wrong, bit for bit against the oracle: lines around one window (62-65 lanes),
partial last tiles, sweeps of one step and around one and two blocks of every
halo depth, NaN and infinite old distances, 1-4 channels in one launch."""
import time

import numpy as np
import pytest
import torch

import fastgeodis_amd as FG
import oracle

pytestmark = pytest.mark.gpu

DEPTHS = [6, 12, 18, 24, 30]


def equal(got, want):
    got, want = np.asarray(got, np.float32), np.asarray(want, np.float32)
    return bool(np.all((got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))))


@pytest.fixture(params=DEPTHS + [0])
def depth(request, device):
    old = FG.get_tuning()
    FG.set_tuning(halo=request.param)
    yield request.param
    FG.set_tuning(**old)


def make(rng, C, H, W, special=False):
    img = rng.random((1, C, H, W), dtype=np.float32)
    m = np.ones((1, 1, H, W), np.float32)
    for _ in range(3):
        m[0, 0, rng.integers(0, H), rng.integers(0, W)] = 0
    if special:
        for value in (np.nan, np.inf, -np.inf, np.nan):
            m[0, 0, rng.integers(0, H), rng.integers(0, W)] = value
        img[0, 0, rng.integers(0, H), rng.integers(0, W)] = np.nan
        img[0, C - 1, rng.integers(0, H), rng.integers(0, W)] = np.inf
    return img, m


def sizes(K):
    """(H, W): lines of one window and of partial last tiles, sweeps of K and
    2K steps and one to either side."""
    K = K or 30
    cap = 64 - 2 * K
    return [(2, 62), (K, 63), (K + 1, 64), (K + 2, 65), (2 * K + 1, 3 * cap + 1), (2 * K + 2, 61), (97, 2), (1, 70)]


@pytest.mark.parametrize("lamb", [1.0, 0.5, 1.5])
@pytest.mark.parametrize("special", [False, True], ids=["finite", "nan-inf"])
def test_sizes(depth, lamb, special):
    rng = np.random.default_rng(7 + depth)
    for k, (H, W) in enumerate(sizes(depth)):
        C = 1 + k % 4
        img, m = make(rng, C, H, W, special)
        print(f"rows K={depth} lamb={lamb} C={C} {H}x{W} special={special}", flush=True)
        with np.errstate(all="ignore"):
            want = oracle.py_geodesic2d(img, m, 1e10, lamb, 2)
        got = FG.generalised_geodesic2d(torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda(), 1e10, lamb, 2)
        assert equal(got.cpu().numpy(), want)


def test_channels_share_a_launch(depth):
    rng = np.random.default_rng(11)
    insts, wants = [], []
    for k in range(12):
        C, H, W = 1 + k % 4, int(rng.integers(2, 200)), int(rng.integers(2, 200))
        op = ("unsigned", "signed", "gsf")[k % 3]
        img, m = make(rng, C, H, W)
        if op != "unsigned":
            m = (rng.random((1, 1, H, W)) > 0.5).astype(np.float32)
        insts.append(FG.Instance(torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda(), 1e10, 1.0, iter=1 + k % 2,
                                 op=op, theta=0.1))
        want = {"unsigned": lambda: oracle.py_geodesic2d(img, m, 1e10, 1.0, 1 + k % 2),
                "signed": lambda: oracle.py_signed_geodesic2d(img, m, 1e10, 1.0, 1 + k % 2),
                "gsf": lambda: oracle.py_gsf2d(img, m, 0.1, 1e10, 1.0, 1 + k % 2)}[op]()
        wants.append(want)
    for got, want in zip(FG.geodesic_batch(insts), wants):
        assert equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("C,H,W", [(1, 1, 1), (1, 2, 3), (1, 63, 64), (1, 64, 65), (1, 65, 97), (1, 96, 128),
                                   (1, 128, 127), (1, 129, 64), (2, 64, 63), (3, 64, 64), (3, 65, 64)])
@pytest.mark.parametrize("lamb", [1.0, 0.5, 1.5])
def test_small_images(device, C, H, W, lamb):
    """Whole transforms in one workgroup, at the sizes around its limits and
    line splits; and several in one call beside images too large for it."""
    rng = np.random.default_rng(H * 131 + W)
    for special in (False, True):
        img, m = make(rng, C, H, W, special)
        ti, tm = torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda()
        print(f"small C={C} {H}x{W} lamb={lamb} special={special}", flush=True)
        with np.errstate(all="ignore"):
            for it in (0, 1, 3):
                assert equal(FG.generalised_geodesic2d(ti, tm, 1e10, lamb, it).cpu().numpy(),
                             oracle.py_geodesic2d(img, m, 1e10, lamb, it))
    mask = (rng.random((1, 2, H, W)) > 0.5).astype(np.float32)
    img, _ = make(rng, C, H, W)
    ti, tm = torch.from_numpy(img).cuda(), torch.from_numpy(mask).cuda()
    assert equal(FG.signed_generalised_geodesic2d(ti, tm, 1e3, lamb, 2).cpu().numpy(),
                 oracle.py_signed_geodesic2d(img, mask, 1e3, lamb, 2))
    want = oracle.py_gsf2d(img, mask, 0.1, 1e3, lamb, 2)
    assert equal(FG.GSF2d(ti, tm, 0.1, 1e3, lamb, 2).cpu().numpy(), want)
    big, bm = make(rng, 1, 150, 70)
    insts = [FG.Instance(torch.from_numpy(big).cuda(), torch.from_numpy(bm).cuda(), 1e10, lamb, iter=2)]
    insts += [FG.Instance(ti, tm, 1e3, lamb, iter=2, op="gsf", theta=0.1) for _ in range(3)]
    assert all(equal(g.cpu().numpy(), want) for g in FG.geodesic_batch(insts[1:]))
    got = FG.geodesic_batch(insts)
    assert equal(got[0].cpu().numpy(), oracle.py_geodesic2d(big, bm, 1e10, lamb, 2))
    assert all(equal(g.cpu().numpy(), want) for g in got[1:])


@pytest.mark.parametrize("lamb", [1.0, 0.5, 1.5])
@pytest.mark.parametrize("K", [0, 6, 12, 18, 24, 30])
def test_many_tiles(device, lamb, K):
    """Launches of more tiles than the front-and-producers form is used for:
    1-4 channels, initialising and later sweeps, lengths around one and two
    blocks, both output layouts, NaN and infinities."""
    rng = np.random.default_rng(23 + K)
    insts, wants = [], []
    for k in range(44):
        C, n = 1 + k % 4, (2, 5, 6, 7, 13, 25, 31, 49)[k % 8]
        H, W = (n, 1200 + k) if k % 2 else (1200 + k, n)
        img, m = make(rng, C, H, W, special=k % 5 == 0)
        with np.errstate(all="ignore"):
            wants.append(oracle.py_geodesic2d(img, m, 1e10, lamb, 2))
        insts.append(FG.Instance(torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda(), 1e10, lamb, iter=2))
    insts, wants = insts + insts, wants + wants  # (rows of one half, columns of the other: > 900 tiles each)
    old = FG.get_tuning()
    FG.set_tuning(halo=K)
    try:
        print(f"many tiles lamb={lamb} K={K}", flush=True)
        for got, want in zip(FG.geodesic_batch(insts), wants):
            assert equal(got.cpu().numpy(), want)
    finally:
        FG.set_tuning(**old)


def test_recording_time_grows_with_the_batch(device):
    """Host work per image does not grow with the batch: four times the images
    take about four times as long (16 times where each image looks at all)."""
    rng = np.random.default_rng(5)
    img, m = make(rng, 1, 130, 20)
    one = FG.Instance(torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda(), 1e10, 1.0, iter=1)

    def took(n):
        insts, best = [one] * n, float("inf")
        for _ in range(4):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            FG.geodesic_batch(insts)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t0)
        return best

    few, many = took(1024), took(4096)
    print(f"1024 images {few * 1e3:.1f} ms, 4096 images {many * 1e3:.1f} ms", flush=True)
    assert many < 7 * few


@pytest.mark.parametrize("lamb", [1.0, 0.5])
@pytest.mark.parametrize("halo,shape", [(30, (9, 4000)), (24, (9, 9600)), (18, (40, 15000)), (30, (33, 1, 4000)),
                                        (24, (9, 1, 9600)), (30, (34, 1, 2500)), (30, (2, 1, 2100)), (6, (13, 1, 40000))])
def test_long_rows_at_a_requested_depth(device, halo, shape, lamb):
    """Rows of more tiles than workgroups with a front and producers are
    resident at the requested depth: 2D rows take a shallower depth, planes of
    one row the one-wave form.  The stepper takes them (their first sweep is
    tiled) and every result is the oracle's."""
    rng = np.random.default_rng(halo + shape[-1])
    img = rng.random((1, 1, *shape), dtype=np.float32)
    m = (rng.random((1, 1, *shape)) > 0.001).astype(np.float32)
    m[(0, 0) + tuple(rng.integers(0, s) for s in shape)] = np.nan
    ti, tm = torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda()
    sp = [1.5, 1.0, 0.7]
    print(f"long rows halo={halo} {shape} lamb={lamb}", flush=True)
    with np.errstate(all="ignore"):
        want = (oracle.py_geodesic2d(img, m, 1e10, lamb, 1) if len(shape) == 2
                else oracle.py_geodesic3d(img, m, sp, 1e10, lamb, 1))
    old = FG.get_tuning()
    FG.set_tuning(halo=halo)
    try:
        got = (FG.generalised_geodesic2d(ti, tm, 1e10, lamb, 1) if len(shape) == 2
               else FG.generalised_geodesic3d(ti, tm, sp, 1e10, lamb, 1))
        assert equal(got.cpu().numpy(), want)
        st = FG.FastGeodisCpp.Stepper(64 << 20, 4, torch.cuda.current_device())
        _, out = st.add(ti, tm, sp, 0, 1e10, lamb, 1.0 - lamb, 1)
        while st.active():
            st.step()
        assert equal(out.cpu().numpy(), want)
    finally:
        FG.set_tuning(**old)


def test_widest_rows(device):
    """Lines of more tiles than the one-wave form's kernel for 1-4 channels holds:
    one channel's kernel holds twice as many.  Alone, beside an image with more
    channels in one call, and on the stepper, which takes tiled sweeps only."""
    rng = np.random.default_rng(31)
    img, m = make(rng, 1, 5, 400000)
    rgb, rm = make(rng, 3, 40, 70)
    ti, tm = torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda()
    want = oracle.py_geodesic2d(img, m, 1e10, 0.5, 1)
    assert equal(FG.generalised_geodesic2d(ti, tm, 1e10, 0.5, 1).cpu().numpy(), want)
    insts = [FG.Instance(ti, tm, 1e10, 0.5, iter=1),
             FG.Instance(torch.from_numpy(rgb).cuda(), torch.from_numpy(rm).cuda(), 1e10, 0.5, iter=1)]
    got = FG.geodesic_batch(insts)
    assert equal(got[0].cpu().numpy(), want)
    assert equal(got[1].cpu().numpy(), oracle.py_geodesic2d(rgb, rm, 1e10, 0.5, 1))
    st = FG.FastGeodisCpp.Stepper(64 << 20, 4, torch.cuda.current_device())
    _, out = st.add(ti, tm, [1.0, 1.0, 1.0], 0, 1e10, 0.5, 0.5, 1)
    while st.active():
        st.step()
    assert equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("lamb", [1.0, 0.5, 1.5])
@pytest.mark.parametrize("what", ["signed", "gsf", "gsf-second-stage", "mixed"])
def test_many_tiles_of_signed_and_filtered_images(device, what, lamb):
    """Signed transforms and the filter on the one-wave form: both ways to
    initialise, the epilogues' combining transposes after sweeps that write their
    own layout, images of both orientations.  gsf-second-stage: 12 images of 30
    tiles (K = 12) are 720 tiles in the first stage, on the front-and-producers
    form, and 1152 (of 24, K = 6) in the second."""
    rng = np.random.default_rng(len(what))
    insts, wants = [], []
    for k in range(12 if what == "gsf-second-stage" else 44):
        C, n = 1 + k % 4, (2, 7, 13, 26)[k % 4]
        op = {"mixed": ("unsigned", "signed", "gsf")[k % 3]}.get(what, what.split("-")[0])
        H, W = (n, 1190) if what == "gsf-second-stage" or k % 2 else (1190 + k, n)
        img, _ = make(rng, C, H, W)
        m = (rng.random((1, 1, H, W)) > 0.4).astype(np.float32)
        it = 2 + k % 2
        wants.append({"unsigned": lambda: oracle.py_geodesic2d(img, m, 1e10, lamb, it),
                      "signed": lambda: oracle.py_signed_geodesic2d(img, m, 1e10, lamb, it),
                      "gsf": lambda: oracle.py_gsf2d(img, m, 0.1, 1e10, lamb, it)}[op]())
        insts.append(FG.Instance(torch.from_numpy(img).cuda(), torch.from_numpy(m).cuda(), 1e10, lamb, iter=it, op=op,
                                 theta=0.1))
    if what != "gsf-second-stage":
        insts, wants = insts + insts, wants + wants  # (> 2000 tiles of rows and of columns)
    print(f"many tiles {what} lamb={lamb}", flush=True)
    for got, want in zip(FG.geodesic_batch(insts), wants):
        assert equal(got.cpu().numpy(), want)
