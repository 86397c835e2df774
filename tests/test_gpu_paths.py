"""Edges of the kernels' tiles, chunks and dispatch rules: the sizes at which a path begins, ends or
hands over to another one, against the FP64 oracle or the other path.

Tolerances are those of test_gpu_fan2d.py / test_gpu_cone3d.py: rel-L2 <= 1e-5 for FP32 storage and
arithmetic against FP64 (the operators' own errors are 1e-7 to 5e-6).
"""
import numpy as np
import pytest
import torch

import curadon_amd as cm
from geoms import as_cone_geometry, as_fan_geometry, cone, fan

pytestmark = pytest.mark.gpu

RTOL_L2 = 1e-5


def rel_l2(a, b):
    a = a.double().cpu().numpy() if isinstance(a, torch.Tensor) else a
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def rand(shape, gpu, seed, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return torch.rand(shape, generator=g).to(device=gpu, dtype=dtype)


@pytest.mark.parametrize("mode", ["reference", "fbp"])
@pytest.mark.parametrize("n,D,A,prec", [
    (34, 64, 4, torch.float32),    # one angle per quarter; quadrant of 17 pixels: ragged tile
    (34, 64, 20, torch.float32),   # quarters of 5: two quarter ends in one chunk of 8
    (64, 91, 36, torch.float32),   # quarters of 9: a chunk across the quarter's end
    (64, 91, 64, torch.bfloat16),  # quarters of 16: whole chunks
    (130, 187, 100, torch.float16),
])
def test_quarter_turns_equal_pixels(gpu, n, D, A, prec, mode):
    """The backprojection by quarter turns (batches with enough tiles) and the per-pixel one (a
    single small image) give the same bits."""
    geom = as_fan_geometry(fan(n, D, A, 2.0 * n, 3.0 * n), vol_prec=prec, sino_prec=prec)
    tiles = ((n // 2 + 15) // 16) ** 2
    assert tiles < 200
    batch = -(-200 // tiles)
    y = rand((3, A, D), gpu, 1, prec)
    many = y.repeat(-(-batch // 3), 1, 1)
    got = cm.backward(many, geom, mode=mode)
    for i in range(3):
        one = cm.backward(y[i].contiguous(), geom, mode=mode)
        assert torch.equal(got[i], one)
        assert torch.equal(got[-3 + i], one)


@pytest.mark.parametrize("A", [1, 2, 3, 5, 9])
@pytest.mark.parametrize("ny,nx", [(5, 1), (3, 63), (4, 65)])
@pytest.mark.parametrize("views", [False, True])
def test_backward_few_angles_ragged(oracle, gpu, A, ny, nx, views):
    """Quarters of the angles that are empty or unequal, tiles of 64 pixels with one lane in use,
    one lane missing and one over."""
    rec = fan(nx, 70, A, 150.0, 220.0, ny=ny)
    y = np.random.RandomState(A).rand(A, 70)
    if views:
        rec.det_offset, rec.det_rotation, rec.COR, rec.exact_geometry = 1.5, 0.05, 0.75, True
        geom = cm.FanGeometry(DSD=rec.DSD, DSO=rec.DSO, angles=rec.angles,
                              vol_shape=rec.vol_shape, det_shape=rec.det_shape, det_offset=1.5,
                              det_rotation=0.05, COR=0.75, exact_geometry=True)
    else:
        geom = as_fan_geometry(rec)
    for mode, wpow in (("reference", 1), ("fbp", 2)):
        ref = oracle.bp2d(geom, y, wpow=wpow)
        got = cm.backward(torch.tensor(y, dtype=torch.float32, device=gpu), geom, mode=mode)
        assert rel_l2(got, ref) <= RTOL_L2


def test_view_rows_batched_equal_single(gpu):
    """Plans from views: a batch large enough for four rows per thread gives the bits of single
    images with one row per thread."""
    geom = cm.FanGeometry(DSD=220.0, DSO=150.0, angles=np.linspace(0, 2, 11), vol_shape=(6, 65),
                          det_shape=90, det_offset=1.5, exact_geometry=True)
    y = rand((3, 11, 90), gpu, 5)
    got = cm.backward(y.repeat(45, 1, 1), geom)    # 135 images x 4 tiles
    for i in range(3):
        one = cm.backward(y[i].contiguous(), geom)
        assert torch.equal(got[i], one) and torch.equal(got[-3 + i], one)


@pytest.mark.parametrize("what,rec", [
    # staged boxes: ragged slabs, one voxel thick along an axis, panels of one tile less and more
    ("thin x", lambda: cone(1, 17, 15, 6, 60.0, 90.0, nz=21, ny=9)),
    ("thin z", lambda: cone(23, 16, 17, 6, 60.0, 90.0, nz=1, ny=11)),
    ("ten slices", lambda: cone(20, 33, 31, 7, 60.0, 90.0, nz=10, ny=30)),
    # boxes too large to stage: every slab from global memory, or some of them
    ("coarse panel", lambda: cone(40, 24, 20, 5, 80.0, 120.0, du=(5.0, 5.0))),
    ("rows too long", lambda: cone(40, 24, 20, 5, 80.0, 120.0, du=(3.0, 1.0))),
    # rays nearly along the diagonals and within the volume's corners
    ("near source", lambda: cone(24, 40, 36, 9, 26.0, 60.0, du=(1.5, 1.5))),
    # FP32 corner rays that lose the voxel: the workgroups march from global memory
    ("far source", lambda: cone(32, 24, 24, 3, 4.0e6, 4.0e6 + 40.0)),
    # tilted trajectory: other march axes and copies
    ("euler", lambda: cone(22, 30, 28, 4, 60.0, 90.0, nz=18, ny=26, angles=np.array(
        [[0.3, 1.9, 3.0, 5.1], [0.7, 1.4, 0.2, 1.5], [0.1, 0.9, 1.5, 0.4]]))),
])
def test_forward_3d_boxes(oracle, gpu, what, rec):
    rec = rec()
    geom = as_cone_geometry(rec)
    vol = np.random.RandomState(4).rand(*rec.vol_shape)
    got = cm.forward(torch.tensor(vol, dtype=torch.float32, device=gpu), geom)
    assert rel_l2(got, oracle.fwd3d(geom, vol)) <= RTOL_L2, what


@pytest.mark.parametrize("views", [False, True])
@pytest.mark.parametrize("ny,nx,D,du", [
    (3, 2, 5, 1.0),        # lines shorter than a wavefront, a segment wider than the detector
    (9, 64, 64, 1.5),      # one line's width, one whole segment
    (67, 150, 129, 1.0),   # chunks of 64 lines and a remainder; a segment of one cell
    (40, 200, 20, 12.0),   # segments wider than the image: walks of several steps
])
def test_backward_transpose_lines(oracle, gpu, views, ny, nx, D, du):
    """Widths, lines and segments at the edges of the walk's steps, chunks and batches."""
    n = max(ny, nx)
    more = {"det_offset": 1.25, "exact_geometry": True} if views else {}
    geom = cm.FanGeometry(DSD=3.0 * n, DSO=2.0 * n, angles=np.linspace(0, 6, 7),
                          vol_shape=(ny, nx), det_shape=D, det_spacing=du, **more)
    v = np.random.RandomState(nx).rand(ny, nx) - 0.3
    x = torch.tensor(v, dtype=torch.float32, device=gpu)
    for mode, wpow in (("reference", 1), ("fbp", 2)):
        got = cm.backward_transpose(x, geom, mode=mode)
        assert rel_l2(got, oracle.bp2d_T(geom, v, wpow=wpow)) <= RTOL_L2
    # the scale's two factors over the range of FP32: powers of two scale the result exactly
    big = cm.backward_transpose(x * 2.0 ** 100, geom, mode="reference")
    assert torch.equal(big, cm.backward_transpose(x, geom, mode="reference") * 2.0 ** 100)


@pytest.mark.parametrize("what,rec", [
    ("one slice", lambda: cone(21, 30, 17, 5, 60.0, 90.0, nz=1, ny=13)),
    ("two chunks", lambda: cone(41, 33, 16, 4, 90.0, 130.0, nz=81, ny=7)),   # 40 slices, and one
    ("one voxel wide", lambda: cone(1, 18, 30, 6, 60.0, 90.0, nz=19, ny=17)),
    # pixels that see a quarter of the volume each: boxes of many steps, and whole slices
    ("wide boxes", lambda: cone(30, 6, 6, 3, 80.0, 120.0, du=(10.0, 10.0))),
    ("whole slices", lambda: cone(30, 5, 5, 3, 45.0, 60.0, du=(40.0, 40.0))),
])
def test_backward_transpose_3d_boxes(oracle, gpu, what, rec):
    rec = rec()
    geom = as_cone_geometry(rec)
    v = np.random.RandomState(3).rand(*rec.vol_shape) - 0.3
    x = torch.tensor(v, dtype=torch.float32, device=gpu)
    for mode, kw in (("reference", {}), ("matched", {"matched": True}),
                     ("fdk", {"matched": True, "fdk": True})):
        got = cm.backward_transpose(x, geom, mode=mode)
        assert rel_l2(got, oracle.bp3d_T(geom, v, **kw)) <= RTOL_L2, (what, mode)
    tiny = cm.backward_transpose(x * 2.0 ** -100, geom, mode="matched")
    assert torch.equal(tiny, cm.backward_transpose(x, geom, mode="matched") * 2.0 ** -100)


TILTED = np.array([[0.3, 1.9, 3.0, 5.1, 5.9], [0.7, 1.4, 0.2, 1.5, 1.1], [0.1, 0.9, 1.5, 0.4, 0.2]])


@pytest.mark.parametrize("what,rec", [
    # circular orbits: runs of 16 y voxels
    ("one angle", lambda: cone(17, 20, 18, 1, 60.0, 90.0, nz=15, ny=5)),
    ("one group", lambda: cone(16, 24, 26, 8, 60.0, 90.0, nz=33, ny=16)),
    ("a group and one", lambda: cone(33, 50, 44, 9, 80.0, 120.0, nz=16, ny=17)),
    # footprints of 30 to 60 rows, and wider or higher than the staged ones (some or all angles)
    ("many rows", lambda: cone(20, 70, 90, 6, 60.0, 90.0, du=(0.45, 0.6))),
    ("too wide", lambda: cone(20, 130, 40, 6, 60.0, 90.0, du=(0.3, 1.0))),
    ("too high", lambda: cone(20, 40, 160, 6, 60.0, 90.0, du=(1.0, 0.25))),
    ("some too wide", lambda: cone(20, 90, 40, 12, 33.0, 66.0, du=(0.6, 1.0))),
    # a ragged tile's corners lie behind the source, its voxels do not
    ("corners behind", lambda: cone(17, 40, 40, 12, 20.0, 44.0)),
    # tilted orbits: runs of 8 y voxels, a divide per voxel
    ("tilted", lambda: cone(17, 30, 28, 5, 60.0, 90.0, nz=18, ny=9, angles=TILTED)),
    ("tilted, too wide", lambda: cone(19, 150, 150, 5, 60.0, 90.0, du=(0.25, 0.25),
                                      angles=TILTED)),
    ("tilted, corners behind", lambda: cone(17, 40, 40, 5, 20.0, 44.0, ny=17, angles=TILTED)),
])
def test_backward_3d_footprints(oracle, gpu, what, rec):
    rec = rec()
    geom = as_cone_geometry(rec)
    y = np.random.RandomState(6).rand(rec.nangles, *rec.det_shape)
    x = torch.tensor(y, dtype=torch.float32, device=gpu)
    for mode, kw in (("reference", {}), ("matched", {"matched": True}),
                     ("fdk", {"matched": True, "fdk": True})):
        got = cm.backward(x, geom, mode=mode)
        assert rel_l2(got, oracle.bp3d(geom, y, **kw)) <= RTOL_L2, (what, mode)


@pytest.mark.parametrize("what,rec", [
    ("one pixel", lambda: fan(1, 9, 5, 6.0, 9.0)),
    ("one tile", lambda: fan(64, 99, 17, 128.0, 192.0, ny=32)),      # 64 x 32: one of each axis
    ("one over", lambda: fan(65, 99, 16, 128.0, 192.0, ny=33)),      # lists of 16 angles: one whole
    ("one less", lambda: fan(31, 99, 33, 128.0, 192.0, ny=63)),      # two and one angle
    # rays along the axes and the diagonals, of slope 0 and 1
    ("axes", lambda: fan(50, 80, 8, 100.0, 150.0, arc=2 * np.pi, ny=70)),
    # fans of more than 90 degrees: rays of both axes and both directions in one angle and tile
    ("wide fan", lambda: fan(40, 220, 11, 30.0, 60.0, du=1.5)),
    ("coarse cells", lambda: fan(90, 13, 21, 150.0, 220.0, du=12.0)),
    ("fine cells", lambda: fan(20, 700, 9, 50.0, 75.0, du=0.06)),     # many rays per texel
    ("spacings", lambda: fan(48, 90, 13, 120.0, 170.0, spacing=(0.7, 1.3), offset=(2.5, -1.5))),
])
def test_adjoint_tiles(oracle, gpu, what, rec):
    """Rows with two terms and with one, tiles of either dominant axis, lists of angles of which
    some have no ray of the tile's axis."""
    rec = rec()
    geom = as_fan_geometry(rec)
    y = np.random.RandomState(8).rand(rec.nangles, rec.det_shape) - 0.3
    got = cm.adjoint(torch.tensor(y, dtype=torch.float32, device=gpu), geom)
    assert rel_l2(got, oracle.adj2d(rec, y)) <= RTOL_L2, what


@pytest.mark.parametrize("what,rec", [
    ("ragged tiles", lambda: cone(17, 30, 28, 5, 60.0, 90.0, nz=33, ny=15)),
    ("one voxel", lambda: cone(1, 5, 5, 3, 6.0, 9.0)),
    ("thin y", lambda: cone(40, 50, 9, 18, 90.0, 130.0, nz=16, ny=1)),    # groups of one angle
    # hundreds of rays through a voxel: the 32-bit sums are moved within an angle
    ("fine panel", lambda: cone(5, 230, 220, 3, 15.0, 22.0, du=(0.06, 0.06))),
    ("tilted", lambda: cone(20, 30, 28, 5, 60.0, 90.0, nz=18, ny=35, angles=TILTED)),
    # corners of a tile's box behind the source: all rays are candidates
    ("near source", lambda: cone(17, 40, 40, 12, 20.0, 44.0)),
])
def test_adjoint_3d_tiles(oracle, gpu, what, rec):
    rec = rec()
    geom = as_cone_geometry(rec)
    y = np.random.RandomState(9).rand(rec.nangles, *rec.det_shape) - 0.3
    got = cm.adjoint(torch.tensor(y, dtype=torch.float32, device=gpu), geom)
    assert rel_l2(got, oracle.adj3d(rec, y)) <= RTOL_L2, what


def test_adjoint_3d_angle_groups(gpu):
    """A tile's only workgroup (a batch of many tiles) and angle groups that share a tile (one
    volume) give the same bits."""
    geom = as_cone_geometry(cone(256, 60, 9, 7, 520.0, 780.0, du=(8.0, 2.0), nz=2, ny=16))
    y = rand((2, 7, 9, 60), gpu, 12) - 0.3
    batch = 1600                                   # x 16 tiles
    many = cm.adjoint(y.repeat(batch // 2, 1, 1, 1), geom)
    for i in range(2):
        one = cm.adjoint(y[i].contiguous(), geom)
        assert torch.equal(many[i], one) and torch.equal(many[batch - 2 + i], one)


@pytest.mark.parametrize("ny,nx", [(1, 40), (12, 33), (15, 64), (27, 90), (28, 29), (59, 31), (150, 140)])
@pytest.mark.parametrize("D,du", [
    (70, 0.4),     # many cells per texel: narrow bands, four groups of threads with rows to spare
    (300, 0.9),    # bands of about 25 quads
    (200, 1.55),   # more than 32 quads: two groups of threads, nine rows each
    (130, 3.0),    # bands too wide for LDS
])
def test_forward_bands(oracle, gpu, ny, nx, D, du):
    """Images whose rows (with the border) end before, at and after a band and a group of rows, in
    both dominant axes; angles on and between the axes."""
    n = max(ny, nx)
    rec = fan(nx, D, 9, 2.0 * n, 3.0 * n, du=du, ny=ny)
    geom = as_fan_geometry(rec)
    img = np.random.RandomState(D + ny).rand(ny, nx)
    got = cm.forward(torch.tensor(img, dtype=torch.float32, device=gpu), geom)
    assert rel_l2(got, oracle.fwd2d(rec, img)) <= RTOL_L2


@pytest.mark.parametrize("prec", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lead,grad", [((), False), ((2,), True)])
@pytest.mark.parametrize("rec", [lambda: fan(33, 51, 7, 70.0, 100.0, ny=21),
                                 lambda: cone(17, 20, 18, 6, 60.0, 90.0, nz=15, ny=5)])
def test_fbp_equals_its_steps(gpu, rec, lead, grad, prec):
    """The filtered projections scaled and cast in one pass are those of `fbp_filter`, rounded."""
    rec = rec()
    as_geom = as_fan_geometry if isinstance(rec.det_shape, int) else as_cone_geometry
    geom = as_geom(rec, vol_prec=prec, sino_prec=prec)
    mode = "fbp" if isinstance(geom, cm.FanGeometry) else "fdk"
    for src in (torch.float32, torch.float64):
        y = rand(lead + tuple(geom.sinogram_shape()), gpu, 3, src).requires_grad_(grad)
        got = cm.fbp(y, geom)
        steps = cm.backward(cm.fbp_filter(y, geom).detach().to(prec), geom, mode=mode)
        assert torch.equal(got, steps) and got.dtype == prec and not got.requires_grad


@pytest.mark.parametrize("A,D", [(1, 1), (3, 256), (5, 257), (65537, 2)])
@pytest.mark.parametrize("one", [True, False])
def test_cosine_weights_equal_host(gpu, A, D, one):
    """The kernel's weights are the host's, bit for bit, as is the scale of equal distances."""
    from curadon_amd import reconstruction as R
    dso = 100.0 + 0.1 * (np.zeros(A) if one else np.arange(A) % 97)
    geom = cm.FanGeometry(DSD=1.37 * dso, DSO=dso, angles=np.linspace(0, 6, A), vol_shape=(8, 8),
                          det_shape=D, det_spacing=0.731)
    host = R.cosine_weights_fan(geom, "cpu")
    assert torch.equal(R.cosine_weights_fan(geom, gpu).cpu(), host)
    c = cm.ConeGeometry(DSD=137.1, DSO=100.3, angles=np.linspace(0, 6, 3), vol_shape=(8, 8, 8),
                        det_shape=(A, D), det_spacing=(0.31, 0.731))
    assert torch.equal(R.cosine_weights_cone(c, gpu).cpu(), R.cosine_weights_cone(c, "cpu"))
    y = rand((A, D), gpu, 7)
    q, scale = R._filtered(y, geom, "ram-lak", 1.0)
    column = (np.pi / A) * torch.as_tensor(dso / (1.37 * dso), dtype=torch.float32, device=gpu)
    assert torch.equal(q * scale, q * column[:, None])


def test_fbp_filter_rows_that_are_not_the_angles(gpu):
    """Equal distances change nothing in which shapes are refused and how others broadcast."""
    A, D = 6, 20
    for dso in (np.full(A, 50.0), 50.0 + np.arange(A)):
        geom = cm.FanGeometry(DSD=1.5 * dso, DSO=dso, angles=np.linspace(0, 5, A),
                              vol_shape=(8, 8), det_shape=D)
        y = rand((2, A, D), gpu, 9)
        with pytest.raises(RuntimeError):
            cm.fbp_filter(y.reshape(2 * A, D), geom)
        assert cm.fbp_filter(y[:, :, None, :], geom).shape == (2, A, A, D)
        assert cm.fbp_filter(y, geom).shape == (2, A, D)
