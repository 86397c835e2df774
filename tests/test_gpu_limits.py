"""Geometries and sizes at the far ends of what the operators accept: sources close to the image and
far from it, rays along an axis, tall panels, infinities. Against the FP64 oracle.

Tolerances are those of test_gpu_fan2d.py / test_gpu_cone3d.py unless a test derives its own.
"""
import numpy as np
import pytest
import torch

import curadon_amd as cm
from geoms import as_cone_geometry, as_fan_geometry, cone, fan

pytestmark = pytest.mark.gpu

RTOL_L2 = 1e-5
MAXABS = 2e-5


def rel_l2(a, b):
    a = a.double().cpu().numpy() if isinstance(a, torch.Tensor) else a
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("rec", [
    lambda: fan(64, 48, 12, 36.0, 60.0, du=4.0),           # a workgroup of one wavefront
    lambda: fan(64, 64, 12, 46.0, 70.0, du=4.0),
    lambda: fan(64, 128, 13, 36.0, 60.0, du=2.5),          # of two
    lambda: fan(256, 128, 12, 190.0, 290.0, du=12.0),
    lambda: fan(300, 100, 9, 60.0, 90.0, du=8.0, ny=40),   # the source inside the image's circle
    lambda: fan(40, 300, 9, 60.0, 90.0, du=4.0, ny=300),
])
def test_forward_wide_fan(oracle, gpu, rec):
    """Fans of more than 90 degrees within one workgroup of the forward: rays of one dominant axis
    go both ways, some of them outside the workgroup's first and last, and rays of the other axis
    follow in a second pass. Such a pass reads the image from global memory."""
    rec = rec()
    geom = as_fan_geometry(rec)
    img = np.random.RandomState(11).rand(*rec.vol_shape)
    x = torch.tensor(img, dtype=torch.float32, device=gpu)
    got = cm.forward(x, geom)
    assert rel_l2(got, oracle.fwd2d(rec, img)) <= RTOL_L2
    for _ in range(3):
        assert torch.equal(cm.forward(x, geom), got)


@pytest.mark.parametrize("dso", [5.0e5, 2.0e6, 4.0e6, 1.0e8])
def test_forward_3d_far_sources(oracle, gpu, dso):
    """Near-parallel rays of a whole panel: the staged boxes hold every sample at any distance of
    the source. One misread sample of the 256 of a ray is 1e-3 of it, fifty times the tolerance."""
    rec = cone(256, 384, 384, 3, dso, dso + 300.0)
    geom = as_cone_geometry(rec)
    vol = np.random.RandomState(2).rand(*rec.vol_shape)
    got = cm.forward(torch.tensor(vol, dtype=torch.float32, device=gpu), geom)
    ref = oracle.fwd3d(geom, vol)
    assert rel_l2(got, ref) <= RTOL_L2
    assert np.abs(got.double().cpu().numpy() - ref).max() <= MAXABS * np.abs(ref).max()


@pytest.mark.parametrize("dso,gap", [(2.0e6, 4e-4), (8.0e5, 3e-4), (5.0e7, 1e-4), (5.0e8, 2e-5)])
@pytest.mark.parametrize("cell", [0, 1])
def test_adjoint_rays_along_tile_edges(oracle, gpu, dso, gap, cell):
    """A ray almost along each axis, `gap` of a texel before (and after) the first texel of a tile
    of 64 columns: all of its rows add that share to the texels before, which are another tile's.
    Terms are rounded to 2^-19 of the largest (0.95e-6 each, three to a texel and ray, two rays) and
    positions to 2e-6 (FP32 at 40 texels from the centre): 1e-5, 6e-6 of the largest sum."""
    rec = fan(1200, 2, 2, dso, 2.0 * dso, du=2.0 * (1.0 - 2.0 * gap), offset=(-40.0, -40.0),
              arc=np.pi)                    # world (0, 0) lies between texels 639 and 640 then
    geom = as_fan_geometry(rec)
    y = np.zeros((2, 2))
    y[:, cell] = 1.0
    ref = oracle.adj2d(rec, y)
    got = cm.adjoint(torch.tensor(y, dtype=torch.float32, device=gpu), geom)
    small = (ref > 0.2 * gap) & (ref < 5 * gap)
    assert small.sum() > 1000               # texels that take the small share alone
    assert np.abs(got.double().cpu().numpy() - ref).max() <= 6e-6 * np.abs(ref).max()


@pytest.mark.parametrize("columns", [0, 1])
@pytest.mark.parametrize("v0", [100, 27600, 55300, 65300])
def test_served_tall_panels(gpu, columns, v0):
    """Rows far down a tall panel are sampled as the same rows of a short one: the staged
    footprints' LDS addresses hold for every panel the server accepts. Positions are quarters of a
    pixel and every weight is exact, so both give the same bits."""
    from curadon_amd import _lib
    A, U, V, n = 3, 40, 65536, 24
    gen = torch.Generator().manual_seed(v0)
    rows = torch.randint(0, 256, (A, 200, U), generator=gen).float()

    def served(first, height):
        panel = torch.zeros((A, height + 4, U + 4))
        panel[:, 2 + first:202 + first, 2:-2] = rows
        panel = panel.to(gpu)
        # (U, V, W) = (x + .25 + 12 + a, y + z + .5 + first + 90 - a, 1)
        M = torch.zeros((A, 3, 4))
        M[:, 0, 0], M[:, 0, 3] = 1.0, torch.arange(A) + 17.25
        M[:, 1, 1], M[:, 1, 2], M[:, 1, 3] = 1.0, 1.0, first + 90.5 - torch.arange(A)
        M[:, 2, 3] = 1.0
        M = M.to(gpu)
        vol = torch.zeros((n, n, n), device=gpu)
        job = _lib.BPJob(kind=_lib.JOB_CONE3D, mode=0, columns=columns, sino=panel.data_ptr(),
                         table=M.data_ptr(), volume=vol.data_ptr(), nx=n, ny=n, nz=n, nu=U,
                         nv=height, nangles=A)
        job.tile_end = _lib.bp_job_tiles(job)
        server = _lib.Server(gpu.index or 0, 4)
        server.backproject([job], torch.float32, torch.float32)
        torch.cuda.synchronize()
        return vol

    tall, short = served(v0, V), served(0, 200)
    assert float(short.min()) > 0.0
    assert torch.equal(tall, short)


@pytest.mark.parametrize("mode", ["matched", "fdk"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_backward_3d_nothing_behind_the_source(gpu, mode, value):
    """Voxels behind the source (W <= 0, tilted orbit) take nothing from a projection, whatever its
    pixels hold."""
    rec = cone(26, 40, 36, 1, 5.0, 30.0, angles=np.array([[0.5], [0.6], [0.3]]))
    geom = as_cone_geometry(rec)
    M = np.asarray(geom.bp_matrices(mode), dtype=np.float64).reshape(3, 4)
    n = rec.vol_shape
    z, y, x = np.meshgrid(*[np.arange(int(k)) - (int(k) - 1) / 2 for k in n], indexing="ij")
    W = M[2, 0] * x + M[2, 1] * y + M[2, 2] * z + M[2, 3]
    assert abs(M[2, 1]) > 1e-3                       # not the layout of a circular orbit
    behind = torch.tensor(W < -1e-4 * np.abs(W).max(), device=gpu)
    assert 1000 < int(behind.sum()) < behind.numel() - 1000
    sino = torch.full(tuple(geom.sinogram_shape()), value, device=gpu)
    got = cm.backward(sino, geom, mode=mode)
    assert not bool(got[~behind].isfinite().all())   # what lies before it does take them
    assert bool((got[behind] == 0).all())


@pytest.mark.parametrize("views", [False, True])
@pytest.mark.parametrize("ny,nx,A,D,du", [
    (40, 30, 7, 255, 0.25),     # a segment of 256 cells, less one
    (40, 30, 7, 257, 0.25),     # and one cell over
    (70, 66, 7, 1100, 0.1),     # lines of a few pixels in segments of ten cells a pixel
    (20, 150, 7, 600, 0.24),    # either side of the lines between the segments' sizes
    (20, 150, 7, 600, 0.26),
    (20, 150, 400, 600, 0.5),
    (150, 20, 400, 400, 0.65),
])
def test_backward_transpose_fine_cells(oracle, gpu, views, ny, nx, A, D, du):
    """FP32 rounds a position of up to D / 2 cells by 2^-24 of that at most in each of its about
    four operations, and a position's error is its weights' (0.58 in the mean square)."""
    n = max(ny, nx)
    more = {"det_offset": 0.25, "exact_geometry": True} if views else {}
    geom = cm.FanGeometry(DSD=3.0 * n, DSO=2.0 * n, angles=np.linspace(0, 6, A),
                          vol_shape=(ny, nx), det_shape=D, det_spacing=1.5 * du, **more)
    v = np.random.RandomState(nx).rand(ny, nx)
    x = torch.tensor(v, dtype=torch.float32, device=gpu)
    tol = max(RTOL_L2, 4 * (D / 2) * 2.0 ** -24 / 0.58)
    for mode, wpow in (("reference", 1), ("fbp", 2)):
        got = cm.backward_transpose(x, geom, mode=mode)
        assert rel_l2(got, oracle.bp2d_T(geom, v, wpow=wpow)) <= tol
    three = cm.backward_transpose(torch.stack([x, 2.0 * x, x.flip(0)]), geom)
    one = cm.backward_transpose(x, geom)
    assert torch.equal(three[0], one) and torch.equal(three[1], 2.0 * one)


@pytest.mark.parametrize("mode,wpow", [("reference", 1), ("fbp", 2)])
def test_backward_quarter_turns_of_rounded_angles(oracle, gpu, mode, wpow):
    """Angles written with ten digits: by quarter turns (a batch) and by pixels (one image), the same
    bits, and the oracle's values."""
    rec = fan(64, 91, 200, 128.0, 192.0)
    rec.angles = np.round(rec.angles, 10)
    geom = as_fan_geometry(rec)
    y = np.random.RandomState(5).rand(200, 91)
    x = torch.tensor(y, dtype=torch.float32, device=gpu)
    one = cm.backward(x, geom, mode=mode)
    assert rel_l2(one, oracle.bp2d(rec, y, wpow=wpow)) <= RTOL_L2
    many = cm.backward(x.expand(60, 200, 91).contiguous(), geom, mode=mode)
    assert torch.equal(many[0], one) and torch.equal(many[59], one)


@pytest.mark.parametrize("views", [False, True])
@pytest.mark.parametrize("ny,nx,A", [(1, 65, 5), (3, 64, 9), (6, 130, 8), (7, 63, 2)])
def test_backward_fine_cells_rows(oracle, gpu, views, ny, nx, A):
    """Fine cells: a batch with enough tiles takes two rows per thread, one image one; the same
    bits, rows left over at the image's edge among them. The oracle's tolerance as for the
    transpose: positions of up to D / 2 cells, four operations of 2^-24 each."""
    more = {"det_offset": 0.25, "exact_geometry": True} if views else {}
    D = 6 * nx
    geom = cm.FanGeometry(DSD=3.0 * nx, DSO=2.0 * nx, angles=np.linspace(0, 5, A),
                          vol_shape=(ny, nx), det_shape=D, det_spacing=0.4, **more)
    y = np.random.RandomState(nx).rand(3, A, D)
    x = torch.tensor(y, dtype=torch.float32, device=gpu)
    tiles = ((nx + 63) // 64) * ((ny + 1) // 2)
    many = x.repeat(-(-1024 // (3 * tiles)), 1, 1).contiguous()
    for mode, wpow in (("reference", 1), ("fbp", 2)):
        got = cm.backward(many, geom, mode=mode)
        for i in range(3):
            one = cm.backward(x[i].contiguous(), geom, mode=mode)
            assert rel_l2(one, oracle.bp2d(geom, y[i], wpow=wpow)) <= 4 * (D / 2) * 2.0 ** -24 / 0.58
            assert torch.equal(got[i], one) and torch.equal(got[-3 + i], one)


@pytest.mark.parametrize("prec", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("ny", [1, 11, 12, 13, 15, 27, 28, 43, 44, 59, 74, 75])
@pytest.mark.parametrize("turned", [False, True])
@pytest.mark.parametrize("D,du", [(70, 0.55), (300, 0.9), (200, 1.55), (130, 3.0)])
def test_forward_half_bands(oracle, gpu, prec, ny, turned, D, du):
    """Images of at least 4 MB in their two copies, whose groups of 31 rows come in two bands: image
    rows (with the border) that end before, at and after a band and a group, in either dominant
    axis, narrow and wide bands. FP32 sinograms of images in either type."""
    nx = 4096 * 1024 // (8 if prec == torch.float32 else 4) // (ny + 4) + 1
    rec = fan(nx, D, 5, 2.0 * nx, 3.0 * nx, du=1.5 * du, ny=ny, arc=0.4)
    rec.angles = rec.angles - 0.15
    img = np.random.RandomState(D + ny).rand(ny, nx)
    if turned:
        rec.vol_shape, img, rec.angles = rec.vol_shape[::-1].copy(), img.T.copy(), rec.angles + np.pi / 2
    geom = as_fan_geometry(rec, vol_prec=prec, sino_prec=torch.float32)
    x = torch.tensor(img, dtype=prec, device=gpu)
    got = cm.forward(x, geom)
    ref = oracle.fwd2d(rec, x.double().cpu().numpy())
    assert np.abs(ref).max() > 0.1
    assert rel_l2(got, ref) <= RTOL_L2


@pytest.mark.parametrize("A", [16, 17, 24])
@pytest.mark.parametrize("batch", [511, 512, 768])
def test_adjoint_3d_few_angles(gpu, A, batch):
    """Volumes of one tile in batches around the number of tiles from which few angles stay one
    group: the same bits as in a batch of three, whose tiles have groups of their own."""
    geom = as_cone_geometry(cone(16, 24, 20, A, 40.0, 60.0, du=(1.0, 1.0)))
    y = torch.tensor(np.random.RandomState(A).rand(3, A, 20, 24) - 0.3, dtype=torch.float32, device=gpu)
    few = cm.adjoint(y, geom)
    many = cm.adjoint(y.repeat((batch + 2) // 3, 1, 1, 1)[:batch].contiguous(), geom)
    for i in range(batch):
        assert torch.equal(many[i], few[i % 3])


@pytest.mark.parametrize("rec", [
    lambda: cone(40, 120, 90, 7, 80.0, 120.0, nz=1, ny=30),           # panels far beyond the volume
    lambda: cone(40, 120, 90, 7, 80.0, 120.0, nz=30, ny=1),
    lambda: cone(1, 120, 90, 7, 80.0, 120.0, nz=30, ny=30),
    lambda: cone(20, 100, 100, 7, 80.0, 120.0, det_offset=(31.0, -23.0), nz=13, ny=17),
    lambda: cone(20, 100, 100, 5, 40.0, 60.0, du=(0.31, 0.29), nz=4,
                 angles=np.array([[0.3, 1.9, 3.0, 5.1, 5.9], [0.7, 1.4, 0.2, 1.5, 1.1],
                                  [0.1, 0.9, 1.5, 0.4, 0.2]])),
])
def test_backward_transpose_3d_tiles_beside_the_volume(oracle, gpu, rec):
    """Panel tiles whose rays pass the volume on any side, next to tiles that see one edge of it:
    the latter keep every voxel, the former are zero.

    A pixel of these fine panels holds few terms, each rounded to units of 2^-18 max|v| wbound
    (wbound = 1, or 1 / min W^2 for FDK): 0.29 units rms, against terms of rms|v| / 3 (two linear
    weights of rms 1 / sqrt(3)). Twice that."""
    rec = rec()
    geom = as_cone_geometry(rec)
    v = np.random.RandomState(5).rand(*rec.vol_shape) - 0.3
    x = torch.tensor(v, dtype=torch.float32, device=gpu)
    wmin = 1.0 - np.linalg.norm(rec.vol_shape) / 2.0 / rec.DSO
    unit = 0.29 * 2.0 ** -18 * np.abs(v).max() / (np.sqrt(np.mean(v * v)) / 3.0)
    for mode, kw, wbound in (("reference", {}, 1.0), ("matched", {"matched": True}, 1.0),
                             ("fdk", {"matched": True, "fdk": True}, 1.0 / wmin ** 2)):
        got = cm.backward_transpose(x, geom, mode=mode)
        want = oracle.bp3d_T(geom, v, **kw)
        assert rel_l2(got, want) <= 2.0 * unit * wbound, mode
        beside = want == 0.0
        assert beside.any() and not got.cpu().numpy()[beside].any()


@pytest.mark.parametrize("views", [False, True])
@pytest.mark.parametrize("ny,nx,D,du", [
    (70, 1, 300, 1.5), (1, 70, 300, 1.5), (130, 7, 400, 1.5), (65, 2, 90, 4.0),
    (40, 31, 100, 1.5), (40, 32, 100, 1.5), (40, 33, 100, 1.5), (33, 40, 40, 9.0),
    (20, 20, 500, 1.5),                    # segments that see no pixel on both sides
])
def test_backward_transpose_thin_images(oracle, gpu, views, ny, nx, D, du):
    """Lines of up to 32 pixels, several to a wavefront, widths around that, and detectors far
    beyond the image on both sides.

    Terms are rounded to units of 2^-18 max|v| bound, 0.29 units rms, against terms of rms|v| w /
    sqrt(3) (w >= 0.6 bound with the source at twice the image's size): twice that, and the rounding
    of positions as above."""
    n = max(ny, nx)
    more = {"det_offset": 0.25, "exact_geometry": True} if views else {}
    geom = cm.FanGeometry(DSD=3.0 * n, DSO=2.0 * n, angles=np.linspace(0, 6, 9),
                          vol_shape=(ny, nx), det_shape=D, det_spacing=du, **more)
    v = np.random.RandomState(ny + nx).rand(ny, nx) - 0.3
    x = torch.tensor(v, dtype=torch.float32, device=gpu)
    units = 0.29 * 2.0 ** -18 * np.abs(v).max() / (np.sqrt(np.mean(v * v)) / 3 ** 0.5)
    for mode, wpow in (("reference", 1), ("fbp", 2)):
        got = cm.backward_transpose(x, geom, mode=mode)
        want = oracle.bp2d_T(geom, v, wpow=wpow)
        assert rel_l2(got, want) <= 2.0 * units / 0.6 ** wpow + 4 * (D / 2) * 2.0 ** -24 / 0.58, mode
        hit = np.pad(want != 0.0, ((0, 0), (1, 1)))
        beside = ~(hit[:, :-2] | hit[:, 1:-1] | hit[:, 2:])
        assert not got.cpu().numpy()[beside].any()
        both = cm.backward_transpose(torch.stack([x, 2.0 * x]), geom, mode=mode)
        assert torch.equal(both[0], got) and torch.equal(both[1], 2.0 * got)


@pytest.mark.parametrize("ny", [1, 3, 4, 5, 8, 9, 12, 13, 17, 20, 21])
def test_backward_3d_thin_runs(oracle, gpu, ny):
    """Tilted orbits: runs of 8 y voxels in batches of four, of which the volume ends within any."""
    rec = cone(18, 36, 34, 5, 60.0, 90.0, nz=9, ny=ny,
               angles=np.array([[0.3, 1.9, 3.0, 5.1, 5.9], [0.7, 1.4, 0.2, 1.5, 1.1],
                                [0.1, 0.9, 1.5, 0.4, 0.2]]))
    geom = as_cone_geometry(rec)
    y = np.random.RandomState(ny).rand(rec.nangles, *rec.det_shape)
    x = torch.tensor(y, dtype=torch.float32, device=gpu)
    for mode, kw in (("reference", {}), ("matched", {"matched": True}),
                     ("fdk", {"matched": True, "fdk": True})):
        got = cm.backward(x, geom, mode=mode)
        assert rel_l2(got, oracle.bp3d(geom, y, **kw)) <= RTOL_L2, mode


@pytest.mark.parametrize("ny,nx,A,D", [(1, 50, 40, 60), (50, 1, 40, 60), (33, 65, 25, 90), (64, 64, 40, 300)])
def test_adjoint_angle_groups(gpu, ny, nx, A, D):
    """One image, whose tiles have many angle groups, and large batches, whose tiles have few: the
    same bits, scaled data by powers of two included."""
    n = max(ny, nx)
    geom = as_fan_geometry(fan(nx, D, A, 2.0 * n, 3.0 * n, du=2.4 * n / D, ny=ny))
    y = torch.tensor(np.random.RandomState(D).rand(A, D) - 0.3, dtype=torch.float32, device=gpu)
    one = cm.adjoint(y, geom)
    scale = torch.tensor([1.0, 4.0, 0.5], device=gpu).repeat(400)[:1000, None, None]
    many = cm.adjoint(y * scale, geom)
    assert torch.equal(many, one * scale)
