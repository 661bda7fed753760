"""GPU: cone Siddon geometries outside the voxel-driven window backprojector's
range, and volumes of 2^29 voxels or more, against the FP64 oracle.

* the ray-driven backprojector (atomic scatter, the reference's transpose;
  cone_bp_mode 2) on the default small case: oracle, dot test, equality with
  the window backprojector;
* the detector of the reference's example/projector.cfg (0.25 mm cells, dsd
  3000, dso 2700) with 1 mm voxels: a voxel shadow of more than 4 cells, so
  the backprojection takes the ray-driven path by itself;
* sources inside and just outside the volume's corner radius;
* z-slabs: small volumes forced into slabs (cone_slab_slices) equal the
  oracle and the unslabbed call; a 1024 x 1024 x 513 volume (more than 2^29
  voxels) on 2 views (the BP there against an FP32 bound: 1e-3, and a tenth
  of the reference arithmetic's own FP32 error).

Each case prints its name before its GPU work."""

import numpy as np
import pytest

from helpers import Geo, rel_l2, small_cone

pytestmark = pytest.mark.gpu
TOL = 1e-4


@pytest.fixture
def tuning():
    from ctprojector_amd import _lib
    keys = []

    def set_(k, v):
        keys.append(k)
        _lib.set_tuning(k, v)
    yield set_
    for k in keys:
        _lib.set_tuning(k, 0)


def _say(*a):
    print('[cone-general]', *a, flush=True)


def _check(oracle, g, geo, img, seed=4, dot=True):
    from ctprojector_amd.projector.numpy import cone
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    p = g.to(ct_projector())
    args = (geo.det_center, geo.det_u, geo.det_v, geo.src)
    fp = cone.siddon_fp_arbitrary(p, img, *args)
    e_fp = rel_l2(fp, oracle.siddon_cone_fp(g, img, *args))
    y = np.random.default_rng(seed).uniform(size=fp.shape).astype(np.float32)
    bp = cone.siddon_bp_arbitrary(p, y, *args)
    e_bp = rel_l2(bp, oracle.siddon_cone_bp(g, y, *args))
    _say('fp %.2e bp %.2e' % (e_fp, e_bp))
    assert e_fp < TOL and e_bp < TOL
    if dot:
        lhs = np.dot(fp.ravel().astype(np.float64), y.ravel().astype(np.float64))
        rhs = np.dot(img.ravel().astype(np.float64), bp.ravel().astype(np.float64))
        assert abs(lhs - rhs) / (np.linalg.norm(fp) * np.linalg.norm(y)) < 1e-6
    return fp, bp


def test_scatter_backprojection(oracle, tuning):
    g, geo, img = small_cone(seed=31)
    _say('default geometry, window backprojector')
    _, a = _check(oracle, g, geo, img)
    tuning('cone_bp_mode', 2)
    _say('default geometry, ray-driven scatter')
    _, b = _check(oracle, g, geo, img)
    assert rel_l2(b, a) < 1e-5


def test_reference_example_detector(oracle):
    """example/projector.cfg: du = dv = 0.25 mm, dsd 3000, dso 2700 (nu, nv
    reduced to the volume's shadow); 48 x 48 x 32 voxels of 1 mm."""
    from ctprojector_amd.phantom import circular_cone_geometry, ellipsoid_phantom
    g = Geo(nx=48, ny=48, nz=32, dx=1.0, dy=1.0, dz=1.0, cx=0.4, cy=-0.3, cz=0.2, nu=256, nv=176, du=0.25, dv=0.25,
            off_u=0.3, off_v=-0.2, dsd=3000.0, dso=2700.0)
    geo = circular_cone_geometry(6, 2700.0, 3000.0, -1.0, 1.0, jitter=0.5, seed=33)
    img = ellipsoid_phantom(32, 48, 48, 1.0, 1.0, 1.0, seed=33)[None]
    _say('example detector 256x176 @0.25 mm, dsd 3000, dso 2700, 48x48x32 @1 mm')
    _check(oracle, g, geo, img)


def test_reference_example_detector_large_volume(oracle):
    """The example detector on a 256 x 256 x 96 volume of 1 mm voxels (ray-driven
    backprojection on a grid where accumulated crossings would drift): FP and
    BP against the FP64 oracle at 1e-4; the reference's own FP32 arithmetic is
    printed beside it."""
    from ctprojector_amd.phantom import circular_cone_geometry, ellipsoid_phantom
    from ctprojector_amd.projector.numpy import cone
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    g = Geo(nx=256, ny=256, nz=96, dx=1.0, dy=1.0, dz=1.0, cx=0.7, cy=-0.4, nu=1200, nv=480, du=0.25, dv=0.25,
            off_u=0.3, off_v=-0.2, dsd=3000.0, dso=2700.0)
    geo = circular_cone_geometry(2, 2700.0, 3000.0, -1.0, 1.0, jitter=0.5, seed=41, angle_range=np.pi / 2)
    img = ellipsoid_phantom(96, 256, 256, 1.0, 1.0, 1.0, seed=41)[None]
    p = g.to(ct_projector())
    args = (geo.det_center, geo.det_u, geo.det_v, geo.src)
    _say('example detector 1200x480 @0.25 mm, 256x256x96 @1 mm: FP')
    fp = cone.siddon_fp_arbitrary(p, img, *args)
    e = rel_l2(fp, oracle.siddon_cone_fp(g, img, *args))
    _say('fp rel-L2 %.2e' % e)
    assert e < TOL
    y = np.random.default_rng(6).uniform(size=fp.shape).astype(np.float32)
    _say('BP (ray-driven)')
    bp = cone.siddon_bp_arbitrary(p, y, *args)
    ref = oracle.siddon_cone_bp(g, y, *args)
    e = rel_l2(bp, ref)
    e32 = rel_l2(oracle.siddon_cone_bp(g, y, *args, prec='f'), ref)
    _say('bp rel-L2 %.2e (the reference arithmetic in FP32: %.2e)' % (e, e32))
    assert e < TOL


@pytest.mark.parametrize('dso', [8.0, 15.0])
def test_source_inside_or_near_volume(oracle, dso):
    """A 24^3 volume of 1 mm voxels (half width 12 mm, corner radius 20.8 mm)
    with the source at 8 mm (inside) or 15 mm (between the faces and the
    corners) from the centre."""
    from ctprojector_amd.phantom import circular_cone_geometry, ellipsoid_phantom
    g = Geo(nx=24, ny=24, nz=24, dx=1.0, dy=1.0, dz=1.0, nu=64, nv=48, du=2.0, dv=2.0, dsd=dso + 40.0, dso=dso)
    geo = circular_cone_geometry(5, dso, dso + 40.0, -2.0, 2.0, jitter=0.3, seed=35)
    img = ellipsoid_phantom(24, 24, 24, 1.0, 1.0, 1.0, seed=35)[None]
    _say('source at %.0f mm from the centre of a 24 mm cube' % dso)
    _check(oracle, g, geo, img)


@pytest.mark.parametrize('slices', [7, 24])
def test_forced_slabs(oracle, tuning, slices):
    from ctprojector_amd.projector.numpy import cone
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    g, geo, img = small_cone(seed=37, c=(0.5, -1.0, 1.5))
    img2 = np.concatenate([img, 0.5 * img[:, ::-1].copy()], 0)
    p = g.to(ct_projector())
    args = (geo.det_center, geo.det_u, geo.det_v, geo.src)
    whole_fp = cone.siddon_fp_arbitrary(p, img2, *args)
    y = np.random.default_rng(3).uniform(size=whole_fp.shape).astype(np.float32)
    whole_bp = cone.siddon_bp_arbitrary(p, y, *args)
    tuning('cone_slab_slices', slices)
    _say('slabs of %d slices, batch of 2' % slices)
    fp = cone.siddon_fp_arbitrary(p, img2, *args)
    bp = cone.siddon_bp_arbitrary(p, y, *args)
    assert rel_l2(fp, oracle.siddon_cone_fp(g, img2, *args)) < TOL
    assert rel_l2(bp, oracle.siddon_cone_bp(g, y, *args)) < TOL
    assert rel_l2(fp, whole_fp) < 1e-5 and rel_l2(bp, whole_bp) < 1e-5


def test_volume_of_more_than_2pow29_voxels(oracle):
    import torch
    from ctprojector_amd.phantom import circular_cone_geometry
    from ctprojector_amd.projector.cupy import cone, ct_projector
    nx, ny, nz = 1024, 1024, 513
    assert nx * ny * nz > 1 << 29
    g = Geo(nx=nx, ny=ny, nz=nz, dx=0.25, dy=0.25, dz=0.25, cz=0.3, nu=96, nv=64, du=5.0, dv=5.0, off_u=0.2,
            dsd=1000.0, dso=600.0)
    geo = circular_cone_geometry(2, 600.0, 1000.0, -3.0, 3.0, jitter=0.5, seed=39, angle_range=np.pi / 2)
    dev = torch.device('cuda', 0)
    x = torch.linspace(0, 6.0, nx, device=dev)
    yv = torch.linspace(0, 4.0, ny, device=dev)
    z = torch.linspace(0, 1.0, nz, device=dev)
    img = (0.01 * (1 + torch.sin(x)[None, None, :] * torch.cos(yv)[None, :, None]) * (1 + z[:, None, None]))[None]
    img = img.contiguous()
    p = g.to(ct_projector())
    gd = [torch.from_numpy(a).to(dev) for a in (geo.det_center, geo.det_u, geo.det_v, geo.src)]
    _say('1024x1024x513 volume (%d voxels), 2 views, 96x64 detector: FP' % (nx * ny * nz))
    fp = cone.siddon_fp_arbitrary(p, img, *gd).cpu().numpy()
    img_h = img.cpu().numpy()
    del img
    hg = (geo.det_center, geo.det_u, geo.det_v, geo.src)
    e = rel_l2(fp, oracle.siddon_cone_fp(g, img_h, *hg))
    _say('fp rel-L2 %.2e' % e)
    assert e < TOL
    del img_h
    y = np.random.default_rng(5).uniform(size=fp.shape).astype(np.float32)
    _say('BP')
    bp = cone.siddon_bp_arbitrary(p, torch.from_numpy(y).to(dev), *gd).cpu().numpy()
    ref = oracle.siddon_cone_bp(g, y, *hg)
    e = rel_l2(bp, ref)
    # FP32 bound: a 0.25 mm voxel seen from 600 mm is ~2400 voxels from the
    # source, so each chord, a difference of ray parameters of that size, is
    # good to ~1e-4 in FP32.  The reference's own FP32 traversal (the oracle's
    # FP32 mirror: crossings accumulated step by step) is 1.6% off here.
    e32 = rel_l2(oracle.siddon_cone_bp(g, y, *hg, prec='f'), ref)
    _say('bp rel-L2 %.2e (the reference arithmetic in FP32: %.2e)' % (e, e32))
    assert e < 1e-3 and e < 0.1 * e32


@pytest.mark.parametrize('case', ['ragged', 'flipped_rows', 'fine_rows', 'more_rows', 'fine_columns', 'axis_parallel', 'truncated',
                                  'batch'])
def test_bp_plane_form(oracle, tuning, case):
    """The plane form of the backprojector (one crossing ray per voxel plane and
    detector column) on signed data against the oracle, and against the candidate
    windows (cone_bp_planes 2): grids that end inside a block, det_v pointing
    down, several rows and several columns per voxel, rays along the axes (no
    jitter, odd panel, source on a voxel plane), planes outside the panel, and
    volumes sharing the geometry.  'fine_rows' has more rows per voxel than the
    plane form takes and keeps the windows; the others differ from them in last
    bits.  The rays of 'axis_parallel' run within voxel faces, where the voxel
    they count for is a tie that both forms decide alike and the oracle
    otherwise: compared with the windows only.

    Largest differences: a chord's two ends are off by up to 1e-4 voxel (a few
    roundings of a ray parameter, over 300 voxels), and at most 36 chords of
    weight below 1 meet in a voxel: 3.6e-3, under a thousandth of the largest
    voxel (about 5); a row more or less is off by a tenth of it."""
    from ctprojector_amd.phantom import circular_cone_geometry
    from ctprojector_amd.projector.numpy import cone
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    kw = dict(nx=23, ny=19, nz=37, dx=1.0, dy=1.0, dz=1.0, cx=0.4, cy=-0.3, cz=0.7, nu=44, nv=45, du=1.7, dv=1.7,
              off_u=0.2, off_v=-0.4, dsd=300.0, dso=180.0)
    jitter, B = 1.0, 1
    if case == 'fine_rows':
        kw.update(dz=1.5, nz=21, dv=0.8, nv=90)
    if case == 'more_rows':
        kw.update(dz=1.5, nz=21, dv=1.1, nv=70)
    if case == 'fine_columns':
        kw.update(du=0.75, nu=100)
    if case == 'axis_parallel':
        kw.update(nx=24, ny=24, nz=24, cx=0.0, cy=0.0, cz=0.0, nu=45, off_u=0.0, off_v=0.0)
        jitter = 0.0
    if case == 'truncated':
        kw.update(nv=7, nu=15, off_v=3.0)
    if case == 'batch':
        B = 3
    g = Geo(**kw)
    z = 0.0 if case == 'axis_parallel' else 6.0
    geo = circular_cone_geometry(12, 180.0, 300.0, -z, z, jitter=jitter, seed=5)
    if case == 'flipped_rows':
        geo.det_v = -geo.det_v
    args = (geo.det_center, geo.det_u, geo.det_v, geo.src)
    y = np.random.default_rng(8).uniform(-1, 1, size=[B, 12, g.nv, g.nu]).astype(np.float32)
    p = g.to(ct_projector())
    a = cone.siddon_bp_arbitrary(p, y, *args)
    tuning('cone_bp_planes', 2)
    b = cone.siddon_bp_arbitrary(p, y, *args)
    ref = oracle.siddon_cone_bp(g, y, *args)
    e, d = rel_l2(a, ref), rel_l2(a, b)
    top = np.abs(ref).max()
    me, md = np.abs(a - ref).max() / top, np.abs(a - b).max() / top
    _say(case, 'plane form against the oracle %.2e (largest %.2e), against the windows %.2e (%.2e)' % (e, me, d, md))
    assert (a != b).any() == (case != 'fine_rows')
    assert d < TOL and md < 1e-3
    assert (e < TOL and me < 1e-3) or case == 'axis_parallel'


# Geometry of the tests below: no ray near an axis direction (so that no ray is
# scattered atomically and results are compared bit for bit), several rows and
# columns of the panel beside the volume, source heights on both sides of it.
def _plane_case(nview=12, B=1, **over):
    from ctprojector_amd.phantom import circular_cone_geometry
    kw = dict(nx=23, ny=19, nz=37, dx=1.0, dy=1.0, dz=1.0, cx=0.4, cy=-0.3, cz=0.7, nu=44, nv=45, du=1.7, dv=1.7,
              off_u=0.2, off_v=-0.4, dsd=300.0, dso=180.0)
    kw.update(over)
    g = Geo(**kw)
    geo = circular_cone_geometry(nview, 180.0, 300.0, -6.0, 6.0, jitter=1.0, seed=5)
    args = (geo.det_center, geo.det_u, geo.det_v, geo.src)
    y = np.random.default_rng(8).uniform(-1, 1, size=[B, nview, g.nv, g.nu]).astype(np.float32)
    return g, args, y


@pytest.mark.parametrize('form', ['planes', 'windows', 'general'])
def test_bp_signed_and_nan_rays(oracle, tuning, form):
    """A ray is weighted alike whatever the sign of its value, so the
    backprojection is odd bit for bit, and a NaN is not dropped: every voxel
    that the ray crosses is NaN."""
    from ctprojector_amd.projector.numpy import cone
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    if form == 'windows':
        tuning('cone_bp_planes', 2)
    if form == 'general':
        tuning('cone_bp_mode', 1)
    g, args, y = _plane_case()
    p = g.to(ct_projector())
    a, b = cone.siddon_bp_arbitrary(p, y, *args), cone.siddon_bp_arbitrary(p, -y, *args)
    e = rel_l2(a, oracle.siddon_cone_bp(g, y, *args))
    _say(form, 'signed sinogram against the oracle %.2e' % e)
    assert e < TOL and np.array_equal(a, -b)
    unit = np.zeros_like(y)
    unit[0, 3, 20, 25] = 1.0
    met = oracle.siddon_cone_bp(g, unit, *args) > 1e-2   # chords of at least a hundredth of a voxel
    y[0, 3, 20, 25] = np.nan
    bad = np.isnan(cone.siddon_bp_arbitrary(p, y, *args))
    _say(form, 'voxels met by the NaN ray', int(met.sum()), 'NaN voxels', int(bad.sum()))
    assert met.sum() > 10 and bad[met].all()


@pytest.mark.parametrize('value', [np.inf, -np.inf, np.nan])
def test_bp_planes_not_finite(oracle, tuning, value):
    """A ray value that is not finite reaches the voxels that the ray crosses,
    as itself, and no others: single calls of every z-run, volumes sharing the
    geometry, and the batch plan.  (Two voxels more are allowed: chords that
    are zero in 64 bits and a rounding error in 32.)"""
    import torch
    from ctprojector_amd.batched import ConeBatch, ConeJob
    from ctprojector_amd.projector.numpy import cone
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    g, args, y = _plane_case(B=2)
    p = g.to(ct_projector())
    at = (1, 7, 14, 22)
    unit = np.zeros_like(y)
    unit[at] = 1.0
    ref = oracle.siddon_cone_bp(g, unit, *args)
    met = ref > 1e-2
    y[at] = value

    def check(name, out, ref=ref, met=met):
        bad = ~np.isfinite(out)
        _say(value, name, 'voxels met', int(met.sum()), 'not finite', int(bad.sum()))
        assert met.sum() > 10 and bad[met].all() and bad.sum() <= (ref > 0).sum() + 2
        assert np.array_equal(out[bad], np.full(bad.sum(), value, np.float32), equal_nan=True)

    check('two volumes', cone.siddon_bp_arbitrary(p, y, *args))
    for z in (1, 2, 4, 8):
        tuning('cone_bp_zrun', z)
        check('z-run %d' % z, cone.siddon_bp_arbitrary(p, y[1:], *args), ref[1:], met[1:])
    tuning('cone_bp_zrun', 0)
    from types import SimpleNamespace
    geo = SimpleNamespace(det_center=args[0], det_u=args[1], det_v=args[2], src=args[3])
    b = ConeBatch([ConeJob(p, geo)])
    b.prj[0].copy_(torch.from_numpy(y[1]))
    b.backward()
    check('plan', b.img[0].cpu().numpy(), ref[1], met[1])


@pytest.mark.parametrize('case', ['default', 'narrow', 'three_columns', 'fine_columns', 'more_rows', 'flipped', 'tall'])
def test_bp_planes_bits_do_not_depend_on_the_run(tuning, case):
    """The plane form gives a voxel the same bits in z-runs of 1, 2, 4 and 8
    slices, alone and among 2, 4 or 5 volumes of one geometry, and the batch
    plan in z-runs of 2, 4 and 8 (which its autotuner chooses by time), with
    planes on both sides of the source and candidate windows of 1 to 4 columns;
    and it is the plane form that runs: the windows round otherwise."""
    import torch
    from types import SimpleNamespace
    from ctprojector_amd.batched import ConeBatch, ConeJob
    from ctprojector_amd.projector.numpy import cone
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    over = {'default': {}, 'narrow': dict(du=3.4, nu=22), 'three_columns': dict(du=1.0, nu=75),
            'fine_columns': dict(du=0.75, nu=100), 'flipped': {},
            'more_rows': dict(dz=1.5, nz=21, dv=1.1, nv=70), 'tall': dict(nz=301, cz=60.0, nv=30)}[case]
    g, args, y = _plane_case(B=5, **over)
    if case == 'flipped':
        args = (args[0], args[1], -args[2], args[3])
    p = g.to(ct_projector())
    ref = cone.siddon_bp_arbitrary(p, y[:1], *args)
    for b in (2, 4, 5):
        out = cone.siddon_bp_arbitrary(p, np.concatenate([y[1:b], y[:1]]), *args)
        assert np.array_equal(out[-1:], ref), '%d volumes' % b
        out = cone.siddon_bp_arbitrary(p, y[:b], *args)
        assert np.array_equal(out[:1], ref), '%d volumes' % b
    geo = SimpleNamespace(det_center=args[0], det_u=args[1], det_v=args[2], src=args[3])
    plans = []
    for z in (1, 2, 4, 8):
        tuning('cone_bp_zrun', z)
        assert np.array_equal(cone.siddon_bp_arbitrary(p, y[:1], *args), ref), 'z-run %d' % z
        if z > 1:
            b = ConeBatch([ConeJob(p, geo)])
            b.prj[0].copy_(torch.from_numpy(y[0]))
            b.backward()
            plans.append(b.img[0].clone())
    assert torch.equal(plans[0], plans[1]) and torch.equal(plans[0], plans[2])
    tuning('cone_bp_zrun', 0)
    tuning('cone_bp_planes', 2)
    windows = cone.siddon_bp_arbitrary(p, y[:1], *args)
    _say(case, 'voxels that the windows round otherwise: %.2f' % (windows != ref).mean())
    assert (windows != ref).any() and rel_l2(windows, ref) < TOL


@pytest.mark.parametrize('case,single,plan', [('thin_1', False, True), ('thin_4', False, True), ('nz_5', True, True),
                                              ('narrow_4', True, True), ('dense_rows', False, True),
                                              ('dense_tall', True, True), ('three_rows', False, True)])
def test_bp_form_by_geometry(oracle, tuning, case, single, plan):
    """Which column-mode backprojections take the plane form, in single calls
    (alone and beside another volume) and in a plan: single calls keep the
    windows for up to 4 slices of wide images and for voxels holding many rows;
    against the oracle."""
    import torch
    from types import SimpleNamespace
    from ctprojector_amd.batched import ConeBatch, ConeJob
    from ctprojector_amd.projector.numpy import cone
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    wide = dict(nx=446, ny=435, dx=0.2, dy=0.2, nu=150, du=1.1)
    over = {'thin_1': dict(nz=1, **wide), 'thin_4': dict(nz=4, **wide), 'nz_5': dict(nz=5, **wide),
            'narrow_4': dict(nz=4), 'dense_rows': dict(dv=1.33, nv=90), 'dense_tall': dict(nz=260, dv=1.33, nv=90),
            'three_rows': dict(dz=1.5, nz=21, dv=0.82, nv=90)}[case]
    g, args, y = _plane_case(nview=3, B=2, **over)
    p = g.to(ct_projector())
    geo = SimpleNamespace(det_center=args[0], det_u=args[1], det_v=args[2], src=args[3])

    def all_ways():
        b = ConeBatch([ConeJob(p, geo)])
        b.prj[0].copy_(torch.from_numpy(y[0]))
        b.backward()
        return (cone.siddon_bp_arbitrary(p, y[:1], *args), cone.siddon_bp_arbitrary(p, y, *args),
                b.img[0].cpu().numpy())

    got = all_ways()
    tuning('cone_bp_planes', 2)
    windows = all_ways()
    ref = oracle.siddon_cone_bp(g, y, *args)
    differs = [bool((a != b).any()) for a, b in zip(got, windows)]
    _say(case, 'against the oracle %.2e %.2e' % (rel_l2(got[1], ref), rel_l2(got[2], ref[0])), 'not the windows', differs)
    assert rel_l2(got[1], ref) < TOL and rel_l2(got[2], ref[0]) < TOL
    assert differs == [single, single, plan]
    assert np.array_equal(got[0], got[1][:1])


def test_bp_plan_of_mixed_widths(oracle, tuning):
    """A batch plan whose jobs have candidate windows of 1 to 4 columns (one
    launch over all of them, compiled for the widest) and one job in the
    windows form: every image the same bit for bit as from a plan of that job
    alone and from one launch per width, and near the oracle's."""
    import torch
    from types import SimpleNamespace
    from ctprojector_amd.batched import ConeBatch, ConeJob
    from ctprojector_amd.projector.numpy.ct_projector import ct_projector
    sizes = [dict(du=3.4, nu=22), dict(), dict(du=1.0, nu=75), dict(du=0.75, nu=100, nz=70),
             dict(nv=260)]   # (rows that far from the source's height cross a plane by more than one within a voxel)
    jobs, ys, refs = [], [], []
    for over in sizes:
        g, args, y = _plane_case(**over)
        jobs.append(ConeJob(g.to(ct_projector()), SimpleNamespace(det_center=args[0], det_u=args[1], det_v=args[2], src=args[3])))
        ys.append(torch.from_numpy(y[0]))
        refs.append(oracle.siddon_cone_bp(g, y, *args)[0])

    def run(picked):
        b = ConeBatch([jobs[j] for j in picked])
        for q, j in zip(b.prj, picked):
            q.copy_(ys[j])
        b.backward()
        return [x.cpu().numpy() for x in b.img]

    every = list(range(len(jobs)))
    alone = [run([j])[0] for j in every]
    for launch in (1, 2):
        tuning('cone_plan_bp_launch', launch)
        for j, x in enumerate(run(every)):
            assert np.array_equal(x, alone[j]), (launch, j)
    errs = [rel_l2(x, r) for x, r in zip(alone, refs)]
    _say('plan of mixed widths', ['%.1e' % e for e in errs])
    assert max(errs) < TOL
