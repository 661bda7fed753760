"""Performance cases of the projector framework: what its users run, from the
smallest call to the largest, each through the public entry points.

``listed()`` names the cases, ``draw(rng)`` makes another one of the same
ranges, ``prepare(case, seed)`` builds what a user's program holds before the
call, ``run(state)`` is one pass, ``work(case)`` the bytes and operations a
pass cannot do without, and ``exact(case, seed)`` the same outputs from plain
torch arithmetic in 64 bits (None where that would take too long).

Kinds of cases
  par_slice   one parallel-beam slice: forward projection, Hann filter, FBP-weighted backprojection
  fan_stack   a stack of fan-beam slices: forward projection and backprojection
  fan_fp, fan_bp, fan_fbp  one direction of a fan-beam volume (projection; backprojection; ramp filter + pixel-driven FBP)
  unrolled    training step of an unrolled SQS-TV network on fan-beam slices (forward, gradient w.r.t. the sinogram)
  dd_batch    uneven fan / parallel jobs in one batch plan, forward and backward
  cone_fp, cone_bp  cone-beam Siddon projection of one volume; its exact transpose
  cone_batch  uneven cone-beam jobs in one batch plan, forward and backward
  cone_sqs    one SQS-TV iteration of a cone-beam reconstruction
  tomo        tomosynthesis forward projection and backprojection

Inputs: volumes of ten random ellipsoids, sinograms their closed-form line
integrals with 1% noise, all drawn from the seed on the GPU.
"""

import math
import random
from types import SimpleNamespace

import numpy as np
import torch

from ctprojector_amd.autograd import FanDD, sqs_tv_unrolled
from ctprojector_amd.batched import ConeBatch, ConeJob, DDBatch, DDJob
from ctprojector_amd.phantom import CONE_SAMPLES, DD_BATCH_SAMPLES, circular_cone_geometry
from ctprojector_amd.projector.cupy import cone, ct_projector, fan_equiangular, parallel, tomo
from ctprojector_amd.recon.cupy.sqs_algorithms import sqs_tv_one_step

F64 = torch.float64


# ------------------------------------------------------------------- the cases
def listed():
    fan512 = dict(nx=512, ny=512, nz=32, dx=0.7, nu=888, nview=984, branchless=False)
    nz, ny, nx, _, _, dx = CONE_SAMPLES[2]
    cone256 = dict(nx=nx, ny=ny, nz=nz, dx=dx, nu=512, nv=384, nview=720)
    return [
        # the smallest calls: a 96^2 parallel slice (the smallest job of the mixed
        # stream); a notebook user's or a small test's single slice, where the
        # launches and the host path count
        dict(name='par_slice_96', kind='par_slice', nx=96, ny=96, dx=2.6, nu=137, nview=128, branchless=False),
        # an ordinary small volume of odd sizes, branchless projector
        dict(name='fan_stack_217x193x5', kind='fan_stack', nx=217, ny=193, nz=5, dx=1.5, nu=355, nview=301,
             branchless=True, fbp=False),
        # a clinical fan-beam volume (the benchmark's): projection, backprojection, FBP
        dict(name='fan_fp_512x32', kind='fan_fp', **fan512),
        dict(name='fan_bp_512x32', kind='fan_bp', fbp=False, **fan512),
        dict(name='fan_fbp_512x32', kind='fan_fbp', **fan512),
        # training step of the unrolled network (the benchmark's)
        dict(name='unrolled_8x256', kind='unrolled', batch=8, nx=256, ny=256, dx=1.4, nu=444, nview=492, niter=10),
        # a mixed stream of sixteen uneven fan / parallel jobs in one plan (the benchmark's)
        dict(name='dd_batch_16', kind='dd_batch', jobs=16, mix=0),
        # cone-beam CT of a 256^3 volume (the benchmark's), each direction
        dict(name='cone_fp_256', kind='cone_fp', **cone256),
        dict(name='cone_bp_256', kind='cone_bp', **cone256),
        # a stream of twelve small uneven cone jobs in one plan (the benchmark's)
        dict(name='cone_batch_12', kind='cone_batch', jobs=12, mix=0),
        # one iteration of an iterative cone-beam reconstruction at the served size
        dict(name='cone_sqs_128', kind='cone_sqs', nx=128, ny=128, nz=128, dx=1.0, nu=256, nv=192, nview=180),
        # breast-tomosynthesis-like scan: nine views of the example configuration
        dict(name='tomo_256x48', kind='tomo', nx=256, ny=256, nz=48, dx=1.0, nu=256, nv=256, nview=9),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(['par_slice', 'fan_stack', 'fan_fp', 'fan_bp', 'fan_fbp', 'unrolled', 'dd_batch', 'cone_fp',
                       'cone_bp', 'cone_batch', 'cone_sqs', 'tomo'])
    if kind == 'par_slice':
        n = log(64, 768)
        return dict(kind=kind, nx=n, ny=max(48, n - rng.randrange(24)), dx=250.0 / n, nu=int(n * 1.43),
                    nview=log(90, 900), branchless=rng.random() < 0.3)
    if kind in ('fan_stack', 'fan_fp', 'fan_bp', 'fan_fbp'):
        n = rng.randrange(160, 513)
        nz = log(1, 32)
        c = dict(kind=kind, nx=n, ny=n - rng.randrange(24), nz=nz, dx=358.4 / n, nu=rng.randrange(int(1.5 * n), 889),
                 nview=rng.randrange(300, 985), branchless=rng.random() < 0.3)
        if kind in ('fan_stack', 'fan_bp'):
            c['fbp'] = rng.random() < 0.4
        return c
    if kind == 'unrolled':
        n = rng.randrange(128, 257)
        return dict(kind=kind, batch=rng.randrange(1, 9), nx=n, ny=n, dx=358.4 / n, nu=int(n * 1.734),
                    nview=rng.randrange(180, 493), niter=rng.randrange(4, 11))
    if kind in ('dd_batch', 'cone_batch'):
        return dict(kind=kind, jobs=rng.randrange(4, 17 if kind == 'dd_batch' else 13), mix=rng.randrange(1, 1 << 20))
    if kind in ('cone_fp', 'cone_bp'):
        n = rng.randrange(64, 257)
        return dict(kind=kind, nx=n, ny=n, nz=max(32, n - rng.randrange(48)), dx=128.0 / n,
                    nu=rng.randrange(300, 513), nv=rng.randrange(200, 385), nview=rng.randrange(90, 721))
    if kind == 'cone_sqs':
        n = rng.randrange(64, 161)
        return dict(kind=kind, nx=n, ny=n, nz=max(32, n - rng.randrange(32)), dx=128.0 / n, nu=rng.randrange(160, 321),
                    nv=rng.randrange(128, 257), nview=rng.randrange(90, 361))
    n = rng.randrange(96, 385)
    return dict(kind=kind, nx=n, ny=n - rng.randrange(24), nz=rng.randrange(12, 65), dx=256.0 / n,
                nu=rng.randrange(128, 385), nv=rng.randrange(128, 321), nview=rng.randrange(5, 26))


def _batch_sizes(case):
    """The jobs of a batch case, as plain cases of one job each."""
    kind, mix, n = case['kind'], case['mix'], case['jobs']
    rng = random.Random(1000 + mix)
    out = []
    for j in range(n):
        if kind == 'dd_batch':
            if mix == 0:
                beam, size, nz, nview, nu, pix = DD_BATCH_SAMPLES[j]
            else:
                beam = rng.choice(['fan', 'parallel'])
                size, nz = rng.randrange(96, 513), rng.choice([1, 1, 1, 2, 3, 4, 8])
                nview, nu, pix = rng.randrange(128, 985), int(1.43 * size) + rng.randrange(160), 358.4 / size
            du = 1.2858 * 888 / nu if beam == 'fan' else 1.4336 * size * pix / nu
            out.append(dict(fan=beam == 'fan', nx=size, ny=size, nz=nz, dx=pix, nu=nu, nview=nview, du=du))
        else:
            size = (48, 64, 80, 96)[j % 4] if mix == 0 else rng.randrange(40, 97)
            nview = (90, 120, 180)[j % 3] if mix == 0 else rng.randrange(90, 181)
            out.append(dict(nx=size, ny=size, nz=size, dx=96.0 / size, nu=64, nv=48, nview=nview, du=4.0, seed=j))
    return out


# ------------------------------------------------------------------- geometry
def _projector(**kw):
    p = ct_projector()
    for k, v in dict(dy=kw.get('dx'), dz=1.0, nv=1, dv=1.0, dsd=1085.6, dso=595.0).items():
        setattr(p, k, v)
    for k, v in kw.items():
        setattr(p, k, v)
    return p


def _dd_projector(c, fan):
    """Stacked 2D slices: the fan spans 888 x 1.2858 mm at dsd, the parallel beam 1.4336 image widths."""
    du = c.get('du') or (1.2858 * 888 / c['nu'] if fan else 1.4336 * c['nx'] * c['dx'] / c['nu'])
    nz = c.get('nz', 1)
    return _projector(nx=c['nx'], ny=c['ny'], nz=nz, dx=c['dx'], nu=c['nu'], nv=nz, du=du, nview=c['nview'])


def _angles(c, fan):
    return (np.arange(c['nview']) * (2 * np.pi if fan else np.pi) / c['nview']).astype(np.float32)


def _cone(c):
    du = c.get('du', 512.0 / c['nu'])
    p = _projector(nx=c['nx'], ny=c['ny'], nz=c['nz'], dx=c['dx'], dz=c['dx'], nu=c['nu'], nv=c['nv'], du=du, dv=du,
                   nview=c['nview'])
    geo = circular_cone_geometry(c['nview'], 595.0, 1085.6, -20.0, 20.0, jitter=2.0, seed=1032 + c.get('seed', 0))
    return p, geo


def _tomo(c):
    p = _projector(nx=c['nx'], ny=c['ny'], nz=c['nz'], dx=c['dx'], cz=c['nz'] / 2.0, nu=c['nu'], nv=c['nv'],
                   du=256.0 / c['nu'], dv=256.0 / c['nv'])
    t = np.linspace(-0.4, 0.4, c['nview'])
    src = np.stack([618 * np.sin(t), 0 * t - 100.0, 618 * np.cos(t) + 32], 1).astype(np.float32)
    dc = np.stack([0 * t, 0 * t, 0 * t - 10.0], 1).astype(np.float32)
    return p, dc, src


# --------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device='cuda').manual_seed(int(seed))


def _ellipsoids(gen, p, n=10):
    """Rows (cx, cy, cz, a, b, c, phi, value) inside the volume of projector p."""
    u = torch.rand([n, 8], generator=gen, device='cuda', dtype=F64)
    r = min(p.nx * p.dx, p.ny * p.dy) / 2
    z = p.nz * p.dz / 2
    return torch.stack([(u[:, 0] - 0.5) * 1.2 * r, (u[:, 1] - 0.5) * 1.2 * r, (u[:, 2] - 0.5) * 1.2 * z + p.cz,
                        (0.05 + 0.35 * u[:, 3]) * r, (0.05 + 0.35 * u[:, 4]) * r, (0.2 + 0.6 * u[:, 5]) * z,
                        u[:, 6] * math.pi, u[:, 7] * 0.02], 1)


def _volume(gen, p, batch=1):
    """[batch, nz, ny, nx] float32 volumes of ellipsoids with 1% noise."""
    x = ((torch.arange(p.nx, device='cuda') - (p.nx - 1) / 2) * p.dx + p.cx)[None, None, :]
    y = ((torch.arange(p.ny, device='cuda') - (p.ny - 1) / 2) * p.dy + p.cy)[None, :, None]
    z = ((torch.arange(p.nz, device='cuda') - (p.nz - 1) / 2) * p.dz + p.cz)[:, None, None]
    out = torch.zeros([batch, p.nz, p.ny, p.nx], device='cuda')
    for b in range(batch):
        for e in _ellipsoids(gen, p).float():
            c, s = torch.cos(e[6]), torch.sin(e[6])
            xr, yr = (x - e[0]) * c + (y - e[1]) * s, (y - e[1]) * c - (x - e[0]) * s
            out[b] += e[7] * (((xr / e[3]) ** 2 + (yr / e[4]) ** 2 + ((z - e[2]) / e[5]) ** 2) <= 1)
    return out + 2e-4 * torch.rand(out.shape, generator=gen, device='cuda')


def _line_integrals(gen, p, origin, direction):
    """Float32 line integrals of ellipsoids along the rays (broadcastable float tensors of
    x, y, z; unit directions), with 1% noise."""
    total = 0
    for e in _ellipsoids(gen, p).float():
        c, s = torch.cos(e[6]), torch.sin(e[6])
        ox, oy, oz = origin[0] - e[0], origin[1] - e[1], (origin[2] - e[2]) / e[5]
        ox, oy = (ox * c + oy * s) / e[3], (oy * c - ox * s) / e[4]
        dx, dy = (direction[0] * c + direction[1] * s) / e[3], (direction[1] * c - direction[0] * s) / e[4]
        dz = direction[2] / e[5]
        a = dx * dx + dy * dy + dz * dz
        b = ox * dx + oy * dy + oz * dz
        d = b * b - a * (ox * ox + oy * oy + oz * oz - 1)
        total = total + e[7] * 2 * torch.sqrt(torch.clamp(d, min=0)) / a
    return total * (1 + 0.01 * torch.randn(total.shape, generator=gen, device='cuda'))


def _dd_sinogram(gen, p, angles, fan, batch=1):
    """[batch, nview, nv, nu] fan or parallel sinograms of ellipsoids."""
    th = torch.from_numpy(angles).cuda()[:, None, None]
    i = torch.arange(p.nu, device='cuda')[None, None, :]
    z = ((torch.arange(p.nv, device='cuda') - (p.nv - 1) / 2) * p.dv)[None, :, None]
    u = -(i - (p.nu - 1) / 2) * (p.du / p.dsd if fan else p.du)
    if fan:
        o = (p.dso * torch.sin(th), -p.dso * torch.cos(th), z)
        d = (torch.sin(u - th), torch.cos(u - th), 0 * z)
    else:
        o = (u * torch.cos(th), u * torch.sin(th), z)
        d = (-torch.sin(th), torch.cos(th), 0 * z)
    return torch.stack([_line_integrals(gen, p, o, d) for _ in range(batch)], 0).contiguous()


def _cone_rays(p, geo, dtype, views=slice(None)):
    """Source [V,1,1] and detector cell [V,nv,nu] coordinates of the views, as triples."""
    dc, du, dv, src = (torch.from_numpy(a[views]).cuda().to(dtype) for a in (geo.det_center, geo.det_u, geo.det_v,
                                                                            geo.src))
    u = ((torch.arange(p.nu, device='cuda', dtype=dtype) - (p.nu - 1) / 2) * p.du)[None, None, :]
    v = ((torch.arange(p.nv, device='cuda', dtype=dtype) - (p.nv - 1) / 2) * p.dv)[None, :, None]
    s = [src[:, k, None, None] for k in range(3)]
    t = [dc[:, k, None, None] + du[:, k, None, None] * u + dv[:, k, None, None] * v for k in range(3)]
    return s, t


def _cone_sinogram(gen, p, geo):
    s, t = _cone_rays(p, geo, torch.float32)
    d = [t[k] - s[k] for k in range(3)]
    n = torch.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
    return _line_integrals(gen, p, s, [x / n for x in d])[None].contiguous()


# -------------------------------------------------------------------- prepare
def prepare(case, seed):
    c, kind, gen = case, case['kind'], _generator(seed)
    s = SimpleNamespace(kind=kind, case=case)
    if kind in ('par_slice', 'fan_stack', 'fan_fp', 'fan_bp', 'fan_fbp'):
        fan = kind != 'par_slice'
        s.p, s.ang = _dd_projector(c, fan), _angles(c, fan)
        s.angles = torch.from_numpy(s.ang).cuda()
        s.img = _volume(gen, s.p) if kind not in ('fan_bp', 'fan_fbp') else None
        s.prj = _dd_sinogram(gen, s.p, s.ang, fan) if kind != 'fan_fp' else None
    elif kind == 'unrolled':
        s.p, s.ang = _dd_projector(c, True), _angles(c, True)
        s.op = FanDD(s.p, torch.from_numpy(s.ang).cuda())
        s.target = _volume(gen, s.p, c['batch'])
        s.prj = _dd_sinogram(gen, s.p, s.ang, True, c['batch'])
        s.weight = torch.exp(-s.prj)
        # an upper bound of the projector's norm (column sums x row sums), for
        # which a constant majorizer is one
        s.pn = math.sqrt(1.3 * c['nview'] * c['dx'] ** 2 / (s.p.du * s.p.dso / s.p.dsd) * c['nx'] * c['dx'])
        s.norm_img = torch.ones_like(s.target)
        s.x0 = torch.zeros_like(s.target)
    elif kind == 'dd_batch':
        s.jobs = [(j, _dd_projector(j, j['fan']), _angles(j, j['fan'])) for j in _batch_sizes(c)]
        s.plan = DDBatch([DDJob(p, a, fan=j['fan']) for j, p, a in s.jobs])
        s.x = [_volume(gen, p) for _, p, _ in s.jobs]
    elif kind in ('cone_fp', 'cone_bp', 'cone_sqs'):
        s.p, s.geo = _cone(c)
        s.g = [torch.from_numpy(a).cuda() for a in (s.geo.det_center, s.geo.det_u, s.geo.det_v, s.geo.src)]
        s.img = _volume(gen, s.p) if kind != 'cone_bp' else None
        s.prj = _cone_sinogram(gen, s.p, s.geo) if kind != 'cone_fp' else None
        if kind == 'cone_sqs':
            kw = dict(zip(('det_center', 'det_u', 'det_v', 'src'), s.g))
            s.p.set_projector(cone.siddon_fp_arbitrary, **kw)
            s.p.set_backprojector(cone.siddon_bp_arbitrary, **kw)
            cell = s.p.du * s.p.dso / s.p.dsd
            s.pn = math.sqrt(1.3 * c['nview'] * c['dx'] ** 3 / cell ** 2 * 1.2 * c['nx'] * c['dx'])
            s.norm_img = torch.ones_like(s.img)
    elif kind == 'cone_batch':
        s.jobs = [_cone(j) for j in _batch_sizes(c)]
        s.plan = ConeBatch([ConeJob(p, g) for p, g in s.jobs])
        s.x = [_volume(gen, p)[0] for p, _ in s.jobs]
    else:
        s.p, s.dc, s.src = _tomo(c)
        s.g = [torch.from_numpy(a).cuda() for a in (s.dc, s.src)]
        s.img = _volume(gen, s.p)
        s.prj = torch.rand([1, c['nview'], c['nv'], c['nu']], generator=gen, device='cuda') * 2.0
    return s


# ------------------------------------------------------------------------ run
def run(s):
    kind, c = s.kind, s.case
    if kind == 'par_slice':
        fp = parallel.distance_driven_fp(s.p, s.img, s.angles, branchless=c['branchless'])
        flt = parallel.ramp_filter(s.p, s.prj, 'hann')
        return {'fp': fp, 'filtered': flt, 'img': parallel.distance_driven_bp(s.p, flt, s.angles, is_fbp=True,
                                                                             branchless=c['branchless'])}
    if kind == 'fan_stack':
        return {'fp': fan_equiangular.distance_driven_fp(s.p, s.img, s.angles, branchless=c['branchless']),
                'bp': fan_equiangular.distance_driven_bp(s.p, s.prj, s.angles, is_fbp=c['fbp'],
                                                         branchless=c['branchless'])}
    if kind == 'fan_fp':
        return fan_equiangular.distance_driven_fp(s.p, s.img, s.angles, branchless=c['branchless'])
    if kind == 'fan_bp':
        return fan_equiangular.distance_driven_bp(s.p, s.prj, s.angles, is_fbp=c['fbp'], branchless=c['branchless'])
    if kind == 'fan_fbp':
        flt = fan_equiangular.ramp_filter(s.p, s.prj, 'hann')
        return {'filtered': flt, 'img': fan_equiangular.fbp_bp(s.p, flt, s.angles)}
    if kind == 'unrolled':
        q = s.prj.detach().clone().requires_grad_(True)
        x = sqs_tv_unrolled(s.op, q, s.x0, s.norm_img, s.pn, 2e-3, c['niter'], weight=s.weight)
        x.backward(2.0 * (x.detach() - s.target))
        return {'x': x.detach(), 'grad': q.grad}
    if kind in ('dd_batch', 'cone_batch'):
        torch._foreach_copy_(s.plan.img, s.x)
        s.plan.forward()
        s.plan.backward()
        return {'prj': s.plan.prj, 'img': s.plan.img}
    if kind == 'cone_fp':
        return cone.siddon_fp_arbitrary(s.p, s.img, *s.g)
    if kind == 'cone_bp':
        return cone.siddon_bp_arbitrary(s.p, s.prj, *s.g)
    if kind == 'cone_sqs':
        return sqs_tv_one_step(s.p, s.img, s.prj, s.norm_img, s.pn, 1e-3)
    return {'fp': tomo.distance_driven_fp(s.p, s.img, *s.g), 'bp': tomo.distance_driven_bp(s.p, s.prj, *s.g)}


# ----------------------------------------------------------------------- work
def work(case):
    """Bytes: every input and output of the pass once; operations: one multiply-add per
    voxel and view of a projection, one per pixel of a filter row's transform stages."""
    c, kind = case, case['kind']
    if kind in ('dd_batch', 'cone_batch'):
        jobs = _batch_sizes(c)
        vol = [j['nx'] * j['ny'] * j['nz'] for j in jobs]
        det = [j['nu'] * (j.get('nv') or j['nz']) * j['nview'] for j in jobs]
        return {'bytes': 4 * (4 * sum(vol) + 2 * sum(det)),
                'flops': 4 * sum(v * j['nview'] for v, j in zip(vol, jobs))}
    vol = c['nx'] * c['ny'] * c.get('nz', 1) * c.get('batch', 1)
    det = c['nu'] * (c.get('nv') or c.get('nz', 1)) * c['nview'] * c.get('batch', 1)
    pair = 2 * vol * c['nview']
    fft = int(det * 10 * math.log2(4 * c['nu']))
    if kind == 'par_slice':
        return {'bytes': 4 * (2 * vol + 4 * det), 'flops': 2 * pair + fft}
    if kind in ('fan_stack', 'tomo'):
        return {'bytes': 8 * (vol + det), 'flops': 2 * pair}
    if kind == 'fan_fbp':
        return {'bytes': 4 * (vol + 3 * det), 'flops': pair + fft}
    if kind == 'unrolled':
        return {'bytes': 4 * (4 * vol + 3 * det), 'flops': 4 * c['niter'] * pair}
    if kind == 'cone_sqs':
        return {'bytes': 4 * (3 * vol + det), 'flops': 2 * pair}
    return {'bytes': 4 * (vol + det), 'flops': pair}


# ---------------------------------------------------------------- 64-bit values
def _chunks(n, per, most=1.2e8):
    """Slices of range(n) of which each holds about `most` values at `per` values an item."""
    k = max(1, int(most / max(per, 1)))
    return [slice(i, min(n, i + k)) for i in range(0, n, k)]


class _DD64:
    """The distance-driven projector of stacked slices in 64 bits; img [C, ny, nx] with C slices
    (batch x nz), prj [C', nview, nu] rows already selected."""

    def __init__(self, p, angles, fan, branchless=False):
        f = np.float32
        self.p, self.fan, self.branchless = p, fan, branchless
        self.du = float(f(p.du / p.dsd if fan else p.du))
        self.dx, self.dy, self.dso = float(f(p.dx)), float(f(p.dy)), float(f(p.dso))
        self.th = torch.from_numpy(angles).cuda().double()
        c, s = torch.cos(self.th), torch.sin(self.th)
        m = float(f(0.12))
        self.ymain = c.abs() > s.abs()
        self.wx = self.ymain.double() if branchless else torch.clamp((c.abs() - s.abs() + m) / (2 * m), 0, 1)
        # the column edges: angles for the fan beam, lengths for the parallel beam
        self.edges = -(torch.arange(p.nu + 1, device='cuda', dtype=F64) - p.nu / 2) * self.du
        self.mid = (self.edges[1:] + self.edges[:-1]) / 2 if fan else torch.zeros(p.nu, device='cuda', dtype=F64)

    def _rows(self, trace):
        """(rows, cells along a row, row centres, pitch along a row) of a trace along y (0) or x (1)."""
        n, m = (self.p.ny, self.p.nx) if trace == 0 else (self.p.nx, self.p.ny)
        d, e = (self.dy, self.dx) if trace == 0 else (self.dx, self.dy)
        return n, m, (torch.arange(n, device='cuda', dtype=F64) + 0.5 - n / 2) * d, e

    def _norm(self, v, trace):
        a = self.th[v, None] - self.mid[None, :]
        if trace == 0:
            return self.wx[v, None] * self.dy / torch.cos(a).abs()
        return (1 - self.wx[v, None]) * self.dx / torch.sin(a).abs()

    def _crossings(self, v, trace):
        """Index coordinate along a row where each column edge crosses the row's centre, [V, nu + 1, rows]."""
        th, e = self.th[v, None, None], self.edges[None, :, None]
        n, m, t, d = self._rows(trace)
        t = t[None, None, :]
        if self.fan:
            sx, sy = self.dso * torch.sin(th), -self.dso * torch.cos(th)
            k = torch.tan(e - th)
            x = sx + (t - sy) * k if trace == 0 else sy + (t - sx) / k
        elif trace == 0:
            x = (e - t * torch.sin(th)) / torch.cos(th)
        else:
            x = (e - t * torch.cos(th)) / torch.sin(th)
        return x / d + m / 2

    def fp(self, img):
        out = torch.zeros([len(self.th), self.p.nu, img.shape[0]], device='cuda', dtype=F64)
        for trace in (0, 1):
            use = torch.nonzero(self.wx > 0 if trace == 0 else self.wx < 1)[:, 0]
            n, m, _, _ = self._rows(trace)
            rows = img.permute(1, 2, 0) if trace == 0 else img.permute(2, 1, 0)       # [rows, cells, C]
            cum = torch.cat([torch.zeros_like(rows[:, :1]), torch.cumsum(rows, 1)], 1).reshape(-1, img.shape[0])
            first = (torch.arange(n, device='cuda') * (m + 1))[None, None, :]
            for k in _chunks(len(use), (self.p.nu + 1) * n * img.shape[0]):
                v = use[k]
                x = self._crossings(v, trace)
                xc = torch.clamp(x, 0, m)
                i = torch.clamp(xc.long(), max=m - 1)
                at = first + i
                g = torch.lerp(cum[at], cum[at + 1], (xc - i)[..., None])
                g = (g[:, 1:] - g[:, :-1]) / (x[:, 1:] - x[:, :-1])[..., None]
                out[v] += g.sum(2) * self._norm(v, trace)[..., None]
        return out.permute(2, 0, 1)

    def adjoint(self, prj):
        """The transpose of fp: prj [C, nview, nu] -> [C, ny, nx]."""
        p, C = self.p, prj.shape[0]
        img = torch.zeros([p.ny, p.nx, C], device='cuda', dtype=F64)
        for trace in (0, 1):
            use = torch.nonzero(self.wx > 0 if trace == 0 else self.wx < 1)[:, 0]
            n, m, t, d = self._rows(trace)
            t = t[None, None, :]
            r = ((torch.arange(m + 1, device='cuda', dtype=F64) - m / 2) * d)[None, :, None]
            for k in _chunks(len(use), (m + 1) * n * C):
                v = use[k]
                th = self.th[v, None, None]
                x, y = (r, t) if trace == 0 else (t, r)
                if self.fan:
                    px, py = x - self.dso * torch.sin(th), y + self.dso * torch.cos(th)
                    # the ray angle e: (px, py) along (sin(e - th), cos(e - th))
                    e = torch.atan2(px * torch.cos(th) + py * torch.sin(th), py * torch.cos(th) - px * torch.sin(th))
                else:
                    e = x * torch.cos(th) + y * torch.sin(th)
                col = torch.clamp((p.nu / 2 - e / self.du).floor().long(), 0, p.nu - 1)      # [V, m + 1, rows]
                edge = self._crossings(v, trace)
                lo, hi = torch.gather(edge, 1, col), torch.gather(edge, 1, col + 1)
                at = torch.arange(m + 1, device='cuda', dtype=F64)[None, :, None]
                frac = torch.clamp((at - lo) / (hi - lo), 0, 1)
                mass = (prj[:, v] * self._norm(v, trace)[None]).permute(1, 2, 0)             # [V, nu, C]
                cum = torch.cat([torch.zeros_like(mass[:, :1]), torch.cumsum(mass, 1)], 1).reshape(-1, C)
                base = torch.arange(len(v), device='cuda')[:, None, None] * (p.nu + 1) + col
                f = torch.lerp(cum[base], cum[base + 1], frac[..., None])
                sign = torch.sign(edge[:, -1] - edge[:, 0])[:, None, :, None]
                part = ((f[:, 1:] - f[:, :-1]) * sign).sum(0)
                img += part.permute(1, 0, 2) if trace == 0 else part
        return img.permute(2, 0, 1)

    def bp(self, prj, fbp):
        """The reference's backprojection (not the transpose of fp): [C, nview, nu] -> [C, ny, nx]."""
        p, C = self.p, prj.shape[0]
        img = torch.zeros([p.ny, p.nx, C], device='cuda', dtype=F64)
        x = ((torch.arange(p.nx, device='cuda', dtype=F64) + 0.5 - p.nx / 2) * self.dx)[None, None, :]
        y = ((torch.arange(p.ny, device='cuda', dtype=F64) + 0.5 - p.ny / 2) * self.dy)[None, :, None]
        if not fbp:
            a = self.th[:, None] - self.mid[None, :]
            prj = prj * torch.where(self.ymain[:, None], self.dy / torch.cos(a).abs(), self.dx / torch.sin(a).abs())
        cum = torch.cumsum(prj.permute(1, 2, 0), 1)
        cum = torch.cat([torch.zeros_like(cum[:, :1]), cum], 1)                              # [nview, nu + 1, C]
        for k in _chunks(len(self.th), p.nx * p.ny * C):
            th = self.th[k, None, None]
            c, s = torch.cos(th), torch.sin(th)
            flat = cum[k].reshape(-1, C)
            base = torch.arange(th.shape[0], device='cuda')[:, None, None] * (p.nu + 1)

            def at(px, py):
                u = torch.atan2(px * c + py * s, py * c - px * s + self.dso) if self.fan else px * c + py * s
                return p.nu / 2 - u / self.du

            def box(u1, u2):
                def upto(u):
                    u = torch.clamp(u, 0, p.nu)
                    i = torch.clamp(u.long(), max=p.nu - 1)
                    return torch.lerp(flat[base + i], flat[base + i + 1], (u - i)[..., None])
                return (upto(u2) - upto(u1)) / (u2 - u1)[..., None]

            hx, hy, one = self.dx / 2, self.dy / 2, torch.zeros_like(x + y)
            if self.fan:
                ym = self.ymain[k, None, None]
                ox, oy = torch.where(ym, hx, 0.0), torch.where(ym, 0.0, hy)
                val = box(at(x - ox, y - oy), at(x + ox, y + oy))
                if fbp:
                    rx, ry = x * c + y * s, y * c - x * s + self.dso
                    val = val * (self.dso ** 2 / (rx * rx + ry * ry))[..., None]
            else:
                # a footprint of no width belongs to a trace of weight 0
                w = self.wx[k, None, None, None]
                val = torch.where(w > 0, w * box(at(x - hx, y + one), at(x + hx, y + one)), 0.0) + \
                    torch.where(w < 1, (1 - w) * box(at(x + one, y - hy), at(x + one, y + hy)), 0.0)
            img += val.sum(0)
        return img.permute(2, 0, 1)

    def fp_rows(self, img):
        """[1, nz, ny, nx] -> [1, nview, nv, nu] with the slice interpolation of the detector rows."""
        p = self.p
        z = torch.clamp((torch.arange(p.nv, device='cuda', dtype=F64) - (p.nv - 1) / 2) * p.dv / p.dz + p.nz / 2 - 0.5,
                        0, p.nz)
        i = torch.clamp(z.long(), max=p.nz - 1)
        j = torch.clamp(i + 1, max=p.nz - 1)
        q, w = self.fp(img[0].double()), (z - i)[:, None, None]
        return ((1 - w) * q[i] + w * q[j]).permute(1, 0, 2)[None]

    def bp_rows(self, prj, fbp):
        """[1, nview, nv, nu] -> [1, nz, ny, nx] (as many detector rows as slices, at their centres)."""
        return self.bp(prj[0].double().permute(1, 0, 2), fbp)[None]


def _ramp64(p, prj, fan):
    """Hann-windowed ramp filter of the rows: the windowed kernel's linear convolution."""
    pi, n = float(np.float32(3.141592657)), p.nu
    du = float(np.float32(p.du / p.dsd if fan else p.du))
    k = torch.arange(-(n - 1), n, device='cuda', dtype=F64)
    den = torch.sin(k * du) if fan else k * du
    r = torch.where(k % 2 == 0, torch.zeros_like(k), -1 / (pi * den) ** 2)
    r[n - 1] = 1 / (4 * du * du)
    h = 0.5 * r + 0.25 * (torch.roll(r, 1) + torch.roll(r, -1))
    m = 1 << (3 * n).bit_length()
    pre = torch.cos((torch.arange(n, device='cuda', dtype=F64) - (n - 1) / 2) * du) if fan else 1.0
    hf = torch.fft.rfft(h, m)
    scale = pi / p.nview * du / (float(np.float32(p.dso)) if fan else 1.0)
    out = torch.empty(prj.shape, device='cuda', dtype=F64)
    for v in _chunks(prj.shape[1], prj.shape[2] * m):
        x = torch.fft.rfft(prj[:, v].double() * pre, m)
        out[:, v] = torch.fft.irfft(x * hf, m)[..., n - 1:2 * n - 1] * scale
    return out


def _pixel_fbp64(p, angles, prj):
    """Pixel-driven fan backprojection: linear interpolation between detector columns."""
    du, dso = float(np.float32(p.du / p.dsd)), float(np.float32(p.dso))
    x = ((torch.arange(p.nx, device='cuda', dtype=F64) + 0.5 - p.nx / 2) * float(np.float32(p.dx)))[None, None, :]
    y = ((torch.arange(p.ny, device='cuda', dtype=F64) + 0.5 - p.ny / 2) * float(np.float32(p.dy)))[None, :, None]
    img = torch.zeros([p.ny, p.nx, p.nz], device='cuda', dtype=F64)
    th = torch.from_numpy(angles).cuda().double()
    for k in _chunks(p.nview, p.nx * p.ny * p.nz):
        c, s = torch.cos(th[k, None, None]), torch.sin(th[k, None, None])
        rx, ry = x * c + y * s, y * c - x * s + dso
        u = (p.nu - 1) / 2 - torch.atan2(rx, ry) / du
        w = (dso ** 2 / (rx * rx + ry * ry)) * ((u >= 0) & (u < p.nu))
        u = torch.clamp(u, 0, p.nu - 1)
        i = u.long()
        flat = prj[0, k].permute(0, 2, 1).reshape(-1, p.nz)
        base = torch.arange(c.shape[0], device='cuda')[:, None, None] * p.nu
        q = torch.lerp(flat[base + i], flat[base + torch.clamp(i + 1, max=p.nu - 1)], (u - i)[..., None])
        img += (q * w[..., None]).sum(0)
    return img.permute(2, 0, 1)[None]


class _Siddon64:
    """Cone-beam line integrals through voxels in 64 bits and their transpose.  Each ray is cut by
    the slabs of its main axis; within a slab it meets at most one plane of either other axis
    (rays no steeper than 45 degrees to the main axis, which the cone scans here are)."""

    def __init__(self, p, geo):
        self.p, self.geo = p, geo

    def _segments(self, v, take):
        """take(cells, lengths) for every slab segment of the rays of views v, where x is (or after
        an exchange of x and y, y is) the main axis; rays keep the shape [V, nv, nu]."""
        p = self.p
        s, t = _cone_rays(p, self.geo, F64, v)
        d = [b - a for a, b in zip(s, t)]
        length = torch.sqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2)
        n, pitch = (p.nx, p.ny, p.nz), [float(np.float32(x)) for x in (p.dx, p.dy, p.dz)]
        o = [a / h + k / 2 for a, h, k in zip(s, pitch, n)]
        d = [a / h for a, h in zip(d, pitch)]
        xmain = (d[0].abs() >= d[1].abs())
        a0, a1 = 0.0, 1.0
        for k in range(3):
            e, f = (0 - o[k]) / d[k], (n[k] - o[k]) / d[k]
            a0, a1 = torch.clamp(torch.minimum(e, f), min=a0), torch.clamp(torch.maximum(e, f), max=a1)
        om, dm = torch.where(xmain, o[0], o[1]), torch.where(xmain, d[0], d[1])       # main axis
        oc, dc = torch.where(xmain, o[1], o[0]), torch.where(xmain, d[1], d[0])       # the other of x, y
        stride_m = torch.where(xmain, 1, p.nx)
        stride_c = torch.where(xmain, p.nx, 1)
        nc = torch.where(xmain, p.ny, p.nx)

        def crossing(org, dirn, lo, hi):
            """The parameter in [lo, hi] where the ray crosses a plane of one axis (lo if it does not)."""
            i, j = torch.floor(org + lo * dirn), torch.floor(org + hi * dirn)
            return torch.where(i != j, torch.minimum(torch.maximum((torch.maximum(i, j) - org) / dirn, lo), hi), lo)

        for slab in range(max(p.nx, p.ny)):
            e, f = (slab - om) / dm, (slab + 1 - om) / dm
            lo, hi = torch.maximum(torch.minimum(e, f), a0), torch.minimum(torch.maximum(e, f), a1)
            hi = torch.maximum(hi, lo)
            b, c = crossing(oc, dc, lo, hi), crossing(o[2], d[2], lo, hi)
            b, c = torch.minimum(b, c), torch.maximum(b, c)
            for q, r in ((lo, b), (b, c), (c, hi)):
                mid = (q + r) / 2
                ic = torch.minimum(torch.clamp((oc + mid * dc).long(), min=0), nc - 1)
                iz = torch.clamp((o[2] + mid * d[2]).long(), 0, p.nz - 1)
                cell = iz * (p.nx * p.ny) + ic * stride_c + slab * stride_m
                take(torch.clamp(cell, max=p.nx * p.ny * p.nz - 1), (r - q) * length)

    def fp(self, img):
        p, flat = self.p, img.double().reshape(-1)
        out = torch.zeros([p.nview, p.nv, p.nu], device='cuda', dtype=F64)
        for k in _chunks(p.nview, p.nu * p.nv, 1.6e7):
            def take(cell, length, o=out[k]):
                o.addcmul_(flat[cell], length)
            self._segments(k, take)
        return out

    def bp(self, prj):
        """The transpose, voxel by voxel: the chords of the rays in each voxel's shadow (det_v along z and
        det_u horizontal, so a ray's extent in x and y depends on its column only)."""
        p = self.p
        n, (dx, dy, dz, du, dv) = (p.nx, p.ny, p.nz), [float(np.float32(x)) for x in (p.dx, p.dy, p.dz, p.du, p.dv)]
        ex, ey, ez = [(torch.arange(k + 1, device='cuda', dtype=F64) - k / 2) * h for k, h in zip(n, (dx, dy, dz))]
        out = torch.zeros([p.nz, p.ny, p.nx], device='cuda', dtype=F64)
        rows = torch.arange(p.nv, device='cuda', dtype=F64) - (p.nv - 1) / 2
        for k in range(p.nview):
            C, U, S = (torch.from_numpy(a[k]).double().tolist() for a in (self.geo.det_center, self.geo.det_u,
                                                                         self.geo.src))
            ax, ay = C[0] - S[0], C[1] - S[1]
            det = ax * U[1] - ay * U[0]
            px, py = (ex - S[0])[None, :], (ey - S[1])[:, None]
            tau = (px * U[1] - py * U[0]) / det                          # voxel corners [ny + 1, nx + 1]
            u = (ax * py - ay * px) / det / tau / du + (p.nu - 1) / 2

            def corners(a):
                a = torch.stack([a[:-1, :-1], a[:-1, 1:], a[1:, :-1], a[1:, 1:]])
                return a.amin(0), a.amax(0)
            ulo, uhi = corners(u)
            tlo, thi = corners(tau)
            zlo, zhi = (ez[:-1] - S[2])[:, None, None], (ez[1:] - S[2])[:, None, None]
            off = (p.nv - 1) / 2 - (C[2] - S[2]) / dv
            vlo = torch.minimum(zlo / tlo, zlo / thi) / dv + off
            vhi = torch.maximum(zhi / tlo, zhi / thi) / dv + off
            iu0, iv0 = torch.ceil(ulo).long(), torch.ceil(vlo).long()
            wu, wv = int(torch.ceil((uhi - ulo).max())), int(torch.ceil((vhi - vlo).max()))
            cu = (torch.arange(p.nu, device='cuda', dtype=F64) - (p.nu - 1) / 2) * du
            dirx, diry, dirz = ax + U[0] * cu, ay + U[1] * cu, C[2] - S[2] + rows * dv
            y = prj[k].double() * torch.sqrt((dirx ** 2 + diry ** 2)[None, :] + (dirz ** 2)[:, None])
            for j in range(wu):
                iu = iu0 + j
                iuc = torch.clamp(iu, 0, p.nu - 1)
                x0, x1 = px[:, :-1] / dirx[iuc], px[:, 1:] / dirx[iuc]
                y0, y1 = py[:-1] / diry[iuc], py[1:] / diry[iuc]
                lo = torch.maximum(torch.minimum(x0, x1), torch.minimum(y0, y1))
                hi = torch.minimum(torch.maximum(x0, x1), torch.maximum(y0, y1))
                hi = torch.where((iu >= 0) & (iu < p.nu), hi, lo)
                for i in range(wv):
                    iv = iv0 + i
                    ivc = torch.clamp(iv, 0, p.nv - 1)
                    r = dirz[ivc]
                    z0, z1 = zlo / r, zhi / r
                    chord = torch.minimum(torch.maximum(z0, z1), hi) - torch.maximum(torch.minimum(z0, z1), lo)
                    chord = torch.clamp(chord, min=0) * (iv == ivc)
                    out.addcmul_(chord, y.reshape(-1)[ivc * p.nu + iuc])
        return out


def _tv64(x, eps=1e-8):
    """(s1, s2) of the anisotropic total variation with unit weights; x [B, nz, ny, nx]."""
    def behind(a, d):
        return torch.cat([torch.zeros_like(a.narrow(d, 0, 1)), torch.diff(a, dim=d)], d)

    d = [behind(x, k) for k in (1, 2, 3)]
    var = torch.sqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2 + eps)
    s1, s2 = (d[0] + d[1] + d[2]) / var, 3 / var
    for k in (1, 2, 3):
        n = x.shape[k]
        nxt = torch.cat([var.narrow(k, 1, n - 1), var.narrow(k, n - 1, 1)], k)
        ahead = torch.cat([-torch.diff(x, dim=k), torch.zeros_like(x.narrow(k, 0, 1))], k)
        s1, s2 = s1 + ahead / nxt, s2 + 1 / nxt
    return s1, s2


class _Pair64(torch.autograd.Function):
    """A linear map with its transpose as the gradient."""

    @staticmethod
    def forward(ctx, x, fwd, adj):
        ctx.adj = adj
        return fwd(x)

    @staticmethod
    def backward(ctx, g):
        return ctx.adj(g), None, None


def _unrolled64(s):
    c, dd = s.case, _DD64(s.p, s.ang, True)

    def fwd(x):
        return dd.fp(x[:, 0])[:, :, None, :]

    def adj(y):
        return dd.adjoint(y[:, :, 0, :])[:, None]

    q = s.prj.double().requires_grad_(True)
    w, x = s.weight.double(), s.x0.double()
    for _ in range(c['niter']):
        r = _Pair64.apply(x, fwd, adj) / s.pn - q / s.pn
        g = _Pair64.apply(r * w, adj, fwd) / s.pn
        s1, s2 = _tv64(x)
        x = x - (g + 2e-3 * s1) / (s.norm_img.double() + 2e-3 * s2)
    x.backward(2.0 * (x.detach() - s.target.double()))
    return {'x': x.detach(), 'grad': q.grad}


def _tomo64(s):
    """Area averages over the footprint boxes, which are products of an interval in x and one in y."""
    p = s.p
    f = [float(np.float32(v)) for v in (p.dx, p.dy, p.dz, p.du, p.dv)]
    dx, dy, dz, du, dv = f
    img, prj = s.img[0].double(), s.prj[0].double()
    u = (torch.arange(p.nu, device='cuda', dtype=F64) - (p.nu - 1) / 2) * du
    v = (torch.arange(p.nv, device='cuda', dtype=F64) - (p.nv - 1) / 2) * dv
    fp, bp = torch.zeros_like(prj), torch.zeros_like(img)

    def overlap(a, b, n):
        """[len(a), n]: share of the interval [a, b] in each cell."""
        i = torch.arange(n, device='cuda', dtype=F64)[None, :]
        return torch.clamp(torch.minimum(b[:, None], i + 1) - torch.maximum(a[:, None], i), min=0) / (b - a)[:, None]

    for k in range(s.case['nview']):
        S, C = (torch.from_numpy(a[k]).double().tolist() for a in (s.src, s.dc))
        ray = torch.sqrt((S[2] - C[2]) ** 2 + (S[1] - C[1] - v[:, None]) ** 2 + (S[0] - C[0] - u[None, :]) ** 2)
        scale = dz / abs(S[2] - C[2]) * ray
        w = prj[k] * scale
        for iz in range(p.nz):
            # projection: the plane at the slice's lower edge
            z = (iz - p.nz / 2) * dz + p.cz
            r = (z - S[2]) / (C[2] - S[2])

            def ends(c0, s0, e, h, d, n):
                return [(s0 + (c0 + e + o - s0) * r) / d + n / 2 for o in (-h / 2, h / 2)]
            bx = overlap(*ends(C[0], S[0], u, du, dx, p.nx), p.nx)
            by = overlap(*ends(C[1], S[1], v, dv, dy, p.ny), p.ny)
            fp[k] += by @ img[iz] @ bx.T
            # backprojection: the voxel's shadow from its centre plane, detector cells indexed from their centres
            q = (C[2] - S[2]) / (z + dz / 2 - S[2])

            def cells(c0, s0, n, d, e, m):
                x = (torch.arange(n, device='cuda', dtype=F64) - (n - 1) / 2) * d
                return [(s0 - c0 + q * (x + o - s0)) / e + (m - 1) / 2 for o in (-d / 2, d / 2)]
            wx = overlap(*cells(C[0], S[0], p.nx, dx, du, p.nu), p.nu)
            wy = overlap(*cells(C[1], S[1], p.ny, dy, dv, p.nv), p.nv)
            bp[iz] += wy @ w @ wx.T
        fp[k] *= scale
    return {'fp': fp[None], 'bp': bp[None]}


def exact(case, seed):
    c, kind, s = case, case['kind'], prepare(case, seed)
    if kind in ('par_slice', 'fan_stack', 'fan_fp', 'fan_bp'):
        fan = kind != 'par_slice'
        dd = _DD64(s.p, s.ang, fan, c['branchless'])
        if kind == 'fan_fp':
            return dd.fp_rows(s.img)
        if kind == 'fan_bp':
            return dd.bp_rows(s.prj, c['fbp'])
        if kind == 'fan_stack':
            return {'fp': dd.fp_rows(s.img), 'bp': dd.bp_rows(s.prj, c['fbp'])}
        flt = _ramp64(s.p, s.prj, False)
        return {'fp': dd.fp_rows(s.img), 'filtered': flt, 'img': dd.bp_rows(flt, True)}
    if kind == 'fan_fbp':
        flt = _ramp64(s.p, s.prj, True)
        return {'filtered': flt, 'img': _pixel_fbp64(s.p, s.ang, flt)}
    if kind == 'unrolled':
        return _unrolled64(s)
    if kind == 'dd_batch':
        ops = [_DD64(p, a, j['fan']) for j, p, a in s.jobs]
        prj = [dd.fp_rows(x) for dd, x in zip(ops, s.x)]
        return {'prj': prj, 'img': [dd.bp_rows(y, False) for dd, y in zip(ops, prj)]}
    if kind == 'cone_batch':
        ops = [_Siddon64(p, g) for p, g in s.jobs]
        prj = [op.fp(x) for op, x in zip(ops, s.x)]
        return {'prj': prj, 'img': [op.bp(y) for op, y in zip(ops, prj)]}
    if kind == 'tomo':
        return _tomo64(s)
    op = _Siddon64(s.p, s.geo)
    if kind == 'cone_fp':
        return op.fp(s.img[0])[None]
    if kind == 'cone_bp':
        return op.bp(s.prj[0])[None]
    r = op.fp(s.img[0]) / s.pn - s.prj[0].double() / s.pn
    x = s.img.double()
    s1, s2 = _tv64(x)
    return x - (op.bp(r)[None] / s.pn + 1e-3 * s1) / (s.norm_img.double() + 1e-3 * s2)
