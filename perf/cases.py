"""The calls this framework is timed on: what a program that turns voxel
volumes into meshes has it do, from the smallest volume to the 512^3 one.

Volumes are head phantoms as in nii2mesh_amd/synth.py (ellipsoid, blobs,
ventricles, two spheres outside it, noise), drawn on the GPU for any size
and seed; atlases are weighted-Voronoi labels.  Device cases read a volume
in HBM and copy the meshes (n2m_ctx_device_mesh) into vertex and index
buffers of the program's own, of a fixed size, as a renderer keeps them: the
context's own arrays last until its next call.  Drop-in cases go from host
arrays to host arrays through the reference's own entry points, as the
linked CLI does.

The differentiable path is not among them: its tests are switched off until
the cause of a stall of their process is known.
"""
import ctypes as C
import math

import numpy as np
import torch

import nii2mesh_amd as n2m

CLASSIC, LEWINER = n2m.CUBES_CLASSIC, n2m.CUBES_LEWINER


def listed():
    return [
        # the smallest useful call (the smoke test's volume): all latency
        dict(name='meshify_tiny', kind='meshify', nx=48, ny=44, nz=40, cubes=LEWINER, bubbles=True, iso=110.0,
             hc=20),
        # the reference's plain run: 128^3, classic cubes, largest cluster,
        # no smoothing of the mesh
        dict(name='meshify_plain_128', kind='meshify', nx=128, ny=128, nz=128, cubes=CLASSIC, bubbles=False,
             iso=128.0, hc=0),
        # a skull-stripped brain scan's size (odd rows), every cleaning
        # option and 100 smoothing iterations (-l 1 -b 1 -s 100)
        dict(name='meshify_brain_142x178x142', kind='meshify', nx=142, ny=178, nz=142, cubes=LEWINER, bubbles=True,
             iso=110.0, hc=100),
        # a low-resolution template through the drop-in entry points, classic
        # cubes and a light smoothing
        dict(name='dropin_91x109x91', kind='dropin', nx=91, ny=109, nz=91, cubes=CLASSIC, bubbles=False, iso=110.0,
             hc=10),
        # the 256^3 drop-in workload: host volume in, smoothed mesh out
        dict(name='dropin_lewiner_256', kind='dropin', nx=256, ny=256, nz=256, cubes=LEWINER, bubbles=True,
             iso=80.0, hc=100),
        # dark / mid / bright surfaces of a scan with odd sides
        dict(name='pipeline_245x347x275', kind='pipeline', nx=245, ny=347, nz=275, modes='123', hc=50),
        # the headline workload: 512^3, three isolevels, 100 iterations each
        dict(name='pipeline_512', kind='pipeline', nx=512, ny=512, nz=512, modes='123', hc=100),
        # the batched atlas workload: every label of a 256^3 parcellation
        dict(name='atlas_256_370', kind='atlas', nx=256, ny=256, nz=256, labels=370, cubes=CLASSIC, post=0),
        # a smaller parcellation with odd sides, Lewiner cubes, the sform and
        # smoothed label surfaces (-a 1 -s 15)
        dict(name='atlas_ragged_60', kind='atlas', nx=117, ny=151, nz=133, labels=60, cubes=LEWINER, post=15),
        # the three automatic isolevels of a scan
        dict(name='thresholds_181x217x181', kind='thresholds', nx=181, ny=217, nz=181),
        # connected components of a noisy mask, all labels, host to host
        dict(name='bwlabel_26_128', kind='bwlabel', nx=128, ny=128, nz=128, conn=26, largest=False),
        # the loader's conversion of a raw int16 scan in HBM
        dict(name='decode_i16_256x256x176', kind='decode', nx=256, ny=256, nz=176, datatype=n2m.DT_INT16),
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, lo, hi):
    """Three sides about one log-uniform size, each up to a quarter off, so
    that rows are odd, even or whole words."""
    n = _loguniform(rng, lo, hi)
    s = [min(hi, max(lo, int(round(n * rng.uniform(0.8, 1.25))))) for _ in range(3)]
    if rng.random() < 0.3:  # scanners' row lengths
        s[0] = min(hi, max(lo, 32 * max(1, round(s[0] / 32))))
    return dict(nx=s[0], ny=s[1], nz=s[2])


def draw(rng):
    kind = rng.choice(['meshify', 'meshify', 'meshify', 'dropin', 'pipeline', 'pipeline', 'atlas', 'atlas',
                       'thresholds', 'bwlabel', 'decode'])
    c = dict(kind=kind)
    if kind in ('meshify', 'dropin'):
        c.update(_sides(rng, 40, 320 if kind == 'meshify' else 256))
        c.update(cubes=rng.choice([CLASSIC, LEWINER]), bubbles=rng.random() < 0.5,
                 iso=float(rng.randint(70, 135)), hc=rng.choice([0, _loguniform(rng, 5, 100)]))
    elif kind == 'pipeline':
        c.update(_sides(rng, 64, 384))
        c.update(modes=rng.choice(['2', '12', '13', '123']), hc=_loguniform(rng, 10, 100))
    elif kind == 'atlas':
        c.update(_sides(rng, 64, 256))
        c.update(labels=_loguniform(rng, 8, 370), cubes=rng.choice([CLASSIC, LEWINER]),
                 post=rng.choice([0, _loguniform(rng, 5, 50)]))
    elif kind == 'thresholds':
        c.update(_sides(rng, 40, 512))
    elif kind == 'bwlabel':
        c.update(_sides(rng, 40, 256))
        c.update(conn=rng.choice([6, 18, 26]), largest=rng.random() < 0.5)
    else:
        c.update(_sides(rng, 40, 512))
        c.update(datatype=rng.choice([n2m.DT_UINT8, n2m.DT_INT16, n2m.DT_UINT16, n2m.DT_FLOAT32]))
    return c


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(int(seed))


def _axes(case):
    """Coordinates of the voxel centres in the phantom's 128^3 frame."""
    ax = [torch.arange(case[k], dtype=torch.float32, device='cuda') * (128.0 / case[k]) for k in ('nx', 'ny', 'nz')]
    return ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]


# centre (in semi-axes of the ellipsoid), sigma and height of the six blobs of
# the 512^3 benchmark volume; a seed moves them a little, as between two scans
BLOBS = [((-0.24, 0.24, 0.67), 4.8, -40.0), ((-0.45, 0.65, 0.28), 5.3, 40.0), ((-0.02, -0.35, 0.93), 8.7, -40.0),
         ((0.01, -0.22, -0.83), 4.2, -40.0), ((0.36, -0.12, -0.57), 8.8, 40.0), ((0.06, -0.34, 0.05), 7.6, 40.0)]


def _head(case, seed, noise=8.0):
    """float32 (nz, ny, nx) phantom, 0..255, in HBM."""
    rng = np.random.Generator(np.random.PCG64(seed))
    x, y, z = _axes(case)
    c, ax = 64.0, (50.0, 40.0, 45.0)
    inside = ((x - c) / ax[0]) ** 2 + ((y - c) / ax[1]) ** 2 + ((z - c) / ax[2]) ** 2 <= 1.0
    vol = torch.where(inside, 160.0, 0.0)
    for p, s, amp in BLOBS:
        p = np.array(p) + rng.uniform(-0.02, 0.02, 3)
        s *= float(rng.uniform(0.98, 1.02))
        g = [torch.exp(-(a - (c + q * h)) ** 2 / (2 * s * s)) for a, q, h in zip((x, y, z), p.tolist(), ax)]
        vol += inside * (amp * g[0] * g[1] * g[2])
    for side in (-1, 1):
        r = ((x - (c + 12.0 * side)) / 6.0) ** 2 + ((y - 60.0) / 12.0) ** 2 + ((z - 66.0) / 8.0) ** 2
        vol = torch.where(r <= 1.0, 40.0, vol)
    r = ((x - c) ** 2 + (y - (c + 52.0)) ** 2 + (z - c) ** 2).sqrt()
    vol = torch.where((r <= 8.0) & (r > 6.0), 200.0, vol)
    r = ((x - 18.0) ** 2 + (y - 18.0) ** 2 + (z - 110.0) ** 2).sqrt()
    vol = torch.where(r <= 6.0, 200.0, vol)
    vol += noise * torch.randn(vol.shape, generator=_gen(seed), device='cuda')
    return vol.clamp_(0, 255).contiguous()


def _parcels(case, seed):
    """float32 labels 0..labels: the ellipsoid split into the cells of a
    multiplicatively weighted Voronoi diagram with log-normal cell sizes."""
    rng = np.random.Generator(np.random.PCG64(seed))
    n = case['labels']
    x, y, z = _axes(case)
    c, ax = 64.0, np.array([50.0, 40.0, 45.0])
    inside = ((x - c) / ax[0]) ** 2 + ((y - c) / ax[1]) ** 2 + ((z - c) / ax[2]) ** 2 <= 1.0
    idx = inside.flatten().nonzero().flatten()
    shape = inside.shape
    P = torch.stack([torch.broadcast_to(a, shape).flatten()[idx] for a in (x, y, z)], 1)
    size = np.exp(rng.normal(0.0, 1.68, n))
    rad = np.cbrt(size / size.sum())
    cand = rng.uniform(-1, 1, (16 * n + 64, 3))
    seeds = c + cand[(cand ** 2).sum(1) <= 1.0][:n] * ax
    S = torch.tensor(seeds, dtype=torch.float32, device='cuda')
    w = torch.tensor(1.0 / rad ** 2, dtype=torch.float32, device='cuda')
    lab = torch.empty(len(idx), dtype=torch.float32, device='cuda')
    for b in range(0, len(idx), 1 << 20):
        q = P[b:b + (1 << 20)]
        best = torch.full((len(q),), float('inf'), device='cuda')
        for k in range(n):
            d = ((q - S[k]) ** 2).sum(1) * w[k]
            near = d < best
            best = torch.where(near, d, best)
            lab[b:b + (1 << 20)][near] = k + 1.0
    vol = torch.zeros(inside.numel(), dtype=torch.float32, device='cuda')
    vol[idx] = lab
    vol = vol.view(shape)
    # every cell keeps its own centre, so that every label has a voxel
    at = [torch.tensor(np.rint(seeds[:, a] * case[k] / 128.0).astype(np.int64), device='cuda')
          for a, k in enumerate(('nx', 'ny', 'nz'))]
    vol[at[2], at[1], at[0]] = torch.arange(1, n + 1, dtype=torch.float32, device='cuda')
    return vol


_TORCH_DT = {n2m.DT_UINT8: torch.uint8, n2m.DT_INT16: torch.int16, n2m.DT_UINT16: torch.uint16,
             n2m.DT_FLOAT32: torch.float32}


def _raw(case, seed):
    """A raw scan as stored: (voxels in HBM, slope, intercept)."""
    v = _head(case, seed)
    t = case['datatype']
    if t == n2m.DT_UINT8:
        return v.round().to(torch.uint8), 0.5, -10.0
    if t == n2m.DT_INT16:
        return (v * 12.0 - 1024.0).round().to(torch.int16), 1.0, 24.0
    if t == n2m.DT_UINT16:
        return (v * 200.0).round().to(torch.int32).to(torch.uint16), 0.01, 0.0
    return v, 2.5, 1.0


def prepare(case, seed):
    kind = case['kind']
    st = dict(case=case, dims=(case['nx'], case['ny'], case['nz']))
    if kind in ('meshify', 'pipeline', 'thresholds'):
        st['vol'] = _head(case, seed)
        if kind == 'meshify':  # meshify works in place: a copy is its input
            st['work'] = torch.empty_like(st['vol'])
            st['buf'] = _buffers(case)
        elif kind == 'pipeline':
            st['buf'] = [_buffers(case, m) for m in case['modes']]
    elif kind == 'dropin':
        st['host'] = _head(case, seed).cpu().numpy()
        st['work'] = np.empty_like(st['host'])
        st['buf'] = _buffers(case, host=True)
    elif kind == 'atlas':
        st['vol'] = _parcels(case, seed)
        st['buf'] = _buffers(case)
        st['srow'] = [-1.5, 0, 0, 90, 0, 1.5, 0, -126, 0, 0, 1.5, -72] if case['post'] else None
    elif kind == 'bwlabel':
        v = _head(case, seed, noise=24.0)
        st['host'] = (v > 150.0).float().cpu().numpy()
        st['work'] = np.empty_like(st['host'])
        st['lib'] = n2m.lib()
    else:
        st['raw'], st['slope'], st['inter'] = _raw(case, seed)
        st['out'] = torch.empty(st['raw'].shape, dtype=torch.float32, device='cuda')
    if 'host' not in st:
        ctx = st['ctx'] = n2m.DeviceContext()
        L = ctx.L
        L.n2m_ctx_device_mesh.argtypes = [C.c_void_p, C.c_int, C.POINTER(C.c_void_p), C.POINTER(C.c_void_p)]
        L.n2m_ctx_atlas_device_mesh.argtypes = [C.c_void_p, C.POINTER(C.c_void_p), C.POINTER(C.c_void_p),
                                                C.POINTER(C.c_int), C.POINTER(C.c_int)]
        L.n2m_ctx_set_thresholds.argtypes = [C.c_void_p, C.c_void_p, C.c_int64, C.c_int, C.POINTER(C.c_int),
                                             C.POINTER(C.c_float)]
        L.n2m_ctx_decode.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int64, C.c_float, C.c_float, C.c_void_p]
        if kind == 'meshify':
            st['prm'] = ctx.params(case['iso'], cubes=case['cubes'], preSmooth=True, onlyLargest=True,
                                   fillBubbles=case['bubbles'])
        elif kind == 'pipeline':
            st['prm'] = ctx.params(0.0, cubes=LEWINER, preSmooth=True, onlyLargest=True, fillBubbles=True)
        elif kind == 'atlas':
            st['prm'] = ctx.params(0.5, cubes=case['cubes'], preSmooth=True, onlyLargest=False, fillBubbles=False)
    torch.cuda.synchronize()  # the library's contexts run on streams of their own
    return st


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def _room(case, mode=None):
    """Triangles the program's buffers hold (half as many vertices): well over
    what the phantom gives, by the surface and, where an isolevel may cut the
    noise, by the volume."""
    n = case['nx'] * case['ny'] * case['nz']
    if case['kind'] == 'atlas':
        return int(2 * _atlas_tris(case)) + 20000
    return int(20 * n ** (2.0 / 3.0) + (0.35 if mode == '3' else 0.12) * n) + 4096


def _buffers(case, mode=None, host=False):
    t = _room(case, mode)
    if host:
        return np.zeros((t, 3), np.int32), np.zeros((t // 2 + 16, 3), np.float64)
    return (torch.zeros((t, 3), dtype=torch.int32, device='cuda'),
            torch.zeros((t // 2 + 16, 3), dtype=torch.float64, device='cuda'))


class _View:
    """Device memory of a context as torch sees it."""

    def __init__(self, ptr, rows, typestr):
        self.__cuda_array_interface__ = dict(shape=(rows, 3), typestr=typestr, data=(ptr, False), version=2)


def _fill(buf, t, p, nt, npt):
    """A context's mesh into the program's buffers: [triangle and vertex
    counts, triangles, vertices]."""
    tris, pts = buf
    if nt:
        tris[:nt].copy_(torch.as_tensor(_View(t, nt, '<i4'), device='cuda'))
    if npt:
        pts[:npt].copy_(torch.as_tensor(_View(p, npt, '<f8'), device='cuda'))
    return [nt, npt, tris, pts]


def _device_mesh(ctx, k, buf):
    t, p = C.c_void_p(), C.c_void_p()
    if ctx.L.n2m_ctx_device_mesh(ctx.h, k, C.byref(t), C.byref(p)) != 0:
        raise IndexError(k)
    nt, npt = ctx.mesh_size(k)
    return _fill(buf, t.value, p.value, nt, npt)


def _thresholds(st, modes):
    m = (C.c_int * len(modes))(*modes)
    out = (C.c_float * len(modes))()
    ctx = st['ctx']
    if ctx.L.n2m_ctx_set_thresholds(ctx.h, C.c_void_p(st['vol'].data_ptr()), st['vol'].numel(), len(modes), m,
                                    out) != 0:
        raise RuntimeError(n2m.last_error())
    return list(out)


def _ok(rc):
    if rc != 0:
        raise RuntimeError('call failed: ' + n2m.last_error())


def _wait():
    """Work queued on torch's stream that touches what the library reads or
    overwrites is complete before a call, as the library asks."""
    torch.cuda.current_stream().synchronize()


def run(st):
    case, kind = st['case'], st['case']['kind']
    if kind == 'meshify':
        ctx = st['ctx']
        st['work'].copy_(st['vol'])
        _wait()
        _ok(ctx.meshify(st['work'].data_ptr(), st['dims'], st['prm']))
        if case['hc']:
            _ok(ctx.smooth_hc(0, 0.1, 0.5, case['hc']))
        return [st['work']] + _device_mesh(ctx, 0, st['buf'])
    if kind == 'pipeline':
        ctx = st['ctx']
        isos = _thresholds(st, [int(m) for m in case['modes']])
        _wait()
        _ok(ctx.pipeline(st['vol'].data_ptr(), st['dims'], st['prm'], isos, 0.1, 0.5, case['hc']))
        return isos + [a for k in range(len(isos)) for a in _device_mesh(ctx, k, st['buf'][k])]
    if kind == 'dropin':
        lib = n2m.lib(case['cubes'])
        vol, (tris, pts) = st['work'], st['buf']
        np.copyto(vol, st['host'])  # the call changes its volume
        rc, t, p = lib.meshify(vol, case['iso'], True, True, case['bubbles'])
        _ok(rc)
        if case['hc']:
            lib.laplacian_smoothHC(p, t, 0.1, 0.5, case['hc'])
        tris[:len(t)] = t
        pts[:len(p)] = p
        return [vol, len(t), len(p), tris, pts]
    if kind == 'atlas':
        ctx = st['ctx']
        _wait()
        _ok(ctx.atlas(st['vol'].data_ptr(), st['dims'], st['prm'], case['post'], st['srow']))
        t, p, nt, npt = C.c_void_p(), C.c_void_p(), C.c_int(), C.c_int()
        ctx.L.n2m_ctx_atlas_device_mesh(ctx.h, C.byref(t), C.byref(p), C.byref(nt), C.byref(npt))
        ent = np.frombuffer(b''.join(map(bytes, ctx.atlas_entries())), np.int32).reshape(-1, 6)
        return [ent] + _fill(st['buf'], t.value, p.value, nt.value, npt.value)
    if kind == 'thresholds':
        return _thresholds(st, [1, 2, 3])
    if kind == 'bwlabel':
        np.copyto(st['work'], st['host'])
        return [st['lib'].bwlabel(st['work'], case['conn'], case['largest'], False), st['work']]
    ctx = st['ctx']
    _ok(ctx.L.n2m_ctx_decode(ctx.h, C.c_void_p(st['raw'].data_ptr()), case['datatype'], st['raw'].numel(),
                             st['slope'], st['inter'], C.c_void_p(st['out'].data_ptr())))
    return st['out']


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _atlas_tris(case):
    n = case['nx'] * case['ny'] * case['nz']
    return 11.0 * case['labels'] * (0.18 * n / case['labels']) ** (2.0 / 3.0)


def work(case):
    """Bytes: the volume in once and the meshes out once (36 bytes per
    triangle with its half a vertex and that vertex's 24); a drop-in call's
    changed volume out too.  Triangles are estimated from the phantom: about
    4.6 per square voxel side for the outer surface, 0.15 per voxel where the
    bright isolevel cuts the noise, 11 per label and cell^(2/3) voxels.
    Operations: 25 per voxel smoothed, 130 per vertex and smoothing
    iteration (two sums over six neighbour pairs of three coordinates)."""
    kind = case['kind']
    n = case['nx'] * case['ny'] * case['nz']
    side2 = n ** (2.0 / 3.0)
    if kind in ('meshify', 'dropin'):
        t = 4.6 * side2
        b = 4.0 * n * (2 if kind == 'dropin' else 1) + 24.0 * t
        return {'bytes': b, 'flops': 25.0 * n + 130.0 * case['hc'] * t / 2}
    if kind == 'pipeline':
        t = sum({'1': 5.8 * side2, '2': 4.6 * side2, '3': 0.15 * n}[m] for m in case['modes'])
        return {'bytes': 4.0 * n + 24.0 * t, 'flops': 25.0 * n + 130.0 * case['hc'] * t / 2}
    if kind == 'atlas':
        t = _atlas_tris(case)
        return {'bytes': 4.0 * n + 24.0 * t, 'flops': 25.0 * n + 130.0 * case['post'] * t / 2}
    if kind == 'thresholds':
        return {'bytes': 4.0 * n, 'flops': 4.0 * n}
    if kind == 'bwlabel':
        return {'bytes': 8.0 * n, 'flops': 1.0 * n}
    size = _TORCH_DT[case['datatype']].itemsize
    return {'bytes': (size + 4.0) * n, 'flops': 2.0 * n}


def exact(case, seed):
    """The decoded voxels.  The other cases have no such value short of the
    whole method again: meshes and labels follow from decisions on 32-bit
    voxels (which side of the isolevel, which bin), made exactly."""
    if case['kind'] != 'decode':
        return None
    raw, slope, inter = _raw(case, seed)
    if raw.dtype == torch.uint16:
        raw = raw.to(torch.int32)
    return raw.double() * float(np.float32(slope)) + float(np.float32(inter))
