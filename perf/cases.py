"""Performance cases of the density-field and power-spectrum path.

Every case is one call, or one short chain of calls, of the public Python API, as a
reference user's script makes it (library/Pk_library/Pk_snapshot.py:77-89: positions ->
MA -> density contrast -> Pk).  Kinds:

  ma      MAS_library.MA, or MA_rsd when "rsd" is set, on GPU positions
  pk      Pk_library.Pk (one field) or XPk (several) on GPU density fields
  batch   MA_batch of the matter and the weighted tracers of many realisations, then
          Pk_batch: auto and cross spectra of each
  map     MA onto a 2D map, then Pk_plane
  host    MA on numpy arrays, then Pk of the contrast: the drop-in use, where the
          particles and the grid live in host memory

Particle orders ("order"): "lattice", Zel'dovich-displaced particles in ID order, as an
unsorted simulation snapshot holds them; "shuffled", the same particles in random order;
"uniform", uniform random positions; "tracers", random points moved by a displacement
field (a halo or galaxy catalogue, in no order).
"""
import math

import numpy as np
import torch

from pylians3_amd import MAS_library as MASL
from pylians3_amd import Pk_library as PKL
from pylians3_amd import batch, workloads

DEV = 'cuda'
SCHEMES = ('NGP', 'CIC', 'TSC', 'PCS')
HUBBLE, REDSHIFT = 100.0, 0.5          # of the redshift-space cases


def listed():
    return [
        # the smallest request a server of the library sees: 1e5 particles on 64^3
        dict(name='ma_cic_64_small', kind='ma', dims=64, n=100_000, mas='CIC', order='tracers',
             weights=False, rsd=False, box=500.0),
        # the small uniform box: 128^3 particles on 128^3, CIC
        dict(name='ma_cic_128_uniform', kind='ma', dims=128, n=128 ** 3, mas='CIC', order='uniform',
             weights=False, rsd=False, box=1000.0),
        # a weighted halo or galaxy catalogue, far fewer objects than cells, on a fine grid
        dict(name='ma_pcs_w_512_catalogue', kind='ma', dims=512, n=2_000_000, mas='PCS', order='tracers',
             weights=True, rsd=False, box=1000.0),
        # a 512^3 snapshot in redshift space on 512^3: density contrast in one call
        dict(name='ma_rsd_tsc_512', kind='ma', dims=512, n=512 ** 3, mas='TSC', order='lattice',
             weights=False, rsd=True, box=1000.0),
        # as many particles out of order (light cones, resampled or domain-decomposed data),
        # on a grid that is no power of two
        dict(name='ma_tsc_500_shuffled', kind='ma', dims=500, n=512 ** 3, mas='TSC', order='shuffled',
             weights=False, rsd=False, box=1000.0),
        # the largest field: 1024^3 particles on 1024^3, PCS
        dict(name='ma_pcs_1024', kind='ma', dims=1024, n=1024 ** 3, mas='PCS', order='lattice',
             weights=False, rsd=False, box=2000.0),
        # spectra of a small field, the reference's default line of sight
        dict(name='pk_64', kind='pk', dims=64, fields=1, axis=2, mas='CIC', box=500.0),
        # a field of ragged size
        dict(name='pk_300', kind='pk', dims=300, fields=1, axis=1, mas='PCS', box=1000.0),
        # auto and cross spectra of two fields of different schemes
        dict(name='xpk_256', kind='pk', dims=256, fields=2, axis=2, mas='TSC', box=1000.0),
        # spectra of the 512^3 field, line of sight along the redshift-space axis
        dict(name='pk_512', kind='pk', dims=512, fields=1, axis=0, mas='TSC', box=1000.0),
        # an ensemble of realisations: matter and weighted tracers, auto and cross spectra
        dict(name='batch_128', kind='batch', dims=128, nreal=32, axis=0, mas='CIC', ntracers=600_000,
             box=500.0),
        # a script on numpy arrays: 256^3 particles onto 256^3, then the spectra
        dict(name='host_cic_256', kind='host', dims=256, n=256 ** 3, mas='CIC', order='lattice', axis=0,
             box=1000.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(('ma', 'ma', 'ma', 'pk', 'pk', 'batch', 'map', 'host'))
    axis = rng.randrange(3)
    box = round(rng.uniform(200.0, 2000.0), 1)
    if kind == 'ma':
        dims = rng.choice((64, 128, 256, 512, 1024)) if rng.random() < 0.4 else _log_int(rng, 60, 800)
        order = rng.choice(('lattice', 'shuffled', 'uniform', 'tracers'))
        n = _log_int(rng, 100_000, 134_217_728)
        if order in ('lattice', 'shuffled'):
            n = min(512, max(47, int(round(n ** (1.0 / 3.0))))) ** 3
        return dict(kind='ma', dims=dims, n=n, mas=rng.choice(SCHEMES), order=order,
                    weights=order == 'tracers' and rng.random() < 0.7,
                    rsd=order == 'lattice' and rng.random() < 0.4, box=box)
    if kind == 'pk':
        dims = rng.choice((64, 128, 256, 512)) if rng.random() < 0.6 else _log_int(rng, 50, 400)
        fields = rng.choice((1, 1, 2, 3)) if dims <= 256 else 1
        return dict(kind='pk', dims=dims, fields=fields, axis=axis, mas=rng.choice(SCHEMES), box=box)
    if kind == 'batch':
        return dict(kind='batch', dims=rng.choice((64, 128)), nreal=rng.randint(4, 48), axis=axis,
                    mas='CIC', ntracers=_log_int(rng, 50_000, 1_000_000), box=box)
    if kind == 'map':
        return dict(kind='map', dims=_log_int(rng, 200, 2048), n=_log_int(rng, 100_000, 20_000_000),
                    mas='CIC', box=box)
    d = rng.randint(64, 256)
    return dict(kind='host', dims=rng.choice((64, 128, 256)), n=d ** 3, mas='CIC', order='lattice',
                axis=axis, box=box)


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7fffffff)


def _wrapped(x, box):
    x = torch.remainder(x, box)
    x[x >= box] = 0.0                  # remainder can round up to box
    return x


def _cube_root(n):
    d = int(round(n ** (1.0 / 3.0)))
    if d ** 3 != n:
        raise ValueError('lattice cases take a cube of particles')
    return d


def _positions(order, n, box, seed, axes=3):
    g = _gen(seed)
    if order == 'lattice':
        return workloads.zeldovich(_cube_root(n), box, seed)
    if order == 'shuffled':
        p = workloads.zeldovich(_cube_root(n), box, seed)
        return p[torch.randperm(n, generator=g, device=DEV)].contiguous()
    q = torch.rand((n, 3), generator=g, device=DEV, dtype=torch.float32) * box
    if order == 'tracers':
        d = 64
        psi = workloads.displacement_field(d, box, seed + 1)
        cell = torch.clamp((q * (d / box)).long(), max=d - 1)
        lin = (cell[:, 0] * d + cell[:, 1]) * d + cell[:, 2]
        q = q + psi.view(3, -1)[:, lin].t()
    q = _wrapped(q, box)
    return q[:, :axes].contiguous()


def _weights(n, seed):
    return torch.exp(torch.randn((n,), generator=_gen(seed + 77), device=DEV, dtype=torch.float32))


def _density(dims, box, seed, shared=0.0):
    """A lognormal density contrast with a falling spectrum; `shared` in [0, 1): how much
    of the modes it takes from the field of seed // 100 (correlated fields)."""
    w = torch.randn((dims,) * 3, generator=_gen(seed), device=DEV, dtype=torch.float32)
    if shared:
        u = torch.randn((dims,) * 3, generator=_gen(seed // 100), device=DEV, dtype=torch.float32)
        w = shared * u + math.sqrt(1.0 - shared * shared) * w
    wk = torch.fft.rfftn(w)
    k1 = torch.fft.fftfreq(dims, 1.0 / dims, device=DEV) * (2 * math.pi / box)
    kz = torch.fft.rfftfreq(dims, 1.0 / dims, device=DEV) * (2 * math.pi / box)
    k2 = k1.view(-1, 1, 1) ** 2 + k1.view(1, -1, 1) ** 2 + kz.view(1, 1, -1) ** 2
    k2[0, 0, 0] = 1.0
    wk *= k2 ** -0.375 * torch.exp(-k2 / 0.5)
    wk[0, 0, 0] = 0.0
    f = torch.fft.irfftn(wk, s=(dims,) * 3)
    f = torch.exp(0.8 * f / f.std())
    return (f / f.mean() - 1.0).contiguous()


def _field_schemes(case):
    first = SCHEMES.index(case['mas'])
    return [SCHEMES[(first + 3 * f) % 4] for f in range(case['fields'])]


def prepare(case, seed):
    kind, box = case['kind'], case['box']
    s = dict(case=case)
    if kind == 'ma':
        s['pos'] = _positions(case['order'], case['n'], box, seed)
        s['W'] = _weights(case['n'], seed) if case['weights'] else None
        if case['rsd']:
            s['vel'] = 300.0 * torch.randn((case['n'], 3), generator=_gen(seed + 5), device=DEV)
    elif kind == 'pk':
        F = case['fields']
        s['fields'] = [_density(case['dims'], box, 100 * seed + f, 0.6 if F > 1 else 0.0)
                       for f in range(F)]
    elif kind == 'batch':
        rng = np.random.default_rng(seed)
        R, d = case['nreal'], case['dims']
        counts = rng.integers(case['ntracers'] // 4, case['ntracers'] + 1, R)
        s['mpos'] = torch.cat([workloads.zeldovich(d, box, seed * 64 + r) for r in range(R)])
        s['moffs'] = np.arange(R + 1, dtype=np.int64) * d ** 3
        s['tpos'] = torch.cat([_positions('tracers', int(counts[r]), box, seed * 64 + r) for r in range(R)])
        s['toffs'] = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
        s['tw'] = _weights(int(s['toffs'][-1]), seed)
        s['mean_m'] = np.full(R, np.float32(1.0))
        sums = torch.stack([x.double().sum() for x in torch.split(s['tw'], [int(c) for c in counts])])
        s['mean_t'] = (sums / d ** 3).float().cpu().numpy()
    elif kind == 'map':
        s['pos'] = _positions('tracers', case['n'], box, seed, axes=2)
    else:
        s['pos'] = _positions(case['order'], case['n'], box, seed).cpu().numpy()
    return s


# ---------------------------------------------------------------- one pass
def _mean(case):
    return float(np.float32(case['n'] / case['dims'] ** 3))


def _pk_out(p):
    return dict(k3D=p.k3D, Pk=p.Pk, Nmodes3D=p.Nmodes3D, k1D=p.k1D, Pk1D=p.Pk1D, Nmodes1D=p.Nmodes1D,
                kpar=p.kpar, kper=p.kper, Pk2D=p.Pk2D, Nmodes2D=p.Nmodes2D, Pkphase=p.Pkphase)


def _xpk_out(p):
    return dict(k3D=p.k3D, Pk=p.Pk, XPk=p.XPk, Nmodes3D=p.Nmodes3D, k1D=p.k1D, Pk1D=p.Pk1D,
                PkX1D=p.PkX1D, Nmodes1D=p.Nmodes1D, kpar=p.kpar, kper=p.kper, Pk2D=p.Pk2D,
                PkX2D=p.PkX2D, Nmodes2D=p.Nmodes2D)


def run(state):
    case = state['case']
    kind, dims, box = case['kind'], case['dims'], case['box']
    if kind == 'ma' and case['rsd']:
        delta = torch.empty((dims,) * 3, dtype=torch.float32, device=DEV)
        MASL.MA_rsd(state['pos'], state['vel'], delta, box, HUBBLE, REDSHIFT, 0, case['mas'],
                    overwrite=True, scale=_mean(case), shift=1.0)
        return delta
    if kind == 'ma':
        grid = torch.zeros((dims,) * 3, dtype=torch.float32, device=DEV)
        MASL.MA(state['pos'], grid, box, case['mas'], W=state['W'])
        return grid
    if kind == 'pk':
        f = state['fields']
        if len(f) == 1:
            return _pk_out(PKL.Pk(f[0], box, case['axis'], case['mas'], verbose=False))
        return _xpk_out(PKL.XPk(f, box, case['axis'], _field_schemes(case)))
    if kind == 'batch':
        R = case['nreal']
        matter = torch.empty((R,) + (dims,) * 3, dtype=torch.float32, device=DEV)
        tracers = torch.empty_like(matter)
        batch.MA_batch(state['mpos'], state['moffs'], matter, box, case['mas'], accumulate=False)
        batch.MA_batch(state['tpos'], state['toffs'], tracers, box, case['mas'], W=state['tw'],
                       accumulate=False)
        res = batch.Pk_batch([matter, tracers], box, case['axis'], (case['mas'],) * 2,
                             scales=np.stack([state['mean_m'], state['mean_t']], 1),
                             shifts=np.ones((R, 2), np.float32))
        keys = ('Pk', 'XPk', 'Pk1D', 'PkX1D', 'Pk2D', 'PkX2D')
        return dict({k: np.stack([getattr(r, k) for r in res]) for k in keys},
                    matter=matter, tracers=tracers, k3D=res[0].k3D, Nmodes3D=res[0].Nmodes3D,
                    Nmodes1D=res[0].Nmodes1D, Nmodes2D=res[0].Nmodes2D)
    if kind == 'map':
        grid = torch.zeros((dims,) * 2, dtype=torch.float32, device=DEV)
        MASL.MA(state['pos'], grid, box, case['mas'])
        p = PKL.Pk_plane(grid, box, case['mas'], verbose=False)
        return dict(grid=grid, k=p.k, Pk=p.Pk, Nmodes=p.Nmodes)
    delta = np.zeros((dims,) * 3, np.float32)
    MASL.MA(state['pos'], delta, box, case['mas'])
    delta /= np.float32(_mean(case))
    delta -= np.float32(1.0)
    p = PKL.Pk(delta, box, case['axis'], case['mas'], verbose=False)
    return dict(_pk_out(p), delta=delta)


# ---------------------------------------------------------------- the work of a pass
def _spectra_bytes(dims, spectra):
    m = dims // 2
    n2 = (m + 1) * (int(math.sqrt(2) * m) + 1)
    return 8.0 * (spectra * (n2 + 3 * int(math.sqrt(3) * m) + m) + 3 * n2)


def _fft_flops(cells):
    return 2.5 * cells * math.log2(cells)


def work(case):
    kind, d = case['kind'], case['dims']
    F = SCHEMES.index(case['mas']) + 1
    if kind == 'ma':
        per = 12 + (4 if case['weights'] else 0) + (4 if case['rsd'] else 0)
        return dict(bytes=float(case['n']) * per + 4.0 * d ** 3, flops=2.0 * case['n'] * F ** 3)
    if kind == 'pk':
        f = case['fields']
        return dict(bytes=4.0 * f * d ** 3 + _spectra_bytes(d, f * (f + 1) // 2),
                    flops=f * _fft_flops(d ** 3) + 20.0 * f * (f + 1) / 2 * d ** 3 / 2)
    if kind == 'batch':
        R, nt = case['nreal'], case['nreal'] * case['ntracers'] * 0.625
        nm = float(R) * d ** 3
        return dict(bytes=12.0 * nm + 16.0 * nt + 8.0 * nm + R * _spectra_bytes(d, 3),
                    flops=2.0 * (nm + nt) * F ** 3 + 2.0 * R * _fft_flops(d ** 3))
    if kind == 'map':
        return dict(bytes=8.0 * case['n'] + 4.0 * d ** 2 + 24.0 * d,
                    flops=2.0 * case['n'] * F ** 2 + _fft_flops(d ** 2))
    return dict(bytes=12.0 * case['n'] + 4.0 * d ** 3 + _spectra_bytes(d, 1),
                flops=2.0 * case['n'] * F ** 3 + _fft_flops(d ** 3))


# ---------------------------------------------------------------- the same in 64 bits
def _axis_weights(x, mas):
    """First node and the node weights of coordinates x (cells, float64)."""
    if mas == 'NGP':
        return torch.floor(x + 0.5).long(), [torch.ones_like(x)]
    if mas == 'CIC':
        i = torch.floor(x)
        return i.long(), [1.0 - (x - i), x - i]
    if mas == 'TSC':
        i = torch.floor(x - 0.5)
        u = x - i - 1.0
        return i.long(), [0.5 * (0.5 - u) ** 2, 0.75 - u * u, 0.5 * (0.5 + u) ** 2]
    i = torch.floor(x) - 1.0
    w = []
    for j in range(4):
        s = torch.abs(x - i - j)
        w.append(torch.where(s < 1.0, (4.0 - 6.0 * s * s + 3.0 * s ** 3) / 6.0, (2.0 - s) ** 3 / 6.0))
    return i.long(), w


def _deposit64(pos, W, dims, box, mas, shift_x=None):
    axes = pos.shape[1]
    grid = torch.zeros(dims ** axes, dtype=torch.float64, device=DEV)
    step = 1 << 24
    for a in range(0, pos.shape[0], step):
        p = torch.as_tensor(pos[a:a + step], device=DEV).double()
        if shift_x is not None:
            p[:, 0] = torch.remainder(p[:, 0] + shift_x[a:a + step].double(), box)
        feet = [_axis_weights(p[:, c] * (dims / box), mas) for c in range(axes)]
        w0 = None if W is None else W[a:a + step].double()
        for ix, wx in enumerate(feet[0][1]):
            nx = torch.remainder(feet[0][0] + ix, dims)
            wx = wx if w0 is None else wx * w0
            for iy, wy in enumerate(feet[1][1]):
                nxy = nx * dims + torch.remainder(feet[1][0] + iy, dims)
                wxy = wx * wy
                if axes == 2:
                    grid.index_add_(0, nxy, wxy)
                    continue
                for iz, wz in enumerate(feet[2][1]):
                    grid.index_add_(0, nxy * dims + torch.remainder(feet[2][0] + iz, dims), wxy * wz)
    return grid.view((dims,) * axes)


def _window(dims, p):
    k = torch.fft.fftfreq(dims, 1.0 / dims, dtype=torch.float64, device=DEV).round()
    x = math.pi / dims * k
    return torch.where(k == 0, torch.ones_like(x), (x / torch.sin(torch.where(k == 0, 1.0, x))) ** p)


def _spectra64(fields, box, axis, schemes):
    """Reference sums over the independent modes of (dims, dims, dims) fields, float64."""
    F, dims = len(fields), fields[0].shape[0]
    m, even = dims // 2, dims % 2 == 0
    kF = 2.0 * math.pi / box
    kmax, kmax_per = int(math.sqrt(3 * m * m)), int(math.sqrt(2 * m * m))
    dk = []
    for f, mas in zip(fields, schemes):
        x = torch.fft.rfftn(f.double())
        c = _window(dims, SCHEMES.index(mas) + 1)
        cz = c[:m + 1].clone()
        for sh, cc in (((dims, 1, 1), c), ((1, dims, 1), c), ((1, 1, m + 1), cz)):
            x *= cc.view(sh)
        dk.append(x)
    kf = torch.arange(dims, device=DEV)
    kf = torch.where(kf > m, kf - dims, kf)
    ky, kz = kf.view(1, -1, 1), torch.arange(m + 1, device=DEV).view(1, 1, -1)
    pairs = [(i, i) for i in range(F)] + [(i, j) for i in range(F) for j in range(i + 1, F)]
    S = len(pairs)
    n2 = (m + 1) * (kmax_per + 1)
    z = lambda n: torch.zeros(n, dtype=torch.float64, device=DEV)  # noqa: E731
    N3, K3, N2, N1, K1, ph = z(kmax + 1), z(kmax + 1), z(n2), z(m + 1), z(m + 1), z(kmax + 1)
    P3, P2, P1 = z((S, 3, kmax + 1)), z((S, n2)), z((S, m + 1))
    slab = max(1, (1 << 23) // (dims * (m + 1)))
    for a in range(0, dims, slab):
        kx = kf[a:a + slab].view(-1, 1, 1)
        plane = (kz == 0) | ((kz == m) & even)
        edge = (kx == 0) | ((kx == m) & even)
        ok = (~(plane & ((kx < 0) | (edge & (ky < 0))))).expand(kx.shape[0], dims, m + 1)
        comp = [t.expand(ok.shape)[ok] for t in (kx, ky, kz)]
        k2 = comp[0] ** 2 + comp[1] ** 2 + comp[2] ** 2
        kpar = comp[axis].abs()
        per2 = k2 - kpar * kpar
        i3 = torch.sqrt(k2.double()).long()
        i2 = (m + 1) * torch.sqrt(per2.double()).long() + kpar
        mu2 = torch.where(k2 == 0, 0.0, (kpar * kpar).double() / k2.clamp(min=1).double())
        L2, L4 = (3 * mu2 - 1) / 2, (35 * mu2 * mu2 - 30 * mu2 + 3) / 8
        one = torch.ones_like(mu2)
        in1 = k2 <= m * m

        def add(out, idx, val):
            out += torch.bincount(idx, weights=val, minlength=out.numel())
        add(N3, i3, one)
        add(K3, i3, torch.sqrt(k2.double()))
        add(N2, i2, one)
        add(N1, kpar[in1], one[in1])
        add(K1, kpar[in1], kpar[in1].double())
        v = [x[a:a + slab][ok] for x in dk]
        for s, (i, j) in enumerate(pairs):
            d2 = v[i].real * v[j].real + v[i].imag * v[j].imag
            add(P3[s, 0], i3, d2)
            add(P3[s, 1], i3, d2 * L2)
            add(P3[s, 2], i3, d2 * L4)
            add(P2[s], i2, d2)
            add(P1[s], kpar[in1], d2[in1])
        if F == 1:
            add(ph, i3, torch.atan2(v[0].real, v[0].abs()) ** 2)
    fact = (box / dims ** 2) ** 3
    kN = m * kF
    k1 = K1 / N1 * kF
    P1 = P1 * fact * (math.pi * (kN ** 2 - k1 ** 2).clamp(min=0) / N1) / (2 * math.pi) ** 2
    P3 = P3 / N3 * fact * torch.tensor([1.0, 5.0, 9.0], dtype=torch.float64, device=DEV).view(1, 3, 1)
    idx = torch.arange(n2, device=DEV)
    per, par = (idx // (m + 1)).double(), (idx % (m + 1)).double()
    host = lambda t: t.cpu().numpy()  # noqa: E731
    out = dict(k3D=host((K3 / N3 * kF)[1:]), Nmodes3D=host(N3[1:]), k1D=host(k1[1:]),
               Nmodes1D=host(N1[1:]), kpar=host((par + 0.5) * kF), kper=host((per + 0.5) * kF),
               Nmodes2D=host(N2))
    p3, p2, p1 = host(P3[:, :, 1:].permute(2, 1, 0)), host((P2 / N2 * fact).t()), host(P1[:, 1:].t())
    if F == 1:
        out.update(Pk=p3[:, :, 0], Pk2D=p2[:, 0], Pk1D=p1[:, 0], Pkphase=host((ph / N3 * fact)[1:]))
    else:
        out.update(Pk=p3[:, :, :F], XPk=p3[:, :, F:], Pk2D=p2[:, :F], PkX2D=p2[:, F:], Pk1D=p1[:, :F],
                   PkX1D=p1[:, F:])
    return out


def _plane64(grid, box, mas):
    dims = grid.shape[0]
    m, even = dims // 2, dims % 2 == 0
    c = _window(dims, SCHEMES.index(mas) + 1)
    x = torch.fft.rfftn(grid.double()) * c.view(-1, 1) * c[:m + 1].view(1, -1)
    kx = torch.arange(dims, device=DEV)
    kx = torch.where(kx > m, kx - dims, kx).view(-1, 1)
    ky = torch.arange(m + 1, device=DEV).view(1, -1)
    ok = ~(((ky == 0) | ((ky == m) & even)) & (kx < 0))
    k2 = (kx ** 2 + ky ** 2)[ok].double()
    b, n = torch.sqrt(k2).long(), int(math.sqrt(2 * m * m)) + 1
    N, K, P = (torch.bincount(b, weights=w, minlength=n)[1:]
               for w in (torch.ones_like(k2), torch.sqrt(k2), (x.real ** 2 + x.imag ** 2)[ok]))
    return dict(k=(K / N * 2 * math.pi / box).cpu().numpy(), Nmodes=N.cpu().numpy(),
                Pk=(P / N * (box / dims ** 2) ** 2).cpu().numpy())


def exact(case, seed):
    kind, dims, box = case['kind'], case['dims'], case['box']
    if kind == 'ma' and case['n'] * (SCHEMES.index(case['mas']) + 1) ** 3 > 1e10:
        return None                    # the 1024^3 deposit in 64 bits takes too long
    s = prepare(case, seed)
    if kind == 'ma':
        shift = s['vel'][:, 0].double() * ((1.0 + REDSHIFT) / HUBBLE) if case['rsd'] else None
        g = _deposit64(s['pos'], s['W'], dims, box, case['mas'], shift)
        return g / _mean(case) - 1.0 if case['rsd'] else g
    if kind == 'pk':
        return _spectra64(s['fields'], box, case['axis'],
                          [case['mas']] if case['fields'] == 1 else _field_schemes(case))
    if kind == 'batch':
        return _batch64(s, case)
    if kind == 'map':
        grid = _deposit64(s['pos'], None, dims, box, case['mas'])
        return dict(_plane64(grid, box, case['mas']), grid=grid)
    delta = _deposit64(s['pos'], None, dims, box, case['mas']) / _mean(case) - 1.0
    return dict(_spectra64([delta], box, case['axis'], [case['mas']]), delta=delta.cpu().numpy())


def _batch64(s, case):
    dims, box, mas = case['dims'], case['box'], case['mas']
    res, grids = [], ([], [])
    for r in range(case['nreal']):
        deltas = []
        for out, pos, offs, W, mean in ((grids[0], 'mpos', 'moffs', None, 'mean_m'),
                                        (grids[1], 'tpos', 'toffs', 'tw', 'mean_t')):
            a, b = int(s[offs][r]), int(s[offs][r + 1])
            g = _deposit64(s[pos][a:b], None if W is None else s[W][a:b], dims, box, mas)
            out.append(g)
            deltas.append(g / float(s[mean][r]) - 1.0)
        res.append(_spectra64(deltas, box, case['axis'], [mas, mas]))
    keys = ('Pk', 'XPk', 'Pk1D', 'PkX1D', 'Pk2D', 'PkX2D')
    one = ('k3D', 'Nmodes3D', 'Nmodes1D', 'Nmodes2D')
    return dict({k: np.stack([x[k] for x in res]) for k in keys}, **{k: res[0][k] for k in one},
                matter=torch.stack(grids[0]), tracers=torch.stack(grids[1]))
