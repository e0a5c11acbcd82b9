"""The calls whose speed this framework answers for, as a user's program makes them.

A case is one whole reconstruction: catalogs in hand, shifted catalogs out.  It names the
reconstruction class, the mesh, the precision, the catalogs (a survey with randoms and a local line
of sight, or a periodic box) and where they live (device tensors or numpy arrays).
"""
import math

import torch  # before pyrecon_amd, so that both use the HIP runtime that torch brings
import numpy as np

import pyrecon_amd

F, BIAS, RADIUS, CELL = 0.8, 2.0, 15., 7.8125
CLASSES = {'multigrid': pyrecon_amd.MultiGridReconstruction,
           'iterative_fft': pyrecon_amd.IterativeFFTReconstruction,
           'plane_parallel': pyrecon_amd.PlaneParallelFFTReconstruction,
           'particle': pyrecon_amd.IterativeFFTParticleReconstruction}


def _case(name, algorithm, nmesh, ndata, nrandoms, precision='plain', dtype='f8', geometry='survey', host=False,
          randoms_field='disp+rsd'):
    n0, n1, n2 = (nmesh,) * 3 if isinstance(nmesh, int) else nmesh
    case = dict(algorithm=algorithm, n0=n0, n1=n1, n2=n2, ndata=ndata, nrandoms=nrandoms, precision=precision,
                dtype=dtype, geometry=geometry, host=host, randoms_field=randoms_field)
    if name is not None: case['name'] = name
    return case


def listed():
    return [
        # a first try or a small mock, called in a loop over mocks: latency and launches count
        _case('mock_64', 'multigrid', 64, 100000, 1000000),
        # the most frequent size of a stream of mocks, in mixed precision
        _case('mock_128_mixed', 'multigrid', 128, 300000, 3000000, precision='mixed'),
        # an ordinary survey at the default precision
        _case('survey_256', 'multigrid', 256, 2000000, 20000000),
        # catalogs and meshes kept in single precision; RecIso (randoms moved by the displacement only)
        _case('survey_256_f4', 'multigrid', 256, 1000000, 10000000, dtype='f4', randoms_field='disp'),
        # a survey that is not cubic, its mesh chosen by cell size
        _case('survey_ragged_mixed', 'multigrid', (384, 320, 448), 3000000, 30000000, precision='mixed'),
        # the headline survey, and the same mesh at the default precision
        _case('survey_512_mixed', 'multigrid', 512, 20000000, 100000000, precision='mixed'),
        _case('survey_512', 'multigrid', 512, 5000000, 50000000),
        # a simulation box: periodic, plane-parallel, no randoms
        _case('box_192', 'multigrid', 192, 2000000, 0, geometry='box'),
        # catalogs that live in numpy arrays: the copies to and from the device are part of the call
        _case('survey_256_numpy', 'multigrid', 256, 2000000, 10000000, precision='mixed', host=True),
        # the field-level iterative reconstruction of a survey
        _case('iterative_fft_384', 'iterative_fft', 384, 4000000, 20000000, randoms_field='disp'),
        # a periodic box through the plane-parallel reconstruction, lengths with factors 3 and 5
        _case('plane_parallel_240', 'plane_parallel', (240, 225, 250), 1000000, 0, geometry='box', host=True),
        # the particle-level iterative reconstruction of a small survey, from and to numpy
        _case('particle_128', 'particle', 128, 300000, 2000000, host=True),
    ]


def draw(rng):
    """Another case of the same ranges; at most as costly as the headline survey."""
    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    algorithm = rng.choice(['multigrid'] * 7 + ['iterative_fft'] * 2 + ['plane_parallel', 'particle'])
    top = {'multigrid': 512, 'iterative_fft': 400, 'plane_parallel': 400, 'particle': 160}[algorithm]
    base = log_uniform(56, top)
    ragged = rng.random() < 0.5
    nmesh = []
    for _ in range(3):
        target = base * (log_uniform(0.75, 1.3) if ragged else 1.)
        if not ragged and nmesh:
            nmesh.append(nmesh[0])
            continue
        if algorithm == 'multigrid':
            # the sizes that the class recommends, now and then any even one with small factors
            steps = [64, 80, 96, 112, 128, 160, 192, 224, 256, 320, 384, 448, 512]
            if rng.random() < 0.25: steps = [n for n in range(48, top + 1, 2) if _smooth(n)]
        else:
            steps = [n for n in range(48, top + 1) if _smooth(n)]
        nmesh.append(min(steps, key=lambda n: abs(n - target)))
    cells = nmesh[0] * nmesh[1] * nmesh[2]
    geometry = 'box' if algorithm == 'plane_parallel' or (algorithm != 'particle' and rng.random() < 0.2) else 'survey'
    host = algorithm == 'particle' or (algorithm == 'plane_parallel') or rng.random() < 0.15
    limit = 1000000 if algorithm in ('plane_parallel', 'particle') else 3000000 if host else 20000000
    ndata = int(min(limit, max(20000, cells * log_uniform(0.02, 0.4))))
    nrandoms = 0 if geometry == 'box' else int(min(100000000, ndata * rng.uniform(4., 10.)))
    if host: nrandoms = min(nrandoms, 10000000 if algorithm == 'multigrid' else 3000000)
    dtype, precision = 'f8', 'plain'
    if algorithm == 'multigrid':
        precision = rng.choice(['plain', 'mixed', 'mixed'])
        if precision == 'plain' and geometry == 'survey' and rng.random() < 0.3: dtype = 'f4'
    return _case(None, algorithm, tuple(nmesh), ndata, nrandoms, precision=precision, dtype=dtype, geometry=geometry,
                 host=host, randoms_field=rng.choice(['disp+rsd', 'disp']))


def _smooth(n):
    for q in (2, 3, 5, 7):
        while n % q == 0: n //= q
    return n == 1


# ------------------------------------------------------------------ inputs

def _geometry(case):
    """Mesh, box and centre: cells of one size; a survey is seen from the origin, outside its box."""
    nmesh = (case['n0'], case['n1'], case['n2'])
    boxsize = [CELL * n for n in nmesh]
    return nmesh, boxsize, [0., 0., 0.75 * boxsize[2]] if case['geometry'] == 'survey' else [0.5 * b for b in boxsize]


def _modes(case, seed):
    """Fourier modes of the displacement that clusters the data: wavevectors, directions k / k^2 and phases."""
    gen = torch.Generator(device='cpu').manual_seed(1000003 * seed + 5)
    _, boxsize, _ = _geometry(case)
    index = torch.randint(-8, 9, (24, 3), generator=gen).double()
    index[:, 0] += (index == 0).all(dim=1)
    k = 2. * math.pi * index / torch.tensor(boxsize, dtype=torch.float64)
    amplitude = k / (k**2).sum(dim=1, keepdim=True).sqrt() * 2.5
    phase = 2. * math.pi * torch.rand(24, generator=gen, dtype=torch.float64)
    return k.cuda(), amplitude.cuda(), phase.cuda()


def _length(x):
    return torch.sqrt(x[:, 0]**2 + x[:, 1]**2 + x[:, 2]**2)


def _catalog(case, size, seed, clustered):
    """Positions and weights: in a box, uniform and (data) displaced, wrapped, unit weights from 0.5 to 1.5; in a
    survey, those of a shell around the observer, thinned with its radial density, with FKP weights."""
    _, boxsize, boxcenter = _geometry(case)
    gen = torch.Generator(device='cuda').manual_seed(1000003 * seed + (1 if clustered else 2))
    box = torch.tensor(boxsize, dtype=torch.float64, device='cuda')
    low = torch.tensor(boxcenter, dtype=torch.float64, device='cuda') - box / 2.
    k, amplitude, phase = _modes(case, seed)
    survey = case['geometry'] == 'survey'
    rmid, width = boxcenter[2], 0.5 * boxsize[2]
    positions = torch.empty((size, 3), dtype=torch.float64, device='cuda')
    filled = 0
    while filled < size:
        batch = min(1 << 23, max(1 << 16, 3 * (size - filled)))
        x = low + box * torch.rand((batch, 3), generator=gen, dtype=torch.float64, device='cuda')
        if clustered:
            psi = torch.zeros_like(x)
            for kk, aa, pp in zip(k, amplitude, phase):
                psi += torch.sin(x[:, 0] * kk[0] + x[:, 1] * kk[1] + x[:, 2] * kk[2] + pp)[:, None] * aa
            if survey:
                los = x / _length(x)[:, None]
                x = x + psi + F * (psi * los).sum(dim=1, keepdim=True) * los
            else:
                x = x + psi
                x[:, 2] += F * psi[:, 2]
                x = (x - low) % box + low
        keep = ((x >= low) & (x <= low + box)).all(dim=1)
        if survey:
            r = _length(x)
            keep &= (r - rmid).abs() < 0.9 * width
            keep &= torch.rand(batch, generator=gen, dtype=torch.float64, device='cuda') \
                < torch.exp(-((r - rmid) / (0.6 * width))**2)
        x = x[keep][:size - filled]
        positions[filled:filled + len(x)] = x
        filled += len(x)
    if survey:
        r = _length(positions)
        weights = 1. / (1. + 3. * torch.exp(-((r - rmid) / (0.6 * width))**2))
    else:
        weights = 0.5 + torch.rand(size, generator=gen, dtype=torch.float64, device='cuda')
    if case['dtype'] == 'f4': positions, weights = positions.float(), weights.float()
    return positions, weights


def _inputs(case, seed):
    out = dict(zip(('data', 'data_weights'), _catalog(case, case['ndata'], seed, True)))
    if case['nrandoms']:
        out.update(zip(('randoms', 'randoms_weights'), _catalog(case, case['nrandoms'], seed, False)))
    return out


def prepare(case, seed):
    state = _inputs(case, seed)
    if case['host']: state = {name: value.cpu().numpy() for name, value in state.items()}
    state['case'] = case
    return state


# ------------------------------------------------------------------ one pass

class _Exported(object):
    """A device array as torch sees it (no copy); the array lives as long as the tensor."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = dict(shape=tuple(array.shape), typestr=np.dtype(array.dtype).str,
                                             data=(array.ptr, False), strides=None, version=2)


def _tensor(array):
    if isinstance(array, np.ndarray): return array
    return torch.as_tensor(_Exported(array), device='cuda')


def run(state):
    case = state['case']
    nmesh, boxsize, boxcenter = _geometry(case)
    kwargs = dict(f=F, bias=BIAS, nmesh=nmesh, boxsize=boxsize, boxcenter=boxcenter, dtype=case['dtype'])
    if case['geometry'] == 'box': kwargs.update(los='z', wrap=True)
    if case['precision'] != 'plain': kwargs['precision'] = case['precision']
    recon = CLASSES[case['algorithm']](**kwargs)
    recon.assign_data(state['data'], state['data_weights'])
    if case['nrandoms']: recon.assign_randoms(state['randoms'], state['randoms_weights'])
    recon.set_density_contrast(smoothing_radius=RADIUS)
    recon.run()
    # the particle reconstruction keeps its data and moves them itself
    out = {'data': _tensor(recon.read_shifted_positions('data' if case['algorithm'] == 'particle' else state['data']))}
    if case['nrandoms']:
        out['randoms'] = _tensor(recon.read_shifted_positions(state['randoms'], field=case['randoms_field']))
    return out


def work(case):
    cells = case['n0'] * case['n1'] * case['n2']
    points = case['ndata'] + case['nrandoms']
    word = 4 if case['dtype'] == 'f4' else 8
    # positions and weights in, shifted positions out
    nbytes = points * 7 * word
    transform = 5. * cells * math.log2(cells)
    flops = points * (40. + 150.)  # paint; gradient or value read and the shift
    flops += (2 if case['nrandoms'] else 1) * transform  # smoothing: forward and inverse, real meshes
    if case['algorithm'] == 'multigrid':
        # six V-cycles a level of ten sweeps, a residual and the transfers, 45 operations a cell
        flops += 6 * 11 * 45. * cells * (8. / 7.)**2
    elif case['algorithm'] == 'plane_parallel':
        flops += 4 * transform / 2.
    else:
        per_iteration = 1 + (6 if case['geometry'] == 'survey' and case['algorithm'] == 'iterative_fft' else 3)
        flops += (3 * per_iteration + 4) * transform / 2.
    return {'bytes': nbytes, 'flops': flops}


# ------------------------------------------------------------------ the same in 64 bits, with torch alone

def _axis(values, axis):
    shape = [1, 1, 1]
    shape[axis] = -1
    return values.reshape(shape)


class _Exact(object):

    def __init__(self, case):
        self.case = case
        self.n, boxsize, boxcenter = _geometry(case)
        to = lambda x: torch.tensor(x, dtype=torch.float64, device='cuda')
        self.box, self.center = to(boxsize), to(boxcenter)
        if case['dtype'] == 'f4': self.box, self.center = self.box.float().double(), self.center.float().double()
        self.low = self.center - self.box / 2.
        self.cell = self.box / to([float(n) for n in self.n])
        self.wrap = case['geometry'] == 'box'
        self.los = to([0., 0., 1.]) if self.wrap else None
        self.beta = F / BIAS
        self.k = [2. * math.pi * torch.fft.fftfreq(n, d=float(c), dtype=torch.float64, device='cuda')
                  for n, c in zip(self.n, self.cell)]
        k2 = sum(_axis(k**2, i) for i, k in enumerate(self.k))
        k2[0, 0, 0] = 1.
        self.k2 = k2
        self.x = [o + c * torch.arange(n, dtype=torch.float64, device='cuda')
                  for n, o, c in zip(self.n, self.low, self.cell)]

    def wrapped(self, x):
        return (x - self.low) % self.box + self.low

    def units(self, x, wrap):
        u = ((self.wrapped(x) if wrap else x) - self.low) / self.cell
        base = u.floor()
        return base.long(), u - base

    def index(self, base, offset):
        i = [(base[:, d] + offset[d]) % self.n[d] for d in range(3)]
        return (i[0] * self.n[1] + i[1]) * self.n[2] + i[2]

    def paint(self, positions, weights, wrap=None):
        mesh = torch.zeros(self.n, dtype=torch.float64, device='cuda')
        for x, w in zip(positions.split(1 << 23), weights.split(1 << 23)):
            base, t = self.units(x.double(), self.wrap if wrap is None else wrap)
            for corner in range(8):
                o = (corner >> 2, corner >> 1 & 1, corner & 1)
                weight = w.double()
                for d in range(3): weight = weight * (t[:, d] if o[d] else 1. - t[:, d])
                mesh.view(-1).scatter_add_(0, self.index(base, o), weight)
        return mesh

    def read(self, mesh, x, wrap):
        """CIC values of ``mesh`` at ``x``; of its central-difference gradient where ``mesh`` is the potential."""
        base, t = self.units(x, wrap)
        flat, gradient = mesh.view(-1), self.case['algorithm'] == 'multigrid'
        out = torch.zeros((len(x), 3) if gradient else len(x), dtype=torch.float64, device='cuda')
        for corner in range(8):
            o = (corner >> 2, corner >> 1 & 1, corner & 1)
            weight = torch.ones(len(x), dtype=torch.float64, device='cuda')
            for d in range(3): weight = weight * (t[:, d] if o[d] else 1. - t[:, d])
            if not gradient:
                out += flat[self.index(base, o)] * weight
                continue
            for d in range(3):
                up, down = ([o[e] + s * (e == d) for e in range(3)] for s in (1, -1))
                out[:, d] += (flat[self.index(base, up)] - flat[self.index(base, down)]) * weight / (2. * self.cell[d])
        return out

    def smooth(self, mesh):
        gain = 1.
        for d in range(3): gain = gain * _axis(torch.exp(-0.5 * (RADIUS * self.k[d])**2), d)
        return torch.fft.ifftn(torch.fft.fftn(mesh) * gain).real

    def contrast(self, data, randoms):
        if randoms is None: return (data / data.mean() - 1.) / BIAS
        alpha = data.sum() / randoms.sum()
        mask = randoms > 0.01 * randoms.sum() / self.case['nrandoms']
        return torch.where(mask, (data - alpha * randoms) / (BIAS * alpha * randoms), torch.zeros_like(data))

    # the multigrid of the redshift-space operator
    def level(self, shape):
        h = [float(b) / n for b, n in zip(self.box, shape)]
        if self.los is None:
            p = [_axis((float(self.low[d]) / h[d]) + torch.arange(shape[d], dtype=torch.float64, device='cuda'), d)
                 for d in range(3)]
        else:
            p = [torch.full((1, 1, 1), float(self.los[d]) / h[d], dtype=torch.float64, device='cuda') for d in range(3)]
        g = self.beta / sum(h[d]**2 * p[d]**2 for d in range(3))
        return p, g, [1. / h[d]**2 + g * p[d]**2 for d in range(3)]

    def off_diagonal(self, v, coefficients):
        p, g, c = coefficients
        edges = torch.zeros_like(v)
        total = torch.zeros_like(v)
        shifted = [(torch.roll(v, -1, d), torch.roll(v, 1, d)) for d in range(3)]
        for d in range(3):
            up, down = shifted[d]
            total += c[d] * (up + down)
            if self.los is None: total += g * p[d] * (up - down)
        for a in range(3):
            for b in range(a + 1, 3):
                up, down = shifted[a]
                edges += p[a] * p[b] * ((torch.roll(up, -1, b) - torch.roll(up, 1, b))
                                        - (torch.roll(down, -1, b) - torch.roll(down, 1, b)))
        return total.add_(g / 2. * edges)

    def sweep(self, v, f, coefficients, count):
        diagonal = 2. * sum(coefficients[2])
        for _ in range(count):
            v = 0.6 * v + 0.4 * (f + self.off_diagonal(v, coefficients)) / diagonal
        return v

    def coarser(self, fine):
        for d in range(3):
            fine = 0.5 * fine + 0.25 * (torch.roll(fine, 1, d) + torch.roll(fine, -1, d))
            fine = fine[tuple(slice(None, None, 2 if e == d else None) for e in range(3))]
        return fine.contiguous()

    def finer(self, coarse):
        for d in range(3):
            coarse = torch.stack([coarse, 0.5 * (coarse + torch.roll(coarse, -1, d))], dim=d + 1)
            coarse = coarse.flatten(d, d + 1)
        return coarse

    def vcycle(self, v, f):
        coefficients = self.level(v.shape)
        v = self.sweep(v, f, coefficients, 5)
        if all(n > 4 and n % 2 == 0 for n in v.shape):
            residual = f - 2. * sum(coefficients[2]) * v + self.off_diagonal(v, coefficients)
            coarse = self.coarser(residual)
            v = v + self.finer(self.vcycle(torch.zeros_like(coarse), coarse))
        return self.sweep(v, f, coefficients, 5)

    def full_multigrid(self, f):
        v = torch.zeros_like(f)
        if all(n > 4 and n % 2 == 0 for n in f.shape): v = self.finer(self.full_multigrid(self.coarser(f)))
        for _ in range(6): v = self.vcycle(v, f)
        return v

    # the reconstructions in Fourier space
    def real(self, spectrum):
        return torch.fft.ifftn(spectrum).real

    def over_k2(self, delta):
        spectrum = torch.fft.fftn(delta) / self.k2
        spectrum[0, 0, 0] = 0.
        return spectrum

    def k_los(self):
        return sum(_axis(self.k[d] * self.los[d], d) for d in range(3))

    def iterated(self, delta):
        current = delta
        for iteration in range(3):
            spectrum = self.over_k2(current)
            factor = self.beta / (1. + self.beta) if iteration == 0 else self.beta
            if self.los is not None:
                current = delta - factor * self.real(self.k_los()**2 * spectrum)
                continue
            x = [_axis(self.x[d], d) for d in range(3)]
            x2 = sum(xx**2 for xx in x)
            current = delta.clone()
            for a in range(3):
                for b in range(a, 3):
                    term = self.real(_axis(self.k[a], a) * _axis(self.k[b], b) * spectrum)
                    current -= (1 + (a != b)) * factor * x[a] * x[b] * term / x2
        return current

    def displacements(self, delta):
        spectrum = self.over_k2(delta)
        if self.case['algorithm'] == 'plane_parallel':
            spectrum = spectrum / (1. + self.beta * self.k_los()**2 / self.k2)
        return [self.real(1j * _axis(self.k[d], d) * spectrum) for d in range(3)]

    def direction(self, x):
        return self.los if self.los is not None else x / _length(x)[:, None]

    def along(self, shifts, los):
        return F * (shifts * los).sum(dim=1, keepdim=True) * los

    def displacement(self, x, wrap):
        if self.case['algorithm'] == 'multigrid': return self.read(self.field, x, wrap)
        return torch.stack([self.read(psi, x, wrap) for psi in self.field], dim=1)

    def shifted(self, positions, field):
        out = torch.empty(positions.shape, dtype=torch.float64, device='cuda')
        for x, y in zip(positions.split(1 << 22), out.split(1 << 22)):
            x = x.double()
            inside = self.wrapped(x) if self.wrap and self.case['algorithm'] != 'multigrid' else x
            shifts = self.displacement(inside, self.wrap)
            if field == 'disp+rsd':
                rsd = self.along(shifts, self.direction(inside))
                if self.case['algorithm'] == 'particle': shifts = self.displacement(inside - rsd, True)
                shifts = shifts + rsd
            y[:] = self.wrapped(x - shifts) if self.wrap else x - shifts
        return out

    def particles(self, data, weights, randoms):
        """Data positions without their redshift-space part; leaves the last displacement meshes."""
        current = data = data.double()
        los = self.direction(data)
        for iteration in range(3):
            mesh = self.smooth(self.paint(current, weights, wrap=iteration > 0 or self.wrap))
            self.field = self.displacements(self.contrast(mesh, randoms))
            shifts = self.displacement(current, True)
            if iteration == 0:
                shifts = shifts - self.beta / (1. + self.beta) * (shifts * los).sum(dim=1, keepdim=True) * los
            current = data - self.along(shifts, los)
        return current


def exact(case, seed):
    state = _inputs(case, seed)
    solver = _Exact(case)
    randoms = solver.smooth(solver.paint(state['randoms'], state['randoms_weights'])) if case['nrandoms'] else None
    if case['algorithm'] == 'particle':
        moved = solver.particles(state['data'], state['data_weights'], randoms)
        out = {'data': moved - solver.displacement(moved, True)}
    else:
        delta = solver.contrast(solver.smooth(solver.paint(state['data'], state['data_weights'])), randoms)
        del randoms
        if case['algorithm'] == 'multigrid':
            solver.field = solver.full_multigrid(delta)
        else:
            if case['algorithm'] == 'iterative_fft': delta = solver.iterated(delta)
            solver.field = solver.displacements(delta)
        out = {'data': solver.shifted(state['data'], 'disp+rsd')}
    if case['nrandoms']: out['randoms'] = solver.shifted(state['randoms'], case['randoms_field'])
    return {name: value.cpu().numpy() for name, value in out.items()} if case['host'] else out
