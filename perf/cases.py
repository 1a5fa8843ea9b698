"""Cases that time the framework's main path through its public entry points.

What a user of the backend has it do: evaluate F and its Jacobian, solve the
Newton-corrector systems of one Jacobian (exact FP64 line factor), run Newton
with a factor kept from an earlier Jacobian (mixed precision), run whole
continuations, solve on 3D grids with the two-grid preconditioner, and train
and apply the convolutional correction network.  ``listed`` holds one or more
sizes of each, ``draw`` gives others of the same ranges.

``exact`` restates the discretisation (staggered finite volumes on a uniform
grid), the gauged Newton systems (block elimination over grid lines) and the
network in 64-bit numpy and torch.
"""
import math

import numpy
import torch

import transiflow_amd as tf
from transiflow_amd.learned import ConvNet

LDC, RB = 'Lid-driven Cavity', 'Rayleigh-Benard'


def listed():
    return [
        # F and J of the smallest grid of a batch of cavities: launches and host work decide
        {'name': 'assemble_2d_32', 'kind': 'assemble', 'problem': LDC, 'nx': 32, 'ny': 32, 'nz': 1, 'mu': 500.0},
        # F and J of the Rayleigh-Benard configuration (four unknowns a cell, lines along y)
        {'name': 'assemble_rb_512x128', 'kind': 'assemble', 'problem': RB, 'nx': 512, 'ny': 128, 'nz': 1,
         'mu': 3000.0},
        # F and J of the largest 3D cavity: arrays beyond the caches
        {'name': 'assemble_3d_64', 'kind': 'assemble', 'problem': LDC, 'nx': 64, 'ny': 64, 'nz': 64, 'mu': 300.0},
        # one Newton-corrector iteration with an FP64 factor on a small, odd grid
        {'name': 'corrector_2d_45x37', 'kind': 'corrector', 'problem': LDC, 'nx': 45, 'ny': 37, 'nz': 1, 'mu': 400.0},
        # the same at the size of the headline continuation
        {'name': 'corrector_2d_256', 'kind': 'corrector', 'problem': LDC, 'nx': 256, 'ny': 256, 'nz': 1,
         'mu': 1000.0},
        # the same over the planes of a 3D grid (few lines, large blocks)
        {'name': 'corrector_3d_20', 'kind': 'corrector', 'problem': LDC, 'nx': 20, 'ny': 20, 'nz': 20, 'mu': 200.0},
        # Newton from a nearby state in mixed precision, with the factor of an earlier
        # Jacobian: what most corrector iterations of a continuation are
        {'name': 'newton_2d_256', 'kind': 'newton', 'nx': 256, 'ny': 256, 'nz': 1, 'mu': 800.0},
        # a whole short continuation in mixed precision, small and in 3D
        {'name': 'continuation_2d_64', 'kind': 'continuation', 'nx': 64, 'ny': 64, 'nz': 1, 'mu': 400.0},
        {'name': 'continuation_3d_32', 'kind': 'continuation', 'nx': 32, 'ny': 32, 'nz': 32, 'mu': 100.0},
        # a solve on a 3D grid whose own planes are too large to factor
        {'name': 'twogrid_3d_64', 'kind': 'twogrid', 'nx': 64, 'ny': 64, 'nz': 64, 'mu': 300.0},
        # one training step of the correction network on the grid that it is trained on in 3D
        {'name': 'train_3d_32', 'kind': 'train', 'nx': 32, 'ny': 32, 'nz': 32},
        # one application of the network on the headline grid
        {'name': 'apply_2d_256', 'kind': 'apply', 'nx': 256, 'ny': 256, 'nz': 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['assemble', 'assemble', 'corrector', 'corrector', 'newton', 'continuation', 'twogrid', 'train',
                       'apply'])
    three = rng.random() < (1.0 if kind == 'twogrid' else 0.35)
    if three:
        hi = {'assemble': 60, 'corrector': 19, 'newton': 20, 'continuation': 16, 'twogrid': 24, 'train': 30,
              'apply': 48}[kind]
        nx = _log(rng, 8, hi)
        ny, nz = (max(6, min(hi, int(nx * rng.uniform(0.7, 1.4)))) for _ in range(2))
        if kind == 'twogrid':
            nx, ny, nz = (2 * max(6, v) for v in (nx, ny, nz))
    else:
        hi = {'assemble': 720, 'corrector': 240, 'newton': 240, 'continuation': 72, 'train': 200, 'apply': 400}[kind]
        nx = _log(rng, 24, hi)
        ny, nz = max(16, min(hi, int(nx * rng.uniform(0.4, 1.2)))), 1
    c = {'kind': kind, 'nx': nx, 'ny': ny, 'nz': nz}
    if kind in ('assemble', 'corrector'):
        c['problem'] = RB if not three and rng.random() < 0.4 else LDC
    if kind not in ('train', 'apply'):
        top = {'assemble': 2000, 'corrector': 1000, 'newton': 400, 'continuation': 300, 'twogrid': 300}[kind]
        c['mu'] = round(rng.uniform(50, top / 2 if three else top), 1)
    return c


# ---- shapes and inputs -------------------------------------------------------------------

def _dim(c):
    return 3 if c['nz'] > 1 else 2


def _dof(c):
    return _dim(c) + (2 if c.get('problem', LDC) == RB else 1)


def _parameter(c):
    return 'Rayleigh Number' if c.get('problem', LDC) == RB else 'Reynolds Number'


def _parameters(c, seed):
    """The problem's parameters; the lid speed differs from seed to seed."""
    if c.get('problem', LDC) == RB:
        return {'Problem Type': RB, 'Prandtl Number': 1.0, 'Biot Number': 1.0, 'X-max': 4.0,
                'Rayleigh Number': c['mu']}
    return {'Reynolds Number': c['mu'], 'Lid Velocity': 1.0 + 0.1 * numpy.random.default_rng(seed).random()}


def _smooth(rng, shape, decay):
    """A field on the unit cube of a few random cosine modes, largest value about one."""
    out = 0.0
    axes = [(numpy.arange(n) + 0.5) / n for n in shape]
    for _ in range(4):
        term = rng.standard_normal()
        for a, p in enumerate(axes):
            wave = numpy.cos(math.pi * rng.integers(0, 4) * p) * (numpy.sin(math.pi * p) if decay else 1.0)
            term = term * wave.reshape([-1 if b == a else 1 for b in range(3)])
        out = out + term
    return out / max(1e-300, numpy.abs(out).max())


def _state(c, seed):
    """A flow-like state [nx, ny, nz, dof]: smooth velocities that vanish at the walls,
    smooth pressure and temperature, and noise a thousandth as large."""
    rng = numpy.random.default_rng(seed + 77)
    shape, dim, dof = (c['nx'], c['ny'], c['nz']), _dim(c), _dof(c)
    x = numpy.zeros(shape + (dof,))
    for d in range(dof):
        x[..., d] = _smooth(rng, shape, d < dim) * (0.4 if d < dim else 0.2) + 1e-3 * rng.standard_normal(shape)
    if dof > dim + 1:   # temperature: the conduction profile, hot below
        x[..., dim + 1] += 1.0 - 0.5 * ((numpy.arange(shape[1]) + 0.5) / shape[1])[None, :, None]
    for a in range(dim):   # the last face along an axis is the wall
        x[tuple(-1 if b == a else slice(None) for b in range(3)) + (a,)] = 0.0
    return x


def _vec(x):
    """[nx, ny, nz, dof] -> state vector (cell i + nx (j + ny k), unknowns fastest)."""
    return numpy.ascontiguousarray(x.transpose(2, 1, 0, 3)).reshape(-1)


def _field(v, c):
    return v.reshape(c['nz'], c['ny'], c['nx'], _dof(c)).transpose(2, 1, 0, 3)


def _near(c, seed):
    """The offset of a Newton start from its solution."""
    d = 1e-2 * _state(c, seed + 5)
    d[0, 0, 0, _dim(c)] = 0.0   # the gauged pressure entry keeps the solution's value
    return d


def _ladder(mu):
    """Parameters on the way from the linear problem to mu."""
    return [0.0] + [mu * (k + 1) / 4 for k in range(4)]


def _net_inputs(c, seed):
    """(input, target, weights and biases of the three layers), FP32."""
    dim = _dim(c)
    n, ch = c['nx'] * c['ny'] * c['nz'] * (dim + 1), [dim + 1, 32, 32, dim + 1]
    rng = numpy.random.default_rng(seed + 3)
    x, t = (rng.standard_normal(n).astype(numpy.float32) for _ in range(2))
    layers = []
    for cin, cout in zip(ch, ch[1:]):
        W = rng.standard_normal((3 ** dim * cin, cout)) * math.sqrt(2.0 / (3 ** dim * cin))
        layers.append((W.astype(numpy.float32), (0.1 * rng.standard_normal(cout)).astype(numpy.float32)))
    return x, t, layers


def prepare(case, seed):
    c = case
    if c['kind'] in ('train', 'apply'):
        net = ConvNet(_dim(c), _dim(c) + 1)
        x, t, layers = _net_inputs(c, seed)
        for i, (W, b) in enumerate(layers):
            net.set_layer(i, W, b)
        x, t = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        return {'case': c, 'net': net, 'x': x, 't': t, 'out': torch.empty_like(x), 'shape': (c['nx'], c['ny'], c['nz'])}
    p = _parameters(c, seed)
    if c['kind'] in ('newton', 'continuation'):
        p['HIP Solver'] = {'Precision': 'mixed'}
    if c['kind'] == 'twogrid':
        p['HIP Solver'] = {'Preconditioner': 'multigrid', 'Restart': 100, 'Maximum Iterations': 600}
    itf = tf.Interface(p, c['nx'], c['ny'], c['nz'])
    s = {'case': c, 'itf': itf}
    if c['kind'] == 'newton':
        s['cont'] = tf.Continuation(itf, newton_tolerance=1e-8, printer=None)
        x = itf.vector()
        for mu in _ladder(c['mu']):
            itf.set_parameter('Reynolds Number', mu)
            x = s['cont'].newton(x, tol=1e-8)
        s['x'] = x + itf.vector_from_array(_vec(_near(c, seed)))
    elif c['kind'] == 'continuation':
        s['x'] = itf.vector_from_array(_vec(1e-3 * _state(c, seed)))
    else:
        s['x'] = itf.vector_from_array(_vec(_state(c, seed)))
    if c['kind'] == 'twogrid':
        s['b'] = itf.vector_from_array(_vec(_state(c, seed + 1)))
    return s


def run(state):
    s = state
    c, kind = s['case'], s['case']['kind']
    if kind == 'apply':
        return s['net'].forward(s['x'], s['shape'], out=s['out'])
    if kind == 'train':
        net = s['net']
        loss = net.mse(net.forward(s['x'], s['shape']), s['t'])
        net.backward(net.g_loss, s['shape'])
        net.adam_step(1e-3)
        return {'loss': loss, 'dW': [L.dW[:L.taps * L.cin, :L.cout] for L in net.layers],
                'db': [L.db for L in net.layers], 'W': [L.W[:L.taps * L.cin, :L.cout] for L in net.layers],
                'b': [L.b for L in net.layers]}
    itf = s['itf']
    if kind == 'assemble':
        F = itf.rhs(s['x'])
        J = itf.jacobian(s['x'])
        return {'F': F.data, 'val': J.val, 'col': J.col, 'row_ptr': J.row_ptr}
    if kind == 'corrector':
        # Continuation's corrector iteration: F, its parameter derivative, J, both solves
        name, mu = _parameter(c), c['mu']
        F = itf.rhs(s['x'])
        itf.set_parameter(name, mu + 1.0)
        dF = itf.rhs(s['x']) - F
        itf.set_parameter(name, mu)
        z1, z2 = itf.solve_pair(itf.jacobian(s['x']), -F, dF)
        return [z1.data, z2.data]
    if kind == 'newton':
        return s['cont'].newton(s['x'], tol=1e-8).data
    if kind == 'twogrid':
        return itf.solve(itf.jacobian(s['x']), s['b']).data
    cont = tf.Continuation(itf, newton_tolerance=1e-8, printer=None)
    itf.set_parameter('Reynolds Number', 0.0)
    x0 = cont.newton(s['x'], tol=1e-8)
    x, mu = cont.continuation(x0, 'Reynolds Number', 0.0, c['mu'], min(100.0, c['mu'] / 2))
    return {'x': x.data, 'mu': float(mu)}


# ---- what a pass cannot do without ---------------------------------------------------------

def _lines(c):
    """(lines, unknowns a line) of the block tridiagonal order along the longest axis."""
    n = (c['nx'], c['ny'], c['nz'])
    N = n[2] if c['nz'] > 1 else max(n)
    return N, n[0] * n[1] * n[2] // N * _dof(c)


def work(case):
    c = case
    cells, dim = c['nx'] * c['ny'] * c['nz'], _dim(c)
    if c['kind'] in ('train', 'apply'):
        taps, ch = 3 ** dim, [dim + 1, 32, 32, dim + 1]
        macs = taps * sum(a * b for a, b in zip(ch, ch[1:]))
        fwd, w = 2.0 * cells * macs, 4.0 * (macs + sum(ch[1:]))
        if c['kind'] == 'apply':
            return {'bytes': 4.0 * cells * 2 * ch[0] + w, 'flops': fwd}
        # the weight gradients, and the data gradients of the second and third layer
        return {'bytes': 4.0 * cells * 2 * ch[0] + 7 * w, 'flops': 2 * fwd + 2.0 * cells * taps * sum(
            a * b for a, b in zip(ch[1:], ch[2:]))}
    n = cells * _dof(c)
    nnz = n * (14 if dim == 3 else 8.6)
    matrix = 12.0 * nnz + 4.0 * (n + 1)
    N, m = _lines(c)
    factor = N * 14 / 3.0 * m ** 3   # block elimination over the lines, two thirds + two + two
    if c['kind'] == 'assemble':
        return {'bytes': matrix + 16.0 * n, 'flops': nnz * 20.0}
    if c['kind'] == 'corrector':
        return {'bytes': 2 * matrix + 32.0 * n, 'flops': factor + 8.0 * N * m * m}
    if c['kind'] == 'newton':      # about three corrections, each at least one pass over a half-size factor
        return {'bytes': 3 * (2 * matrix + 16.0 * n + 4.0 * N * m * m), 'flops': 3 * 4.0 * N * m * m}
    if c['kind'] == 'continuation':   # at least one factorisation
        return {'bytes': 6 * (2 * matrix + 16.0 * n), 'flops': factor}
    Nc, mc = N // 2, m // 4
    return {'bytes': 20 * 2 * matrix, 'flops': Nc * 14 / 3.0 * mc ** 3 + cells / c['nx'] * 2.0 * (c['nx'] * 4) ** 3}


# ---- the same in 64 bits ---------------------------------------------------------------------

class _Model:
    """F on a uniform grid, and its Jacobian by probing (F is quadratic in the state, so
    central differences of unit size are exact)."""

    def __init__(self, c, p, mu=None):
        self.c, self.dim, self.dof = c, _dim(c), _dof(c)
        self.shape = (c['nx'], c['ny'], c['nz'])
        size = (p.get('X-max', 1.0), 1.0, 1.0)
        self.h = [size[a] / self.shape[a] if a < self.dim else 1.0 for a in range(3)]
        self.vol = self.h[0] * self.h[1] * self.h[2]
        mu = c['mu'] if mu is None else mu
        self.rb = self.dof > self.dim + 1
        if self.rb:
            gr = mu / p['Prandtl Number'] if mu else 1.0 / p['Prandtl Number']
            self.nu, self.kappa = 1.0 / math.sqrt(gr), 1.0 / (p['Prandtl Number'] * math.sqrt(gr))
            b = self.h[1] * p['Biot Number'] / 2
            self.top = (1 - b) / (1 + b)
            self.lid = 0.0
        else:
            self.nu, self.lid = 1.0 / (mu or 1.0), p['Lid Velocity']
        self.convect = self.rb or mu != 0

    def _at(self, a, i):
        return tuple(i if b == a else slice(None) for b in range(3))

    def _ghosts(self, u, d, a):
        """(value before the first, value after the last) of unknown d along axis a."""
        lo, hi = u[self._at(a, slice(0, 1))], u[self._at(a, slice(-1, None))]
        if d < self.dim:
            if d == a:
                return 0 * lo, 0 * hi
            if self.rb and a == 1:
                return -lo, hi
            lid = 2 * self.lid if (a == self.dim - 1 and d == 0) else 0.0
            return -lo, lid - hi
        if a == 1:
            return 2.0 - lo, self.top * hi
        return lo, hi

    def _pad(self, u, d, a):
        lo, hi = self._ghosts(u, d, a)
        return numpy.concatenate([lo, u, hi], axis=a)

    def _next(self, u, a):
        """u of the next cell along a (zero past the last: those rows are the walls')."""
        return numpy.concatenate([u[self._at(a, slice(1, None))], 0 * u[self._at(a, slice(0, 1))]], axis=a)

    def F(self, x):
        dim, h = self.dim, self.h
        x = x.copy()
        walls = []
        for a in range(dim):
            walls.append(x[self._at(a, -1) + (a,)].copy())
            x[self._at(a, -1) + (a,)] = 0.0
        out = numpy.zeros_like(x)
        n = self.shape
        for d in list(range(dim)) + ([dim + 1] if self.rb else []):
            u = x[..., d]
            f = out[..., d]
            for a in range(dim):
                q = self._pad(u, d, a)
                lo, mid, hi = (q[self._at(a, slice(s, s + n[a]))] for s in range(3))
                f += (self.kappa if d > dim else self.nu) * (lo - 2 * mid + hi) * self.vol / h[a] ** 2
                if not self.convect:
                    continue
                if d == a:       # its own direction: faces at cell centres
                    fl, fr = ((lo + mid) / 2) ** 2, ((mid + hi) / 2) ** 2
                else:            # carried by x[..., a], averaged to this unknown's faces
                    v = x[..., a]
                    v = (v + self._next(v, d)) / 2 if d < dim else v
                    before = numpy.concatenate([0 * v[self._at(a, slice(0, 1))], v[self._at(a, slice(0, -1))]], axis=a)
                    fl, fr = before * (lo + mid) / 2, v * (mid + hi) / 2
                f -= (fr - fl) * self.vol / h[a]
            if d < dim:
                f -= (self._next(x[..., dim], d) - x[..., dim]) * self.vol / h[d]
                if self.rb and d == 1:
                    T = x[..., dim + 1]
                    f += (T + self._next(T, 1)) / 2 * self.vol
        for a in range(dim):
            u = x[..., a]
            before = numpy.concatenate([0 * u[self._at(a, slice(0, 1))], u[self._at(a, slice(0, -1))]], axis=a)
            out[..., dim] += (u - before) * self.vol / h[a]
            out[self._at(a, -1) + (a,)] = -walls[a]
        return out

    def jacobian(self, x):
        """(rows, columns, values) of dF/dx, entries that vanish left out, sorted."""
        dof, n = self.dof, self.shape
        step = [3 if a < self.dim else 1 for a in range(3)]
        number = _vec_index(n, dof)
        idx = numpy.meshgrid(*[numpy.arange(m) for m in n], indexing='ij')
        R, C, V = [], [], []
        for color in numpy.ndindex(*step):
            # the cell of this colour within reach of each cell
            near, ok = [], numpy.ones(n, dtype=bool)
            for a in range(3):
                off = (color[a] - idx[a] + 1) % 3 - 1 if step[a] == 3 else 0 * idx[a]
                near.append(idx[a] + off)
                ok &= (near[a] >= 0) & (near[a] < n[a])
            here = tuple(slice(color[a], None, step[a]) for a in range(3))
            for d in range(dof):
                e = numpy.zeros_like(x)
                e[here + (d,)] = 1.0
                j = (self.F(x + e) - self.F(x - e)) / 2
                for d1 in range(dof):
                    v = j[..., d1]
                    keep = ok & (numpy.abs(v) > 1e-13 * max(1.0, self.nu) * self.vol ** (1.0 / 3))
                    R.append(number[..., d1][keep])
                    C.append(number[..., d][tuple(q[keep] for q in near)])
                    V.append(v[keep])
        R, C, V = (numpy.concatenate(q) for q in (R, C, V))
        order = numpy.lexsort((C, R))
        return R[order], C[order], V[order]


def _vec_index(n, dof):
    i, j, k = numpy.meshgrid(*[numpy.arange(m) for m in n], indexing='ij')
    return (i + n[0] * (j + n[1] * k))[..., None] * dof + numpy.arange(dof)


def _solve(c, J, rhs):
    """The gauged systems J y = rhs (columns) by block elimination over the lines."""
    dim, dof = _dim(c), _dof(c)
    N, m = _lines(c)
    n = (c['nx'], c['ny'], c['nz'])
    axis = 2 if c['nz'] > 1 else (0 if n[0] >= n[1] else 1)
    number = _vec_index(n, dof)
    order = numpy.moveaxis(number, axis, 0).reshape(N, m)      # unknowns of each line
    line, place = (numpy.empty(N * m, dtype=numpy.int64) for _ in range(2))
    line[order.reshape(-1)] = numpy.repeat(numpy.arange(N), m)
    place[order.reshape(-1)] = numpy.tile(numpy.arange(m), N)
    R, C, V = J
    keep = (R != dim) & (C != dim)
    R, C, V = (numpy.append(q[keep], w) for q, w in ((R, dim), (C, dim), (V, -1.0)))
    b = rhs.copy()
    b[dim] = 0.0
    b = b[order]                                                  # [N, m, columns]
    by = numpy.argsort(line[R], kind='stable')
    R, C, V = R[by], C[by], V[by]
    first = numpy.searchsorted(line[R], numpy.arange(N + 1))
    X, y = [], []
    for j in range(N):
        r, q, v = (w[first[j]:first[j + 1]] for w in (R, C, V))
        A = numpy.zeros((3, m, m))
        numpy.add.at(A, (line[q] - j + 1, place[r], place[q]), v)
        D, g = A[1], b[j]
        if j:
            D = D - A[0] @ X[-1]
            g = g - A[0] @ y[-1]
        s = numpy.linalg.solve(D, numpy.concatenate([A[2], g], axis=1) if j + 1 < N else g)
        X.append(s[:, :m])
        y.append(s[:, m:] if j + 1 < N else s)
    for j in range(N - 2, -1, -1):
        y[j] = y[j] - X[j] @ y[j + 1]
    out = numpy.empty_like(rhs)
    out[order.reshape(-1)] = numpy.concatenate(y)
    return out


def _newton(c, p, mu, x, most=10):
    model = _Model(c, p, mu)
    for _ in range(most):
        f = model.F(x)
        dx = _solve(c, model.jacobian(x), -_vec(f)[:, None])[:, 0]
        x = x + _field(dx, c)
        if numpy.linalg.norm(dx) < 1e-10 * numpy.linalg.norm(x):
            break
    return x


def _net_exact(c, seed):
    dim = _dim(c)
    par = []
    x, t, layers = _net_inputs(c, seed)
    for W, b in layers:
        par += [torch.from_numpy(W).double().requires_grad_(), torch.from_numpy(b).double().requires_grad_()]
    x, t = torch.from_numpy(x).double(), torch.from_numpy(t).double()
    shape = (c['nz'], c['ny'], c['nx'])
    y = x.reshape(shape + (-1,))
    for k in range(3):
        W, b = par[2 * k], par[2 * k + 1]
        q = torch.nn.functional.pad(y, (0, 0, 1, 1, 1, 1, 1, 1) if dim == 3 else (0, 0, 1, 1, 1, 1, 0, 0))
        cin, z = y.shape[-1], b
        for tap in range(3 ** dim):
            dx, dy, dz = tap % 3, tap // 3 % 3, tap // 9
            z = z + q[dz:dz + shape[0], dy:dy + shape[1], dx:dx + shape[2]] @ W[tap * cin:(tap + 1) * cin]
        y = torch.relu(z) if k < 2 else z
    y = y.reshape(-1)
    if c['kind'] == 'apply':
        return y.detach()
    loss = ((y - t) ** 2).mean()
    loss.backward()
    dW, db, W, b = [], [], [], []
    for k, q in enumerate(par):
        g = q.grad.detach()
        (db if k % 2 else dW).append(g)
        (b if k % 2 else W).append(q.detach() - 1e-3 * g / (g.abs() + 1e-8))   # Adam's first step
    return {'loss': float(loss), 'dW': dW, 'db': db, 'W': W, 'b': b}


def exact(case, seed):
    c = case
    if c['kind'] in ('train', 'apply'):
        return _net_exact(c, seed)
    p = _parameters(c, seed)
    if c['kind'] == 'assemble':
        model, x = _Model(c, p), _state(c, seed)
        return {'F': _vec(model.F(x)), 'val': model.jacobian(x)[2], 'col': None, 'row_ptr': None}
    N, m = _lines(c)
    solves = {'corrector': 1, 'twogrid': 1, 'newton': 4, 'continuation': 16}[c['kind']]
    if solves * N * 14 / 3.0 * m ** 3 > 2.5e12:
        return None
    if c['kind'] == 'corrector':
        model, x = _Model(c, p), _state(c, seed)
        F = model.F(x)
        dF = _Model(c, p, c['mu'] + 1.0).F(x) - F
        z = _solve(c, model.jacobian(x), numpy.stack([-_vec(F), _vec(dF)], axis=1))
        return [z[:, 0].copy(), z[:, 1].copy()]
    if c['kind'] == 'twogrid':
        return _solve(c, _Model(c, p).jacobian(_state(c, seed)), _vec(_state(c, seed + 1))[:, None])[:, 0].copy()
    if c['kind'] == 'newton':
        x = numpy.zeros((c['nx'], c['ny'], c['nz'], _dof(c)))
        for mu in _ladder(c['mu']):
            x = _newton(c, p, mu, x, 10 if mu == c['mu'] else 2)
        return _vec(x)
    x = 1e-3 * _state(c, seed)
    for mu in _ladder(c['mu']):
        x = _newton(c, p, mu, x)
    return {'x': _vec(x), 'mu': c['mu']}
