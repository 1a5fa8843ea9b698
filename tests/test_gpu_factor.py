"""One application of the line factor against scipy's sparse LU, over the block sizes
at which the blocked inversion and the products change their ways: below, at and above
one and two Gauss-Jordan panel halves (64) and panels (128), whole and ragged last
panels, rows that are and are not whole 16-byte units.

Tolerance: the application is a direct solve, so its relative error is bounded by a
modest multiple of (rows per block) x (condition number) x (unit roundoff); the
condition number is estimated from the sparse LU.
"""
import numpy
import pytest
from scipy.sparse.linalg import LinearOperator, onenormest, splu

from tests.helpers import seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('single', [False, True])
@pytest.mark.parametrize('problem,nx', [('ldc', 1), ('ldc', 5), ('ldc', 21), ('rb', 16), ('ldc', 22), ('rb', 32),
                                        ('ldc', 43), ('ldc', 64), ('ldc', 86)])
def test_line_factor_applies_the_inverse(hip, problem, nx, single):
    from oracle.interface import Interface as OracleInterface
    from transiflow_amd.solver import LineFactor
    T = hip.vector.torch()
    params = {'Reynolds Number': 100} if problem == 'ldc' else {
        'Problem Type': 'Rayleigh-Benard', 'Prandtl Number': 1.0, 'Rayleigh Number': 500.0, 'Biot Number': 1.0}
    shape = (nx, max(nx + 2, 4))    # x-lines: nx dof rows per block
    itf, ref = hip.Interface(dict(params), *shape), OracleInterface(dict(params), *shape)
    state = 0.1 * seeded_state(itf.n, nx)
    J = itf.jacobian(state)
    A = ref.compute_bordered_matrix(ref.jacobian(state), fix_pressure_row=True).tocsc()
    lu = splu(A)
    inverse = LinearOperator(A.shape, matvec=lu.solve, rmatvec=lambda v: lu.solve(v, 'T'),
                             matmat=lu.solve, rmatmat=lambda v: lu.solve(v, 'T'))
    cond = onenormest(inverse) * onenormest(A)
    b = seeded_state(itf.n, nx + 1)
    r = T.from_numpy(b).cuda()
    factor = LineFactor(itf, J, itf.solver.gauge(), single=single)
    assert factor.m == nx * itf.dof and factor.perturbed == 0
    if single:
        z = factor.apply32(r.float(), T.empty_like(r, dtype=T.float32)).double().cpu().numpy()
    else:
        z = factor.apply(r, T.empty_like(r)).cpu().numpy()
    x = lu.solve(b)
    err = numpy.linalg.norm(z - x) / numpy.linalg.norm(x)
    tol = factor.m * cond * numpy.finfo(numpy.float32 if single else numpy.float64).eps
    print('%s m %d single %s: cond %.1e, error %.1e, bound %.1e' % (problem, factor.m, single, cond, err, tol), flush=True)
    assert err <= min(tol, 0.1)


@pytest.mark.parametrize('shape', [(32, 24, 5), (64, 12, 3), (28, 28, 2), (56, 14, 4)])
def test_chain_matches_reduction(hip, shape):
    """Planes of 3072 rows and more, eliminated one after the other when the factor does
    not keep Y L and Y U, against the reduction that does: the same inverse to rounding
    (1e-10, as for the two forms of the reduction), the same bits for one column and two,
    replayed and eager; a handle that is set back and forth before it is factored ends up
    with the order of its last setting."""
    import torch
    from transiflow_amd.solver import LineFactor
    itf = hip.Interface({'Reynolds Number': 100}, *shape)
    g = itf.solver.gauge()
    rng = numpy.random.default_rng(9)
    J = itf.jacobian(itf.vector_from_array(rng.uniform(-1, 1, itf.n) * 0.1))
    r = [torch.from_numpy(rng.uniform(-1, 1, itf.n)).cuda() for _ in range(2)]
    for v in r:
        v[g] = 0.0
    out = {}
    for order in ((True,), (False,), (True, False), (False, True)):
        f = LineFactor(itf, J, g, single=False, factor=False)
        for fused in order:
            f.set_fused(fused)
        f.refactor(J, g)
        got = []
        for graph in (False, True, True):
            f.set_graph(graph)
            z = [torch.full_like(v, numpy.nan) for v in r]
            p = [torch.full_like(v, numpy.nan) for v in r]
            for a, b in zip(r, z):
                f.apply(a, b)
            f.apply_pair(r[0], r[1], p[0], p[1], single=False)
            torch.cuda.synchronize()
            got.append([v.cpu().numpy() for v in z + p])
        for zs in got:
            for i in range(2):
                assert numpy.isfinite(zs[i]).all()
                assert numpy.array_equal(zs[i], got[0][i]) and numpy.array_equal(zs[2 + i], got[0][i])
        out[order] = got[0][0]
    diff = numpy.linalg.norm(out[(False,)] - out[(True,)]) / numpy.linalg.norm(out[(True,)])
    assert diff <= 1e-10
    assert numpy.array_equal(out[(True, False)], out[(False,)])
    assert numpy.array_equal(out[(False, True)], out[(True,)])


@pytest.mark.parametrize('shape,single', [((32, 24, 5), False), ((56, 14, 4), True), ((40, 20, 9), True),
                                          ((40, 20, 9), False)])
def test_look_ahead_keeps_the_bits(hip, shape, single):
    """Inversions whose next diagonal block is updated and inverted beside the rest of the
    update (3072 and 3136 rows, the last panel half filled; 3200 rows with a batch of up to
    five), against the same launches one after the other, which the kernel profiler asks
    for: the same bits, also from a factor made twice."""
    import torch
    from transiflow_amd import _lib
    from transiflow_amd.solver import LineFactor
    itf = hip.Interface({'Reynolds Number': 100}, *shape)
    g = itf.solver.gauge()
    rng = numpy.random.default_rng(10)
    J = itf.jacobian(itf.vector_from_array(rng.uniform(-1, 1, itf.n) * 0.1))
    r = torch.from_numpy(rng.uniform(-1, 1, itf.n)).cuda()
    r[g] = 0.0
    r = r.float() if single else r
    out = []
    f = LineFactor(itf, J, g, single=single, factor=False)
    f.set_fused(True)
    f.set_graph(False)
    for prof in (1, 0, 0):
        _lib.call('tf_prof_enable', prof)
        try:
            f.refactor(J, g)
        finally:
            _lib.call('tf_prof_enable', 0)
        z = torch.empty_like(r)
        (f.apply32 if single else f.apply)(r, z)
        torch.cuda.synchronize()
        out.append(z.cpu().numpy())
    assert numpy.isfinite(out[0]).all()
    assert numpy.array_equal(out[1], out[0]) and numpy.array_equal(out[2], out[0])


def _flow(itf, seed):
    """A flow-like state: a few smooth modes per unknown, velocities zero at the walls,
    and noise a thousandth as large."""
    rng = numpy.random.default_rng(seed)
    at = [(numpy.arange(n) + 0.5) / n for n in (itf.nx, itf.ny, itf.nz)]
    x = numpy.zeros((itf.nz, itf.ny, itf.nx, itf.dof))
    for d in range(itf.dof):
        field = 0.0
        for _ in range(4):
            term = [numpy.cos(numpy.pi * rng.integers(0, 4) * p) * (numpy.sin(numpy.pi * p) if d < 3 else 1.0)
                    for p in at]
            field = field + rng.standard_normal() * numpy.einsum('i,j,k->kji', *term)
        x[..., d] = field / numpy.abs(field).max() * (0.4 if d < 3 else 0.2)
    x += 1e-3 * rng.standard_normal(x.shape)
    x[:, :, -1, 0] = x[:, -1, :, 1] = x[-1, :, :, 2] = 0.0
    return x.reshape(-1)


@pytest.mark.parametrize('shape,re', [((31, 31, 26), 340.0), ((29, 29, 18), 440.0), ((30, 30, 31), 460.0),
                                      ((31, 30, 32), 480.0)])
def test_direct_factor_of_long_lines_is_as_accurate_without_products(hip, shape, re):
    """Planes of 3072 rows and more at Reynolds numbers where convection dominates: a
    factor without Y L and Y U eliminates the planes in the order of the one with them, so
    the nearly singular pivots that set the residual of an application are the same ones:
    within a factor of 10 of each other."""
    import torch
    from transiflow_amd.solver import LineFactor
    itf = hip.Interface({'Reynolds Number': re}, *shape)
    g = itf.solver.gauge()
    seed = int(re - 340) // 20
    J = itf.jacobian(itf.vector_from_array(_flow(itf, seed)))
    r = torch.from_numpy(seeded_state(itf.n, seed)).cuda()
    r[g] = 0.0
    res = {}
    for fused in (True, False):
        f = LineFactor(itf, J, g, single=False, factor=False)
        f.set_fused(fused)
        f.refactor(J, g)
        z = f.apply(r, torch.empty_like(r))
        res[fused] = float(torch.linalg.norm(r - J.matvec(z, gauge=g)) / torch.linalg.norm(r))
        assert f.perturbed == 0
    print('%s Re %g: residual %.1e with, %.1e without products' % (shape, re, res[True], res[False]), flush=True)
    assert res[False] <= 10 * res[True]


@pytest.mark.parametrize('shape', [(32, 24, 1), (32, 24, 2), (28, 28, 5), (56, 14, 32), (32, 24, 65), (30, 25, 4)])
def test_inner_factor_matches_direct(hip, shape):
    """The factor that a preconditioner may ask for: FP64 planes of 3072 rows and more are
    eliminated one after the other from 2 to 64 planes, the same inverse at Re 100 to
    rounding (1e-10, as for the two forms of the reduction) with the same bits for one
    column and two, replayed and eager; one plane, 65 planes or 3000 rows give the direct
    factor's bits.  In order no products are formed, and asking for them is refused."""
    import torch
    from transiflow_amd._lib import BackendError
    from transiflow_amd.solver import LineFactor
    itf = hip.Interface({'Reynolds Number': 100}, *shape)
    g = itf.solver.gauge()
    J = itf.jacobian(itf.vector_from_array(0.1 * seeded_state(itf.n, 11)))
    r = [torch.from_numpy(seeded_state(itf.n, 12 + i)).cuda() for i in range(2)]
    for v in r:
        v[g] = 0.0
    out = {}
    for inner in (False, True):
        f = LineFactor(itf, J, g, single=False, inner=inner)
        got = []
        for graph in (False, True, True):
            f.set_graph(graph)
            z = [torch.full_like(v, numpy.nan) for v in r]
            p = [torch.full_like(v, numpy.nan) for v in r]
            for a, b in zip(r, z):
                f.apply(a, b)
            f.apply_pair(r[0], r[1], p[0], p[1], single=False)
            torch.cuda.synchronize()
            got.append([v.cpu().numpy() for v in z + p])
        for zs in got:
            for i in range(2):
                assert numpy.isfinite(zs[i]).all()
                assert numpy.array_equal(zs[i], got[0][i]) and numpy.array_equal(zs[2 + i], got[0][i])
        out[inner] = got[0][0]
        del f
    if shape[2] in (1, 65) or shape == (30, 25, 4):
        assert numpy.array_equal(out[True], out[False])
    else:
        assert numpy.linalg.norm(out[True] - out[False]) <= 1e-10 * numpy.linalg.norm(out[False])
        with pytest.raises(BackendError):
            LineFactor(itf, J, g, single=False, factor=False, inner=True).set_fused(True)


@pytest.mark.parametrize('shape,re', [((56, 56, 12), 150.0), ((56, 60, 16), 300.0)])
def test_two_grid_coarse_order_leaves_the_solve_alone(hip, shape, re):
    """The two-grid solve with its coarse planes (3136 and 3360 rows) one after the other,
    and by the reduction ('Fused Apply'): the same number of iterations to the tolerance."""
    import torch
    count = []
    for fused in (None, True):
        itf = hip.Interface({'Reynolds Number': re, 'HIP Solver': {
            'Preconditioner': 'multigrid', 'Restart': 100, 'Maximum Iterations': 600, 'Fused Apply': fused}}, *shape)
        J = itf.jacobian(itf.vector_from_array(_flow(itf, 3)))
        b = itf.vector_from_array(_flow(itf, 4))
        x = itf.solve(J, b)
        r = b.data - J.matvec(x.data)
        r[itf.solver.gauge()] = 0.0
        assert float(torch.linalg.norm(r) / torch.linalg.norm(b.data)) <= 1.1e-10
        count.append(itf.solver.log[-1][0])
    assert count[0] == count[1]


@pytest.mark.parametrize('m', [20, 100, 300])
@pytest.mark.parametrize('single,scale', [(False, 1.0), (False, 2.0 ** 150), (True, 1.0), (True, 2.0 ** 124),
                                          (False, numpy.inf), (True, numpy.inf)])
def test_zero_pivot_at_large_scales(hip, m, single, scale):
    """A line with an empty row and column, its other entries near the end of the exponent
    range: the one zero pivot is found, counted and replaced (by 1e-3 of the largest entry)
    as at scale one, and the rest is inverted.  Rows sum to less than half their diagonal:
    the inverse's error is below 10 m units of rounding.  An infinite entry makes every
    finite pivot of its block a small one, which is counted too."""
    import types

    import torch
    from scipy import sparse
    from transiflow_amd.solver import LineILU
    from transiflow_amd.vector import DeviceCsrMatrix
    rng = numpy.random.default_rng(m)
    A = numpy.diag(numpy.ones(m))
    for off in (1, 2, 3):
        A += 0.07 * numpy.diag(rng.uniform(-1, 1, m - off), off) + 0.07 * numpy.diag(rng.uniform(-1, 1, m - off), -off)
    p = m // 2 + 3
    A[p, :] = A[:, p] = 0.0
    S = sparse.csr_matrix(A)
    if numpy.isinf(scale):
        S.data[3] = numpy.inf
    else:
        S.data *= scale
    t = lambda v, dt: torch.from_numpy(numpy.ascontiguousarray(v)).to(dt).cuda()
    M = DeviceCsrMatrix(t(S.indptr, torch.int32), t(S.indices, torch.int32), t(S.data, torch.float64), m)
    P = LineILU(types.SimpleNamespace(nx=m, ny=1, nz=1, dof=1), single)
    P.refactor(M, -1)
    if numpy.isinf(scale):
        assert P.perturbed > 1
        return
    r = rng.uniform(-1, 1, m)
    dt = torch.float32 if single else torch.float64
    out = torch.empty(m, dtype=dt, device='cuda')
    (P.apply32 if single else P.apply)(t(r * scale, dt), out)
    got, keep = out.double().cpu().numpy(), numpy.arange(m) != p
    ref = numpy.linalg.solve(A[numpy.ix_(keep, keep)], r[keep])
    assert P.perturbed == 1
    assert numpy.max(numpy.abs(got[keep] - ref)) <= 10 * m * numpy.finfo(numpy.float32 if single else float).eps
    assert abs(got[p] / r[p]) >= 500


@pytest.mark.parametrize('single', [False, True])
@pytest.mark.parametrize('shape', [(21, 23), (22, 24), (43, 45), (64, 66), (86, 88), (20, 20, 4), (40, 33, 3), (48, 44, 2)])
def test_line_factor_backward_error(hip, shape, single):
    """The residual of an application against the size of what it is made of,
    |b - A z| / (|A| |z| + |b|) in the maximum norm, which no condition number enters: the
    rounding of sums over a block's rows grows like a random walk, so at most 10 units of
    it times the square root of the rows.  The sizes take every way of forming the
    level-0 products (eight, four or two rows of a block in LDS, or the multipliers in
    memory: 1600, 5280 and 8448 rows, FP64 and FP32), with and without Y L and Y U and,
    FP64, in order."""
    import torch
    from scipy import sparse
    from transiflow_amd.solver import LineFactor
    itf = hip.Interface({'Reynolds Number': 100}, *shape)
    g = itf.solver.gauge()
    J = itf.jacobian(itf.vector_from_array(0.1 * seeded_state(itf.n, 21)))
    A = sparse.csr_matrix(tuple(v.cpu().numpy() for v in (J.val, J.col, J.row_ptr)), shape=(itf.n, itf.n))
    norm = abs(A).sum(axis=1).max()
    r = torch.from_numpy(seeded_state(itf.n, 22)).cuda()
    r[g] = 0.0
    for kind in ('fused', 'plain') + (() if single else ('inner',)):
        f = LineFactor(itf, J, g, single=single, factor=False, inner=kind == 'inner')
        f.set_fused(kind == 'fused')
        f.refactor(J, g)
        if single:
            z = f.apply32(r.float(), torch.empty_like(r, dtype=torch.float32)).double()
            b = r.float().double()
        else:
            z, b = f.apply(r, torch.empty_like(r)), r
        res = float((b - J.matvec(z, gauge=g)).abs().max())
        err = res / (norm * float(z.abs().max()) + float(b.abs().max()))
        bound = 10 * numpy.sqrt(f.m) * numpy.finfo(numpy.float32 if single else numpy.float64).eps
        print('%s m %d single %s %s: %.1e, bound %.1e' % (shape, f.m, single, kind, err, bound), flush=True)
        assert f.perturbed == 0 and err <= bound
        del f
