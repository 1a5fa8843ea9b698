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
