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
