"""The line solver at the edges of its preconditioner's forms: columns that
share a workgroup's LDS 16 at a time, long ones that do so by fewer, columns
too long for the LDS, and launches of more rows than the iteration's scalars
are formed in line for (131072).

Against the oracle's direct solve, or the multigrid solver where the grid is
too large for that: each leaves |b - A x| <= 1e-12 |b| or less, the pressure's
error is that times the condition of the system (below 1e5 with cells as wide
as the water is deep and at most 33 levels), and the velocities take dt/rho of
its gradient: 1e-7 on P and 1e-8 on the rest, relative to each field's largest
value.  The long columns' systems are worse than that; they have to converge,
in no more iterations than the shorter ones' count times the ratio of their
levels, which only the right preconditioner does."""
import numpy as np
import pytest

import oracle as O
from nhwave_amd import capi
from nhwave_amd import scenario as S
from nhwave_amd.model import Model

pytestmark = pytest.mark.gpu
FIELDS = ("Eta", "U", "V", "W", "P")


def case(m, n, k, tol=1e-12):
    return S.random_scenario(9, mglob=m, nglob=n, kglob=k, steps=1, dry=False, tol=tol)


def interior(get):
    return {q: (lambda v: v[(slice(2, -2),) * v.ndim])(np.asarray(get(q))) for q in FIELDS}


@pytest.mark.parametrize("m,n,k", [(40, 1, 17), (17, 5, 33), (16, 3, 2), (31, 9, 20), (130, 70, 16)])
def test_line_solver(gpu, m, n, k):
    s = case(m, n, k)
    if m * n * k > 100_000:
        with Model(s) as a:
            a.step(1)
            ref = interior(a.field)
    else:
        o = O.Oracle(s)
        o.step(1)
        ref = interior(o.field)
    with Model(s, solver=capi.NHW_SOLVER_LINE) as a:
        a.step(1)
        assert a.stats().not_converged == 0
        got = interior(a.field)
    for q in FIELDS:
        top = max(float(np.abs(ref[q]).max()), 1e-300)
        assert float(np.abs(got[q] - ref[q]).max()) / top < (1e-7 if q == "P" else 1e-8), q


@pytest.mark.parametrize("k", [128, 129, 600, 2049])
def test_long_columns_converge(gpu, k):
    count = {}
    for levels in (64, k):
        with Model(case(20, 1, levels, 1e-6), solver=capi.NHW_SOLVER_LINE) as a:
            a.step(1)
            st = a.stats()
            assert st.not_converged == 0
            count[levels] = st.total_iters
    assert count[k] <= count[64] * k / 64
