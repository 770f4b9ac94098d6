"""The two-sweep SOR preconditioner with the operator product in one kernel
(a separable operator and pc_maxit 2) at the edges of its regions: 64 x 24
columns of which the outer four hold no tile unless they end the domain, and
chunks of one plane up.  The first iterations follow the oracle's and the
general path's (seven columns, half-sweeps one by one): 1e-11, the solver
tests' bar for iterations in which rounding has not been amplified; 2e-5 in
float, a hundred float roundings.  Every coefficient differs from its
neighbours' and is nonzero on the domain's ends too."""
import numpy as np
import pytest

from falm_amd import _abi as abi
from oracle import pyoracle as O
from tests.helpers import domain, from_dev, interior_mask, rel_err, to_dev

pytestmark = pytest.mark.gpu


def separable(dom, rng):
    nx, ny, nz = dom.shape
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    off = [rng.uniform(0.5, 1.5, n)[q] for n, q in ((nx, i), (nx, i), (ny, j), (ny, j), (nz, k), (nz, k))]
    diag = -sum(off) * rng.uniform(1.0, 1.3, k.shape)
    return np.concatenate([c.reshape(-1) for c in (diag, *off)])


@pytest.mark.parametrize("n", [(64, 24, 1), (65, 25, 2), (120, 40, 9), (121, 41, 5), (7, 81, 31), (180, 3, 64), (127, 4, 64),
                               (600, 470, 1), (130, 70, 3), (66, 100, 4)])
@pytest.mark.parametrize("offset", [(0, 0, 0), (1, 2, 4)])
@pytest.mark.parametrize("precision", [abi.SOLVE_F64, abi.SOLVE_MIXED])
def test_two_sweeps_at_edges(gpu, n, offset, precision):
    dom = domain(n)
    for m, o in enumerate(offset):
        dom.offset[m] = o
        dom.gshape[m] = dom.shape[m] + o
    rng = np.random.default_rng(sum(n))
    a, m = separable(dom, rng), interior_mask(dom)
    b = rng.standard_normal(dom.ncell) * m
    cfg = abi.solver_config(maxit=3, tol=1e-30, pc_type=abi.LS_SOR, pc_maxit=2, pc_relax=1.3, precision=precision)
    x_ref, r_ref = np.zeros(dom.ncell), np.zeros(dom.ncell)
    info_ref = O.Solver(dom, cfg).solve(a, x_ref, b, r_ref)
    da, db = to_dev(a), to_dev(b)
    bar = 1e-11 if precision == abi.SOLVE_F64 else 2e-5
    for declared in (True, False):
        S = gpu.Solver(dom, cfg)
        if declared:
            S.set_matrix(da)
        dx, dr = to_dev(np.zeros(dom.ncell)), to_dev(np.zeros(dom.ncell))
        info = S.solve(da, dx, db, dr)
        assert info.it == info_ref.it == 3
        assert rel_err(from_dev(dx), x_ref) < bar, declared
        if precision == abi.SOLVE_F64:
            assert rel_err(from_dev(dr), r_ref) < 1e-9


@pytest.mark.parametrize("precision", [abi.SOLVE_F64, abi.SOLVE_MIXED])
def test_two_sweeps_beyond_4096_columns(gpu, precision):
    """41 x 106 = 4346 tiles of whole columns, more than a reduction's usual
    number of partial sums: the oracle's first iterations as above."""
    dom = domain((2300, 1700, 1))
    rng = np.random.default_rng(9)
    a, m = separable(dom, rng), interior_mask(dom)
    b = rng.standard_normal(dom.ncell) * m
    cfg = abi.solver_config(maxit=2, tol=1e-30, pc_type=abi.LS_SOR, pc_maxit=2, pc_relax=1.3, precision=precision)
    x_ref, r_ref = np.zeros(dom.ncell), np.zeros(dom.ncell)
    info_ref = O.Solver(dom, cfg).solve(a, x_ref, b, r_ref)
    S = gpu.Solver(dom, cfg)
    da, db, dx = to_dev(a), to_dev(b), to_dev(np.zeros(dom.ncell))
    S.set_matrix(da)
    info = S.solve(da, dx, db, None)
    assert info.it == info_ref.it == 2
    assert rel_err(from_dev(dx), x_ref) < (1e-11 if precision == abi.SOLVE_F64 else 2e-5)
