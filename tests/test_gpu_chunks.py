"""The k-marching kernels' chunk lengths: one plane a chunk on the smallest
domains, a few on middle ones and a shorter last chunk, in the step driver
(every stencil, the one- and the two-sweep preconditioner) against the
oracle's steps.  The solve is cut at four iterations, where rounding has not
been amplified (as in the solver tests): 1e-10, the step tests' bar."""
import numpy as np
import pytest

from falm_amd import _abi as abi
from falm_amd import cases
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


# columns of 64 x 8 cells, and the chunk length that fills 512 workgroups
@pytest.mark.parametrize("n,pc_maxit", [((66, 9, 5), 1),       # 4 columns: chunks of 1 plane
                                        ((66, 9, 5), 2),
                                        ((130, 70, 37), 1),    # 27 columns: 2 planes, the last chunk 1
                                        ((130, 70, 37), 2),
                                        ((200, 136, 70), 1)])  # 68 columns: 9 planes, the last chunk 7
def test_chunk_lengths(gpu, n, pc_maxit):
    kw = dict(n=n, cells_per_d=8, pc_maxit=pc_maxit, pc_relax=1.0 if pc_maxit == 1 else 1.5, hub_x_d=1.0, tol=1e-30, maxit=4,
              with_rotor=n[2] > 8, rotor_kw=dict(n_ap_per_blade=6))
    ref, dev = O.Case(cases.windtunnel(**kw)), gpu.Case(cases.windtunnel(**kw))
    for _ in range(2):
        ir, ig = ref.step(1), dev.step(1)
    assert ig.solver_it == ir.solver_it == 4
    for f in (abi.FIELD_U, abi.FIELD_UU, abi.FIELD_NUT, abi.FIELD_P):
        a, b = dev.get(f), ref.get(f)
        assert np.max(np.abs(a - b)) <= 1e-10 * np.max(np.abs(b)), f
    assert abs(ig.div - ir.div) <= 1e-9 * ir.div
