"""The single operations that take their k-marching form on large domains
(pseudo-velocity with every scheme, Smagorinsky) against the oracle, just above
the sizes where they do (2 M cells in double; in float also planes of 70 k
cells), with a partial tile in x and y, a shorter last chunk and a stretched
mesh.  The expressions are those of the
small-domain kernels: the same bars (1e-12 in double, 1e-5 in float; 1e-11
for the eddy viscosity, whose cube root differs by an ulp or two)."""
import ctypes as C

import numpy as np
import pytest

from falm_amd import _abi as abi
from oracle import pyoracle as O
from tests.helpers import Keep, domain, from_dev, interior_mask, rel_err, smooth_field, to_dev, uniform_metrics

pytestmark = pytest.mark.gpu

# 2 029 170 cells in 3 x 17 columns, planes of 16 770 (in float the small-domain
# form); 2 074 051 cells in 10 x 15 columns, planes of 71 519
@pytest.fixture(scope="module", params=[(130, 129, 121), (601, 119, 29)])
def F(request):
    dom = domain(request.param)
    rng = np.random.default_rng(8)
    _, (xyz, kx, g, ja) = uniform_metrics(dom, stretch=0.004)
    u = smooth_field(dom, 3, rng, base=0.8, amp=0.5)
    return dict(dom=dom, u=u, un=u + 0.01 * smooth_field(dom, 3, rng, base=0.0, amp=1.0),
                uu=smooth_field(dom, 3, rng, base=0.1, amp=0.1), ff=smooth_field(dom, 3, rng, base=0.0, amp=0.3),
                nut=np.abs(smooth_field(dom, 1, rng, base=1e-3, amp=1e-3)),
                kx=kx, g=g, ja=ja)


def _dtype(prec):
    import torch
    return torch.float64 if prec == abi.F64 else torch.float32


@pytest.mark.parametrize("scheme", [abi.ADV_UPWIND1, abi.ADV_UPWIND3, abi.ADV_QUICK, abi.ADV_UTOPIA, abi.ADV_KK])
def test_pseudo_u_large(gpu, F, scheme):
    dom, m = F["dom"], interior_mask(F["dom"], 3)
    ref = O.pseudo_u(dom, scheme, 1e-3, 1e-3, F["un"], F["u"], F["uu"], F["nut"], F["kx"], F["g"], F["ja"], F["ff"])
    for prec, tol in ((abi.F64, 1e-12), (abi.F32, 1e-5)):
        K = Keep()
        ua = to_dev(np.full(3 * dom.ncell, 9.0), _dtype(prec))
        gpu.call("falm_pseudo_u", C.byref(dom), prec, scheme, 1e-3, 1e-3,
                 *[K(F[k], _dtype(prec)) for k in ("un", "u", "uu")], K(ua),
                 *[K(F[k], _dtype(prec)) for k in ("nut", "kx", "g", "ja", "ff")], None)
        got = from_dev(ua)
        assert rel_err(got, ref, m) < tol
        assert np.all(got[~m] == 9.0)


def test_smagorinsky_large(gpu, F):
    dom, m = F["dom"], interior_mask(F["dom"])
    ref = O.sgs(dom, abi.SGS_SMAGORINSKY, 0.1, F["u"], F["kx"], F["ja"])
    for prec, tol in ((abi.F64, 1e-11), (abi.F32, 1e-5)):
        K = Keep()
        nut = to_dev(np.full(dom.ncell, 9.0), _dtype(prec))
        gpu.call("falm_sgs", C.byref(dom), prec, abi.SGS_SMAGORINSKY, 0.1, K(F["u"], _dtype(prec)), K(nut),
                 K(F["kx"], _dtype(prec)), K(F["ja"], _dtype(prec)), None)
        got = from_dev(nut)
        assert rel_err(got, ref, m) < tol
        assert np.all(got[~m] == 9.0)
