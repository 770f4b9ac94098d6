"""A full write of the rotor's force field: exact zeros in every interior cell
outside the force box over whatever was there, ghost cells untouched, the
oracle's sums inside, with the rotor in the middle, over an edge of the domain
and outside it (an empty box).  1e-12 as the other projection tests."""
import numpy as np
import pytest

from falm_amd import _abi as abi
from falm_amd import cases
from oracle import pyoracle as O
from tests.helpers import Keep, domain, from_dev, interior_mask, rel_err, smooth_field, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(70, 27, 25), (24, 9, 7)])
@pytest.mark.parametrize("at", [(0.5, 0.5, 0.5), (0.02, 0.95, 0.1), (3.0, 0.5, 0.5)])
@pytest.mark.parametrize("prec", [abi.F64, abi.F32])
def test_full_write(gpu, n, at, prec):
    import torch
    K = Keep()
    dom, h = domain(n), 1.0 / 8.0
    setup = cases.rotor(h, base=tuple(a * m * h for a, m in zip(at, n)), n_ap_per_blade=5)
    xs = [(np.arange(s) - 1.5) * h for s in dom.shape]
    u = smooth_field(dom, 3, np.random.default_rng(3), base=1.0, amp=0.2)
    dt = torch.float64 if prec == abi.F64 else torch.float32
    ud = to_dev(u, dt)
    ref, ff_ref = O.Alm(dom, setup, *xs), np.zeros(3 * dom.ncell)
    ref.step(ud.double().cpu().numpy(), ff_ref, 0.2)
    A = gpu.Alm(dom, setup, *xs)
    ff = to_dev(np.full(3 * dom.ncell, 7.0), dt)
    for t in (1.1, 0.2):  # the second write covers what the first left
        A.step(prec, K(ud), ff, t)
    got, m = from_dev(ff), interior_mask(dom, 3)
    assert np.all(got[~m] == 7.0)
    assert rel_err(got, ff_ref, m) < (1e-12 if prec == abi.F64 else 1e-6)
    tq, th = A.get()[2:]
    tq_r, th_r = ref.get()[2:]
    assert rel_err(tq, tq_r) < 1e-12 and rel_err(th, th_r) < 1e-12
    if at[0] > 1.0:
        assert np.all(got[m] == 0.0)
