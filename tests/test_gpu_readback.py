"""Host copies of a case's fields: every value as it is on the device, below
and above the size from which several threads share the copy, before and after
the case has copied enough for that, with a last chunk that is short, and with
two callers at once.  Exact (mixed: the float the device holds, widened)."""
import threading

import numpy as np
import pytest

from falm_amd import _abi as abi
from falm_amd import cases

pytestmark = pytest.mark.gpu


# velocity values: 3 (n + 4)^3 = 517 k and 526 k (below four chunks of 2^18),
# 3.5 M, and 8.1 M with a last chunk of 237 k, more than a first copy needs
@pytest.mark.parametrize("n", [(51, 51, 53), (52, 53, 51), (101, 101, 101), (135, 135, 136)])
@pytest.mark.parametrize("precision", [abi.CASE_F64, abi.CASE_MIXED])
def test_get_returns_the_field(gpu, n, precision):
    c = gpu.Case(cases.windtunnel(n=n, cells_per_d=8, precision=precision, with_rotor=False))
    rng = np.random.default_rng(5)
    want = {f: rng.standard_normal(c.dom.ncell * abi.FIELD_NCOL[f]) for f in (abi.FIELD_U, abi.FIELD_P)}
    for f, v in want.items():
        c.set(f, v)
    if precision == abi.CASE_MIXED:
        want[abi.FIELD_U] = want[abi.FIELD_U].astype(np.float32).astype(np.float64)
    got = {}

    def fetch(f):
        got[f] = [c.get(f) for _ in range(2)]

    ts = [threading.Thread(target=fetch, args=(f,)) for f in want]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for f, v in want.items():
        for g in got[f]:
            np.testing.assert_array_equal(g, v)


@pytest.mark.parametrize("precision", [abi.CASE_F64, abi.CASE_MIXED])
def test_repeated_gets(gpu, precision):
    """1 058 610 values (four chunks and one of 10 034), ten times: the plain
    copy until 8 M values have been copied, then the threads."""
    c = gpu.Case(cases.windtunnel(n=(67, 67, 66), cells_per_d=8, precision=precision, with_rotor=False))
    v = np.random.default_rng(6).standard_normal(3 * c.dom.ncell)
    c.set(abi.FIELD_U, v)
    if precision == abi.CASE_MIXED:
        v = v.astype(np.float32).astype(np.float64)
    for _ in range(10):
        np.testing.assert_array_equal(c.get(abi.FIELD_U), v)
