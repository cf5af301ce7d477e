"""The mixed-precision M2L on the f16 matrix cores (simplefmm_amd/csrc/m2l_dense.hpp):
the components of an expansion do not share their range.

Charges and lengths are scaled by powers of two, which every step of the path
passes on exactly (FP32 copy, f16 split, products, sums), so each output column
has to be the scaled column of the unscaled problem bit for bit, however much
larger another component is.
"""
import numpy as np
import pytest

from simplefmm_amd import api, workloads as W
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

# both operands are split to 2^-22 each; twice that again for the FP32 sums
TOLERANCE = 4 * 2.0**-22


def _plan(pos, p, scale=1.0, **kw):
    box = api.Box(corner=[-64.0 * scale] * 3, width=128.0 * scale)
    return api.FMM3D(api.OctreePartitioner(pos * scale, box).refine(20, 32), p, **kw)


def _far(fmm, kind, nq, Q, nout):
    U = np.zeros((len(Q), nout))
    fmm._eval(kind, nq, Q, U, api.FAR)
    return U


@pytest.mark.parametrize("p", [1, 4, 7, 10, 12])
@pytest.mark.parametrize("powers", [(0, -20), (-40, 0, -20), (0, 30, -50, 10)], ids=["two", "three", "four"])
def test_unequal_charges_keep_their_bits(p, powers):
    n, nq = 6000, len(powers)
    pos, q = W.plummer(n, seed=31)
    print(f"n={n} p={p} powers={powers}", flush=True)
    scale = 2.0 ** np.array(powers, dtype=np.float64)
    Q = q.reshape(n, 1) * scale
    u = _far(_plan(pos, p, ncharge=nq, precision=api.MIXED), api.POTENTIAL, nq, Q, nq)
    one = _far(_plan(pos, p, ncharge=1), api.POTENTIAL, 1, q.reshape(n, 1), 1)[:, 0]
    equal = _far(_plan(pos, p, ncharge=nq, precision=api.MIXED), api.POTENTIAL, nq, Q / scale, nq)
    for c in range(nq):
        assert np.array_equal(u[:, c], equal[:, c] * scale[c]), c
        assert rel_l2(u[:, c] / scale[c], one) < TOLERANCE, c


@pytest.mark.parametrize("power", [-30, 30])
@pytest.mark.parametrize("p", [4, 12])
def test_gradient_and_potential_in_any_unit_of_length(p, power):
    # potentials go with 1 / length, gradients with 1 / length^2
    n = 6000
    pos, q = W.plummer(n, seed=32)
    print(f"n={n} p={p} lengths x 2^{power}", flush=True)
    Q = q.reshape(n, 1)
    unit = _far(_plan(pos, p, ncharge=1, precision=api.MIXED), api.POTGRAD, 1, Q, 4)
    u = _far(_plan(pos, p, 2.0**power, ncharge=1, precision=api.MIXED), api.POTGRAD, 1, Q, 4)
    ref = _far(_plan(pos, p, 2.0**power, ncharge=1), api.POTGRAD, 1, Q, 4)
    assert np.array_equal(u * 2.0 ** (power * np.array([1, 2, 2, 2])), unit)
    for cols in (slice(0, 1), slice(1, 4)):
        assert rel_l2(u[:, cols], ref[:, cols]) < TOLERANCE


def test_infinite_charge_stays_in_its_component():
    n, p = 6000, 8
    pos, q = W.plummer(n, seed=33)
    print(f"n={n} p={p} one infinite charge", flush=True)
    Q = np.stack([q, q, q], 1)
    plan = _plan(pos, p, ncharge=3, precision=api.MIXED)
    clean = _far(plan, api.POTENTIAL, 3, Q, 3)
    Q[n // 2, 1] = np.inf
    u = _far(plan, api.POTENTIAL, 3, Q, 3)
    assert np.array_equal(u[:, [0, 2]], clean[:, [0, 2]])
    assert not np.isfinite(u[:, 1]).all()
