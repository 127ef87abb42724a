"""Kernels at the sizes where their tilings can go wrong (remainders, the
smallest and largest of a range), each against the CPU oracle."""
import numpy as np
import pytest

from test_gpu_parity import assert_close, make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jtot", [8, 60, 64, 512, 540, 2048, 2250])
def test_diagnostics_partial_counts(sns, jtot):
    """The last reduction of the monitors over few slots, one full round of
    its threads (64 slots), whole and ragged unrolled rounds (512, 540) and
    the most slots (2048; 2250 rows share them): sums of jtot*itot terms of
    one sign to 1e-12, as the sequential ones."""
    o, inst = make_pair(sns, 8, jtot, 3.0, seed=jtot)
    d = inst.diagnostics()
    ene, nu = o.energy(), o.nusselt()
    assert d["divmax"] == o.divergence()[0]
    for k, ref in (("energy_ux", ene[0]), ("energy_uy", ene[1]), ("energy_t", ene[2]),
                   ("nu_eps_k", nu[2]), ("nu_eps_h", nu[3])):
        assert abs(d[k] - ref) <= 1e-12 * abs(ref), (k, d[k], ref)
    inst.close()
