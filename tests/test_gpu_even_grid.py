"""Evenly spaced imaginary-time grids (EvenSpaced_TF), which take any number of points from any first
time, against the FP64 oracle.

Bars: the FP64 chi0 blocks as elsewhere, 1e-9 of the largest element."""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth
from oracle import rpa

pytestmark = pytest.mark.gpu

EVEN_TF = 5


def _metal():
    """Every band partly occupied, so that G(+tau) and G(-tau) both take all bands."""
    s = synth.tiny(natom=2, period=(2, 1, 1), nao=(3, 2), nabf=(4, 3), nocc=(1, 1), a=7.0, nfreq=6)
    s.occ[:] = 0.2 + 1.6 / (1.0 + np.exp(4.0 * (s.eps - s.efermi)))
    return s


def _options(nfreq, first, step):
    return L.Options(nfreq=nfreq, tfgrids_type=EVEN_TF, parallel_routing=L.LIBRI, tfgrids_freq_min=0.1,
                     tfgrids_freq_interval=0.05, tfgrids_time_min=first, tfgrids_time_interval=step)


def _check_chi0(s, o):
    h = L.Handler()
    L.load_system(h, s)
    h.set_keep_chi0(True)
    h.get_rpa_correlation_energy(o, s.nk)
    grid = h.get_tfgrids(o)
    for t, ref in enumerate(rpa.chi0s_all_tau(s, grid)):
        big = max(np.abs(b).max() for b in ref.values())
        for (I, J, R), b in ref.items():
            got = h.get_chi0s_block(t, I, J, R, int(s.nabf[I]), int(s.nabf[J]))
            assert np.abs(got - b).max() <= 1e-9 * big, (grid["tau"][t], I, J, R)


@pytest.mark.parametrize("first", [0.0, -0.4, 0.3])
def test_first_time(lib, first):
    """G(R, tau) changes sign for tau < 0 only: at tau = 0 both G keep theirs."""
    print(f"even grid from tau = {first}", flush=True)
    _check_chi0(_metal(), _options(6, first, 0.2))
