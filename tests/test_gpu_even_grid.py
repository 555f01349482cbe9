"""Evenly spaced imaginary-time grids (EvenSpaced_TF), which take any number of points from any first
time, against the FP64 oracle.

Bars: the FP64 chi0 blocks as elsewhere, 1e-9 of the largest element; Ec 1e-10 (a few hundred FP64 roundings
and a 14 x 14 log-determinant); the same sums in another order 1e-12."""
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


@pytest.mark.parametrize("nfreq", [34, 35, 40, 70])
def test_more_points_than_a_pass(lib, nfreq):
    """A pass takes at most 34 tau points; the chi0(R, omega) store takes as many, longer grids go without."""
    print(f"even grid of {nfreq} points", flush=True)
    s = synth.tiny(natom=2, period=(2, 1, 1), nao=(3, 2), nabf=(4, 3), nocc=(1, 1), a=7.0, nfreq=nfreq)
    o = _options(nfreq, 0.1, 0.05)
    _check_chi0(s, o)
    h = L.Handler()
    L.load_system(h, s)
    ec, contrib = h.get_rpa_correlation_energy(o, s.nk)
    acc = {}
    grid = h.get_tfgrids(o)
    for it, blocks in enumerate(rpa.chi0s_all_tau(s, grid)):
        rpa.freq_accumulate(s, grid, blocks, it, acc)
    ref, _ = rpa.rpa_ec_streamed(s, grid, acc)
    print(f"  Ec {ec!r} oracle {ref!r}", flush=True)
    assert abs(ec - ref) <= 1e-10 * abs(ref)


def test_self_energy_on_a_long_grid(lib, monkeypatch):
    """G0W0 on 40 points: passes of several tau points and one at a time give the same Sigma."""
    s = synth.tiny(natom=2, period=(2, 1, 1), nao=(3, 2), nabf=(4, 3), nocc=(1, 1), a=7.0, nfreq=40,
                   real_gamma_v=True)
    o = _options(40, 0.1, 0.05)
    out = []
    for batch in (None, "1"):
        print(f"Sigma on 40 points, tau points a pass {batch}", flush=True)
        if batch:
            monkeypatch.setenv("LIBRPA_AMD_TAU_BATCH", batch)
        h = L.Handler()
        L.load_system(h, s, vq_cut=True)
        h.build_g0w0_sigma(o)
        out.append(np.array([[h.get_sigc_ks(0, k, n, 40) for n in range(s.nbands)] for k in range(s.nk)]))
    assert np.abs(out[0] - out[1]).max() <= 1e-12 * np.abs(out[1]).max()
