"""Sigma with U and Y of one sign of tau at a time (what a system does whose two signs do not fit), against
both signs at once: the same sums over other passes.

Bars: FP64 1e-12 of the largest element (order of the atomic adds); FP32 2^-24 sqrt(1e4) times the entries
of up to 1e2 of the six-point transforms, 6e-4, so 1e-3."""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth

pytestmark = pytest.mark.gpu

SYSTEMS = {
    "gamma_odd": dict(nao=(17, 33), nabf=(48, 65), period=(1, 1, 1)),
    "k_small": dict(nao=(3, 5), nabf=(11, 16), period=(3, 1, 1)),
    "k_two_fragments": dict(nao=(16, 20), nabf=(31, 33), period=(2, 1, 1)),
}


def _sigma(s, prec=L.FP64):
    h = L.Handler()
    L.load_system(h, s, vq_cut=True)
    h.set_precision(prec, prec)
    h.build_g0w0_sigma(L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI))
    return np.array([[[h.get_sigc_ks(sp, k, n, s.nfreq) for n in range(0, s.nbands, 5)] for k in range(s.nk)]
                     for sp in range(s.nspin)])


@pytest.mark.parametrize("nspin", [1, 2])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_one_sign_at_a_time(lib, monkeypatch, name, nspin):
    s = synth.tiny(natom=2, nocc=(1, 1), a=7.0, nfreq=6, seed=7, real_gamma_v=True, **SYSTEMS[name])
    if nspin == 2:
        s = synth.spin_polarised(s)
    print(f"Sigma by signs, {name}, spins {nspin}", flush=True)
    ref = _sigma(s)
    big = np.abs(ref).max()
    monkeypatch.setenv("LIBRPA_AMD_SIGMA_SIGNS", "1")
    assert np.abs(_sigma(s) - ref).max() <= 1e-12 * big
    assert np.abs(_sigma(s, L.FP32) - ref).max() <= 1e-3 * big
    monkeypatch.setenv("LIBRPA_AMD_CHUNK_BYTES", "1")
    assert np.abs(_sigma(s) - ref).max() <= 1e-12 * big
