"""W in passes of several q points with a shorter last pass, and in chunks of the frequencies of one q (what
large systems do), against one pass over all; with equal and with truncated Coulomb matrices, filtered
roots and a replaced head.  FP32 Sigma with several tau points in a pass.

Bars: the same FP64 sums in another order, 1e-12 of the largest element; a root from the eigen-solver
repeats to rounding times the condition number of v (1e4 here), 1e-11.  FP32 as elsewhere, 2^-24 sqrt(1e4)
x 1e2 = 6e-4, so 1e-3."""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth

pytestmark = pytest.mark.gpu

PASSES = [{"LIBRPA_AMD_W_QGROUP": "2"}, {"LIBRPA_AMD_W_FREQS": "4"}, {"LIBRPA_AMD_W_QGROUP": "1"}, {"LIBRPA_AMD_W_FREQS": "1"}]


def _system():
    return synth.tiny(natom=2, period=(3, 1, 1), nao=(3, 4), nabf=(9, 14), nocc=(1, 1), a=7.0, nfreq=6, seed=9,
                      real_gamma_v=True)


def _w(s, cut=True, threshold=0.0, head=False):
    h = L.Handler()
    L.load_system(h, s, vq_cut=cut)
    o = L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI, sqrt_coulomb_threshold=threshold,
                  replace_w_head=1 if head else 0)
    if head:
        h.set_dielect_func_imagfreq(h.get_tfgrids(o)["omega"], 1.5 + np.arange(s.nfreq) / 10.0)
    h.build_g0w0_sigma(o)
    return np.concatenate([h.get_wc_block(t, I, J, (R, 0, 0), int(s.nabf[I]), int(s.nabf[J])).ravel()
                           for t in range(s.nfreq) for I in range(2) for J in range(2) for R in (-1, 0, 1)])


def _sigma(s, prec):
    h = L.Handler()
    L.load_system(h, s, vq_cut=True)
    h.set_precision(prec, prec)
    h.build_g0w0_sigma(L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI))
    return np.array([[h.get_sigc_ks(0, k, n, s.nfreq) for n in range(s.nbands)] for k in range(s.nk)])


@pytest.mark.parametrize("kind", ["equal", "truncated", "filtered", "head", "truncated_head"])
def test_w_passes(lib, monkeypatch, kind):
    s = _system()
    rng = np.random.default_rng(4)
    d = 0.6 + 0.3 * rng.random(s.nabf_tot)
    cut = s.vq * d[None, :, None] * d[None, None, :] if kind.startswith("truncated") else True
    kw = dict(cut=cut, threshold=1e-4 if kind == "filtered" else 0.0, head=kind.endswith("head"))
    ref = _w(s, **kw)
    bar = 1e-11 if kind in ("filtered", "head", "truncated_head") else 1e-12
    for env in PASSES:
        print(f"W passes {kind} {env}", flush=True)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        assert np.abs(_w(s, **kw) - ref).max() <= bar * np.abs(ref).max()
        for k in env:
            monkeypatch.delenv(k)


def test_fp32_sigma_of_several_tau_points(lib, monkeypatch):
    s = _system()
    ref = _sigma(s, L.FP64)
    low = _sigma(s, L.FP32)
    assert np.abs(low - ref).max() <= 1e-3 * np.abs(ref).max()
    monkeypatch.setenv("LIBRPA_AMD_TAU_BATCH", "4")  # passes of 3 and 3
    assert np.abs(_sigma(s, L.FP32) - ref).max() <= 1e-3 * np.abs(ref).max()
    assert np.abs(_sigma(s, L.FP64) - ref).max() <= 1e-12 * np.abs(ref).max()
