"""Device memory of G0W0 builds: what a handle keeps between builds, after a failed build, and beside
another handle.  Free device memory is asked of the driver; sizes are chosen so that the kept buffers (over
100 MB) stand out against its granularity (2 MB a buffer)."""
import numpy as np
import pytest
import torch

import librpa_amd as L
from librpa_amd import synth

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _system(nabf=220):
    s = synth.tiny(natom=2, period=(2, 1, 1), nao=(12, 9), nabf=(nabf, nabf - 20), nocc=(2, 1), a=7.0, nfreq=12,
                   real_gamma_v=True)
    n = s.nabf_tot
    s.vq[:] = np.eye(n)  # its largest eigenvalue is degenerate: no head can be replaced
    return s


def _options(s, **kw):
    return L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI, **kw)


def _fail(h, s):
    h.set_dielect_func_imagfreq(h.get_tfgrids(_options(s))["omega"], np.full(s.nfreq, 2.0))
    with pytest.raises(L.LibrpaError, match="degenerate"):
        h.build_g0w0_sigma(_options(s, replace_w_head=1))


def test_failed_build(lib, monkeypatch):
    """With nothing to be kept, a build that fails gives the memory back as one that ends does."""
    print("failed G0W0 build", flush=True)
    monkeypatch.setenv("LIBRPA_AMD_KEEP_BYTES", "0")
    s = _system()
    h = L.Handler()
    L.load_system(h, s, vq_cut=True)
    _fail(h, s)  # (the eigen-solver library takes its own work memory on first use)
    h.free()
    h = L.Handler()
    L.load_system(h, s, vq_cut=True)
    h.build_g0w0_sigma(_options(s))
    good = np.array([h.get_sigc_ks(0, 0, n, s.nfreq) for n in range(3)])
    before = _free()
    _fail(h, s)
    after = _free()
    print(f"  free memory {before / MB:.0f} MB before, {after / MB:.0f} MB after the failed build", flush=True)
    assert after >= before - 8 * MB
    # the earlier results stay, and the next build needs nothing of the failed one
    assert np.array_equal(np.array([h.get_sigc_ks(0, 0, n, s.nfreq) for n in range(3)]), good)
    h.build_g0w0_sigma(_options(s))
    again = np.array([h.get_sigc_ks(0, 0, n, s.nfreq) for n in range(3)])
    assert np.abs(again - good).max() <= 1e-11 * np.abs(good).max()


def test_nothing_kept(lib, monkeypatch):
    """LIBRPA_AMD_KEEP_BYTES=0: a second build leaves as much free as the first; by default it keeps its buffers."""
    s = _system()
    used = {}
    for keep in ("0", None):
        if keep:
            monkeypatch.setenv("LIBRPA_AMD_KEEP_BYTES", keep)
        else:
            monkeypatch.delenv("LIBRPA_AMD_KEEP_BYTES")
        h = L.Handler()
        L.load_system(h, s, vq_cut=True)
        start = _free()
        h.build_g0w0_sigma(_options(s))
        used[keep] = start - _free()
        h.build_g0w0_sigma(_options(s))
        assert abs(start - _free() - used[keep]) <= 8 * MB
        h.free()
    print(f"  kept: {used['0'] / MB:.0f} MB with a limit of 0, {used[None] / MB:.0f} MB by default", flush=True)
    assert used[None] - used["0"] > 100 * MB


def test_changed_precision(lib):
    """A build in another precision plans with the old engine's memory free: after one that failed there is the
    new engine (half the bytes) beside the old results, not both engines."""
    print("G0W0 in another precision", flush=True)
    s = _system()
    h = L.Handler()
    L.load_system(h, s, vq_cut=True)
    _fail(h, s)
    h.free()
    h = L.Handler()
    L.load_system(h, s, vq_cut=True)
    start = _free()
    h.build_g0w0_sigma(_options(s))
    good = np.array([h.get_sigc_ks(0, 0, n, s.nfreq) for n in range(3)])
    both = start - _free()
    h.set_precision(L.FP32, L.FP32)
    _fail(h, s)
    used = start - _free()
    print(f"  {both / MB:.0f} MB after the FP64 build, {used / MB:.0f} MB after the failed FP32 one", flush=True)
    assert used <= both + 8 * MB
    assert np.array_equal(np.array([h.get_sigc_ks(0, 0, n, s.nfreq) for n in range(3)]), good)
    h.build_g0w0_sigma(_options(s))
    low = np.array([h.get_sigc_ks(0, 0, n, s.nfreq) for n in range(3)])
    assert 0 < np.abs(low - good).max() <= 1e-2 * np.abs(good).max()


def test_given_back_to_another_handle(lib):
    """What an idle handle keeps goes back when another plans with less than half of the device free, and not
    before; the idle handle's next calls allocate again."""
    print("two handles", flush=True)
    s = _system()
    a = L.Handler()
    L.load_system(a, s, vq_cut=True)
    a.build_g0w0_sigma(_options(s))
    ec = a.get_rpa_correlation_energy(_options(s), s.nk)[0]
    good = np.array([a.get_sigc_ks(0, 0, n, s.nfreq) for n in range(3)])
    small = synth.tiny(natom=2, period=(2, 1, 1), nao=(3, 2), nabf=(4, 3), nocc=(1, 1), a=7.0, nfreq=6)

    def plan():
        h = L.Handler()
        L.load_system(h, small)
        h.get_rpa_correlation_energy(_options(small), small.nk)
        h.free()

    plan()
    free = _free()
    plan()
    assert abs(_free() - free) <= 8 * MB
    total = torch.cuda.mem_get_info()[1]
    fill = torch.empty(max(0, free - int(0.4 * total)), dtype=torch.uint8, device="cuda")
    free = _free()
    plan()
    got = _free() - free
    del fill
    torch.cuda.empty_cache()
    print(f"  {got / MB:.0f} MB came back", flush=True)
    assert got > 100 * MB
    again = a.get_rpa_correlation_energy(_options(s), s.nk)[0]
    assert abs(again - ec) <= 1e-11 * abs(ec)
    a.build_g0w0_sigma(_options(s))
    again = np.array([a.get_sigc_ks(0, 0, n, s.nfreq) for n in range(3)])
    assert np.abs(again - good).max() <= 1e-11 * np.abs(good).max()
