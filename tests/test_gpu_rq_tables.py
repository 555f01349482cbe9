"""The tau -> omega and R -> q sums with their tables as kernel arguments (up to 448 values) and in memory
(24 x 24 transform entries, 8 q of 30 or 36 cells), eight q at a time with a shorter last group and one at a
time, against the oracle.

Bar: 1e-10 of Ec, as for the factorisation's other tests."""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth
from oracle import rpa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("period,nfreq", [((3, 3, 3), 6), ((5, 6, 1), 6), ((6, 6, 1), 10), ((2, 1, 1), 24)])
def test_tables(lib, monkeypatch, period, nfreq):
    s = synth.tiny(natom=2, period=period, nao=(2, 3), nabf=(5, 7), nocc=(1, 1), a=7.0, nfreq=nfreq, seed=13)
    o = L.Options(nfreq=nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
    ref = None
    for group in (None, "1", "3"):
        print(f"R -> q tables {period} nfreq {nfreq}, q a pass {group}", flush=True)
        if group:
            monkeypatch.setenv("LIBRPA_AMD_EC_QGROUP", group)
        h = L.Handler()
        L.load_system(h, s)
        ec, contrib = h.get_rpa_correlation_energy(o, s.nk)
        if ref is None:
            grid = h.get_tfgrids(o)
            acc = {}
            for it, blocks in enumerate(rpa.chi0s_all_tau(s, grid)):
                rpa.freq_accumulate(s, grid, blocks, it, acc)
            ref, rc = rpa.rpa_ec_streamed(s, grid, acc)
        assert abs(ec - ref) <= 1e-10 * abs(ref)
        assert np.abs(contrib.real - rc.real).max() <= 1e-10 * abs(ref)
