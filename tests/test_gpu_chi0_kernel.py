"""The chi0 contraction kernel at the edges of its tiles, against the oracle.

A wave covers 16 FM rows (FM = 2, 4, 6, 8; more rows take several waves), 32 (FP64) or 64 (FP32)
columns, 16 or 32 functions of I and 16, 32 or any number of J per pass, with the first 128 of them
in LDS.  The sizes below sit on and next to those lines.

Bars: FP64 sums of at most 1e6 products agree to about 1e-16 sqrt(1e6) = 1e-13 of the largest
element; 1e-12 leaves the intermediate W and G their share.  FP32: 6e-8 sqrt(1e6) = 6e-5, so 1e-4.
"""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth
from oracle import rpa

pytestmark = pytest.mark.gpu

# (functions per atom, auxiliary functions per atom, k mesh)
SIZES = {
    "one_function": ((2, 1), (1, 2), (2, 1, 1)),
    "full_tiles": ((16, 32), (32, 64), (2, 1, 1)),
    "past_a_tile": ((17, 33), (33, 65), (2, 1, 1)),
    "short_of_a_tile": ((15, 31), (31, 63), (3, 1, 1)),
    "two_row_strips": ((8, 16), (128, 129), (1, 1, 1)),
    "five_row_fragments": ((12, 27), (80, 96), (1, 1, 1)),
    "large_basis": ((5, 70), (17, 140), (1, 1, 1)),
    "past_the_lds_share": ((3, 131), (4, 9), (1, 1, 1)),
}


def _system(name, nspin=1):
    nao, nabf, period = SIZES[name]
    s = synth.tiny(natom=2, period=period, nao=nao, nabf=nabf, nocc=(1, 1), a=7.0, nfreq=6, seed=11)
    return synth.spin_polarised(s) if nspin == 2 else s


def _blocks(h, s, taus):
    return {(t, I, J, R): h.get_chi0s_block(t, I, J, R, int(s.nabf[I]), int(s.nabf[J]))
            for t in taus for I in range(s.natom) for J in range(I, s.natom) for R in rpa.r_grid(s.period)}


@pytest.mark.parametrize("prec,bar", [(L.FP64, 1e-12), (L.FP32, 1e-4)])
@pytest.mark.parametrize("name", sorted(SIZES))
def test_tile_edges(name, prec, bar, monkeypatch):
    s = _system(name)
    taus = (0, 3)
    ref = None
    for splitk in (None, "1", "5"):
        print(f"chi0 kernel {name} prec={prec} parts={splitk}", flush=True)
        if splitk:
            monkeypatch.setenv("LIBRPA_AMD_SPLITK", splitk)
        h = L.Handler()
        L.load_system(h, s)
        h.set_precision(prec, L.FP64)
        h.set_keep_chi0(True)
        o = L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
        h.get_rpa_correlation_energy(o, s.nk)
        if ref is None:
            ref = rpa.chi0s_all_tau(s, h.get_tfgrids(o))
        got = _blocks(h, s, taus)
        for t in taus:
            big = max(np.abs(b).max() for b in ref[t].values())
            for (I, J, R), b in ref[t].items():
                assert np.abs(got[(t, I, J, R)] - b).max() <= bar * big, (t, I, J, R)


def test_two_spins_accumulate():
    s = _system("past_a_tile", nspin=2)
    print("chi0 kernel, two spins", flush=True)
    h = L.Handler()
    L.load_system(h, s)
    h.set_keep_chi0(True)
    o = L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
    h.get_rpa_correlation_energy(o, s.nk)
    ref = rpa.chi0s_all_tau(s, h.get_tfgrids(o))
    got = _blocks(h, s, (0, 5))
    for t in (0, 5):
        big = max(np.abs(b).max() for b in ref[t].values())
        for (I, J, R), b in ref[t].items():
            assert np.abs(got[(t, I, J, R)] - b).max() <= 1e-12 * big
