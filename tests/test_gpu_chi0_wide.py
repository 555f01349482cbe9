"""The chi0 contraction kernel on atoms with more than 32 functions or more than 128 auxiliary functions,
against the oracle: W steps in a loop of groups of 4 or 8; strips of up to 192 (FP64) or 128 rows, and of
half the columns and up to 320 or 256 rows past that; G in LDS for up to 192 functions of J, from memory past
them.

Bars: FP64 sums of at most 1e6 products agree to about 1e-16 sqrt(1e6) = 1e-13 of the largest
element; 1e-12 leaves the intermediate W and G their share.  FP32: 6e-8 sqrt(1e6) = 6e-5, so 1e-4."""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth
from oracle import rpa

pytestmark = pytest.mark.gpu

# (functions per atom, auxiliary functions per atom, k mesh)
SIZES = {
    "first_past_32": ((33, 34), (40, 50), (2, 1, 1)),
    "groups": ((40, 41), (96, 128), (1, 1, 1)),
    "first_past_128_rows": ((5, 17), (129, 145), (2, 1, 1)),
    "full_strip_of_half_columns": ((33, 40), (256, 160), (1, 1, 1)),
    "11_and_13_fragments": ((9, 48), (176, 208), (2, 1, 1)),
    "many_rows_few_columns": ((35, 36), (129, 20), (1, 1, 1)),
    "17_and_19_fragments": ((16, 35), (257, 290), (1, 1, 1)),
    "two_strips": ((34, 33), (321, 500), (1, 1, 1)),
    "fragments_10_12_14_16": ((33, 4), (192, 193), (1, 1, 1)),
    "fragments_18_20": ((15, 36), (288, 320), (1, 1, 1)),
    "lds_share": ((17, 192), (20, 130), (1, 1, 1)),
    "past_the_lds_share": ((20, 194), (20, 140), (1, 1, 1)),
    "far_past_the_lds_share": ((2, 258), (5, 3), (1, 1, 1)),
}


@pytest.mark.parametrize("prec,bar", [(L.FP64, 1e-12), (L.FP32, 1e-4)])
@pytest.mark.parametrize("name", sorted(SIZES))
def test_classes(lib, name, prec, bar, monkeypatch):
    nao, nabf, period = SIZES[name]
    s = synth.tiny(natom=2, period=period, nao=nao, nabf=nabf, nocc=(1, 1), a=7.0, nfreq=6, seed=11)
    o = L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
    ref = None
    for splitk in (None, "1", "5"):
        print(f"chi0 kernel {name} prec={prec} parts={splitk}", flush=True)
        if splitk:
            monkeypatch.setenv("LIBRPA_AMD_SPLITK", splitk)
        h = L.Handler()
        L.load_system(h, s)
        h.set_precision(prec, L.FP64)
        h.set_keep_chi0(True)
        h.get_rpa_correlation_energy(o, s.nk)
        if ref is None:
            grid = h.get_tfgrids(o)
            ref = rpa.chi0s_all_tau(s, {"tau": [grid["tau"][0], grid["tau"][3]]})
        for it, t in enumerate((0, 3)):
            big = max(np.abs(b).max() for b in ref[it].values())
            for (I, J, R), b in ref[it].items():
                got = h.get_chi0s_block(t, I, J, R, int(s.nabf[I]), int(s.nabf[J]))
                assert np.abs(got - b).max() <= bar * big, (t, I, J, R)
