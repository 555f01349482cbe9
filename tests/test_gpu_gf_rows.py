"""G(R, +-tau) by strips of rows: bases around the lines where the strips of 64 rows begin (2 n = 64, 512,
1024 rows) and a k mesh of 8 points that takes whole matrices, through chi0 against the oracle.

Bar: as the other FP64 parity tests, 1e-9 of the largest element."""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth
from oracle import rpa

pytestmark = pytest.mark.gpu

SIZES = [((16, 16), (1, 1, 1)), ((16, 17), (1, 1, 1)), ((16, 17), (2, 1, 1)), ((128, 128), (1, 1, 1)),
         ((128, 129), (1, 1, 1)), ((200, 257), (1, 1, 1)), ((16, 17), (2, 2, 2)), ((20, 13), (7, 1, 1))]


@pytest.mark.parametrize("nao,period", SIZES)
def test_rows(lib, nao, period):
    print(f"G rows nao={nao} period={period}", flush=True)
    s = synth.tiny(natom=2, period=period, nao=nao, nabf=(3, 4), nocc=(3, 2), a=7.0, nfreq=6, seed=3)
    o = L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
    h = L.Handler()
    L.load_system(h, s)
    h.set_keep_chi0(True)
    h.get_rpa_correlation_energy(o, s.nk)
    tau = h.get_tfgrids(o)["tau"]
    for t, ref in zip((0, 4), rpa.chi0s_all_tau(s, {"tau": [tau[0], tau[4]]})):
        big = max(np.abs(b).max() for b in ref.values())
        for (I, J, R), b in ref.items():
            got = h.get_chi0s_block(t, I, J, R, int(s.nabf[I]), int(s.nabf[J]))
            assert np.abs(got - b).max() <= 1e-9 * big, (t, I, J, R)
