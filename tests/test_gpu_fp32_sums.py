"""The length of FP32 sums in the chi0 contraction of a large cell: FP32 blocks of the 128-atom cell
against FP64 ones (V = 1; only chi0 is looked at).

Bar, rms over the diagonal blocks (the largest) of a tau point: n adds of either sign into one FP32 accumulator are off by about
2^-24 sqrt(n / 2) / sqrt(3) x 0.72 of the sum (rounding errors uniform in half a unit of the running sum,
which grows like sqrt(n)).  At most 1600 adds into an accumulator: 7.0e-7; W, 640 adds (K = 2560 by fours):
4.4e-7; together 8.3e-7, so 8.5e-7.  Two accumulators for a whole list, 6400 adds each, would be at 1.4e-6."""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth

pytestmark = pytest.mark.gpu


def test_large_cell(lib, monkeypatch):
    monkeypatch.setenv("LIBRPA_AMD_AUTOTUNE", "0")
    s = synth.cubic128(nfreq=6, with_vq=False)
    print("128 atoms: system made", flush=True)
    o = L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
    blocks = {}
    for prec in (L.FP64, L.FP32):
        h = L.Handler()
        L.load_system(h, s, vq=False)
        for I, n in enumerate(s.nabf):
            h.set_aux_bare_coulomb_k_atom_pair(0, I, I, int(n), int(n), np.eye(n), np.zeros((n, n)), 0.0)
        h.set_precision(prec, L.FP32)
        h.set_keep_chi0(True)
        print(f"128 atoms: chi0, precision {prec}", flush=True)
        h.get_rpa_correlation_energy(o, s.nk)
        blocks[prec] = [np.concatenate([h.get_chi0s_block(t, I, I, (0, 0, 0), int(n), int(n)).ravel()
                                        for I, n in enumerate(s.nabf)]) for t in range(0, s.nfreq, 2)]
        h.free()
    for a, b in zip(blocks[L.FP32], blocks[L.FP64]):
        rms = np.linalg.norm(a - b) / np.linalg.norm(b)
        print(f"  rms error {rms:.2e}", flush=True)
        assert rms <= 8.5e-7
