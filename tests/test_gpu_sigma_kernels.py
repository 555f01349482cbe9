"""Sigma_c(R, i omega) at the edges of the self-energy kernels' fragments (16 and 32 orbitals, 16 and 64
auxiliary functions, 64 and 128 segments), in one pass over all tau points and one at a time, and with
C W cut into one chunk per atom, against the FP64 oracle; the FP32 kernels against the FP64 ones.

Bars: FP64 1e-10 of the largest element (as for the other self-energy parity tests).  FP32: operands
and sums carry 2^-24 each; the longest sum has some 10^4 terms of either sign (random-walk growth 100)
and the six-point transforms add entries of up to 10^2: 2^-24 * 100 * 100 = 6e-4, so 1e-3."""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth
from oracle import gw, rpa

pytestmark = pytest.mark.gpu

SIZES = [
    ((1, 2), (3, 15), (1, 1, 1)),
    ((15, 16), (16, 17), (2, 1, 1)),
    ((16, 17), (31, 33), (1, 1, 1)),
    ((17, 33), (48, 65), (2, 1, 1)),
    ((32, 31), (63, 64), (1, 1, 1)),
    ((33, 4), (66, 130), (3, 1, 1)),
]


def _system(nao, nabf, period):
    return synth.tiny(natom=2, period=period, nao=nao, nabf=nabf, nocc=(1, 1), a=7.0, nfreq=6, seed=7, real_gamma_v=True)


def _sigma(s, prec=L.FP64):
    h = L.Handler()
    L.load_system(h, s, vq_cut=True)
    h.set_precision(prec, prec)
    o = L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
    h.build_g0w0_sigma(o)
    ao = rpa.Basis(s.nao)
    out = {}
    for iw in range(s.nfreq):
        for R in rpa.r_grid(s.period):
            m = np.zeros((int(sum(s.nao)), int(sum(s.nao))), dtype=complex)
            for I in range(s.natom):
                for J in range(s.natom):
                    m[ao.sl(I), ao.sl(J)] = h.get_sigma_block(0, iw, I, J, R, int(s.nao[I]), int(s.nao[J]))
            out[(iw, R)] = m
    return out, h.get_tfgrids(o)


def _rel(a, b):
    return max(np.abs(a[k] - b[k]).max() for k in b) / max(np.abs(b[k]).max() for k in b)


@pytest.mark.parametrize("nao,nabf,period", SIZES)
def test_fragment_edges(lib, monkeypatch, nao, nabf, period):
    print(f"Sigma nao={nao} nabf={nabf} period={period}", flush=True)
    s = _system(nao, nabf, period)
    got, grid = _sigma(s)
    chi0s = rpa.chi0s_all_tau(s, grid)
    ref = gw.sigma_all(s, grid, gw.w_r_tau(s, grid, gw.wc_q_omega(s, grid, rpa.chi0_q_omega(s, grid, chi0s))))
    print(f"  against the oracle {_rel(got, ref):.2e}", flush=True)
    assert _rel(got, ref) < 1e-10
    monkeypatch.setenv("LIBRPA_AMD_TAU_BATCH", "1")
    monkeypatch.setenv("LIBRPA_AMD_CHUNK_BYTES", "1")
    one, _ = _sigma(s)
    print(f"  one tau point a pass, one atom a chunk {_rel(one, ref):.2e}", flush=True)
    assert _rel(one, ref) < 1e-10
    low, _ = _sigma(s, L.FP32)
    print(f"  FP32 {_rel(low, ref):.2e}", flush=True)
    assert _rel(low, ref) < 1e-3
