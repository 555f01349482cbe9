"""Atoms without basis functions, without auxiliary functions or without both (ghosts, point charges),
first, in the middle and last, against the FP64 oracle's label-by-label sums.

Bars: as the other FP64 parity tests, 1e-9 of the largest chi0 element, 1e-10 of Ec and of the largest
self-energy element."""
import dataclasses

import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth
from oracle import gw, rpa

pytestmark = pytest.mark.gpu

SIZES = [((3, 2, 0), (4, 3, 0)), ((3, 2, 0), (4, 3, 5)), ((3, 2, 2), (4, 3, 0)), ((3, 0, 2), (4, 3, 2)),
         ((0, 3, 2), (0, 3, 4)), ((0, 3, 2), (2, 3, 4))]


@pytest.mark.parametrize("nao,nabf", SIZES)
@pytest.mark.parametrize("period", [(1, 1, 1), (2, 1, 1)])
def test_empty_atoms(lib, nao, nabf, period):
    print(f"empty atoms nao={nao} nabf={nabf} period={period}", flush=True)
    s = synth.tiny(natom=3, period=period, nao=nao, nabf=nabf, nocc=(1, 1, 0), a=7.0, nfreq=6, real_gamma_v=True)
    o = L.Options(nfreq=6, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
    h = L.Handler()
    L.load_system(h, s, vq_cut=True)
    h.set_keep_chi0(True)
    ec, _ = h.get_rpa_correlation_energy(o, s.nk)
    grid = h.get_tfgrids(o)
    ref = dataclasses.replace(s, cs=[c for c in s.cs if c[3].size])
    chi0s = rpa.chi0s_all_tau(ref, grid, method="bruteforce")
    for t in (0, 5):
        big = max(np.abs(b).max() for b in chi0s[t].values() if b.size)
        for (I, J, R), b in chi0s[t].items():
            if b.size:
                got = h.get_chi0s_block(t, I, J, R, nabf[I], nabf[J])
                assert np.abs(got - b).max() <= 1e-9 * big, (t, I, J, R)
    chi0q = rpa.chi0_q_omega(ref, grid, chi0s)
    want, _ = rpa.rpa_ec(ref, grid, chi0q)
    print(f"  Ec {ec!r} oracle {want!r}", flush=True)
    assert abs(ec - want) <= 1e-10 * abs(want)
    h.build_g0w0_sigma(o)
    sig = gw.sigma_all(ref, grid, gw.w_r_tau(ref, grid, gw.wc_q_omega(ref, grid, chi0q)), method="labels")
    ao = rpa.Basis(s.nao)
    big = max(np.abs(m).max() for m in sig.values())
    for (iw, R), m in sig.items():
        for I in range(3):
            for J in range(3):
                if nao[I] * nao[J]:
                    got = h.get_sigma_block(0, iw, I, J, R, nao[I], nao[J])
                    assert np.abs(got - m[ao.sl(I), ao.sl(J)]).max() <= 1e-10 * big, (iw, I, J, R)
