"""Ec at the edges of the Cholesky blocks (16 and 64 real or 32 complex columns; panels of 512 / 256;
outer panels from n = 4096 / 2048), at Gamma (real) and with k points (Hermitian, two planes),
against the oracle's LU form, with a positive-definite and an indefinite Coulomb matrix.

Bar: 1e-10 of Ec.  The factorisation's own error is about n eps (2055 x 1e-16 = 2e-13); the 6-point
minimax transforms, which both sides share to 1e-13, multiply that by less than 100.
"""
import numpy as np
import pytest

import librpa_amd as L
from librpa_amd import synth
from oracle import rpa

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (7, 8), (8, 8), (8, 9), (15, 17), (16, 17), (31, 33), (32, 33), (60, 70), (128, 129), (200, 313)]


def _check(nabf, period, indefinite=False):
    s = synth.tiny(natom=2, period=period, nao=(2, 3), nabf=nabf, nocc=(1, 1), a=7.0, nfreq=6, seed=5)
    if indefinite:
        n = s.nabf_tot
        rng = np.random.default_rng(3)
        for k in range(s.nk):
            u = rng.standard_normal(n) + 1j * rng.standard_normal(n) * (s.nk > 1)
            u /= np.linalg.norm(u)
            s.vq[k] -= 0.05 * np.outer(u, u.conj())
            assert np.linalg.eigvalsh(s.vq[k].real if s.nk == 1 else s.vq[k])[0] < 0
    h = L.Handler()
    L.load_system(h, s)
    o = L.Options(nfreq=s.nfreq, tfgrids_type=L.MINIMAX, parallel_routing=L.LIBRI)
    ec, contrib = h.get_rpa_correlation_energy(o, s.nk)
    grid = h.get_tfgrids(o)
    acc = {}
    for it, blocks in enumerate(rpa.chi0s_all_tau(s, grid)):
        rpa.freq_accumulate(s, grid, blocks, it, acc)
    ref, rc = rpa.rpa_ec_streamed(s, grid, acc)
    print(f"Ec nabf={nabf} period={period} indefinite={indefinite}: {ec!r} oracle {ref!r}", flush=True)
    assert abs(ec - ref) <= 1e-10 * abs(ref)
    assert np.abs(contrib.real - rc.real).max() <= 1e-10 * abs(ref)


@pytest.mark.parametrize("period", [(1, 1, 1), (2, 1, 1), (3, 1, 1)])
@pytest.mark.parametrize("nabf", SIZES)
def test_block_edges(nabf, period):
    _check(nabf, period)


@pytest.mark.parametrize("period", [(1, 1, 1), (3, 1, 1)])
@pytest.mark.parametrize("nabf", [(16, 17), (60, 70)])
def test_indefinite_coulomb(nabf, period):
    _check(nabf, period, indefinite=True)


def test_outer_panels_of_a_hermitian_matrix():
    _check((1025, 1030), (2, 1, 1))
