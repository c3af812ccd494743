"""The orbital-size kernels and the Sigma products at the edges of their blocks, against the oracle (needs an
MI355X): every block count of the 4 x 4 x 4 kernels (nao <= 64) with a partial quad of auxiliary indices, with
two and four spin blocks where G takes several passes through LDS, the half product of a Hermitian P-tilde at
the edges of its 64-wide blocks, and k maps whose pairs are not each other's adjoint.

FP64 within 1e-10 relative, split precision within 1e-8, as everywhere."""
import numpy as np
import pytest

from gwhip import lib as gl
from helpers import min_eig_I_minus_P0, rel_err, synthetic
from oracle import gw_oracle as go
from oracle import hf_oracle as ho
from test_hf_oracle import random_system

pytestmark = pytest.mark.gpu


def _system(nk, nao, NQ, hermitian=True, **kw):
    # V ~ N(0, (0.5 / nao)^2) keeps I - P0 positive definite, also for a G that is not Hermitian
    G, V, T, d = synthetic(nk, nao, NQ, beta=20.0, lam=1e3, mesh=(nk, 1, 1), seed=31, sigma=0.5 / max(nao, 5), **kw)
    if not hermitian:
        rng = np.random.default_rng(8)
        G = G + 1e-3 * (rng.standard_normal(G.shape) + 1j * rng.standard_normal(G.shape))
    assert min_eig_I_minus_P0(G, V, T, d) > 0.3
    return G, V, T, d


def _check(G, V, T, d, maps=None):
    k = gl.GwHipKernel(d["nk"], d["nao"], d["nso"], d["ns"], d["NQ"], T.nts, T.nw_b, d["beta"], mesh=d["mesh"])
    try:
        k.set_grid(T.T_bt, T.T_tb)
        if maps is not None:
            k.set_kq_maps(*maps)
        k.upload_V(V)
        S = k.solve(G)
        P = k.P_tilde()
        S_split = k.solve(G, gl.PREC_SPLIT)
    finally:
        k.close()
    S_ref, P_ref = go.gw_sigma(G, V, T.T_bt, T.T_tb, d["nk"], d["nao"], d["nso"], d["ns"], d["NQ"], mesh=d["mesh"],
                               return_P=True)
    print(f"P {rel_err(P, P_ref):.2e}, Sigma {rel_err(S, S_ref):.2e}, split {rel_err(S_split, S_ref):.2e}", flush=True)
    assert rel_err(P, P_ref) < 1e-10
    assert rel_err(S, S_ref) < 1e-10
    assert rel_err(S_split, S_ref) < 1e-8


@pytest.mark.parametrize("hermitian", [True, False])
@pytest.mark.parametrize("nao", [1, 4, 5, 9, 12, 13, 20, 21, 25, 28, 29, 36, 37, 41, 44, 49, 53, 56, 57, 64])
def test_every_block_count(nao, hermitian):
    _check(*_system(3, nao, 6, hermitian))


@pytest.mark.parametrize("case", [
    dict(nao=30, ns=2), dict(nao=39, ns=2), dict(nao=44, ns=2), dict(nao=52, ns=2), dict(nao=64, ns=2),
    dict(nao=9, nso=18), dict(nao=22, nso=44), dict(nao=31, nso=62), dict(nao=52, nso=104),
])
def test_spin_blocks(case):
    _check(*_system(2, case["nao"], 5, ns=case.get("ns", 1), nso=case.get("nso")))


@pytest.mark.parametrize("case", [
    dict(nao=12), dict(nao=13), dict(nao=16), dict(nao=17), dict(nao=16, ns=2), dict(nao=14, nso=28), dict(nao=24),
    dict(nao=25), dict(nao=32), dict(nao=33), dict(nao=31, ns=2), dict(nao=26, nso=52), dict(nao=41), dict(nao=48),
    dict(nao=45, ns=2), dict(nao=44, nso=88), dict(nao=48, nso=96),
])
def test_wide_blocks(case):
    """The P0 operand on 16-wide blocks at the edges of its sizes, with more auxiliary indices than a work-group takes
    and several q per launch."""
    _check(*_system(2, case["nao"], 19, ns=case.get("ns", 1), nso=case.get("nso")))


@pytest.mark.parametrize("hermitian", [True, False])
@pytest.mark.parametrize("NQ", [63, 64, 65, 128, 129, 200])
def test_half_product_block_edges(NQ, hermitian):
    _check(*_system(2, 3, NQ, hermitian))


def test_maps_without_adjoint_pairs(monkeypatch):
    """k - q rows that are rows of the k + q map, as the store requires, but not their inverses: rows whose
    reversed pair is not the adjoint are read directly."""
    G, V, T, d = _system(4, 5, 7)
    rng = np.random.default_rng(3)
    kp = np.stack([rng.permutation(4) for _ in range(4)]).astype(np.int32)
    km = kp[rng.permutation(4)]
    monkeypatch.setattr(go, "k_add", lambda k, q, mesh, sign: int((kp if sign > 0 else km)[q, k]))
    assert min_eig_I_minus_P0(G, V, T, d) > 0.3
    _check(G, V, T, d, maps=(kp, km))


@pytest.mark.parametrize("hermitian", [True, False])
@pytest.mark.parametrize("nao", [1, 4, 5, 12, 13, 28, 29, 36, 37, 49, 56, 57, 64])
def test_exchange_every_block_count(nao, hermitian):
    dm, V, S, mad = random_system(3, nao, nao, 1, 6, 500 + nao)
    if not hermitian:
        rng = np.random.default_rng(nao)
        dm = dm + 0.1 * (rng.standard_normal(dm.shape) + 1j * rng.standard_normal(dm.shape))
    k = gl.GwHipKernel(3, nao, nao, 1, 6, 4, 3, 10.0, mesh=(3, 1, 1))
    try:
        k.upload_V(V)
        F = k.hf(dm, S, mad)
    finally:
        k.close()
    assert rel_err(F, ho.hf_fock(dm, V, S, mad, 3, nao, nao, 1, 6)) < 1e-10


@pytest.mark.parametrize("hermitian", [True, False])
@pytest.mark.parametrize("nk,nao,NQ", [(8, 2, 16), (9, 3, 130), (10, 2, 129)])
def test_several_q_per_launch(nk, nao, NQ, hermitian):
    """P0 of several q in one launch: all of them at once, and groups with a shorter last one."""
    _check(*_system(nk, nao, NQ, hermitian))
