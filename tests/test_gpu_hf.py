"""Device Hartree-Fock Fock contribution (gwhip_hf) -- needs an MI355X.

All through the C ABI, against the oracle (oracle/hf_oracle.py, itself pinned by the reference's
HF_X2C fixture and a brute-force einsum in test_hf_oracle.py):
* the HF_X2C fixture of test/solvers_test.cpp:388 (nk = 1, X2C, nao = 10, NQ = 154): the
  reference's 1e-6 and 1e-10 absolute;
* random ns = 1, ns = 2 and X2C systems with a non-zero Madelung constant, up to nk = 27
  (3x3x3), nao = 26, naux = 250: 1e-10 relative (FP64 throughout);
* the device-pointer entry point gives the same F as the host one, and a second call on the
  same handle (scratch reused) gives it again;
* the exchange as batched FP64 GEMMs (tuning key orbital_gemm; always so for nao > 48): against
  the register-chained kernels at small nao, and against the oracle at nao = 50 (ns = 1, X2C).
"""
import os

import numpy as np
import pytest

from gwhip import lib as gl
from helpers import GOLDEN, rel_err
from oracle import hf_oracle as ho
from test_hf_oracle import random_system

pytestmark = pytest.mark.gpu


def _kernel(nk, nao, nso, ns, NQ, mesh=None):
    # the HF entry point uses only the integrals and the k + q maps; any valid tau grid will do
    return gl.GwHipKernel(nk, nao, nso, ns, NQ, 4, 3, 10.0, mesh=mesh)


def test_hf_x2c_fixture():
    z = np.load(os.path.join(GOLDEN, "hf_x2c.npz"), allow_pickle=False)
    nao, nso, ns, NQ, nk = (int(z[k]) for k in ("nao", "nso", "ns", "NQ", "nk"))
    dm = ho.dm_from_G(z["G_beta"], ns, nso != nao)
    k = _kernel(nk, nao, nso, ns, NQ)
    try:
        k.upload_V(z["V"])
        F = k.hf(dm, z["S_k"], float(z["madelung"]))
    finally:
        k.close()
    err = np.abs(F - z["Sigma1"]).max()
    print(f"HF_X2C fixture: max abs err {err:.2e}")
    assert err < 1e-6
    assert err < 1e-10


CASES = [
    dict(nk=3, mesh=(3, 1, 1), nao=3, nso=3, ns=1, NQ=5),
    dict(nk=4, mesh=(2, 2, 1), nao=2, nso=2, ns=2, NQ=4),
    dict(nk=2, mesh=(2, 1, 1), nao=2, nso=4, ns=1, NQ=3),
    dict(nk=8, mesh=(2, 2, 2), nao=17, nso=17, ns=2, NQ=33),
    dict(nk=8, mesh=(2, 2, 2), nao=11, nso=22, ns=1, NQ=40),
    dict(nk=27, mesh=(3, 3, 3), nao=26, nso=26, ns=1, NQ=250),
]


@pytest.mark.parametrize("ci", range(len(CASES)))
def test_hf_random_systems(ci):
    c = CASES[ci]
    dm, Vp, S, mad = random_system(c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"], 100 + ci)
    F_ref = ho.hf_fock(dm, Vp, S, mad, c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"])
    k = _kernel(c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"], mesh=c["mesh"])
    try:
        k.upload_V(Vp)
        F = k.hf(dm, S, mad)
        F0 = k.hf(dm, S, 0.0)
        ms = k.hf_ms()
    finally:
        k.close()
    err = rel_err(F, F_ref)
    err0 = rel_err(F0, ho.hf_fock(dm, Vp, S, 0.0, c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"]))
    print(f"case {c}: rel err {err:.2e} (madelung 0: {err0:.2e}), {ms:.3f} ms")
    assert err < 1e-10 and err0 < 1e-10


def test_hf_device_pointers_and_reuse():
    import torch
    c = dict(nk=8, mesh=(2, 2, 2), nao=11, nso=22, ns=1, NQ=40)
    dm, Vp, S, mad = random_system(c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"], 7)
    k = _kernel(c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"], mesh=c["mesh"])
    try:
        k.upload_V(Vp)
        F_host = k.hf(dm, S, mad)
        d_dm = torch.from_numpy(np.ascontiguousarray(dm)).to("cuda:0")
        d_S = torch.from_numpy(np.ascontiguousarray(S)).to("cuda:0")
        out = []
        for _ in range(2):
            d_F = torch.full_like(d_dm, float("nan"))
            k.hf_device(d_dm.data_ptr(), d_S.data_ptr(), mad, d_F.data_ptr())
            out.append(d_F.cpu().numpy())
    finally:
        k.close()
    for F in out:
        assert np.array_equal(F, F_host)


@pytest.mark.parametrize("c", [
    dict(nk=4, mesh=(2, 2, 1), nao=9, nso=9, ns=2, NQ=21, gemm_only=False),
    dict(nk=2, mesh=(2, 1, 1), nao=7, nso=14, ns=1, NQ=12, gemm_only=False),
    dict(nk=2, mesh=(2, 1, 1), nao=50, nso=50, ns=1, NQ=16, gemm_only=True),
    dict(nk=2, mesh=(2, 1, 1), nao=50, nso=100, ns=1, NQ=6, gemm_only=True),
])
def test_hf_gemm_form(c):
    dm, Vp, S, mad = random_system(c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"], 300 + c["nao"])
    F_ref = ho.hf_fock(dm, Vp, S, mad, c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"])
    k = _kernel(c["nk"], c["nao"], c["nso"], c["ns"], c["NQ"], mesh=c["mesh"])
    try:
        k.upload_V(Vp)
        if not c["gemm_only"]:
            F_kern = k.hf(dm, S, mad)
            k.set_tuning(orbital_gemm=1)
        F = k.hf(dm, S, mad)
    finally:
        k.close()
    print(f"HF GEMM form {c}: rel err {rel_err(F, F_ref):.2e}", flush=True)
    assert rel_err(F, F_ref) < 1e-10
    if not c["gemm_only"]:
        assert rel_err(F, F_kern) < 1e-13


@pytest.mark.parametrize("nao", [49, 64])
def test_exchange_above_48_is_the_gemm_form(nao):
    """By itself above nao = 48, where the exchange kernel is slower: the same bits as with the GEMM form asked for."""
    dm, Vp, S, mad = random_system(3, nao, nao, 1, 6, 700 + nao)
    k = _kernel(3, nao, nao, 1, 6, mesh=(3, 1, 1))
    try:
        k.upload_V(Vp)
        F = k.hf(dm, S, mad)
        k.set_tuning(orbital_gemm=1)
        F_gemm = k.hf(dm, S, mad)
    finally:
        k.close()
    assert np.array_equal(F, F_gemm)


@pytest.mark.parametrize("c", [
    dict(nk=13, nao=45, nso=45, ns=1), dict(nk=14, nao=41, nso=41, ns=2), dict(nk=14, nao=48, nso=48, ns=1),
    dict(nk=14, nao=45, nso=90, ns=1), dict(nk=17, nao=44, nso=44, ns=1),
])
@pytest.mark.parametrize("hermitian", [True, False])
def test_exchange_of_three_blocks(c, hermitian):
    """nao of 41 to 48, where the number of pairs decides between the two exchange kernels."""
    dm, Vp, S, mad = random_system(c["nk"], c["nao"], c["nso"], c["ns"], 3, 800 + c["nk"])
    if not hermitian:
        rng = np.random.default_rng(c["nk"])
        dm = dm + 0.1 * (rng.standard_normal(dm.shape) + 1j * rng.standard_normal(dm.shape))
    k = _kernel(c["nk"], c["nao"], c["nso"], c["ns"], 3, mesh=(c["nk"], 1, 1))
    try:
        k.upload_V(Vp)
        F = k.hf(dm, S, mad)
    finally:
        k.close()
    assert rel_err(F, ho.hf_fock(dm, Vp, S, mad, c["nk"], c["nao"], c["nso"], c["ns"], 3)) < 1e-10


@pytest.mark.parametrize("nao", [3, 5, 9, 13, 17, 21, 28, 29, 33, 37, 40, 41, 48])
@pytest.mark.parametrize("work", [6e6, 8e6])
def test_hermitian_density_matrix(nao, work):
    """On both sides of the work from which on a Hermitian density matrix is looked for, at the block counts of the
    exchange kernel."""
    NQ = int(work / (16.0 * nao ** 3)) + 1
    dm, Vp, S, mad = random_system(2, nao, nao, 1, NQ, 900 + nao)
    dm = 0.5 * (dm + np.conj(np.swapaxes(dm, -1, -2)))
    k = _kernel(2, nao, nao, 1, NQ, mesh=(2, 1, 1))
    try:
        k.upload_V(Vp)
        F = k.hf(dm, S, mad)
    finally:
        k.close()
    assert rel_err(F, ho.hf_fock(dm, Vp, S, mad, 2, nao, nao, 1, NQ)) < 1e-10
