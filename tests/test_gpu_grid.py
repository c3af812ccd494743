"""Transforms whose P-tilde(tau) is not Hermitian: the imaginary parts of T_tb do not cancel over +-Omega.  The
library takes the whole Sigma product for them, and the product of one triangle otherwise (needs an MI355X).

* a batch whose graph was captured with a grid of the one kind follows a grid of the other kind on the same
  pointers, bit for bit as a stand-alone kernel;
* Sigma is that of the oracle, which is not Hermitian there, within 1e-10 in FP64 and 1e-8 in split precision, as
  everywhere, also where the tilt is so small (3e-12) that it changes Sigma by no more than 2e-9."""
import numpy as np
import pytest

from gwhip import lib as gl
from helpers import min_eig_I_minus_P0, rel_err, synthetic
from oracle import gw_oracle as go
from test_gpu_batch import _batch, _make, _standalone

pytestmark = pytest.mark.gpu


class Tilted:
    """T with i rel max|T_tb| added to every element of T_tb (the same at tau and beta - tau)."""

    def __init__(self, T, rel):
        self.nts, self.nw_b, self.T_bt = T.nts, T.nw_b, np.asarray(T.T_bt)
        self.T_tb = np.asarray(T.T_tb) + 1j * rel * np.abs(T.T_tb).max()


@pytest.mark.parametrize("precision", [gl.PREC_FP64, gl.PREC_SPLIT])
def test_batch_follows_a_grid_of_the_other_kind(precision):
    import torch

    systems = _make()
    G, V, T, d = systems[1]
    tilted = Tilted(T, 1e-3)
    ref = [_standalone(*s, precision) for s in systems]
    ref_tilted = _standalone(G, V, tilted, d, precision)
    assert rel_err(ref_tilted, ref[1]) > 1e-6
    G_d = [torch.tensor(s[0], device="cuda:0") for s in systems]
    S_d = [torch.empty_like(g) for g in G_d]
    gp, sp = [g.data_ptr() for g in G_d], [s.data_ptr() for s in S_d]
    b = _batch(systems)
    try:
        torch.cuda.synchronize()
        for grid, want in ((T, ref[1]), (tilted, ref_tilted), (tilted, ref_tilted), (T, ref[1]), (T, ref[1])):
            b.systems[1].set_grid(grid.T_bt, grid.T_tb)
            before = b.stats()["captures"]
            b.eval_device(gp, sp, precision)
            again = b.stats()["captures"]
            b.eval_device(gp, sp, precision)
            assert b.stats()["captures"] == again <= before + 1
            for i, s in enumerate(S_d):
                assert np.array_equal(s.cpu().numpy(), want if i == 1 else ref[i]), i
        assert b.stats()["captures"] <= 3  # a grid of the same kind replays the graph
    finally:
        b.close()


@pytest.mark.parametrize("case", [
    dict(nao=5, NQ=130),                    # several tiles of P-tilde
    dict(nao=5, NQ=40, ns=2),
    dict(nao=4, NQ=30, nso=8),              # X2C
    dict(nao=5, NQ=40, orbital_gemm=1),
])
@pytest.mark.parametrize("rel", [1e-3, 3e-12])
def test_sigma_of_a_tilted_grid(case, rel):
    G, V, T, d = synthetic(2, case["nao"], case["NQ"], ns=case.get("ns", 1), nso=case.get("nso"), beta=20.0, lam=1e3,
                           mesh=(2, 1, 1), seed=31, sigma=0.1)
    assert min_eig_I_minus_P0(G, V, T, d) > 0.5
    T = Tilted(T, rel)
    k = gl.GwHipKernel(d["nk"], d["nao"], d["nso"], d["ns"], d["NQ"], T.nts, T.nw_b, d["beta"], mesh=d["mesh"])
    try:
        k.set_grid(T.T_bt, T.T_tb)
        k.upload_V(V)
        if "orbital_gemm" in case:
            k.set_tuning(orbital_gemm=1)
        S, S_split = k.solve(G), k.solve(G, gl.PREC_SPLIT)
    finally:
        k.close()
    S_ref = go.gw_sigma(G, V, T.T_bt, T.T_tb, d["nk"], d["nao"], d["nso"], d["ns"], d["NQ"], mesh=d["mesh"])
    print(f"{case} tilt {rel}: FP64 {rel_err(S, S_ref):.2e}, split {rel_err(S_split, S_ref):.2e}, Sigma - Sigma^H "
          f"{rel_err(S_ref, np.conj(np.swapaxes(S_ref, -1, -2))):.2e}", flush=True)
    assert rel_err(S, S_ref) < 1e-10
    assert rel_err(S_split, S_ref) < 1e-8
