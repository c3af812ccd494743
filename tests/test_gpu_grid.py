"""Transforms whose P-tilde(tau) is not Hermitian: the imaginary parts of T_tb do not cancel over +-Omega.  The
library takes the whole Sigma product for them, and the product of one triangle otherwise (needs an MI355X).

* a batch whose graph was captured with a grid of the one kind follows a grid of the other kind on the same
  pointers, bit for bit as a stand-alone kernel."""
import numpy as np
import pytest

from gwhip import lib as gl
from helpers import rel_err
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
