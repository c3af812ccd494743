"""The register-resident inverses at the edges of their sizes, against the oracle (needs an MI355X).

* Dyson step: nso around every change of the lane group (16, 32, 64 lanes), of the register count (multiples
  of 4) and of the kernel (48 / 49), with one matrix more or less than a wave holds; the diagonal of
  mu S - H is zero, so that the elimination has to exchange rows;
* the pivot blocks of I - P0: naux around one and two blocks of 64 and their 16-column parts.

Within 1e-10 relative, as the FP64 results everywhere."""
import numpy as np
import pytest

from helpers import rel_err
from oracle import dyson as od
from test_gpu_dyson import _dyson, _fixture, _random
from test_gpu_orbital import _check, _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nso", [1, 2, 3, 4, 5, 15, 16, 17, 20, 26, 31, 32, 33, 36, 37, 45, 48, 49])
@pytest.mark.parametrize("ink", [1, 3])
def test_dyson_sizes(nso, ink):
    _, T, wn = _fixture()
    H, S, S1, St = _random(1, ink, nso, nso, 11 + nso, T.nts)
    i = np.arange(nso)
    H[..., i, i] = 0.1 * S[..., i, i]
    d = _dyson(T, wn, 1, ink, ink, nso, nso)
    try:
        d.set_system(H, S, None)
        G = d.compute_G(S1, St, 0.1)
        N = d.number_of_electrons(S1, St, 0.1)
    finally:
        d.close()
    G_or = od.compute_G(H, S, S1, St, 0.1, T.T_ft, T.T_tf, wn)
    e = od.eigenspectra(H, S, S1, St, T.T_ft)
    N_or = od.number_of_electrons(0.1, e, wn, T.T_tf, [1.0] * ink, ink, 1, X2C=False)
    print(f"nso {nso} ink {ink}: G {rel_err(G, G_or):.2e}, N {N:.12f} vs {N_or:.12f}", flush=True)
    assert rel_err(G, G_or) < 1e-10
    assert abs(N - N_or) < 1e-9 * max(1.0, abs(N_or))


@pytest.mark.parametrize("NQ", [1, 15, 16, 17, 33, 63, 64, 65, 80, 81, 127, 128, 130])
def test_pivot_blocks(NQ):
    _check(*_system(2, 4, NQ))
