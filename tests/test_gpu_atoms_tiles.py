"""The GPU atom expansion at the edges of its tiles against the oracle: one atom,
atoms around a wavefront's 256 and a chunk's 1024, one q, q around a tile's 16 and
a block's 48, expansion orders with one, four and five column tiles (L = 0, 9, 10)
and the largest order (L = 40), and arguments q r up to 75, whose Bessel
series have more terms than the reciprocal table.  The bar is that of the parity
test of the expansion: only the order of the sums over atoms differs (1e-12 of
the largest value)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F():
    import libfmftsaxs_amd as F
    if F.device_count() < 1:
        pytest.fail("no HIP device visible")
    return F


@pytest.mark.parametrize("L,natoms,Q,qmax", [(1, 1, 1, 0.3), (9, 255, 16, 0.5), (10, 257, 17, 0.5),
                                             (4, 1024, 48, 0.5), (5, 1025, 49, 0.5),
                                             (40, 60, 5, 0.5), (3, 120, 7, 8.0)])
def test_tile_edges_vs_oracle(F, L, natoms, Q, qmax):
    from libfmftsaxs_amd import synthetic as S
    rec = S.random_chain(natoms, 23)
    xyz = rec.coords - rec.coords.mean(axis=0) + np.array([1.0, 0.5, 0.25])
    sa = np.linspace(0.0, 40.0, natoms)
    q = np.linspace(0.0, qmax, Q) if Q > 1 else np.array([qmax])
    print(f"L={L} {natoms} atoms, {Q} q up to {qmax}", flush=True)
    rg, ig, rmg = F.atoms2spf(xyz, rec.vac, rec.dum, sa, rec.vdw, q, L)
    ro, io, rmo = O.atoms2spf(xyz, rec.vac, rec.dum, sa, rec.vdw, q, L)
    assert rmg == rmo
    scale = np.maximum(np.abs(ro).max(axis=2, keepdims=True), np.abs(io).max(axis=2, keepdims=True))
    assert np.all(np.abs(rg - ro) <= 1e-12 * scale)
    assert np.all(np.abs(ig - io) <= 1e-12 * scale)
