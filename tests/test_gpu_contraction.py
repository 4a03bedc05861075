"""FP64 contraction (energies and Qss through get_soap_energy_and_forces) at the sizes where its
GEMMs change tile: numpy in FP64 is the reference."""
import numpy as np
import pytest

from turbogap_amd import structures as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from turbogap_amd import Context
    with Context(0) as c:
        yield c


# rows either side of the lines between the K-split, 64-row, 64 x 64 and 128 x 128 tiles (D = 324:
# 3 column tiles of Qss; 1,700 sparse points: 14 of K), one row, and the widest descriptor
@pytest.mark.parametrize("n,n_max,n_sparse,zeta", [(1, 8, 1700, 4.0), (129, 8, 1700, 2.5), (768, 8, 1700, 4.0),
                                                   (769, 8, 1700, 4.0), (2049, 8, 1700, 4.0), (4640, 8, 130, 1.0),
                                                   (13185, 16, 130, 2.0)])
def test_contraction_tiles(ctx, n, n_max, n_sparse, zeta):
    h = S.soap_hypers([S.CARBON], n_max=n_max)
    h.zeta = zeta
    rng = np.random.default_rng(n)
    D = h.dim
    q = rng.random((n, D)) ** 4
    q /= np.linalg.norm(q, axis=1)[:, None]
    Qs = rng.random((n_sparse, D)) ** 4
    Qs /= np.linalg.norm(Qs, axis=1)[:, None]
    al = rng.normal(size=n_sparse)
    der = rng.normal(size=(n, D, 3))
    ctx.set_system(np.zeros((1, 3)), np.full(1, S.CARBON, np.int32), S.cubic_box(20.0))
    mid = ctx.soap_model(h, Qs, al)
    ctx.soap_backend_begin(mid)
    # one entry per centre: its own atom, so the force on it is Qss . dq/dr
    E, F, _ = ctx.get_soap_energy_and_forces(q, der, np.ones(n, np.int32), np.arange(1, n + 1), np.zeros((n, 3)), n)
    ctx.soap_backend_end()
    K = q @ Qs.T
    Eo = (K ** zeta) @ al
    Qss = -zeta * (K ** (zeta - 1.0) * al) @ Qs
    Fo = np.einsum("id,idk->ik", Qss, der)
    # worst-case rounding: zeta D products inside K^zeta, n_sparse and D in the sums; |K|, |Qs| <= 1
    eps = 2.0 ** -53
    bound = np.abs(al).sum() * eps
    assert np.abs(E - Eo).max() <= 2 * (zeta * D + n_sparse + 8) * bound
    assert np.abs(F - Fo).max() <= 2 * zeta * (zeta * D + n_sparse + D + 8) * bound * np.linalg.norm(der, axis=1).max()
