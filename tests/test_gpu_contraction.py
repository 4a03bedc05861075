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


# By 128 x 128 tiles of the kernel product (14 columns of 1,700 sparse points, 2 of 130) the rows are on
# both sides of the lines between K-split (below 96 tiles), 64-row and 128-row workgroups (from 512):
# 14, 28, 74, 84, 98, 208, 238, 518, integer and other zeta on each; of the Qss product (3 columns of D = 324,
# 10 of D = 1,224) between K-split (below 48), 64 x 64 and 128 x 128 (from 1,024): 3, 6, 18, 21, 51, 111, 1,040.
# One row and the widest descriptor among them.
@pytest.mark.parametrize("n,n_max,n_sparse,zeta", [(1, 8, 1700, 4.0), (129, 8, 1700, 2.5), (768, 8, 1700, 4.0),
                                                   (769, 8, 1700, 4.0), (2049, 8, 1700, 4.0), (2049, 8, 1700, 2.5),
                                                   (4640, 8, 130, 1.0), (4700, 8, 1700, 4.0), (4700, 8, 1700, 2.5),
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


def test_qss_tiles_beside_another_block():
    """540 tiles of the Qss product: 128 x 128 ones where the two blocks run at once, 64 x 64 ones in turn.
    Both add an element's products in the same order."""
    from turbogap_amd import Context
    rng = np.random.default_rng(2)
    sysm = S.binary_system(13700, seed=5)
    with Context(0) as c:
        c.set_system(sysm.positions, sysm.species, sysm.box)
        c.build_neighbors_list(3.7, fetch=False)
        for h in S.soap_binary():
            Qs = rng.random((200, h.dim))
            c.soap_model(h, Qs / np.linalg.norm(Qs, axis=1, keepdims=True), rng.normal(scale=1e-2, size=200))
        out = []
        for streams in (0, 1):
            c.set_block_streams(streams)
            out.append(c.compute("fp64_adjoint") + c.results())
    assert all(np.array_equal(a, b) for a, b in zip(*out)) and np.abs(out[0][3]).max() > 0.0
