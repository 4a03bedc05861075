"""dq/dr of the FP64 plain path where the pairs of a centre fill less than one, one or several of the
32-pair chunks they are prepared in, and a chunk's last group and rows only in part."""
import numpy as np
import pytest

from turbogap_amd import structures as S

pytestmark = pytest.mark.gpu


# atoms in a box of 8 A, i.e. 212 / 512 of them within the cutoff: 0, ~3, ~30, ~50 and ~75 pairs a centre
@pytest.mark.parametrize("n,species,n_max", [(1, 1, 8), (8, 1, 8), (75, 2, 8), (76, 2, 3), (120, 1, 7), (180, 2, 8)])
def test_derivatives_match_oracle(ctx, orc, n, species, n_max):
    rng = np.random.default_rng(n)
    pos = S.rsa(n, 8.0, 0.9, 3 * n)
    codes = [S.SPECIES_A, S.SPECIES_B][:species]
    sp = np.array(codes, np.int32)[rng.integers(0, species, n)]
    ctx.set_system(pos, sp, S.cubic_box(8.0))
    nl = ctx.build_neighbors_list(3.7)
    if n == 180:
        assert nl["n_neigh"].max() > 1 + 64
    h = S.soap_hypers(codes, central_species=0, n_max=n_max)
    mid = ctx.soap_model(h, np.zeros((1, h.dim)), np.zeros(1))
    ctx.soap_backend_begin(mid)
    q, der = ctx.get_soap(derivatives=True)
    ctx.soap_backend_end()
    spi = orc.species_index(nl["neighbor_species"], h.species_types)
    qo, dero = orc.get_soap(h, nl["n_neigh"], spi, nl["rjs"], nl["xyz"], derivatives=True)
    # as at the ordinary density: 1e-12 in q; derivatives to 1e-11 of the largest, a self entry sums
    # up to 80 others
    np.testing.assert_allclose(q, qo, rtol=0, atol=1e-12)
    np.testing.assert_allclose(der, dero, rtol=0, atol=1e-11 * max(1.0, np.abs(dero).max()))


@pytest.mark.parametrize("n,species,n_max", [(8, 1, 8), (75, 2, 8), (76, 2, 3), (120, 1, 7), (180, 2, 8)])
def test_adjoint_matches_plain(ctx, n, species, n_max):
    rng = np.random.default_rng(n)
    codes = [S.SPECIES_A, S.SPECIES_B][:species]
    sp = np.array(codes, np.int32)[rng.integers(0, species, n)]
    ctx.set_system(S.rsa(n, 8.0, 0.9, 3 * n), sp, S.cubic_box(8.0))
    ctx.build_neighbors_list(3.7, fetch=False)
    h = S.soap_hypers(codes, central_species=0, n_max=n_max)
    Qs = rng.random((40, h.dim))
    ctx.soap_model(h, Qs / np.linalg.norm(Qs, axis=1, keepdims=True), rng.normal(scale=1e-2, size=40))
    Ep, Wp = ctx.compute("fp64_plain")
    ep, fp = ctx.results()
    Ea, Wa = ctx.compute("fp64_adjoint")
    ea, fa = ctx.results()
    # the same sums in another order: up to 1,224 components by 80 pairs of one sign at most, 2^-53 each
    tol = 1e-12 * max(1.0, np.abs(fp).max())
    assert np.abs(ea - ep).max() <= 1e-13 and abs(Ea - Ep) <= 1e-13 * n
    assert np.abs(fa - fp).max() <= tol
    assert np.abs(Wa - Wp).max() <= tol * n * 3.7
