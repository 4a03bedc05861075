"""Selection and scans of all blocks in shared launches: more blocks than one launch takes, several
blocks on the same centres, and atom counts on both sides of the scan's borders."""
import numpy as np
import pytest

from turbogap_amd import structures as S

pytestmark = pytest.mark.gpu


# one workgroup a scan up to 8,192 atoms, two launches up to 65,536, three above
@pytest.mark.parametrize("n", [40, 8192, 8193, 65537])
def test_many_blocks_match_two(n):
    from turbogap_amd import Context
    rng = np.random.default_rng(n)
    sysm = S.binary_system(n, seed=7)
    hyp = S.soap_binary()
    Qs = [rng.random((6, h.dim)) for h in hyp]
    Qs = [q / np.linalg.norm(q, axis=1, keepdims=True) for q in Qs]
    al = [rng.normal(scale=1e-2, size=6) for _ in hyp]
    res = []
    for copies in ((1, 1), (6, 5)):  # 11 blocks: the alphas shared out over the copies
        with Context(0) as ctx:
            ctx.set_system(sysm.positions, sysm.species, sysm.box)
            ctx.build_neighbors_list(3.7, fetch=False)
            for k in range(max(copies)):
                for h, q, a, c in zip(hyp, Qs, al, copies):
                    if k < c:
                        ctx.soap_model(h, q, a / c)
            E, W = ctx.compute("fp64_adjoint")
            e, f = ctx.results()
            E2, W2 = ctx.compute("fp64_adjoint")
            e2, f2 = ctx.results()
            assert E2 == E and np.array_equal(W2, W)
            assert np.array_equal(e2, e) and np.array_equal(f2, f)
            res.append((E, W, e, f))
    (E0, W0, e0, f0), (E1, W1, e1, f1) = res
    # an atom's energy is 6 terms |alpha k| of some 1e-2 each, shared out and summed again in at most 32
    # roundings (kernel values with q.q_s <= 1); forces and sums over atoms the same, relative to their terms
    assert np.abs(e1 - e0).max() <= 32 * 2.0 ** -53 * 6 * 1e-2 * 6
    assert np.abs(f1 - f0).max() <= 1e-12 * np.abs(f0).max()
    assert abs(E1 - E0) <= 1e-12 * np.abs(e0).sum()
    assert np.abs(W1 - W0).max() <= 1e-12 * n * np.abs(f0).max() * 3.7
