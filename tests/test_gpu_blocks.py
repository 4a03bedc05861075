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


# central_species counts within the block's own species list: entry 1 of (A, B) and entry 2 of (B, A) are
# the same atoms
@pytest.mark.parametrize("path", ["mixed", "fp64_plain", "fp64_adjoint", "surrogate"])
def test_blocks_on_the_same_atoms_under_another_species_order(path):
    from turbogap_amd import Context
    from turbogap_amd import surrogate as SG
    rng = np.random.default_rng(3)
    sysm = S.binary_system(1500, seed=9)
    blocks = []
    for k, (types, central) in enumerate([((S.SPECIES_A, S.SPECIES_B), 1), ((S.SPECIES_B, S.SPECIES_A), 2)]):
        h = S.soap_hypers(list(types), central_species=central)
        Qs = rng.random((30, h.dim))
        blocks.append((k, h, Qs / np.linalg.norm(Qs, axis=1, keepdims=True), rng.normal(scale=1e-2, size=30)))

    def step(chosen, streams):
        with Context(0) as ctx:
            ctx.set_system(sysm.positions, sysm.species, sysm.box)
            ctx.build_neighbors_list(3.7, fetch=False)
            ctx.set_block_streams(streams)
            for k, h, Qs, al in chosen:
                mid = ctx.soap_model(h, Qs, al)
                if path == "surrogate":
                    for i in range(2):
                        net = SG.MLP(ctx, h.dim, 128, 128, seed=11 + 5 * k + i)
                        net.set_normalization(-0.5, 0.03 + 0.01 * i)
                        net.install(mid, i)
            if path == "surrogate":
                SG.set_gate(ctx, 2, 1e9)
            E, W = ctx.compute(path)
            return (E, W) + ctx.results()

    (Ea, Wa, ea, fa), (Eb, Wb, eb, fb) = [step([b], 1) for b in blocks]
    on_a = sysm.species == S.SPECIES_A
    assert np.all(ea[on_a] != 0.0) and np.all(eb[on_a] != 0.0) and not ea[~on_a].any() and not eb[~on_a].any()
    for streams in (0, 1, 2):
        E, W, e, f = step(blocks, streams)
        # the blocks' energies and pair forces are the same numbers, added in FP64
        assert np.array_equal(e, ea + eb), streams
        assert np.abs(f - (fa + fb)).max() <= 1e-12 * (np.abs(fa).max() + np.abs(fb).max())
        assert abs(E - (Ea + Eb)) <= 1e-12 * (np.abs(ea).sum() + np.abs(eb).sum())
        assert np.abs(W - (Wa + Wb)).max() <= 1e-12 * sysm.n * 3.7 * (np.abs(fa).max() + np.abs(fb).max())


# results pass through pinned memory of up to 2,048 atoms that the context always holds, of a size of their
# own above, grown where a system is larger than any before it, and by a copy above 16,384 atoms
def test_results_of_systems_of_changing_size():
    from turbogap_amd import Context
    rng = np.random.default_rng(1)
    hyp = S.soap_binary()
    Qs = rng.random((5, hyp[0].dim))
    Qs /= np.linalg.norm(Qs, axis=1, keepdims=True)
    al = rng.normal(scale=1e-2, size=5)

    def step(ctx, sysm):
        ctx.set_system(sysm.positions, sysm.species, sysm.box)
        ctx.build_neighbors_list(3.7, fetch=False)
        E, _ = ctx.compute("fp64_adjoint")
        return (E,) + ctx.results() + ctx.get_gap_soap("fp64_adjoint")[:2]

    with Context(0) as one:
        one.soap_backend_begin(one.soap_model(hyp[0], Qs, al))
        for n in (300, 2048, 2049, 40, 2500, 9000, 16384, 16385, 700):
            sysm = S.binary_system(n, seed=n)
            got = step(one, sysm)
            with Context(0) as fresh:
                fresh.soap_backend_begin(fresh.soap_model(hyp[0], Qs, al))
                want = step(fresh, sysm)
            # the same calls on the same numbers: whether the context is new does not matter
            assert all(np.array_equal(a, b) for a, b in zip(got, want)), n
            assert abs(got[0] - got[1].sum()) <= 1e-12 * np.abs(got[1]).sum()


# a block assigns the energies of its centres and the forces of the atoms its pairs reach, and nothing else,
# in one batch and in several
@pytest.mark.parametrize("n,budget", [(400, 0.0), (3000, 0.0), (3000, 0.05)])
def test_get_gap_soap_assigns_what_the_block_touches(n, budget):
    from turbogap_amd import Context
    rng = np.random.default_rng(n)
    sysm = S.binary_system(n, seed=n)
    pos, box = np.vstack([sysm.positions, sysm.box.diagonal() + 20.0]), sysm.box + np.diag([40.0, 40.0, 40.0])
    species = np.append(sysm.species, S.SPECIES_B).astype(np.int32)  # the last atom is alone and no centre
    h = S.soap_binary()[0]
    Qs = rng.random((5, h.dim))
    Qs /= np.linalg.norm(Qs, axis=1, keepdims=True)
    al = rng.normal(scale=1e-2, size=5)
    with Context(0) as ctx:
        ctx.set_system(pos, species, box)
        nl = ctx.build_neighbors_list(3.7)
        ctx.soap_backend_begin(ctx.soap_model(h, Qs, al))
        ctx.set_memory_budget(budget)
        e, f = np.full(n + 1, 7.0), np.full((n + 1, 3), 7.0)
        _, _, w, ns, _ = ctx.get_gap_soap("fp64_plain", energies=e, forces=f)
        e2, f2 = np.full(n + 1, 7.0), np.full((n + 1, 3), 7.0)
        _, _, w2, ns2, _ = ctx.get_gap_soap("fp64_plain", do_forces=False, energies=e2, forces=f2)
        E, W = ctx.compute("fp64_adjoint")
        e3, f3 = ctx.results()
    centre = species == S.SPECIES_A
    reached = np.zeros(n + 1, bool)
    first = np.concatenate([[0], np.cumsum(nl["n_neigh"])])
    for i in np.flatnonzero(centre):
        near = nl["rjs"][first[i]:first[i + 1]] < h.rcut_max
        reached[(nl["neighbors_list"][first[i]:first[i + 1]][near] - 1) % (n + 1)] = True
    assert ns == ns2 == centre.sum() and not reached[n]
    for en in (e, e2):
        assert (en[~centre] == 7.0).all() and np.abs(en - e3)[centre].max() <= 1e-13
    assert (f[~reached] == 7.0).all() and np.abs(f - f3)[reached].max() <= 1e-10 and (f2 == 7.0).all()
    assert np.abs(w - W).max() <= 1e-10 * n and not w2.any()
