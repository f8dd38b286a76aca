"""The kernels that work on batches of primitive quartets, at the edges of their batches and tiles,
against the oracle: contractions longer than a batch, uneven contractions in one class, sizes around
the 64 x 64 tiles of the density-fitting products, blocks in every order of their shells.

Tolerances: FP64 sums of at most a few thousand terms in another order, 1e-12 relative with a floor
of 1e-13 of the largest element (the other parity tests'); the gradient 1e-10 relative as in
test_jk_grad."""
import numpy as np
import pytest

from lible_amd import basis as B

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lbx():
    from lible_amd import lbx as L
    L.lib()
    return L


@pytest.fixture(scope="module")
def oracle():
    from oracle import oracle as O
    return O


def close(gpu, ref, rel=1e-12, floor=1e-13):
    gpu, ref = np.asarray(gpu), np.asarray(ref)
    err, tol = np.abs(gpu - ref), rel * np.abs(ref) + floor * np.abs(ref).max()
    assert (err <= tol).all(), f"{(err > tol).sum()} of {ref.size}, worst {(err / np.maximum(tol, 1e-300)).max():.2f} tol"


def uneven_molecule(seed, contractions):
    """Two atoms 1.6 bohr apart; contractions: [(l, K), ...] on the first, reversed on the second."""
    rng = np.random.default_rng(seed)
    per_atom = []
    for order in (1, -1):
        per_atom.append([(l, list(np.exp(rng.uniform(np.log(0.2), np.log(40.0), K))), list(rng.uniform(0.1, 1.0, K)))
                         for l, K in contractions[::order]])
    coords = np.array([[0.0, 0.1, -0.2], [0.9, 0.8, 1.1]])
    return B.Molecule(coords, B.Shells.from_lists(per_atom))


CLASS_PAIRS = [(la, lb, lc, ld) for la in range(4) for lb in range(la + 1) for lc in range(4) for ld in range(lc + 1)
               if la * (la + 1) // 2 + lb >= lc * (lc + 1) // 2 + ld]

# class pairs whose one-lane number (0, 1; FP32 3, 4) runs the one-wave form: at most three column passes,
# or seven of at least three columns, and 5500 FMAs are built as one-lane forms
STAND_IN = {
    0: "2111 2121 2211 2220 3021 3022 3030 3111 3120", 1: "2211 3021 3130 3211 3220 3310",
    3: "2222 3022 3122 3131 3211 3221 3222 3230 3231 3311 3320",
    4: "2220 3120 3122 3130 3210 3211 3220 3221 3222 3230 3231 3310 3311 3320 3321 3330"}
STAND_IN = {v: [tuple(map(int, c)) for c in cs.split()] for v, cs in STAND_IN.items()}


def profiled(ctx, lbx, D, fp32):
    """The kernel of each class pair of one J/K build: the FP64 ones, or with every quartet in FP32."""
    ctx.profile(True)
    ctx.jk(D, schwarz=0.0, **(dict(precision=lbx.LBX_MIXED, mixed_thresh=1e30) if fp32 else {}))
    out = {p["class"]: p["kernel"] for p in ctx.profile_read() if p["quartets"] > 0}
    ctx.profile(False)
    return out


def fix_variant(ctx, lbx, variant):
    """Fixes a variant wherever it is accepted; returns the class pairs that run it themselves."""
    used = [c for c in CLASS_PAIRS if ctx.set_variant(c, variant)]
    assert len(used) == {0: 31, 1: 30, 3: 48, 4: 42}.get(variant, 55)
    return [c for c in used if c not in STAND_IN.get(variant, [])]


# (l, K) lists: K_ab up to 121 (s, s), 81 (p, p) and 25 (f, d), beyond every batch (64 primitive
# quartets at low L, 3 at (ff|ff)), next to single primitives
UNEVEN = [[(0, 11), (0, 1), (1, 2)], [(1, 9), (0, 2), (2, 1)], [(2, 5), (1, 1), (3, 1), (0, 1)],
          [(3, 5), (2, 5), (0, 1), (1, 1)]]


@pytest.mark.parametrize("contractions", UNEVEN)
@pytest.mark.parametrize("variant", [None, 2, 6])
def test_jk_uneven_contractions(lbx, oracle, contractions, variant):
    import torch
    m = uneven_molecule(5, contractions)
    D = B.density_from_orbitals(3, m.shells.nbf, 3, 0.3)
    Jr, Kr, _ = oracle.Structure(m).jk(D, thresh=0.0)
    ctx = lbx.Context(m)
    if variant is not None:
        assert fix_variant(ctx, lbx, variant) == CLASS_PAIRS
        kernels = profiled(ctx, lbx, torch.tensor(D, device="cuda"), False)
        assert kernels and set(kernels.values()) == {lbx.VARIANTS[variant]}
    J, K, _ = ctx.jk(torch.tensor(D, device="cuda"), schwarz=0.0)
    close(J.cpu().numpy(), Jr)
    close(K.cpu().numpy(), Kr)


def test_jk_graph_replays_with_parts_of_J(lbx):
    """Replays of a build whose J is made in parts (420 functions) after the density's contents changed,
    against eager builds: the order of atomic additions, 1e-12 of the largest element."""
    import torch
    m = B.synthetic_molecule(79, 14, 9.0, B.RECIPE_MAIN)
    ctx, eager = lbx.Context(m), lbx.Context(m)
    ctx.set_graphs(True)
    D = torch.empty((ctx.nbf, ctx.nbf), dtype=torch.float64, device="cuda")
    J, K = torch.empty_like(D), torch.empty_like(D)
    for seed in range(4):
        D.copy_(torch.tensor(B.density_from_orbitals(seed, ctx.nbf, 20, 0.1)))
        ctx.jk(D, schwarz=1e-10, J=J, K=K)
        Je, Ke, _ = eager.jk(D, schwarz=1e-10)
        close(J.cpu().numpy(), Je.cpu().numpy(), rel=0.0, floor=1e-12)
        close(K.cpu().numpy(), Ke.cpu().numpy(), rel=0.0, floor=1e-12)


@pytest.mark.parametrize("contractions", UNEVEN)
def test_jk_grad_uneven_contractions(lbx, oracle, contractions):
    import torch
    m = uneven_molecule(6, contractions)
    D = B.density_from_orbitals(4, m.shells.nbf, 3, 0.3)
    ref = oracle.Structure(m).jk_grad(D, thresh=0.0)
    g, _ = lbx.Context(m).jk_grad(torch.tensor(D, device="cuda"), schwarz=0.0)
    close(g.cpu().numpy(), ref, rel=1e-10, floor=1e-10)


@pytest.mark.parametrize("contractions", [[(2, 5), (3, 2)], [(2, 9)], [(3, 4), (2, 1), (3, 1)]])
def test_jk_grad_fp32_sums(lbx, contractions):
    """The FP32 tier sums over primitives in FP64 (class pairs of d and f shells: the one-wave form):
    every primitive listed twice with half its coefficient is the same function, its E matrices scale
    by exact powers of two, and the gradients differ by the rounding of FP64 sums of up to 1e6 terms
    that cancel to about a tenth: 1e-11 of the largest component (FP32 sums: 1e-8 and more).  Against
    FP64: R and E rounded to FP32, about 20 roundings of 6e-8 per term: 1e-5 of the largest component."""
    import torch
    m = uneven_molecule(7, contractions)

    def doubled(exps, coeffs, nprim):
        e, c, at = [], [], 0
        for k in nprim:
            e += [np.tile(exps[at:at + k], 2)]
            c += [np.tile(0.5 * coeffs[at:at + k], 2)]
            at += k
        return np.concatenate(e), np.concatenate(c)

    sh = m.shells
    e2, c2 = doubled(sh.exps, sh.coeffs, sh.nprim)
    m2 = B.Molecule(m.coords, B.Shells(sh.atom, sh.l, 2 * sh.nprim, e2, c2))
    D = torch.tensor(B.density_from_orbitals(4, m.shells.nbf, 3, 0.3), device="cuda")
    mixed = dict(schwarz=0.0, precision=lbx.LBX_MIXED, mixed_thresh=1e30)
    ref, _ = lbx.Context(m).jk_grad(D, schwarz=0.0)
    g, st = lbx.Context(m).jk_grad(D, **mixed)
    g2, _ = lbx.Context(m2).jk_grad(D, **mixed)
    assert st["quartets_fp32"] == st["quartets"]
    close(g2.cpu().numpy(), g.cpu().numpy(), rel=0.0, floor=1e-11)
    close(g.cpu().numpy(), ref.cpu().numpy(), rel=0.0, floor=1e-5)


@pytest.mark.parametrize("natoms", [1, 3, 16])
def test_dense_uneven(lbx, oracle, natoms):
    """Dense eri4 / diagonal of 1 to 16 one-shell atoms (the largest has more pairs than lanes)."""
    rng = np.random.default_rng(natoms)
    per_atom = [[(k % 2, list(rng.uniform(0.3, 3.0, 1 + k % 3)), list(rng.uniform(0.2, 1.0, 1 + k % 3)))]
                for k in range(natoms)]
    m = B.Molecule(B.random_atoms(rng, natoms, 5.0, 0.8), B.Shells.from_lists(per_atom))
    s, ctx = oracle.Structure(m), lbx.Context(m)
    for _ in range(2):   # the second call reuses the task tables
        close(ctx.eri4().cpu().numpy(), s.eri4(), floor=1e-14)
        close(ctx.eri4_diag().cpu().numpy(), s.eri4_diag(), floor=1e-14)


@pytest.fixture(scope="module")
def block_case(oracle):
    m = B.synthetic_molecule(77, 2, 3.0, B.RECIPE_MAIN)
    return m, oracle.Structure(m).eri4()


@pytest.mark.parametrize("perm", [(0, 1, 2, 3), (1, 0, 2, 3), (0, 1, 3, 2), (2, 3, 0, 1), (3, 2, 1, 0)])
@pytest.mark.parametrize("ls", [(3, 1, 2, 0), (0, 0, 3, 2), (1, 1, 1, 1), (2, 0, 2, 2)])
def test_eri4_block_orders(lbx, block_case, ls, perm):
    """Blocks of shells in the caller's order, the side with the higher class first or last."""
    m, e4 = block_case
    off = np.concatenate([[0], np.cumsum(2 * m.shells.l + 1)])
    rng = np.random.default_rng(8)
    shells = np.stack([rng.choice(np.flatnonzero(m.shells.l == ls[p]), 67) for p in perm], 1).astype(np.int32)
    got = lbx.Context(m).blocks(shells).cpu().numpy()[:, 0]
    ref = np.stack([e4[tuple(slice(off[s], off[s + 1]) for s in q)] for q in shells])
    close(got, ref, floor=1e-13 * np.abs(e4).max() / np.abs(ref).max())


def ri_line_molecule(nmain, naux):
    """s shells spread over a line, a well-conditioned auxiliary set."""
    rng = np.random.default_rng(nmain)
    nat = max(nmain, naux)
    coords = np.stack([1.5 * np.arange(nat), rng.uniform(0, 1, nat), rng.uniform(0, 1, nat)], 1)
    main = B.Shells.from_lists([[(0, [0.8], [1.0])] if k < nmain else [] for k in range(nat)])
    aux = B.Shells.from_lists([[(0, [1.1], [1.0])] if k < naux else [] for k in range(nat)])
    return B.Molecule(coords, main, aux)


@pytest.mark.parametrize("nmain,naux", [(1, 1), (5, 3), (63, 7), (64, 2), (65, 9), (130, 5)])
def test_ri_jk_sizes(lbx, oracle, nmain, naux):
    """Density-fitted J and K at sizes around the 64 x 64 tiles and 16-step k loop, against numpy on
    the library's own eri3 / eri2 (pinned to the oracle elsewhere): 1e-11 of the
    largest element."""
    import torch
    from scipy.linalg import cho_solve, solve_triangular
    ctx = lbx.Context(ri_line_molecule(nmain, naux))
    e3, e2 = ctx.eri3().cpu().numpy(), ctx.eri2().cpu().numpy()
    D = B.density_from_orbitals(2, nmain, 4, 0.3)
    L = np.linalg.cholesky(e2)
    Jr = e3 @ cho_solve((L, True), np.einsum("mnp,mn->p", e3, D))
    W = solve_triangular(L, e3.reshape(nmain * nmain, naux).T, lower=True).reshape(naux, nmain, nmain)
    Kr = np.einsum("pmn,nl,pkl->mk", W, D, W, optimize=True)
    for _ in range(2):
        J, K = ctx.ri_jk(torch.tensor(D, device="cuda"))
        close(J.cpu().numpy(), Jr, rel=0.0, floor=1e-11)
        close(K.cpu().numpy(), Kr, rel=0.0, floor=1e-11)
    J, _ = ctx.ri_jk(torch.tensor(D, device="cuda"), exchange=False)
    close(J.cpu().numpy(), Jr, rel=0.0, floor=1e-11)


@pytest.mark.parametrize("nmain,naux", [(5, 3), (65, 9), (130, 5)])
def test_ri_jk_density_not_symmetric(lbx, nmain, naux):
    """J and K of a density that is not symmetric (all of it, or one element of it), in both triangles;
    tolerance as above."""
    import torch
    from scipy.linalg import solve_triangular
    ctx = lbx.Context(ri_line_molecule(nmain, naux))
    e3, e2 = ctx.eri3().cpu().numpy(), ctx.eri2().cpu().numpy()
    W = solve_triangular(np.linalg.cholesky(e2), e3.reshape(nmain * nmain, naux).T, lower=True).reshape(naux, nmain, nmain)
    one = B.density_from_orbitals(2, nmain, 4, 0.3)
    one[0, nmain - 1] += 0.5
    for D in (np.random.default_rng(3).normal(size=(nmain, nmain)), one):
        Jr = np.einsum("pmn,p->mn", W, np.einsum("pmn,mn->p", W, D))
        Kr = np.einsum("pmn,nl,pkl->mk", W, D, W, optimize=True)
        J, K = ctx.ri_jk(torch.tensor(D, device="cuda"))
        close(J.cpu().numpy(), Jr, rel=0.0, floor=1e-11)
        close(K.cpu().numpy(), Kr, rel=0.0, floor=1e-11)


@pytest.mark.parametrize("nmain,naux", [(30, 56), (65, 200), (180, 90)])
def test_ri_jk_repeats(lbx, nmain, naux):
    """The same density gives the same bits again (K and J are added up from parts in a fixed order)."""
    import torch
    ctx = lbx.Context(ri_line_molecule(nmain, naux))
    D = torch.tensor(B.density_from_orbitals(2, nmain, 4, 0.3), device="cuda")
    J, K = ctx.ri_jk(D)
    Jo, _ = ctx.ri_jk(D, exchange=False)
    for _ in range(5):
        J2, K2 = ctx.ri_jk(D)
        assert torch.equal(J, J2) and torch.equal(K, K2)
        assert torch.equal(Jo, ctx.ri_jk(D, exchange=False)[0])


@pytest.mark.parametrize("variant", range(8))
def test_profile_names_the_form_that_ran(lbx, variant):
    """With a variant fixed wherever it is accepted, the profile reports that form, or the one-wave form
    where the number stands for it."""
    import torch
    m = B.synthetic_molecule(81, 3, 4.5, B.RECIPE_MAIN)
    D = torch.tensor(B.density_from_orbitals(3, m.shells.nbf, 6, 0.2), device="cuda")
    ctx = lbx.Context(m)
    own = fix_variant(ctx, lbx, variant)
    kernels = profiled(ctx, lbx, D, variant in (3, 4, 5, 7))
    assert all(kernels[c] == lbx.VARIANTS[variant] for c in own)
    assert all(kernels[c] == lbx.VARIANTS[5 if variant > 2 else 2] for c in STAND_IN.get(variant, []))


def test_tune_times_each_form_once(lbx):
    """The tuner's choice is a form that the class pair has, never a one-lane number that stands for the
    one-wave form."""
    import torch
    m = B.synthetic_molecule(81, 3, 4.5, B.RECIPE_MAIN)
    D = torch.tensor(B.density_from_orbitals(3, m.shells.nbf, 6, 0.2), device="cuda")
    for fp32, variants in ((False, (0, 1)), (True, (3, 4))):
        ctx = lbx.Context(m)
        ctx.tune(D)
        kernels = profiled(ctx, lbx, D, fp32)
        assert len(kernels) == 55
        for v in variants:
            assert not [c for c in STAND_IN[v] if kernels[c] == lbx.VARIANTS[v]]


def until_it_fits(ctx, call, lbx):
    """call() under a memory limit raised in steps of a tenth until it goes through -> its result and
    the number of calls that ran out of memory."""
    limit, refused = 1 << 10, 0
    while True:
        ctx.set_memory_limit(limit)
        try:
            return call(), refused, limit
        except lbx.LbxError as e:
            assert "lbx error -3" in str(e)
            refused += 1
            limit = limit * 11 // 10


@pytest.mark.parametrize("what", ["jk", "grad", "one_electron_grad", "ri_jk", "sums"])
def test_calls_after_running_out_of_memory(lbx, what):
    """A call that ran out of memory leaves a context on which a later one gives the results of a fresh
    context.  Tolerances: the order of atomic additions (1e-12), FP32 tiers the same kernels (the mixed
    sums under the limit run FP64 ones: test_sums_without_room_for_copies)."""
    import torch
    mixed = dict(precision=lbx.LBX_MIXED, mixed_thresh=1e-2)
    m = B.synthetic_molecule(78, 2, 3.0, B.RECIPE_MAIN, B.RECIPE_AUX)
    D = torch.tensor(B.density_from_orbitals(3, m.shells.nbf, 6, 0.2), device="cuda")
    charges = np.column_stack([m.coords, [6.0, 7.0]])
    calls = {"jk": lambda c: c.jk(D, schwarz=0.0, **mixed)[:2], "grad": lambda c: c.jk_grad(D, schwarz=0.0, **mixed)[:1],
             "one_electron_grad": lambda c: c.one_electron_grad(D, D, charges), "ri_jk": lambda c: c.ri_jk(D),
             "sums": lambda c: c.ri_sums(**mixed)[:1]}
    make = lambda: lbx.Context.batch([m, m]) if what == "sums" else lbx.Context(m)
    ref = calls[what](make())
    ctx = make()
    got, refused, _ = until_it_fits(ctx, lambda: calls[what](ctx), lbx)
    assert refused > 10
    ctx.set_memory_limit(0)
    for out in [calls[what](ctx)] + ([got] if what != "sums" else []):
        for a, b in zip(out, ref):
            close(a.cpu().numpy(), b.cpu().numpy(), rel=0.0, floor=1e-12)


@pytest.mark.parametrize("variant", [0, 3])
@pytest.mark.parametrize("graphs", [False, True])
def test_jk_without_room_for_copies(lbx, variant, graphs):
    """A J/K build under the least memory limit that it goes through with: without the one-lane kernels'
    copies of E and the parts of J (420 functions) it runs the one-wave forms with one J, at no more
    memory than a context that is told to.  FP64: the order of the sums, 1e-12 of the largest element;
    FP32 tier 1e-5 (the other parity tests')."""
    import torch
    m = B.synthetic_molecule(79, 14, 9.0, B.RECIPE_MAIN)
    D = torch.tensor(B.density_from_orbitals(3, m.shells.nbf, 20, 0.1), device="cuda")
    mixed = dict(precision=lbx.LBX_MIXED, mixed_thresh=1e30) if variant == 3 else {}
    J, K = torch.empty_like(D), torch.empty_like(D)
    run = lambda c: c.jk(D, schwarz=1e-10, J=J, K=K, **mixed)[:2]
    wave = lbx.Context(m)
    fix_variant(wave, lbx, 5 if variant == 3 else 2)
    ref = [x.clone() for x in run(wave)]
    wave = lbx.Context(m)
    fix_variant(wave, lbx, 5 if variant == 3 else 2)
    _, _, least = until_it_fits(wave, lambda: run(wave), lbx)
    ctx = lbx.Context(m)
    fix_variant(ctx, lbx, variant)
    ctx.set_graphs(graphs)
    _, _, limit = until_it_fits(ctx, lambda: run(ctx), lbx)
    assert limit <= least * 1.25 + (2 << 20)   # the lane orders
    for unbounded in (False, False, False, True, True):
        if unbounded:
            ctx.set_memory_limit(0)
            ctx.set_graphs(False)
        for got, want in zip(run(ctx), ref):
            close(got.cpu().numpy(), want.cpu().numpy(), rel=0.0, floor=1e-5 if variant == 3 else 1e-12)


@pytest.mark.parametrize("mixed", [False, True])
def test_sums_without_room_for_copies(lbx, mixed):
    """RI sums under the least memory limit against the unbounded ones: without the copies of E the
    triplets that had an FP32 one-lane form run in FP64.  1e-12 (FP64), 1e-6 of the largest sum."""
    mols = [B.synthetic_molecule(80 + k, 3, 4.5, B.RECIPE_MAIN, B.RECIPE_AUX) for k in range(3)]
    kw = dict(precision=lbx.LBX_MIXED, mixed_thresh=1e-2) if mixed else {}
    ref, sr = lbx.Context.batch(mols).ri_sums(**kw)
    ctx = lbx.Context.batch(mols)
    (got, st), refused, _ = until_it_fits(ctx, lambda: ctx.ri_sums(**kw), lbx)
    assert refused > 0 and st["triplets"] == sr["triplets"]
    assert st["triplets_fp32"] < sr["triplets_fp32"] or not mixed
    close(got.cpu().numpy(), ref.cpu().numpy(), rel=0.0, floor=1e-6 if mixed else 1e-12)


def test_copies_freed_before_a_call_fails(lbx):
    """A call that cannot have its memory (the fitted tensor of 1000 functions and 60000 auxiliary ones,
    480 GB) frees the parts of J (14 of 8 MB) before it fails, and J and K are the same without them."""
    import torch
    rng = np.random.default_rng(5)
    nat = 1000
    coords = np.stack([1.5 * np.arange(nat), rng.uniform(0, 1, nat), rng.uniform(0, 1, nat)], 1)
    main = B.Shells.from_lists([[(0, [0.8], [1.0])] for _ in range(nat)])
    aux = B.Shells.from_lists([[(0, [float(e)], [1.0]) for e in rng.uniform(0.5, 4.0, 60)] for _ in range(nat)])
    ctx = lbx.Context(B.Molecule(coords, main, aux))
    D = torch.tensor(B.density_from_orbitals(3, nat, 20, 0.1), device="cuda")
    J, K, _ = ctx.jk(D)
    free = torch.cuda.mem_get_info()[0]
    with pytest.raises(lbx.LbxError, match="lbx error -3"):
        ctx.ri_jk(D, exchange=False)
    assert torch.cuda.mem_get_info()[0] - free >= 100 << 20
    J2, K2, _ = ctx.jk(D)
    close(J2.cpu().numpy(), J.cpu().numpy(), rel=0.0, floor=1e-12)
    close(K2.cpu().numpy(), K.cpu().numpy(), rel=0.0, floor=1e-12)


@pytest.mark.parametrize("ns", [14, 15, 16, 19, 23])
@pytest.mark.parametrize("variant", [0, 1, 3, 4])
def test_jk_one_lane_pair_counts(lbx, oracle, ns, variant):
    """One-lane J/K at pair counts around those where K rows move to LDS (more than two 64-pair
    blocks: 105, 120 | 136, 190, 276 (ss) pairs), the last blocks of a group past the end, uneven
    contractions among a block's lanes.  FP32 forms: 1e-5 of the largest element (the other parity
    tests')."""
    import torch
    rng = np.random.default_rng(ns)
    per_atom = [[(0, list(rng.uniform(0.2, 4.0, 1 + k % 4)), list(rng.uniform(0.2, 1.0, 1 + k % 4)))] for k in range(ns)]
    for l in (1, 2, 3):
        per_atom[l].append((l, [0.7, 1.3], [0.6, 0.5]))
    m = B.Molecule(B.random_atoms(rng, ns, 5.0, 0.8), B.Shells.from_lists(per_atom))
    D = B.density_from_orbitals(9, m.shells.nbf, 3, 0.3)
    Jr, Kr, _ = oracle.Structure(m).jk(D, thresh=1e-10)
    ctx = lbx.Context(m)
    own = fix_variant(ctx, lbx, variant)
    kernels = profiled(ctx, lbx, torch.tensor(D, device="cuda"), variant >= 3)
    # (ss) pairs on the lanes, more and fewer than 128 of them, against every uniform side
    assert ((1, 0, 0, 0) if variant in (1, 4) else (0, 0, 0, 0)) in own
    assert all(kernels[c] == lbx.VARIANTS[variant] for c in own)
    mixed = dict(precision=lbx.LBX_MIXED, mixed_thresh=1e9) if variant >= 3 else {}
    for _ in range(2):
        J, K, _ = ctx.jk(torch.tensor(D, device="cuda"), schwarz=1e-10, **mixed)
        for got, ref in ((J, Jr), (K, Kr)):
            close(got.cpu().numpy(), ref, **(dict(rel=0.0, floor=1e-5) if variant >= 3 else dict(floor=1e-12)))
