"""Blocks whose ACA runs over several workgroups (m + n above 1024 on these
meshes): factors, ranks and evaluation counts bit-identical to the CPU
restatement in FP64, and the batched, multi-mesh and single launches
bit-identical to each other in both precisions."""
import numpy as np
import pytest

from helpers import sphere_problem, upload_problem

pytestmark = pytest.mark.gpu
WIDE = 1024


def same(x, y):
    return np.array_equal(np.ascontiguousarray(x).view(np.uint64), np.ascontiguousarray(y).view(np.uint64))


def capsule_problem(O, meshes, edge, freq, impedance=0.3, plane=None):
    """capsule with a lined patchwork (columns of both boundary-condition
    forms in one block), ragged block sizes"""
    tri = meshes.capsule(2.0, 0.25, edge)
    bc = meshes.impedance_bc(len(tri), 2 * np.pi * freq / 343.0, impedance, 4)
    P = O.Problem(tri, bc, leaf=32, eta=2.0)
    P.set_frequency(freq, 343.0, 1)
    if plane is not None:
        P.set_plane(*plane)
    wide = [b for b in range(len(P.blocks)) if P.blocks[b][4] and P.blocks[b][1] + P.blocks[b][3] > WIDE]
    assert wide, "no block is large enough"
    return P, wide


@pytest.mark.parametrize("edge,tol,maxrank,plane", [
    (0.055, 1e-4, 0, None),
    (0.055, 1e-9, 0, None),       # ranks beyond the first capacity: run again with the full one
    (0.055, 1e-9, 7, None),       # stopped by the rank limit
    (0.061, 1e-5, 0, (np.array([0.0, 0.0, -1.5]), np.array([0.0, 0.0, 1.0]))),
])
def test_wide_blocks_bit_exact(bem, O, meshes, edge, tol, maxrank, plane):
    P, wide = capsule_problem(O, meshes, edge, 800.0, plane=plane)
    ctx = upload_problem(bem, P)
    if plane is not None:
        ctx.set_plane(*plane)
        prm = P.params()
        ctx.set_frequency(prm["k"], prm["cc"])
    for kind in (0, 1):
        H = P.assemble(kind, tol, maxrank, 5)
        G = ctx.assemble(kind, tol, maxrank, seed=5)
        ranks = [H.rank(b) for b in wide]
        print("wide blocks", len(wide), "kind", kind, "tol", tol, "ranks", min(ranks), max(ranks), flush=True)
        for b in wide:
            assert G.rank(b) == H.rank(b), (kind, b)
            for x, y in zip(G.block(b), H.block(b)):
                assert same(x, y), (kind, b)
        assert G.stats()["evaluated"] == H.evaluated
        G.close()
    ctx.close()


def test_wide_launch_forms_agree(bem, O, meshes):
    freqs = [600.0, 800.0]
    P, wide = capsule_problem(O, meshes, 0.055, freqs[0], impedance=0.0)
    Q, wide2 = capsule_problem(O, meshes, 0.061, 700.0)
    ctx, ctx2 = upload_problem(bem, P), upload_problem(bem, Q)
    kcc = []
    for f in freqs:
        P.set_frequency(f, 343.0, 1)
        prm = P.params()
        kcc.append([prm["k"], prm["cc"].real, prm["cc"].imag])
    for prec in (bem.FP64, bem.FP32):
        for kind in (0, 1):
            batch = ctx.assemble_batch(kind, kcc, 1e-4, precision=prec, seed=3)
            for f in range(len(freqs)):
                ctx.set_frequency(kcc[f][0], complex(kcc[f][1], kcc[f][2]))
                single = ctx.assemble(kind, 1e-4, precision=prec, seed=3)
                assert batch[f].stats()["evaluated"] == single.stats()["evaluated"]
                assert all(same(x, y) for b in wide for x, y in zip(batch[f].block(b), single.block(b)))
                batch[f].close()
                if f == len(freqs) - 1:
                    multi = bem.assemble_multi([ctx, ctx2], kind, 1e-4, precision=prec, seed=3)
                    other = ctx2.assemble(kind, 1e-4, precision=prec, seed=3)
                    assert all(same(x, y) for b in wide for x, y in zip(multi[0].block(b), single.block(b)))
                    assert all(same(x, y) for b in wide2 for x, y in zip(multi[1].block(b), other.block(b)))
                    for h in (*multi, other):
                        h.close()
                single.close()
    ctx.close()
    ctx2.close()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("level", [1, 2, 3])
def test_class_bounds_keep_factors(bem, O, meshes, level, prec):
    """The bounds that depend on the launch's total (no schedule set) give the
    factors of the fixed schedules, to the bit: small bound at, below and
    above the blocks' extents, the largest class empty and not."""
    P = sphere_problem(O, meshes, level=level, leaf=12, eta=2.0, freq=400.0)
    adm = [b for b in range(len(P.blocks)) if P.blocks[b][4]]
    ctx = upload_problem(bem, P)
    for kind in (0, 1):
        ref = ctx.assemble(kind, 1e-6, 0, precision=prec, seed=5)
        other = upload_problem(bem, P)
        for small, huge in ((0, 0), (64, 96), (384, 2048), (385, 2048)):
            other.set_aca_schedule(prec, small, huge)
            G = other.assemble(kind, 1e-6, 0, precision=prec, seed=5)
            for b in adm:
                assert all(same(x, y) for x, y in zip(G.block(b), ref.block(b))), (kind, small, huge, b)
            G.close()
        ref.close()
        other.close()
    ctx.close()


@pytest.mark.parametrize("far,near,tol,maxrank", [(1500, 500, 1e-5, 0), (4000, 300, 1e-8, 0), (1500, 500, 1e-5, 3),
                                                  (300, 900, 1e-5, 0)])
def test_field_chains_side_by_side(bem, O, meshes, far, near, tol, maxrank):
    """Both field operators' wide blocks at once, against the restatement (its
    ranks and counts; 1e-12 for products summed in another order) and, to the
    bit, against a repeated call."""
    P = sphere_problem(O, meshes, level=4, leaf=32, eta=2.0, freq=700.0)
    ctx = upload_problem(bem, P)
    rng = np.random.default_rng(3)
    phi, dphi = (rng.standard_normal(P.n) + 1j * rng.standard_normal(P.n) for _ in range(2))
    d = rng.standard_normal((near, 3))
    obs = np.concatenate([rng.uniform(0.9, 2.0, near)[:, None] * d / np.linalg.norm(d, axis=1)[:, None],
                          rng.uniform(-1, 1, (far, 3)) + [0, 0, 6.0]])   # a far cluster: a large admissible block
    perm, b5 = P.field_partition(obs, leaf=50, eta=3.0)
    mn = (b5[:, 1] + b5[:, 3])[b5[:, 4] != 0]
    print("field points", len(obs), "largest", mn.max(), flush=True)
    assert mn.max() > WIDE and mn.sum() < 800 * WIDE
    x = ctx.array(phi), ctx.array(dphi)
    ctx.profile(1)
    runs = [ctx.field_hmat(obs[perm], b5, *x, tol, maxrank=maxrank, seed=7)]
    # launches of the profile: both operators' size classes (the bounds of an
    # FP64 launch with this total) and both wide chains, in each pass
    small = max(64, min(384, mn.sum() // 3200))
    classes = int((mn <= small).any()) + int(((mn > small) & (mn <= WIDE)).any()) + 1
    launches = int(ctx.profile(0)[7 + 2])
    print("size classes", classes, "launches", launches, flush=True)
    assert launches == 2 * classes or (maxrank == 0 and launches > 2 * classes)
    runs.append(ctx.field_hmat(obs[perm], b5, *x, tol, maxrank=maxrank, seed=7))
    got = np.empty_like(runs[0][0])
    got[perm] = runs[0][0]
    ref, (nadm, maxr, ev) = P.field_hmat(obs, phi, dphi, tol, maxrank=maxrank, seed=7, leaf=50, eta=3.0)
    st = runs[0][1]
    assert int(st[1]) == nadm and int(st[2]) == maxr and int(st[3]) == ev, (st, nadm, maxr, ev)
    assert np.linalg.norm(got - ref) < 1e-12 * np.linalg.norm(ref)
    assert same(runs[0][0], runs[1][0])
    ctx.close()


def ulps(x):
    return int(np.float64(x).view(np.int64))


def flip_tolerance(rank, lo, hi):
    """adjacent tolerances t0 < t1 with rank(t0) = rank(lo) > rank(t1), by bisection"""
    r0, a, b = rank(lo), ulps(lo), ulps(hi)
    assert rank(hi) < r0
    while b - a > 1:
        mid = (a + b) // 2
        if rank(np.int64(mid).view(np.float64)) < r0:
            b = mid
        else:
            a = mid
    return float(np.int64(a).view(np.float64)), float(np.int64(b).view(np.float64))


@pytest.mark.parametrize("kind", [0, 1])
def test_stopping_rule_in_every_launch_form(bem, O, meshes, kind):
    """The bound above which a block runs over several workgroups depends on
    the launch's total: blocks of m + n from 1024 to 3500 run so in a single
    assembly and in one workgroup in a batch of 16.  At tolerances where the stopping
    rule of such a block turns from one representable number to the next, so
    that the last bit of its norm estimate decides, both forms give the same
    ranks and evaluation counts, and the restatement's."""
    P, wide = capsule_problem(O, meshes, 0.055, 800.0, impedance=0.0)
    nf = 16
    mn = P.blocks[:, 1] + P.blocks[:, 3]
    total = int(mn[P.blocks[:, 4] != 0].sum())
    assert total < 800 * WIDE < nf * total   # one bound at its least, the other above it
    both = [b for b in wide if mn[b] <= min(4096, nf * total // 800)]
    ctx = upload_problem(bem, P)
    prm = P.params()
    kcc = np.array([[prm["k"], prm["cc"].real, prm["cc"].imag]] * nf)

    def single(tol, b):
        G = ctx.assemble(kind, tol, seed=5)
        r = G.rank(b)
        G.close()
        return r

    tested = 0
    for lo in (1e-6, 2e-5):
        for b in both:
            if single(1e-3, b) >= single(lo, b):
                continue
            for t in flip_tolerance(lambda x: single(x, b), lo, 1e-3):
                G = ctx.assemble(kind, t, seed=5)
                batch = ctx.assemble_batch(kind, kcc, t, seed=5)
                rs = [G.rank(w) for w in wide]
                rb = [[H.rank(w) for w in wide] for H in batch]
                ev = [H.stats()["evaluated"] for H in (G, *batch)]
                if tested == 0:
                    # blocks above the first capacity of one workgroup: their
                    # second pass, a shorter list, has the lower bound
                    assert all(H.stats()["overflow_blocks"] > 0 for H in batch) and max(rs) > 48
                    assert all(same(x, y) for w in wide for x, y in zip(G.block(w), batch[-1].block(w)))
                for H in (G, *batch):
                    H.close()
                print("kind", kind, "block", b, "m+n", mn[b], "tol", t, "ranks", rs, rb[0], ev[:2], flush=True)
                assert all(r == rs for r in rb) and len(set(ev)) == 1, (b, t)
                if tested < 2:
                    H = P.assemble(kind, t, 0, 5)
                    assert [H.rank(w) for w in wide] == rs and H.evaluated == ev[0], (b, t)
            tested += 1
    assert tested >= 8, tested
    ctx.close()
