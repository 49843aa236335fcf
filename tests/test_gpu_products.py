"""The product kernels at the edges of their tiles: block ranks around the
four rows of a phase-1 task and the sixteen of its matrix-core form, blocks
narrower than one load group, partly filled near-field tiles and 64-row
chunks."""
import numpy as np
import pytest

from helpers import sphere_problem, upload_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("leaf,maxrank", [(5, 1), (5, 0), (23, 4), (23, 5), (67, 16), (67, 17), (90, 0)])
def test_products_equal_stored_operator(bem, O, meshes, leaf, maxrank, prec):
    """Y = H X against the dense product of the stored operator for 1, 2, 4
    and 8 columns, VALU and matrix cores, plain and accumulating: FP64
    round-off of sums of at most n + rank terms."""
    P = sphere_problem(O, meshes, level=2 if leaf < 30 else 3, leaf=leaf, eta=2.0, freq=400.0)
    ctx = upload_problem(bem, P)
    G = ctx.assemble(1, 1e-9 if maxrank else 1e-5, maxrank, precision=prec, seed=3)
    full = G.to_full()
    ranks = [G.rank(b) for b in range(len(P.blocks)) if P.blocks[b][4]]
    print("leaf", leaf, "maxrank", maxrank, "prec", prec, "ranks", min(ranks), max(ranks), flush=True)
    assert maxrank == 0 or max(ranks) == maxrank
    rng = np.random.default_rng(7)
    for q in (1, 2, 4, 8):
        X = rng.standard_normal((P.n, q)) + 1j * rng.standard_normal((P.n, q))
        ref = full @ X
        for mf in (True, False):
            ctx.set_mfma(mf)
            Y = G.mvm_multi(X)
            for k in range(q):
                assert np.linalg.norm(Y[:, k] - ref[:, k]) < 1e-13 * np.linalg.norm(ref[:, k]), (q, mf, k)
    x, y0 = X[:, 0], X[:, 1]
    y = G.mvm(x, y0, accumulate=True)
    assert np.linalg.norm(y - y0 - full @ x) < 1e-13 * np.linalg.norm(full @ x) + 1e-15 * np.linalg.norm(y0)
    G.close()
    ctx.close()
