"""The sparse PT2's ket batches at their edges: Fock blocks of one, some, 64
and 125 kets (the dense engine takes no larger slices), and one to three
roots; and its bound weights, at thresholds that discard most contributions:
two to four clusters of 2 to 4 orbitals, whose terms have up to 68 weights and so
sixteen down to two lanes each.  A weight summed short drops contributions
that the threshold keeps.

Reference: the dense-target engine on the same state and threshold.  Bar 1e-10
of e2: both sum at most 1e6 contributions per root in FP64, each of them
rounded to 1e-16 of the largest.
"""
import numpy as np
import pytest

from fermicg_amd.state import TPSCIstate
from fermicg_amd.tpsci import Engine, compute_pt2_energy, orthonormalize
from fermicg_amd.workloads import build_problem
from tests.test_gpu_sparse_fill import _space

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("clusters,M,transfer,R", [(3, 1, 2, 1), (3, 2, 1, 2), (3, 4, 1, 1),
                                                   (3, 5, 1, 3)])
def test_pt2_sparse_equals_dense(clusters, M, transfer, R):
    p = build_problem(4 * clusters, clusters, M, 8 * clusters, seed=M, max_transfer=transfer)
    st = TPSCIstate.full_blocks(p.bases, p.focks, R=R)
    rng = np.random.Generator(np.random.PCG64(M))
    st.set_vector(orthonormalize(rng.normal(size=(len(st), R))))
    eng = Engine(0)
    e = {m: compute_pt2_energy(st, p.cluster_ops, p.clustered_ham, thresh_foi=0.0, verbose=0,
                               method=m, engine=eng) for m in ("dense", "sparse")}
    print(clusters, M, len(st), int(np.diff(st.fock_start).max()), e, flush=True)
    assert np.abs(e["sparse"] - e["dense"]).max() < 1e-10 * np.abs(e["dense"]).max()


@pytest.mark.parametrize("sizes,M,R,thresh", [((4, 4, 4, 4), 3, 2, 1e-3), ((4, 4, 4, 4), 2, 1, 1e-2),
                                              ((2, 4, 3, 4), 3, 1, 3e-3), ((4, 3, 4), 3, 3, 1e-3),
                                              ((4, 4, 4), 4, 2, 1e-2), ((3, 4), 6, 1, 1e-3)])
def test_screened_pt2_equals_dense(sizes, M, R, thresh):
    ops, ham, st = _space(sizes, M, 1, 0.7, seed=len(sizes) + M)
    rng = np.random.Generator(np.random.PCG64(M))
    # amplitudes over four decades, so that the bounds cut at every size
    c = rng.normal(size=(len(st), R)) * 10.0 ** -rng.uniform(0, 4, size=(len(st), 1))
    s = TPSCIstate(st.N, R)
    s.fock, s.fock_start, s.cfg = st.fock, st.fock_start, st.cfg
    s.set_vector(orthonormalize(c))
    eng = Engine(0)
    kw = dict(verbose=0, engine=eng)
    d = compute_pt2_energy(s, ops, ham, thresh_foi=thresh, method="dense", **kw)
    e = compute_pt2_energy(s, ops, ham, thresh_foi=thresh, method="sparse", **kw)
    kept = compute_pt2_energy.last_stats["n_contributions"]
    compute_pt2_energy(s, ops, ham, thresh_foi=0.0, method="sparse", **kw)
    share = kept / compute_pt2_energy.last_stats["n_contributions"]
    print(sizes, M, len(s), "kept %.3f" % share, d, flush=True)
    assert 0.005 < share < 0.3
    assert np.abs(e - d).max() < 1e-10 * np.abs(d).max()
    eng.drop_plans()
