"""The sparse PT2's ket batches and bound weights at their edges: Fock blocks of
one, some, 64 and 125 kets (the dense engine takes no larger slices), and
one to three roots.

Reference: the dense-target engine on the same state, unscreened.  Bar 1e-10
of e2: both sum at most 1e6 contributions per root in FP64, each of them
rounded to 1e-16 of the largest.
"""
import numpy as np
import pytest

from fermicg_amd.state import TPSCIstate
from fermicg_amd.tpsci import Engine, compute_pt2_energy, orthonormalize
from fermicg_amd.workloads import build_problem

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
