"""The matrix-free sigma where its stages have edges: clusters of up to 36
states (w_ij in several tiles), sectors of one state, fewer and more than 64
connected ket blocks and 32 terms per pair, and root counts around a launch's
four.

Oracle: the C restatement of tps_ci_matvec / compute_diagonal.  Bars as in the
other matrix-free tests, relative to the largest element: FP64 1e-12, FP32
1e-5, diagonal 1e-12.
"""
import numpy as np
import pytest

from fermicg_amd.marshal import flatten_ham, flatten_ops
from fermicg_amd.state import TPSCIstate
from fermicg_amd.tpsci import Engine, cluster_sizes_of
from fermicg_amd.workloads import build_problem, rank1_space
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("clusters,M,transfer,frac,R", [(2, 36, 2, 1.0, 1), (3, 36, 1, 1.0, 4),
                                                        (3, 1, 2, 1.0, 2), (3, 2, 2, 0.5, 5),
                                                        (4, 33, 1, 0.2, 3), (7, 3, 1, 1.0, 1)])
def test_matrix_free_edges(clusters, M, transfer, frac, R):
    p = build_problem(4 * clusters, clusters, M, 8 * clusters, seed=M, max_transfer=transfer)
    st = (rank1_space(p, R=R, frac=frac, seed=M) if M > 1  # one state: only ground configurations
          else TPSCIstate.full_blocks(p.bases, p.focks, R=R))
    st.set_vector(np.random.Generator(np.random.PCG64(R)).normal(size=(len(st), R)))
    print(clusters, M, transfer, len(st), flush=True)
    eng = Engine(0)
    pl = eng.tpsci_plan(st, p.cluster_ops, p.clustered_ham, precisions=("fp64", "fp32"),
                        matrix_free=True)
    orc = Oracle(flatten_ops(p.cluster_ops, cluster_sizes_of(p.cluster_ops)),
                 flatten_ham(p.clustered_ham), st)
    ref = orc.sigma(st.coeffs)
    scale = np.abs(ref).max()
    assert np.abs(pl.sigma(st.coeffs) - ref).max() < 1e-12 * scale
    assert np.abs(pl.sigma(st.coeffs, "fp32") - ref).max() < 1e-5 * scale
    hd = orc.diagonal()
    assert np.abs(pl.diagonal() - hd).max() < 1e-12 * np.abs(hd).max()
