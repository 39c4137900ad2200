"""The sparse plan's fill at the edges of its dispatch: Fock pairs with few and
many elements (whole and factored contraction), configurations with more
excited clusters than a factored element may have and cluster sizes without
a factored shape, each with its bra blocks cut into eight parts (spaces of
fewer than 1,024 Fock blocks); and larger spaces in four, two and one.

Oracle: the C restatement of tps_ci_matvec / compute_diagonal; bar 1e-12 of
the largest element in FP64, as for the other sparse tests.
"""
import numpy as np
import pytest

from fermicg_amd.cluster_ops import add_cmf_operators, compute_cluster_eigenbasis, compute_cluster_ops
from fermicg_amd.cluster_ops import product_state_rdm1
from fermicg_amd.integrals import synthetic_ints
from fermicg_amd.marshal import flatten_ham, flatten_ops
from fermicg_amd.operator import extract_ClusteredTerms
from fermicg_amd.state import TPSCIstate, fock_configs_within
from fermicg_amd.tpsci import Engine, cluster_sizes_of
from fermicg_amd.workloads import build_problem, rank1_space
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


def _space(sizes, M, transfer, keep, seed):
    """Clusters of the given sizes at half filling; a seeded share of each Fock
    block's configurations, never all of them."""
    n = sum(sizes)
    clusters, at = [], 0
    for s in sizes:
        clusters.append(list(range(at, at + s)))
        at += s
    ref = tuple((s // 2, s // 2) for s in sizes)
    ints = synthetic_ints(n, 2 * n, seed)
    bases = compute_cluster_eigenbasis(ints, clusters, max_roots=M)
    ops = compute_cluster_ops(bases, ints)
    add_cmf_operators(ops, bases, ints, *product_state_rdm1(bases, n, ref))
    full = TPSCIstate.full_blocks(bases, fock_configs_within(bases, ref, transfer))
    rng = np.random.Generator(np.random.PCG64(seed))
    blocks = []
    for fi, a, b in full.blocks():
        k = min(max(1, int(keep * (b - a))), b - a - 1, 250) if b - a > 1 else 1
        idx = np.sort(rng.choice(np.arange(a, b), k, replace=False))
        blocks.append((full.focks()[fi], [tuple(int(x) for x in full.cfg[i]) for i in idx]))
    return ops, extract_ClusteredTerms(ints, clusters), TPSCIstate.from_blocks(len(sizes), blocks)


def _check(ops, ham, st, label):
    c = np.random.Generator(np.random.PCG64(1)).normal(size=(len(st), 2))
    st.set_vector(c)
    print(label, st.n_fock, len(st), int(np.diff(st.fock_start).max()), flush=True)
    orc = Oracle(flatten_ops(ops, cluster_sizes_of(ops)), flatten_ham(ham), st)
    ref = orc.sigma(c)
    pl = Engine(0).tpsci_plan(st, ops, ham)
    assert np.abs(pl.sigma(c) - ref).max() < 1e-12 * np.abs(ref).max()
    hd = orc.diagonal()
    assert np.abs(pl.diagonal() - hd).max() < 1e-12 * np.abs(hd).max()


@pytest.mark.parametrize("sizes,M,transfer,keep", [
    ((4, 4, 4, 4), 3, 2, 0.6), ((4, 4, 4, 4), 4, 1, 0.9), ((4, 4, 4, 4, 4), 2, 2, 0.5),
    ((4, 4, 4), 9, 2, 0.4), ((2, 4, 3, 4), 3, 2, 0.7), ((4, 4), 12, 2, 0.8),
    ((4, 4, 4, 4, 4), 2, 2, 0.03)])
def test_sparse_fill(sizes, M, transfer, keep):
    ops, ham, st = _space(sizes, M, transfer, keep, seed=len(sizes) + M)
    _check(ops, ham, st, sizes)


@pytest.mark.parametrize("clusters,M,frac,blocks", [(6, 6, 0.3, (1024, 2048)), (7, 5, 0.2, (2048, 4096)),
                                                    (8, 4, 0.2, (4096, 8192))])
def test_sparse_fill_in_parts(clusters, M, frac, blocks):
    """Fock block counts of four, two and one parts, of up to 18 configurations."""
    p = build_problem(4 * clusters, clusters, M, 8 * clusters, seed=clusters, max_transfer=2)
    st = rank1_space(p, R=2, frac=frac, seed=2)
    assert blocks[0] <= st.n_fock < blocks[1]
    _check(p.cluster_ops, p.clustered_ham, st, clusters)
