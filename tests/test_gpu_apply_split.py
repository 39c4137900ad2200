"""The sigma apply where panels and rows are shared between wavefronts: boxes
of 1 to 64 rows (dimensions that do and do not divide a wavefront), column
counts that leave the last wavefronts little or nothing, and every root count
with its own compiled form.

Oracle: the C restatements of tps_ci_matvec and build_sigma!.  Bars as for the
other sigma tests, relative to the largest element: FP64 1e-12, FP32 and split
BF16 1e-5 and 1e-4, BF16 and a bf16 c 1e-2 (2e-3 per rounded factor).
"""
import numpy as np
import pytest
import torch

from fermicg_amd import _lib
from fermicg_amd.bst import bst_pq_state, cache_hamiltonian
from fermicg_amd.marshal import flatten_ham, flatten_ops
from fermicg_amd.state import TPSCIstate
from fermicg_amd.tpsci import Engine, cluster_sizes_of
from fermicg_amd.workloads import build_problem, rank1_space
from oracle.pyoracle import BstOracle, Oracle

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5, "bf16x2": 1e-4, "bf16": 1e-2, "fp32_bf16c": 1e-2}


@pytest.fixture(scope="module")
def eng():
    return Engine(0)


def _check(plan, ref, c, label):
    for prec, tol in TOL.items():
        s = plan.sigma(c, prec)
        err = np.abs(s - ref).max() / np.abs(ref).max()
        print(label, prec, "%.2e" % err, flush=True)
        assert err < tol


@pytest.mark.parametrize("clusters,M,transfer,R", [(2, 3, 1, 1), (2, 7, 2, 3), (3, 3, 2, 2),
                                                   (3, 4, 1, 4), (3, 5, 2, 1), (3, 4, 2, 5),
                                                   (3, 4, 2, 16)])
def test_full_blocks(eng, clusters, M, transfer, R):
    p = build_problem(4 * clusters, clusters, M, 8 * clusters, seed=M, max_transfer=transfer)
    st = TPSCIstate.full_blocks(p.bases, p.focks, R=R)
    c = np.random.Generator(np.random.PCG64(R)).normal(size=(len(st), R))
    st.set_vector(c)
    ref = Oracle(flatten_ops(p.cluster_ops, cluster_sizes_of(p.cluster_ops)),
                 flatten_ham(p.clustered_ham), st).sigma(c)
    plan = eng.tpsci_plan(st, p.cluster_ops, p.clustered_ham, precisions=tuple(TOL))
    _check(plan, ref, c, (clusters, M, transfer, R))
    eng.drop_plans()


@pytest.mark.parametrize("clusters,M,rank,R", [(2, 6, 5, 1), (3, 9, 8, 2), (3, 7, 6, 4), (3, 5, 3, 7)])
def test_tucker_boxes(eng, clusters, M, rank, R):
    p = build_problem(4 * clusters, clusters, M, 8 * clusters, seed=M, max_transfer=2)
    st = bst_pq_state(p.bases, p.focks, p.ref_fock, max_rank=rank, R=R, seed=rank)
    ref = BstOracle(flatten_ops(p.cluster_ops, cluster_sizes_of(p.cluster_ops)),
                    flatten_ham(p.clustered_ham), st).sigma_rows(st.coeffs,
                                                                np.arange(len(st.blocks)))[0]
    plan = cache_hamiltonian(st, st, p.cluster_ops, p.clustered_ham, precisions=tuple(TOL),
                             engine=eng)
    _check(plan, ref, st.coeffs, (clusters, M, rank, R))
    eng.drop_plans()


@pytest.mark.parametrize("clusters,M,rank,R", [(3, 5, 2, 1), (3, 8, 4, 2), (3, 12, 6, 4), (2, 3, 1, 3),
                                               (3, 8, 4, 6), (3, 12, 6, 5), (3, 9, 7, 12)])
def test_shared_and_unshared_panels(eng, clusters, M, rank, R):
    """Panels of a few to 60,000 elements through every form of the multi-row
    apply, the ones that share a panel and the ones that do not: the same
    bits (up to four roots; above, the one the rule takes), and the oracle's
    sigma."""
    p = build_problem(4 * clusters, clusters, M, 8 * clusters, seed=M, max_transfer=2)
    st = bst_pq_state(p.bases, p.focks, p.ref_fock, max_rank=rank, R=R, seed=rank)
    ref = BstOracle(flatten_ops(p.cluster_ops, cluster_sizes_of(p.cluster_ops)),
                    flatten_ham(p.clustered_ham), st).sigma_rows(st.coeffs,
                                                                np.arange(len(st.blocks)))[0]
    plan = cache_hamiltonian(st, st, p.cluster_ops, p.clustered_ham, precisions=tuple(TOL),
                             engine=eng)
    nm, nr, max_r = _lib.apply_variant_counts()
    _check(plan, ref, st.coeffs, (clusters, M, rank, R))
    for prec in TOL if R <= max_r else ():
        got = []
        for v in range(nm):
            plan.set_apply_variant(prec, R, v, 0)
            got.append(plan.sigma(st.coeffs, prec))
        assert all(np.array_equal(g, got[0]) for g in got), prec
    eng.drop_plans()


@pytest.mark.parametrize("R", [1, 2, 5, 9, 16])
def test_row_sums_do_not_depend_on_the_number_of_rows(eng, R):
    """One-row boxes below and above the count (2,048) from which a wavefront
    takes a row alone: a row's sigma has the same bits in a bra space of 2,449
    rows and in one of a few Fock blocks of it."""
    p = build_problem(12, 3, 13, 24, seed=3, max_transfer=2)
    ket = rank1_space(p, R=R, frac=1.0, seed=2)
    assert len(ket) >= 2048
    c = np.random.Generator(np.random.PCG64(R)).normal(size=(len(ket), R))
    ham, ops = eng.ham(p.clustered_ham), eng.ops(p.cluster_ops)
    dket = _lib.DeviceSpace.tpsci(eng.ctx, ket)
    whole = _lib.Plan.create_pair(eng.ctx, ham, ops, _lib.DeviceSpace.tpsci(eng.ctx, ket), dket).sigma(c)
    few = TPSCIstate(ket.N, R)
    few.fock, few.fock_start = ket.fock[:9], ket.fock_start[:10]
    few.cfg = ket.cfg[:few.fock_start[-1]]
    few.coeffs = np.zeros((len(few.cfg), R))
    part = _lib.Plan.create_pair(eng.ctx, ham, ops, _lib.DeviceSpace.tpsci(eng.ctx, few), dket).sigma(c)
    print(len(ket), len(few), flush=True)
    assert np.array_equal(part, whole[:len(few)])
    ref = Oracle(flatten_ops(p.cluster_ops, cluster_sizes_of(p.cluster_ops)),
                 flatten_ham(p.clustered_ham), ket).sigma(c)
    assert np.abs(whole - ref).max() < 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("shift", [0, 1, 5])
def test_sigma_over_its_vector(eng, shift):
    """sigma_device with sigma over c, or overlapping it, gives what separate
    buffers give (one FP64 vector, the case that is applied without a copy)."""
    p = build_problem(12, 3, 4, 24, seed=4, max_transfer=1)
    st = TPSCIstate.full_blocks(p.bases, p.focks, R=1)
    n = len(st)
    c = np.random.Generator(np.random.PCG64(1)).normal(size=(n, 1))
    plan = eng.tpsci_plan(st, p.cluster_ops, p.clustered_ham)
    ref = plan.sigma(c)[:, 0]
    buf = torch.zeros(n + 8, dtype=torch.float64, device="cuda:0")
    buf[shift:shift + n] = torch.from_numpy(c[:, 0]).to("cuda:0")
    torch.cuda.synchronize()
    plan.sigma_device(buf[shift:].data_ptr(), buf.data_ptr(), 1)
    eng.ctx.synchronize()
    assert np.array_equal(buf[:n].cpu().numpy(), ref)
    eng.drop_plans()


@pytest.mark.parametrize("prec,R", [("fp64", 1), ("fp64", 3), ("fp32", 2)])
def test_first_sigma_over_its_vector(eng, prec, R):
    """The same on a plan's first sigma, whose timing runs must not read what
    they have written."""
    p = build_problem(12, 3, 4, 24, seed=4, max_transfer=1)
    st = TPSCIstate.full_blocks(p.bases, p.focks, R=R)
    c = np.random.Generator(np.random.PCG64(1)).normal(size=(len(st), R))
    ref = eng.tpsci_plan(st, p.cluster_ops, p.clustered_ham, precisions=("fp64", prec)).sigma(c, prec)
    eng.drop_plans()
    plan = eng.tpsci_plan(st, p.cluster_ops, p.clustered_ham, precisions=("fp64", prec))
    buf = torch.from_numpy(np.ascontiguousarray(c.T)).to("cuda:0")
    torch.cuda.synchronize()
    plan.sigma_device(buf.data_ptr(), buf.data_ptr(), R, prec)
    eng.ctx.synchronize()
    assert np.array_equal(buf.cpu().numpy().T, ref)
    assert plan.apply_variant(prec, R) == (-1, -1)  # not timed yet
    assert np.array_equal(plan.sigma(c, prec), ref)
    assert min(plan.apply_variant(prec, R)) >= 0
    eng.drop_plans()
