"""The performance cases of the package: what a program that uses it has it do.

A case names a kind of call and its sizes.  Problems are the seeded synthetic
ones of fermicg_amd.workloads (clusters of 4 orbitals at half filling);
the trial vectors, Tucker factors of a new space and cores come from the seed.

kind     the call                                            in real use
sigma    Plan.sigma_device on a stored plan, device vectors  one Davidson or response iteration
free     the same on a matrix-free plan                      spaces whose H does not fit the card
new      tps_ci_matvec / build_sigma on a space seen first   selected CI and BST loops, whose
         (plan build and one sigma, host vectors)            spaces change every iteration
solve    tps_ci_davidson on a space seen first               the variational step, a served request
pt2      compute_pt2_energy ("dense" or "sparse" engine)     the perturbative correction

space    full   every configuration of each Fock block (few clusters)
         rank1  rank <= 1 configurations, a fraction kept by hash (many clusters)
         bst    Tucker P/Q blocks with factors
"""
import math

import numpy as np
import torch

from fermicg_amd import _lib, tpsci
from fermicg_amd.bst import BSTstate, bst_pq_state, build_sigma
from fermicg_amd.state import TPSCIstate
from fermicg_amd.tpsci import compute_pt2_energy, default_engine, tps_ci_davidson, tps_ci_matvec
from fermicg_amd.workloads import build_problem, rank1_space


def _case(name, kind, space, clusters, M, transfer, R, precision="fp64", frac=1.0, rank=8,
          thresh=1e-9):
    return {"name": name, "kind": kind, "space": space, "clusters": clusters, "M": M,
            "transfer": transfer, "R": R, "precision": precision, "frac": frac, "rank": rank,
            "thresh": thresh}


def listed():
    return [
        # the small space of the tests and examples: one iteration is all launch latency
        _case("sigma_full_small", "sigma", "full", 3, 4, 2, 1),
        # Tucker spaces: FP64 iterations (residual refreshes) and the FP32 ones between them
        _case("sigma_bst_fp64", "sigma", "bst", 5, 16, 2, 2, rank=8),
        _case("sigma_bst_fp32", "sigma", "bst", 4, 11, 2, 2, "fp32", rank=8),
        # sparse spaces of many clusters, as the benchmark's, in the precisions of the solver
        _case("sigma_rank1_fp64", "sigma", "rank1", 8, 16, 2, 4, frac=0.45),
        _case("sigma_rank1_fp32", "sigma", "rank1", 8, 16, 2, 4, "fp32", frac=0.159),
        _case("sigma_rank1_bf16c", "sigma", "rank1", 8, 16, 2, 3, "fp32_bf16c", frac=0.25),
        # the same kind of space without a stored Hamiltonian
        _case("sigma_matrix_free", "free", "rank1", 6, 13, 2, 2),
        # spaces seen for the first time: plan build and one sigma
        _case("new_rank1", "new", "rank1", 7, 11, 2, 3, frac=0.37),
        _case("new_bst", "new", "bst", 4, 12, 2, 1, rank=6),
        # a whole variational solve of a space seen first
        _case("solve_full", "solve", "full", 3, 5, 2, 2),
        # second-order energies: whole target blocks, and the reached configurations alone
        _case("pt2_dense", "pt2", "full", 4, 5, 1, 2),
        _case("pt2_sparse", "pt2", "rank1", 6, 8, 2, 2, frac=0.3, thresh=1e-4),
    ]


def draw(rng):
    def lg(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    what = rng.choice(["full", "bst64", "bst32", "r64", "r64", "r32", "r32", "rbf", "free",
                       "new_rank1", "new_rank1", "new_bst", "solve", "dense", "sparse"])
    if what == "full":
        c = _case("", "sigma", "full", 3, rng.randint(2, 6), rng.randint(1, 2), rng.randint(1, 4),
                  rng.choice(["fp64", "fp32"]))
    elif what == "bst64":
        c = _case("", "sigma", "bst", rng.randint(3, 5), rng.randint(5, 16), 2, rng.randint(1, 3),
                  rank=rng.randint(2, 8))
    elif what == "bst32":
        c = _case("", "sigma", "bst", rng.randint(3, 4), rng.randint(5, 12), 2, rng.randint(1, 4),
                  "fp32", rank=rng.randint(3, 8))
    elif what == "r64":
        c = _case("", "sigma", "rank1", rng.randint(5, 8), rng.randint(6, 16), 2,
                  rng.randint(1, 6), frac=round(lg(0.05, 0.4), 3))
    elif what in ("r32", "rbf"):
        c = _case("", "sigma", "rank1", rng.randint(5, 8), rng.randint(6, 16), 2,
                  rng.randint(1, 6), "fp32" if what == "r32" else "fp32_bf16c",
                  frac=round(lg(0.05, 0.25), 3))
    elif what == "free":
        c = _case("", "free", "rank1", rng.randint(4, 6), rng.randint(4, 13), 2, rng.randint(1, 3),
                  frac=round(lg(0.2, 1.0), 3))
    elif what == "new_rank1":
        c = _case("", "new", "rank1", rng.randint(4, 7), rng.randint(5, 14), 2, rng.randint(1, 4),
                  frac=round(lg(0.1, 0.35), 3))
    elif what == "new_bst":
        c = _case("", "new", "bst", rng.randint(3, 4), rng.randint(4, 12), 2, rng.randint(1, 2),
                  rank=rng.randint(2, 6))
    elif what == "solve":
        c = _case("", "solve", "full", 3, rng.randint(2, 5), rng.randint(1, 2), rng.randint(1, 3))
    elif what == "dense":
        c = _case("", "pt2", "full", rng.randint(3, 4), rng.randint(2, 5), 1, rng.randint(1, 3))
    else:
        c = _case("", "pt2", "rank1", rng.randint(5, 6), rng.randint(4, 8), 2, rng.randint(1, 3),
                  frac=round(lg(0.1, 0.3), 3), thresh=float("%.2g" % lg(1e-4, 1e-3)))
    del c["name"]
    return c


# ---- inputs ----

_PROBLEMS = {}


def _problem(case):
    """The Hamiltonian of the case's system, which a program keeps for all its spaces."""
    key = (case["clusters"], case["M"], case["transfer"])
    if key not in _PROBLEMS:
        n = case["clusters"]
        _PROBLEMS[key] = build_problem(4 * n, n, case["M"], 8 * n, seed=n,
                                       max_transfer=case["transfer"])
    return _PROBLEMS[key]


_BST = {}


def _rotated(st, rng):
    """The same blocks with other factors: each range turned by an orthogonal matrix."""
    turn, out = {}, BSTstate(st.N, st.R)
    for fi, rgs, facs in st.blocks:
        new = []
        for c, F in enumerate(facs):
            if F is not None:
                n = len(F)
                if (c, n) not in turn:
                    turn[c, n] = np.linalg.qr(rng.normal(size=(n, n)))[0]
                F = np.asfortranarray(turn[c, n] @ F)
            new.append(F)
        out.add_block(st.focks[fi], rgs, new)
    return out


def _space(case, p, seed):
    """The state whose configurations or blocks the case's call works on."""
    rng = np.random.Generator(np.random.PCG64(seed + 1000))
    R = case["R"]
    if case["space"] == "bst":
        key = (case["clusters"], case["M"], case["transfer"], case["rank"])
        if key not in _BST:
            st = bst_pq_state(p.bases, p.focks, p.ref_fock, max_q=2, max_rank=case["rank"], R=1,
                              seed=2001)
            ref = np.array(p.ref_fock)
            damp = [10.0 ** -np.clip(np.array(f) - ref, 0, None).sum() for f in st.focks]
            _BST[key] = st, np.repeat([damp[fi] for fi, _, _ in st.blocks], st.dims())
        st, damp = _BST[key]
        if case["kind"] == "new":
            st = _rotated(st, rng)
        out = st.copy_structure(R)
        out.set_vector(rng.normal(size=(len(damp), R)) * damp[:, None])
        return out
    if case["space"] == "full":
        key = ("full", case["clusters"], case["M"], case["transfer"])
        if key not in _BST:
            _BST[key] = TPSCIstate.full_blocks(p.bases, p.focks, R=1)
        st = TPSCIstate(p.clustered_ham.n_clusters, R)
        base = _BST[key]
        st.fock, st.fock_start, st.cfg = base.fock, base.fock_start, base.cfg
    else:
        st = rank1_space(p, R=R, frac=case["frac"], seed=2)
    v = rng.normal(size=(len(st), R))
    if case["kind"] == "pt2" and case["space"] == "rank1":
        # a reference with small amplitudes, as a CI vector has them
        moved = np.clip(st.fock.astype(np.int64) - np.array(p.ref_fock), 0, None).sum(axis=(1, 2))
        exc = (st.cfg > 1).sum(axis=1)
        v *= (0.03 * 10.0 ** -(moved[st.fock_of_cfg()] + exc))[:, None]
        ref = p.focks.index(p.ref_fock)
        for r in range(R):
            v[int(st.fock_start[ref]) + r, r] = 1.0
    v /= np.linalg.norm(v, axis=0)
    if case["kind"] == "pt2":
        v = tpsci.orthonormalize(v)
    st.set_vector(v)
    return st


def prepare(case, seed):
    p = _problem(case)
    st = _space(case, p, seed)
    eng = default_engine()
    s = {"case": case, "p": p, "st": st, "eng": eng}
    if case["kind"] in ("sigma", "free"):
        if case["space"] == "bst":
            sp = _lib.DeviceSpace.bst(eng.ctx, st.flat())
        else:
            sp = _lib.DeviceSpace.tpsci(eng.ctx, st)
        make = _lib.Plan.create_matrix_free if case["kind"] == "free" else _lib.Plan.create
        s["plan"] = make(eng.ctx, eng.ham(p.clustered_ham), eng.ops(p.cluster_ops), sp,
                         precisions=tuple(sorted({"fp64", case["precision"]})))
        s["c"] = torch.from_numpy(np.ascontiguousarray(st.coeffs.T)).to("cuda:0")
        s["sigma"] = torch.empty_like(s["c"])
    return s


# ---- the calls ----

def run(s):
    case, p, st, eng = s["case"], s["p"], s["st"], s["eng"]
    if case["kind"] in ("sigma", "free"):
        s["plan"].sigma_device(s["c"].data_ptr(), s["sigma"].data_ptr(), case["R"],
                               case["precision"])
        return s["sigma"]
    if case["kind"] == "new":
        if case["space"] == "bst":
            out = build_sigma(st.copy_structure(), st, p.cluster_ops, p.clustered_ham,
                              precision=case["precision"], engine=eng).coeffs
        else:
            out = tps_ci_matvec(st, p.cluster_ops, p.clustered_ham, precision=case["precision"],
                                engine=eng)
        eng.drop_plans()
        return out
    if case["kind"] == "solve":
        e, out = tps_ci_davidson(st, p.cluster_ops, p.clustered_ham, conv_thresh=1e-10,
                                 max_iter=400, precision=case["precision"], engine=eng)
        eng.drop_plans()
        return {"energies": e, "vectors": out.coeffs}
    e2 = compute_pt2_energy(st, p.cluster_ops, p.clustered_ham, thresh_foi=case["thresh"],
                            verbose=0, method="sparse" if case["space"] == "rank1" else "dense",
                            engine=eng)
    eng.drop_plans()
    return e2


# ---- what a call cannot do without ----

_WORK = {}


def work(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key in _WORK:
        return _WORK[key]
    s = prepare(case, 1)
    p, st, R = s["p"], s["st"], case["R"]
    n = len(st)
    io = 16.0 * n * R
    ops = 8.0 * sum(G.size for o in p.cluster_ops for d in o.values() for G in d.values())
    ints = 8.0 * sum(t.ints.size for _, t in p.clustered_ham.terms())
    if case["kind"] == "sigma":
        # the stored elements once, the vectors in and out
        el = s["plan"].stats()["block_elems"]
        w = {"bytes": el * (8.0 if case["precision"] == "fp64" else 4.0) + io,
             "flops": 2.0 * el * R}
    elif case["kind"] == "free":
        # the integrals of every connected (block pair, term) contracted once
        have, fl = set(p.focks), 0.0
        for tc, terms in p.clustered_ham:
            hit = sum(tuple((a + x, b + y) for (a, b), (x, y) in zip(f, tc)) in have
                      for f in p.focks)
            fl += hit * sum(2.0 * t.ints.size for t in terms)
        w = {"bytes": io + ops + ints, "flops": fl}
    elif case["kind"] in ("new", "solve"):
        eng = s["eng"]
        sp = (_lib.DeviceSpace.bst(eng.ctx, st.flat()) if case["space"] == "bst"
              else _lib.DeviceSpace.tpsci(eng.ctx, st))
        q = _lib.Plan.create(eng.ctx, eng.ham(p.clustered_ham), eng.ops(p.cluster_ops), sp).stats()
        # the elements written once and read once (a solve: once per iteration, at least 10)
        times = 2.0 if case["kind"] == "new" else 11.0
        w = {"bytes": io + ops + ints + times * 8.0 * q["block_elems"],
             "flops": q["build_flops"] + 2.0 * (times - 1.0) * R * q["block_elems"]}
    else:
        run(s)
        q = compute_pt2_energy.last_stats
        w = {"bytes": io + ops + ints, "flops": float(q.get("build_flops") or q["chain_flops"])}
    _WORK[key] = w
    return w


# ---- the same in 64 bits, from the inputs alone ----

def _apply_h(p, fock, fock_start, cfg, c):
    """H c over explicit configurations (fock [F, N, 2], cfg [n, N] 1-based), term by term: the
    configuration pairs a term connects agree on the clusters it does not touch (matched by
    64-bit hashes), its element is the integrals contracted with the clusters' Γ columns, its
    sign the electrons its odd operators pass."""
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    n, N = cfg.shape
    F = np.repeat(np.arange(len(fock)), np.diff(fock_start))
    S = int(fock.max()) + 2
    sec = torch.from_numpy((fock[..., 0].astype(np.int64) * S + fock[..., 1])[F]).to(dev)  # n, N
    state = torch.from_numpy(cfg.astype(np.int64) - 1).to(dev)
    before = torch.from_numpy(np.concatenate(
        [np.zeros((len(fock), 1), np.int64),
         np.cumsum(fock.astype(np.int64).sum(axis=2), axis=1)[:, :-1]], axis=1)[F]).to(dev)
    nst = int(cfg.max())
    g = np.random.Generator(np.random.PCG64(7))
    big = 2 ** 62
    h_sec = torch.from_numpy(g.integers(-big, big, (N, S * S))).to(dev)
    h_state = torch.from_numpy(g.integers(-big, big, (N, nst))).to(dev)
    full = sum(h_sec[k][sec[:, k]] + h_state[k][state[:, k]] for k in range(N))  # wraps
    part = [h_state[k][state[:, k]] for k in range(N)]
    hsec = [h_sec[k][sec[:, k]] for k in range(N)]
    v = torch.from_numpy(np.ascontiguousarray(c)).to(dev)
    out = torch.zeros_like(v)
    tables, sorted_keys = {}, {}

    def table(k, op):
        """Every Γ column of the operator on cluster k, and where each sector's block starts."""
        if (k, op) not in tables:
            start = torch.full((S * S,), -1, dtype=torch.int64)
            mbra = torch.ones(S * S, dtype=torch.int64)
            cols, at = [], 0
            for (sb, sk), G in p.cluster_ops[k][op].items():
                if max(sk) >= S or max(sb) >= S:
                    continue
                G3 = np.asarray(G).reshape((-1,) + G.shape[-2:], order="F")
                q = sk[0] * S + sk[1]
                start[q], mbra[q] = at, G3.shape[1]
                cols.append(G3.transpose(2, 1, 0).reshape(-1, G3.shape[0]))
                at += G3.shape[1] * G3.shape[2]
            tables[k, op] = (torch.from_numpy(np.ascontiguousarray(np.concatenate(cols))).to(dev),
                             start.to(dev), mbra.to(dev))
        return tables[k, op]

    for tc, terms in p.clustered_ham:
        for t in terms:
            A = t.clusters
            tabs = [table(k, o) for k, o in zip(A, t.ops)]
            ok = torch.ones(n, dtype=torch.bool, device=dev)
            move = torch.zeros(n, dtype=torch.int64, device=dev)
            odd = torch.zeros(n, dtype=torch.int64, device=dev)
            for k, (T, start, _), d, par in zip(A, tabs, t.delta, t.parity):
                ok &= start[sec[:, k]] >= 0
                shift = d[0] * S + d[1]
                move += h_sec[k][(sec[:, k] + shift).clamp(0, S * S - 1)] - hsec[k]
                if par:
                    odd += before[:, k]
            if A not in sorted_keys:
                key = full.clone()
                for k in A:
                    key -= part[k]
                sorted_keys[A] = torch.sort(key) + (key,)
            skey, order, key = sorted_keys[A]
            J = torch.nonzero(ok)[:, 0]
            want = key[J] + move[J]
            lo = torch.searchsorted(skey, want)
            cnt = torch.searchsorted(skey, want, right=True) - lo
            keep = cnt > 0
            J, lo, cnt = J[keep], lo[keep], cnt[keep]
            V = torch.from_numpy(np.ascontiguousarray(np.asarray(t.ints, np.float64))).to(dev)
            sign = 1.0 - 2.0 * (odd % 2).to(torch.float64)
            step = 1 << 21
            ends = torch.cumsum(cnt, 0)
            at = 0
            while at < len(J):
                base = int(ends[at - 1]) if at else 0
                to = max(int(torch.searchsorted(ends, base + step, right=True)), at + 1)
                m = cnt[at:to]
                j = torch.repeat_interleave(J[at:to], m)
                first = torch.repeat_interleave(lo[at:to] - (ends[at:to] - m), m)
                i = order[first + torch.arange(base, base + len(j), device=dev)]
                x = None
                for q, (k, (T, start, mbra)) in enumerate(zip(A, tabs)):
                    sk = sec[j, k]
                    col = T[start[sk] + state[i, k] + mbra[sk] * state[j, k]]
                    if len(A) == 1:
                        x = col[:, 0]
                    elif q == 0:
                        x = col @ V.reshape(V.shape[0], -1)
                    else:
                        x = (x.reshape(len(j), col.shape[1], -1) * col[:, :, None]).sum(1)
                x = x.reshape(-1) * sign[j]
                out.index_add_(0, i, x[:, None] * v[j])
                at = to
    return out.cpu().numpy()


def _bst_as_configurations(p, st):
    """The configurations of a P/Q state's Fock blocks and, per block, where its ranges lie in
    them and the Kronecker product of its factors (ranges' product x rank)."""
    N, per = st.N, [[] for _ in st.focks]
    for b, (fi, rgs, facs) in enumerate(st.blocks):
        per[fi].append(b)
    cfgs, start, rows, mats = [], [0], {}, {}
    for fi in range(len(st.focks)):
        for b in per[fi]:
            _, rgs, facs = st.blocks[b]
            dims = [hi - lo + 1 for lo, hi in rgs]
            idx = np.indices(dims[::-1]).reshape(N, -1)[::-1].T + np.array([r[0] for r in rgs])
            at = start[-1] if not rows or b == per[fi][0] else rows[prev][1]
            rows[b], prev = (at, at + len(idx)), b
            K = np.ones((1, 1))
            for c in range(N):
                K = np.kron(np.eye(dims[c]) if facs[c] is None else facs[c], K)
            mats[b] = K
            cfgs.append(idx)
        start.append(rows[prev][1])
    return (np.array(st.focks, np.int64), np.array(start), np.concatenate(cfgs), rows, mats)


def exact(case, seed):
    if case["kind"] == "pt2":
        return None
    p = _problem(case)
    st = _space(case, p, seed)
    if case["space"] == "bst":
        fock, start, cfg, rows, mats = _bst_as_configurations(p, st)
        if len(cfg) > 150000:
            return None  # minutes
        off = st.var_offsets()
        c = np.zeros((len(cfg), case["R"]))
        for b, (lo, hi) in rows.items():
            c[lo:hi] = mats[b] @ st.coeffs[off[b]:off[b + 1]]
        s = _apply_h(p, fock, start, cfg, c)
        out = np.concatenate([mats[b].T @ s[rows[b][0]:rows[b][1]] for b in range(len(st.blocks))])
    elif case["kind"] == "solve":
        n = len(st)
        H = np.concatenate([_apply_h(p, st.fock, st.fock_start, st.cfg, np.eye(n)[:, a:a + 2048])
                            for a in range(0, n, 2048)], axis=1) if n <= 10000 else None
        if H is None:
            return None
        w = torch.linalg.eigvalsh(torch.from_numpy(0.5 * (H + H.T))).numpy()
        return {"energies": w[:case["R"]], "vectors": None}
    else:
        out = _apply_h(p, st.fock, st.fock_start, st.cfg, st.coeffs)
    return torch.from_numpy(np.ascontiguousarray(out.T)) if case["kind"] in ("sigma", "free") else out
