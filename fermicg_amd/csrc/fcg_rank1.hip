// Matrix-free sigma for TPSCI spaces of rank <= 1.
//
// A configuration of rank <= 1 has every cluster in the lowest state of its
// sector except at most one (the spaces the large benchmark systems use:
// 9.0e6 configurations at 12 clusters of M=32, whose stored Hamiltonian
// would hold 2.4e11-4.3e11 elements).  For such spaces the reference's
// tps_ci_matvec (src/tpsci_outer.jl:462-527, contract_matrix_element
// src/tpsci_inner.jl:10-216) factorises.  Per bra Fock block F_b, ket Fock
// block F_k = F_b - Δ and term t on active clusters A with integrals V and
// sign s (compute_terms_state_sign, src/type_ClusteredTerm.jl:181-197),
// writing g_a = Γ_a[:, 0, 0] (state 0 = the sector's lowest state):
//
//   e      = sum_p V[p] prod_a g_a[p_a]                          (ref <- ref)
//   W_a    = V contracted with g_b on every b != a               (length n_a)
//   W_ab   = V contracted with g_c on every c not in {a, b}      (n_a x n_b)
//   u_b    = sum_{j>=1} Γ_b[:, 0, j] c_(b,j)                      (length n_b)
//
//   y_ref   += s (e c_ref + sum_b W_b . u_b)
//   y_(a,i) += s (sum_j (W_a . Γ_a[:, i, j]) c_(a,j) [j = 0: c_ref]
//                 + sum_{b != a} Γ_a[:, i, 0]' W_ab u_b)          (a in A, i >= 1)
//   y_(x,i) += s e c_(x,i)                                        (x not in A)
//
// -- every other (bra, ket) pair breaks check_term (src/type_ClusteredTerm.jl:
// 92-176) on an inactive cluster.  Vectors live in a layout that holds every
// rank <= 1 configuration of the space's Fock blocks (ref, then cluster by
// cluster states 1..M-1); the caller's configurations are scattered into it
// and gathered back, so a subset of the rank <= 1 configurations works too.
//
// One workgroup per bra Fock block owns that block's rows of sigma in LDS;
// each output value is updated by one thread in a fixed term order, so the
// result is bit-reproducible.  T = double (FP64) or float (the mixed form:
// FP32 arithmetic on an FP32 copy of the Γ tensors and integrals).
#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "fcg_internal.h"

struct R1Term {
  int32_t nbody;
  int32_t cl[4];
  int32_t op[4];
  int32_t dims[4];
  int32_t odd;
  int32_t pad;
  int64_t ioff;
};

struct fcg_rank1 {
  int N = 0, S = 0, n_ops = 0, nbody = 4;
  int64_t n_fock = 0, n_lay = 0, n_var = 0, n_pairs = 0;
  int lmax = 0;            // largest block layout
  int64_t *d_foff = nullptr;   // [n_fock+1]
  int32_t *d_meta = nullptr;   // [n_fock][2N]: M_c then slot offset of cluster c
  int16_t *d_fock = nullptr;   // [n_fock][N][2]
  int64_t *d_fp_ptr = nullptr;
  int32_t *d_fp_fk = nullptr, *d_fp_g = nullptr;
  int32_t *d_tcs = nullptr;
  R1Term *d_terms = nullptr;
  int32_t *d_gblock = nullptr;
  int64_t *d_perm = nullptr;   // [n_var] caller's configuration -> layout slot
  float *d_g32 = nullptr;      // FP32 copy of the Γ data
  float *d_i32 = nullptr;      // FP32 copy of the integrals
  unsigned int *d_err = nullptr;
  uint8_t *d_nzb = nullptr;    // [n_fock] per-call flags of nonzero ket blocks
  bool checked = false;
};

int fcg_rank1_check(fcg_ctx *ctx, fcg_plan *pl);

namespace {

constexpr int RT = 256;      // threads per workgroup
constexpr int RC = 4;        // roots per launch
constexpr int LMAX = 512;    // layout slots of one Fock block
constexpr int VMX = 1024;    // staged integrals
constexpr int NPX = 64;      // largest leading dimension of a Γ block

template <typename T>
struct R1Args {
  int N, S, n_ops, nbody, R;
  int64_t fb_base, n_lay;
  const int64_t *foff;
  const int32_t *meta;
  const int16_t *fock;
  const int64_t *fp_ptr;
  const int32_t *fp_fk, *fp_g;
  const int32_t *tc_start;
  const R1Term *terms;
  const T *ints;
  const int32_t *gblock;
  const int64_t *gb_off;
  const int32_t *gb_dims;
  const T *gdata;
  const T *x;  // [R][n_lay] (R <= RC in this launch)
  T *y;        // [R][n_lay]
  double *diag;  // DIAG: [n_lay]
  const uint8_t *nzb;  // [n_fock] ket blocks with a nonzero coefficient (others skipped)
  unsigned int *err;
};

constexpr int RP = 64;      // connected ket blocks looked up at a time
constexpr int TS = 32;      // terms of a pair prepared at a time
constexpr int NPS = 80;     // index values of a term's clusters together, and W_ab entries of
constexpr int WABX = 768;   // its cluster pairs: at most 76 and 600 where every index count is
                            // <= NPX, every pair's product <= 256 and the whole <= VMX
constexpr int WIJ = 1024;   // staged w_ij values

// the six pairs of a term's clusters, and the other two of each
__device__ constexpr int kPa[6] = {0, 0, 0, 1, 1, 2}, kPb[6] = {1, 2, 3, 2, 3, 3};
__device__ constexpr int kPc[6] = {2, 1, 1, 0, 0, 0}, kPd[6] = {3, 3, 2, 3, 2, 1};

// a value every lane of the wavefront holds, in a scalar register
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uni64(int64_t v) {
  const uint32_t lo = (uint32_t)uni((int)(uint32_t)v), hi = (uint32_t)uni((int)(v >> 32));
  return (int64_t)((uint64_t)hi << 32 | lo);
}

// s + sum_k g[gs k] w[ws k], eight global loads in flight
template <typename T>
__device__ __forceinline__ T strided_dot(int n, const T *__restrict__ g, int64_t gs, const T *w,
                                         int ws, T s) {
  int k = 0;
  for (; k + 8 <= n; k += 8) {
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = g[gs * (k + u)];
#pragma unroll
    for (int u = 0; u < 8; u++) s += v[u] * w[ws * (k + u)];
  }
  if (k < n) {  // the rest, with valid loads and zero weights past the end
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = g[gs * min(k + u, n - 1)];
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (k + u < n) s += v[u] * w[ws * (k + u)];
  }
  return s;
}

// a term prepared for the pair in hand
struct R1Ready {
  int64_t goff[4], ioff;
  int32_t nb, nv, ok;
  float sgn;
  int16_t cl[4], np[4], mb[4], mk[4], poff[4];  // poff: first place among the NPS index values
};

// One workgroup per bra Fock block.  Per connected ket block and term the
// work is a few thousand multiply-adds on small arrays, so what bounds it is
// the number of dependent steps -- global round trips and barriers -- and
// serial loops on few threads.  Hence: ket blocks are looked up RP at a time
// and a pair's terms prepared TS at a time by one thread per (term, cluster);
// W_a and e come from W_ab instead of from V again; the cross part W_ab u_b is
// formed once per (a, p) instead of once per state of a; and the state
// blocks' w_ij = W_a . Γ_a[:, i, j] are spread over all threads.  Barriers per
// term: three up to W_a and z_a, one after each cluster's tile of w_ij and one
// before every tile but the first: 4, 6, 8, 10 for one to four clusters whose
// w_ij fit one tile each.  102,673 configurations of 6 clusters, 2 roots, FP64:
// 508 ms with each bra state forming its own cross part and every W_a summing V,
// 65 ms without, 50 ms with the shape in scalar registers and eight loads in
// flight per dot product; 2,000,089 of 8 clusters, 4 roots: 7.6 s.
template <typename T, bool DIAG>
__global__ __launch_bounds__(RT) void k_rank1(R1Args<T> a) {
  __shared__ T sY[LMAX * RC];
  __shared__ T sX[LMAX * RC];
  __shared__ T sV[VMX];
  __shared__ T sG[2][NPS];      // Γ_q[:, 0, 0], of this term and the last
  __shared__ T sWa[NPS];        // W_a
  __shared__ T sWab[WABX];      // W_ab of the cluster pairs, [p_a + n_a p_b]
  __shared__ T sU[NPS * RC];    // u_b[p][r]
  __shared__ T sZ[NPS * RC];    // z_a[p][r] = sum_{b != a} W_ab u_b
  __shared__ T sW[WIJ];         // w_ij of a tile of bra states
  __shared__ R1Ready sT[TS];
  __shared__ int sMb[FCG_MAXN], sOb[FCG_MAXN], sMk[FCG_MAXN], sOk[FCG_MAXN];
  __shared__ int16_t sFb[2 * FCG_MAXN], sFk[2 * FCG_MAXN];
  __shared__ uint8_t sCl[LMAX];  // cluster of each layout slot of F_b
  __shared__ int32_t sPk[RP], sPt0[RP], sPt1[RP], sPl[RP];
  __shared__ int64_t sPx[RP];

  const int tid = threadIdx.x;
  const int64_t fb = a.fb_base + blockIdx.x;
  const int N = a.N, S = a.S, R = a.R;
  if (tid < N) {
    sMb[tid] = a.meta[fb * 2 * N + tid];
    sOb[tid] = a.meta[fb * 2 * N + N + tid];
  }
  if (tid < 2 * N) sFb[tid] = a.fock[fb * 2 * N + tid];
  const int64_t o0 = a.foff[fb];
  const int Lb = (int)(a.foff[fb + 1] - o0);
  for (int e = tid; e < Lb * RC; e += RT) sY[e] = (T)0;
  __syncthreads();
  for (int e = tid + 1; e < Lb; e += RT) {
    int x = 0;
    while (x + 1 < N && sOb[x + 1] <= e) x++;
    sCl[e] = (uint8_t)x;
  }
  int flip = 0;
  const int64_t q_end = a.fp_ptr[fb + 1];
  for (int64_t qb = a.fp_ptr[fb]; qb < q_end; qb += RP) {
    const int np_here = (int)std::min<int64_t>(RP, q_end - qb);
    __syncthreads();  // the last pair's readers are done
    if (tid < np_here) {
      const int32_t fk = a.fp_fk[qb + tid], g = a.fp_g[qb + tid];
      // only the Δ = 0 pair reaches the diagonal; a ket block of zeros
      // contributes nothing
      const bool use = DIAG ? fk == fb : a.nzb[fk] != 0;
      sPk[tid] = use ? fk : -1;
      sPt0[tid] = a.tc_start[g];
      sPt1[tid] = a.tc_start[g + 1];
      sPx[tid] = a.foff[fk];
      sPl[tid] = (int)(a.foff[fk + 1] - a.foff[fk]);
    }
    __syncthreads();
    for (int pi = 0; pi < np_here; pi++) {
      const int64_t fk = sPk[pi];
      if (fk < 0) continue;  // uniform
      const int Lk = sPl[pi];
      __syncthreads();  // the last term's readers of sX, sMk and sOk are done
      if (tid < N) {
        sMk[tid] = a.meta[fk * 2 * N + tid];
        sOk[tid] = a.meta[fk * 2 * N + N + tid];
      }
      if (tid >= 64 && tid < 64 + 2 * N) sFk[tid - 64] = a.fock[fk * 2 * N + tid - 64];
      if (!DIAG)
        for (int r = 0; r < R; r++)
          for (int i = tid; i < Lk; i += RT) sX[i + Lk * r] = a.x[(int64_t)r * a.n_lay + sPx[pi] + i];
      const int t1 = sPt1[pi];
      for (int tb = sPt0[pi]; tb < t1; tb += TS) {
        const int nt = min(TS, t1 - tb);
        __syncthreads();  // sFk is there; the last batch's readers are done
        if (tid < 4 * nt) {
          const R1Term Tm = a.terms[tb + tid / 4];
          R1Ready &o = sT[tid / 4];
          const int qq = tid & 3, nb = Tm.nbody;
          bool ok = nb <= a.nbody;
          int np = 0;
          if (ok && qq < nb) {
            const int c = qq == 0 ? Tm.cl[0] : qq == 1 ? Tm.cl[1] : qq == 2 ? Tm.cl[2] : Tm.cl[3];
            const int op = qq == 0 ? Tm.op[0] : qq == 1 ? Tm.op[1] : qq == 2 ? Tm.op[2] : Tm.op[3];
            const int cb = sFb[2 * c] * S + sFb[2 * c + 1], ck = sFk[2 * c] * S + sFk[2 * c + 1];
            const int SS = S * S;
            const int blk = a.gblock[(((int64_t)c * a.n_ops + op) * SS + cb) * SS + ck];
            if (blk < 0) {
              ok = false;
            } else {
              np = a.gb_dims[3 * blk];
              const int mb = a.gb_dims[3 * blk + 1], mk = a.gb_dims[3 * blk + 2];
              ok = np <= NPX && mb == sMb[c] && mk == sMk[c];
              o.goff[qq] = a.gb_off[blk];
              o.mb[qq] = (int16_t)mb;
              o.mk[qq] = (int16_t)mk;
            }
            if (!ok) atomicOr(a.err, 1u);
            o.cl[qq] = (int16_t)c;
          }
          o.np[qq] = (int16_t)np;
          // the four threads of a term agree (lanes of one wavefront)
          const int base = (threadIdx.x & 63) & ~3;
          bool all = true;
          int before = 0, tot = 0;
#pragma unroll
          for (int k = 0; k < 4; k++) {
            all = all && __shfl((int)ok, base + k, 64);
            const int n = __shfl(np, base + k, 64);
            if (k < qq) before += n;
            tot += n;
          }
          o.poff[qq] = (int16_t)before;
          if (qq == 0) {
            // sign from the ket Fock configuration
            int par = 0, nv = 1;
#pragma unroll
            for (int k = 0; k < 4; k++) {
              if (k >= nb) continue;
              if (nb > 1) nv *= Tm.dims[k];
              if (!((Tm.odd >> k) & 1)) continue;
              for (int c2 = 0; c2 < Tm.cl[k]; c2++) par ^= sFk[2 * c2] + sFk[2 * c2 + 1];
            }
            o.sgn = (par & 1) ? -1.f : 1.f;
            o.nb = nb;
            o.nv = nv;
            o.ioff = Tm.ioff;
            o.ok = all && tot <= NPS;
          }
        }
        __syncthreads();
        for (int ti = 0; ti < nt; ti++) {
          const R1Ready &t = sT[ti];
          if (!t.ok) continue;  // uniform: dropped by nbody, or reported through err
          // the term's shape in scalar registers: read from LDS where it is
          // used, each read would cost its latency again
          const int nb = uni(t.nb), nv = uni(t.nv);
          int np[4], po[4], off[6];
          const T *Gq[4];
#pragma unroll
          for (int q = 0; q < 4; q++) {
            np[q] = q < nb ? uni(t.np[q]) : 0;
            po[q] = uni(t.poff[q]);
            Gq[q] = a.gdata + (q < nb ? uni64(t.goff[q]) : 0);
          }
#pragma unroll
          for (int k = 0, at = 0; k < 6; k++) {
            off[k] = at;
            at += np[kPa[k]] * np[kPb[k]];
          }
          const T sg = (T)t.sgn;
          // integrals and Γ_q[:, 0, 0]: a thread may still be in the last
          // term's updates, which use neither this V nor this half of sG
          flip ^= 1;
          T *sG0 = sG[flip];
          const T *ints = a.ints + uni64(t.ioff);
          for (int e = tid; e < nv; e += RT) sV[e] = nb > 1 ? ints[e] : (T)1;
          if (tid < NPS) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
              const int p = tid - po[q];
              if (p >= 0 && p < np[q]) sG0[tid] = Gq[q][p];
            }
          }
          __syncthreads();
          // W_ab of every cluster pair: V summed over the other clusters' g;
          // W_ab for two clusters is V itself
          if (nb > 1) {
            const int str[4] = {1, np[0], np[0] * np[1], np[0] * np[1] * np[2]};
#pragma unroll
            for (int k = 0; k < 6; k++) {
              const int qa = kPa[k], qb = kPb[k];
              if (qb >= nb) continue;
              const int qc = kPc[k], qd = kPd[k];  // the other two, in order
              const int na = np[qa], nc = qc < nb ? np[qc] : 1, nd = qd < nb ? np[qd] : 1;
              for (int e = tid; e < na * np[qb]; e += RT) {
                const T *v = sV + (e % na) * str[qa] + (e / na) * str[qb];
                T s = (T)0;
                if (nb == 2) {
                  s = v[0];
                } else {
                  for (int pd = 0; pd < nd; pd++) {
                    T s1 = (T)0;
                    for (int pc = 0; pc < nc; pc++)
                      s1 += v[pc * str[qc] + pd * str[qd]] * (qc < nb ? sG0[po[qc] + pc] : (T)1);
                    s += qd < nb ? s1 * sG0[po[qd] + pd] : s1;
                  }
                }
                sWab[off[k] + e] = s;
              }
            }
          }
          // u_b[p][r] = sum_{j>=1} Γ_b[p, 0, j] x_(b,j)
          if (!DIAG)
            for (int e = tid; e < NPS * R; e += RT) {
              const int pp = e % NPS, r = e / NPS;
#pragma unroll
              for (int q = 0; q < 4; q++) {
                const int p = pp - po[q];
                if (p < 0 || p >= np[q]) continue;
                const int mk = t.mk[q];
                sU[pp + NPS * r] = strided_dot(mk - 1, Gq[q] + p + (int64_t)np[q] * t.mb[q],
                                               (int64_t)np[q] * t.mb[q],
                                               sX + sOk[t.cl[q]] + Lk * r, 1, (T)0);
              }
            }
          __syncthreads();
          // W_a from one W_ab, and z_a from all of them
          for (int e = tid; e < NPS * (DIAG ? 1 : 1 + R); e += RT) {
            const int pp = e % NPS, r = e / NPS - 1;  // r = -1: W_a
#pragma unroll
            for (int q = 0; q < 4; q++) {
              const int p = pp - po[q];
              if (p < 0 || p >= np[q]) continue;
              T s = nb == 1 && r < 0 ? (T)1 : (T)0;
#pragma unroll
              for (int k = 0; k < 6; k++) {
                if (kPa[k] != q && kPb[k] != q) continue;
                const int o = kPa[k] == q ? kPb[k] : kPa[k];
                if (o >= nb || q >= nb || (r < 0 && o != (q == 0 ? 1 : 0))) continue;
                const T *w = sWab + off[k] + (kPa[k] == q ? p : np[o] * p);
                const int st = kPa[k] == q ? np[q] : 1;
                const T *f = r < 0 ? sG0 + po[o] : sU + po[o] + NPS * r;
                for (int x = 0; x < np[o]; x++) s += w[st * x] * f[x];
              }
              if (r < 0) sWa[pp] = s;
              else sZ[pp + NPS * r] = s;
            }
          }
          __syncthreads();
          T ev = (T)0;  // e, by every thread
          for (int p = 0; p < np[0]; p++) ev += sWa[p] * sG0[p];
          // the ground configuration's row
          if (tid < (DIAG ? 1 : R)) {
            T v = DIAG ? ev : ev * sX[Lk * tid];
            if (!DIAG) {
              const int np_all = np[0] + np[1] + np[2] + np[3];
              for (int p = 0; p < np_all; p++) v += sWa[p] * sU[p + NPS * tid];
            }
            sY[Lb * tid] += sg * v;
          }
          // clusters outside the term: (x, i) <- (x, i) with e
          const int c0 = uni(t.cl[0]), c1 = nb > 1 ? uni(t.cl[1]) : -1;
          const int c2 = nb > 2 ? uni(t.cl[2]) : -1, c3 = nb > 3 ? uni(t.cl[3]) : -1;
          for (int e = RT - 1 - tid; e < Lb - 1; e += RT) {
            const int slot = e + 1, x = sCl[slot];
            if (x == c0 || x == c1 || x == c2 || x == c3) continue;
            if (DIAG) {
              sY[slot] += sg * ev;
            } else {
              const int xs = sOk[x] + slot - sOb[x];  // the same state in the ket block
              for (int r = 0; r < R; r++) sY[slot + Lb * r] += sg * ev * sX[xs + Lk * r];
            }
          }
          // the term's clusters, states i >= 1, in tiles of bra states whose
          // w_ij = W_a . Γ_a[:, i, j] fit the stage
#pragma unroll
          for (int q = 0; q < 4; q++) {
            if (q >= nb) continue;
            const int mb = uni(t.mb[q]), mk = uni(t.mk[q]);
            const int ob = sOb[t.cl[q]] - 1, ok = sOk[t.cl[q]] - 1;
            const T *wa = sWa + po[q];
            if (DIAG) {  // I = J = (c, i): W_a . Γ_a[:, i, i]
              for (int i = 1 + tid; i < mb; i += RT)
                sY[ob + i] += sg * strided_dot(np[q], Gq[q] + (int64_t)np[q] * (i + (int64_t)mb * i),
                                               1, wa, 1, (T)0);
              continue;
            }
            const int tile = min(mb - 1, WIJ / mk);
            for (int i0 = 1; i0 < mb; i0 += tile) {
              const int ni = min(tile, mb - i0);
              if (q > 0 || i0 > 1) __syncthreads();  // the last tile's readers are done
              for (int e = tid; e < ni * mk; e += RT) {
                const int i = i0 + e % ni, j = e / ni;
                sW[e] = strided_dot(np[q], Gq[q] + (int64_t)np[q] * (i + (int64_t)mb * j), 1, wa, 1,
                                    (T)0);
              }
              __syncthreads();
              for (int e = tid; e < ni * R; e += RT) {
                const int k = e % ni, i = i0 + k, r = e / ni;
                const T *x = sX + Lk * r;
                T s = sW[k] * x[0];
                for (int j = 1; j < mk; j++) s += sW[k + ni * j] * x[ok + j];
                if (nb > 1)  // cross terms: Γ_a[:, i, 0]' sum_b W_ab u_b
                  s = strided_dot(np[q], Gq[q] + (int64_t)np[q] * i, 1, sZ + po[q] + NPS * r, 1, s);
                sY[ob + i + Lb * r] += sg * s;
              }
            }
          }
        }
      }
    }
  }
  __syncthreads();
  if (DIAG) {
    for (int i = tid; i < Lb; i += RT) a.diag[o0 + i] = (double)sY[i];
  } else {
    for (int e = tid; e < Lb * R; e += RT) {
      const int i = e % Lb, r = e / Lb;
      a.y[(int64_t)r * a.n_lay + o0 + i] = sY[i + Lb * r];
    }
  }
}

// x_lay[r][perm[i]] = c[r][i] (layout zeroed first); sigma[r][i] = y_lay[r][perm[i]]
template <typename T>
__global__ void k_r1_scatter(int64_t n, int R, int64_t n_lay, const int64_t *perm, const double *c,
                             T *x) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n * R;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = e % n, r = e / n;
    x[r * n_lay + perm[i]] = (T)c[e];
  }
}

template <typename T>
__global__ void k_r1_gather(int64_t n, int R, int64_t n_lay, const int64_t *perm, const T *y,
                            double *s) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n * R;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = e % n, r = e / n;
    s[e] = (double)y[r * n_lay + perm[i]];
  }
}

__global__ void k_r1_gather_diag(int64_t n, const int64_t *perm, const double *d, double *hd) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    hd[i] = d[perm[i]];
}

// nzb[f] = 1 when some root's coefficient in Fock block f's layout is nonzero
template <typename T>
__global__ void k_r1_nonzero(int64_t n_fock, int R, int64_t n_lay, const int64_t *foff,
                             const T *x, uint8_t *nzb) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= n_fock) return;
  uint8_t nz = 0;
  for (int r = 0; r < R && !nz; r++)
    for (int64_t i = foff[f]; i < foff[f + 1]; i++)
      if (x[(int64_t)r * n_lay + i] != (T)0) {
        nz = 1;
        break;
      }
  nzb[f] = nz;
}

__global__ void k_to_float(int64_t n, const double *a, float *b) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    b[i] = (float)a[i];
}

__global__ void k_zero(int64_t n, double *p) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0.0;
}

constexpr int64_t FB_CHUNK = 65535;

template <typename T>
int launch_rank1(fcg_ctx *ctx, fcg_plan *pl, R1Args<T> a, bool diag) {
  const fcg_rank1 *r1 = pl->r1;
  for (int64_t f0 = 0; f0 < r1->n_fock; f0 += FB_CHUNK) {
    a.fb_base = f0;
    const unsigned nb = (unsigned)std::min(FB_CHUNK, r1->n_fock - f0);
    if (diag)
      hipLaunchKernelGGL((k_rank1<T, true>), dim3(nb), dim3(RT), 0, ctx->stream, a);
    else
      hipLaunchKernelGGL((k_rank1<T, false>), dim3(nb), dim3(RT), 0, ctx->stream, a);
  }
  FCG_HIP(hipGetLastError(), ctx);
  return FCG_OK;
}

template <typename T>
R1Args<T> base_args(const fcg_plan *pl, const fcg_ham *h, const fcg_ops *o) {
  const fcg_rank1 *r1 = pl->r1;
  R1Args<T> a{};
  a.N = r1->N;
  a.S = r1->S;
  a.n_ops = r1->n_ops;
  a.nbody = r1->nbody;
  a.n_lay = r1->n_lay;
  a.foff = r1->d_foff;
  a.meta = r1->d_meta;
  a.fock = r1->d_fock;
  a.fp_ptr = r1->d_fp_ptr;
  a.fp_fk = r1->d_fp_fk;
  a.fp_g = r1->d_fp_g;
  a.tc_start = r1->d_tcs;
  a.terms = r1->d_terms;
  a.gblock = r1->d_gblock;
  a.gb_off = o->d_gb_off;
  a.gb_dims = o->d_gb_dims;
  a.err = r1->d_err;
  a.nzb = r1->d_nzb;
  return a;
}

}  // namespace

void fcg_rank1_free(fcg_ctx *ctx, fcg_plan *pl) {
  fcg_rank1 *r = pl->r1;
  if (!r) return;
  fcg_dfree(ctx, r->d_foff);
  fcg_dfree(ctx, r->d_meta);
  fcg_dfree(ctx, r->d_fock);
  fcg_dfree(ctx, r->d_fp_ptr);
  fcg_dfree(ctx, r->d_fp_fk);
  fcg_dfree(ctx, r->d_fp_g);
  fcg_dfree(ctx, r->d_tcs);
  fcg_dfree(ctx, r->d_terms);
  fcg_dfree(ctx, r->d_gblock);
  fcg_dfree(ctx, r->d_perm);
  fcg_dfree(ctx, r->d_g32);
  fcg_dfree(ctx, r->d_i32);
  fcg_dfree(ctx, r->d_err);
  fcg_dfree(ctx, r->d_nzb);
  delete r;
  pl->r1 = nullptr;
}

namespace {
int ensure_r1_buffers(fcg_ctx *ctx, int64_t n) {
  if (n <= ctx->r1_elems) return FCG_OK;
  if (ctx->d_r1x) fcg_dfree(ctx, ctx->d_r1x);
  if (ctx->d_r1y) fcg_dfree(ctx, ctx->d_r1y);
  ctx->d_r1x = static_cast<double *>(fcg_dmalloc(ctx, sizeof(double) * std::max<int64_t>(n, 1)));
  ctx->d_r1y = static_cast<double *>(fcg_dmalloc(ctx, sizeof(double) * std::max<int64_t>(n, 1)));
  ctx->r1_elems = 0;
  if (!ctx->d_r1x || !ctx->d_r1y) return FCG_ENOMEM;
  ctx->r1_elems = n;
  return FCG_OK;
}
}  // namespace

int fcg_rank1_sigma(fcg_ctx *ctx, fcg_plan *pl, int R, const double *c, double *sigma,
                    int precision) {
  fcg_rank1 *r1 = pl->r1;
  const fcg_ham *h = pl->r1_ham;
  const fcg_ops *o = pl->r1_ops;
  const int64_t L = r1->n_lay, n = r1->n_var;
  if (int rc = ensure_r1_buffers(ctx, L * R)) {
    ctx->err = "matrix-free sigma buffers allocation failed";
    return rc;
  }
  hipStream_t s = ctx->stream;
  const bool f32 = precision != FCG_FP64;
  // layout vectors (the slots no configuration maps to stay zero)
  hipLaunchKernelGGL(k_zero, dim3(1024), dim3(256), 0, s, L * R, ctx->d_r1x);
  if (f32)
    hipLaunchKernelGGL(k_r1_scatter<float>, dim3(1024), dim3(256), 0, s, n, R, L, r1->d_perm, c,
                       reinterpret_cast<float *>(ctx->d_r1x));
  else
    hipLaunchKernelGGL(k_r1_scatter<double>, dim3(1024), dim3(256), 0, s, n, R, L, r1->d_perm, c,
                       ctx->d_r1x);
  const unsigned nfb = (unsigned)((r1->n_fock + 255) / 256);
  if (f32)
    hipLaunchKernelGGL(k_r1_nonzero<float>, dim3(nfb), dim3(256), 0, s, r1->n_fock, R, L,
                       r1->d_foff, reinterpret_cast<const float *>(ctx->d_r1x), r1->d_nzb);
  else
    hipLaunchKernelGGL(k_r1_nonzero<double>, dim3(nfb), dim3(256), 0, s, r1->n_fock, R, L,
                       r1->d_foff, ctx->d_r1x, r1->d_nzb);
  FCG_HIP(hipEventRecord(ctx->ev0, s), ctx);
  for (int r0 = 0; r0 < R; r0 += RC) {
    const int rn = std::min(RC, R - r0);
    if (f32) {
      R1Args<float> a = base_args<float>(pl, h, o);
      a.R = rn;
      a.ints = r1->d_i32;
      a.gdata = r1->d_g32;
      a.x = reinterpret_cast<const float *>(ctx->d_r1x) + (int64_t)r0 * L;
      a.y = reinterpret_cast<float *>(ctx->d_r1y) + (int64_t)r0 * L;
      if (int rc = launch_rank1<float>(ctx, pl, a, false)) return rc;
    } else {
      R1Args<double> a = base_args<double>(pl, h, o);
      a.R = rn;
      a.ints = h->d_ints;
      a.gdata = o->d_gdata;
      a.x = ctx->d_r1x + (int64_t)r0 * L;
      a.y = ctx->d_r1y + (int64_t)r0 * L;
      if (int rc = launch_rank1<double>(ctx, pl, a, false)) return rc;
    }
  }
  FCG_HIP(hipEventRecord(ctx->ev1, s), ctx);
  if (!r1->checked) {  // the first sigma visits every term: missing Γ blocks show here
    if (int rc = fcg_rank1_check(ctx, pl)) return rc;
    r1->checked = true;
  }
  if (f32)
    hipLaunchKernelGGL(k_r1_gather<float>, dim3(1024), dim3(256), 0, s, n, R, L, r1->d_perm,
                       reinterpret_cast<const float *>(ctx->d_r1y), sigma);
  else
    hipLaunchKernelGGL(k_r1_gather<double>, dim3(1024), dim3(256), 0, s, n, R, L, r1->d_perm,
                       ctx->d_r1y, sigma);
  FCG_HIP(hipGetLastError(), ctx);
  return FCG_OK;
}

int fcg_rank1_diag(fcg_ctx *ctx, fcg_plan *pl, double *hd) {
  fcg_rank1 *r1 = pl->r1;
  const int64_t L = r1->n_lay;
  if (int rc = ensure_r1_buffers(ctx, L)) {
    ctx->err = "matrix-free diagonal buffers allocation failed";
    return rc;
  }
  R1Args<double> a = base_args<double>(pl, pl->r1_ham, pl->r1_ops);
  a.R = 1;
  a.ints = pl->r1_ham->d_ints;
  a.gdata = pl->r1_ops->d_gdata;
  a.diag = ctx->d_r1y;
  if (int rc = launch_rank1<double>(ctx, pl, a, true)) return rc;
  if (int rc = fcg_rank1_check(ctx, pl)) return rc;
  hipLaunchKernelGGL(k_r1_gather_diag, dim3(1024), dim3(256), 0, ctx->stream, r1->n_var,
                     r1->d_perm, ctx->d_r1y, hd);
  FCG_HIP(hipGetLastError(), ctx);
  return FCG_OK;
}

extern "C" int fcg_plan_create_matrix_free(fcg_ctx_t ctx, fcg_ham_t h, fcg_ops_t o,
                                           fcg_space_t sp, int nbody, int precisions,
                                           fcg_plan_t *out) {
  if (!ctx || !h || !o || !sp || !out || nbody < 1 || nbody > 4) return FCG_EINVAL;
  if (!sp->tpsci) {
    ctx->err = "matrix-free plans need a TPSCI space";
    return FCG_EINVAL;
  }
  if (precisions & ~((1 << FCG_FP64) | (1 << FCG_FP32))) {
    ctx->err = "matrix-free plans compute in FP64 and FP32 only";
    return FCG_EINVAL;
  }
  (void)hipSetDevice(ctx->device);
  if (int rc = fcg_form_boxes(ctx, o, sp)) return rc;
  const int N = sp->N, S = o->S;
  const int64_t n_fock = sp->n_fock, n_var = sp->nvar;
  // layout: per Fock block the ground configuration, then cluster by
  // cluster its states 1..M-1
  std::vector<int64_t> foff(n_fock + 1, 0);
  std::vector<int32_t> meta((size_t)n_fock * 2 * N);
  int lmax = 0;
  for (int64_t f = 0; f < n_fock; f++) {
    int off = 1;
    for (int c = 0; c < N; c++) {
      const int na = sp->fock[(f * N + c) * 2], nb = sp->fock[(f * N + c) * 2 + 1];
      const int m = (na >= 0 && nb >= 0 && na < S && nb < S)
                        ? o->nstates[(int64_t)c * S * S + na * S + nb] : 0;
      if (m < 1) {
        ctx->err = "matrix-free plan: a Fock block's sector has no states";
        return FCG_EINVAL;
      }
      meta[f * 2 * N + c] = m;
      meta[f * 2 * N + N + c] = off;
      off += m - 1;
    }
    foff[f + 1] = foff[f] + off;
    lmax = std::max(lmax, off);
  }
  if (lmax > LMAX) {
    ctx->err = "matrix-free plan: a Fock block holds more than " + std::to_string(LMAX) +
               " rank <= 1 configurations";
    return FCG_EOVERFLOW;
  }
  // the caller's configurations in the layout
  std::vector<int64_t> perm(std::max<int64_t>(n_var, 1));
  std::vector<uint8_t> used(std::max<int64_t>(foff[n_fock], 1), 0);
  for (int64_t b = 0; b < sp->n_box; b++) {
    const int64_t f = sp->box_fock[b];
    const int64_t v0 = sp->var_off[b], d = sp->var_off[b + 1] - v0;
    for (int64_t e = 0; e < d; e++) {
      int64_t r = e;
      int exc = -1, st = 0;
      for (int c = 0; c < N; c++) {
        const int rk = sp->rank[b * N + c];
        const int s0 = (int)(r % rk) + sp->lo[b * N + c] - 1;
        r /= rk;
        if (s0 != 0) {
          if (exc >= 0) {
            ctx->err = "matrix-free plan: a configuration has more than one excited cluster";
            return FCG_EINVAL;
          }
          exc = c;
          st = s0;
        }
      }
      const int64_t slot = foff[f] + (exc < 0 ? 0 : meta[f * 2 * N + N + exc] + st - 1);
      if (exc >= 0 && st >= meta[f * 2 * N + exc]) {
        ctx->err = "matrix-free plan: state outside its sector";
        return FCG_EINVAL;
      }
      if (used[slot]) {
        ctx->err = "matrix-free plan: a configuration appears twice";
        return FCG_EINVAL;
      }
      used[slot] = 1;
      perm[v0 + e] = slot;
    }
  }
  fcg_rank1 *r1 = new fcg_rank1();
  r1->N = N;
  r1->S = S;
  r1->n_ops = o->n_ops;
  r1->nbody = nbody;
  r1->n_fock = n_fock;
  r1->n_lay = foff[n_fock];
  r1->n_var = n_var;
  r1->lmax = lmax;
  std::vector<R1Term> terms(h->n_terms);
  for (int t = 0; t < h->n_terms; t++) {
    R1Term &T = terms[t];
    T = R1Term{};
    T.nbody = h->nbody[t];
    T.ioff = h->ioff[t];
    int nv = 1;
    for (int q = 0; q < 4; q++) {
      T.cl[q] = h->clusters[4 * t + q];
      T.op[q] = h->ops[4 * t + q];
      T.dims[q] = h->dims[4 * t + q];
      if (q < T.nbody && h->parity[4 * t + q] == 1) T.odd |= 1 << q;
      if (q < T.nbody && T.nbody > 1) nv *= T.dims[q];
    }
    if (nv > VMX) {
      delete r1;
      ctx->err = "matrix-free plan: a term's integrals exceed the staged size";
      return FCG_EOVERFLOW;
    }
    if (T.nbody > 1)
      for (int qa = 0; qa < T.nbody; qa++)
        for (int qb = qa + 1; qb < T.nbody; qb++)
          if (T.dims[qa] * T.dims[qb] > 256 || T.dims[qa] > NPX) {
            delete r1;
            ctx->err = "matrix-free plan: a term's index pair exceeds the staged size";
            return FCG_EOVERFLOW;
          }
  }
  {  // every term's Γ blocks shaped as its integrals (the kernel relies on it)
    const int64_t SS = (int64_t)S * S;
    std::vector<uint8_t> seen((size_t)N * o->n_ops, 0);
    for (int t = 0; t < h->n_terms; t++)
      for (int q = 0; q < h->nbody[t]; q++) {
        const int cl = h->clusters[4 * t + q], op = h->ops[4 * t + q];
        if (cl < 0 || cl >= N || op < 0 || op >= o->n_ops) {
          delete r1;
          ctx->err = "matrix-free plan: term cluster or operator out of range";
          return FCG_EINVAL;
        }
        if (seen[(size_t)cl * o->n_ops + op]) continue;
        seen[(size_t)cl * o->n_ops + op] = 1;
        const int want = h->nbody[t] == 1 ? 1 : h->dims[4 * t + q];
        for (int64_t e = 0; e < SS * SS; e++) {
          const int blk = o->gblock[((int64_t)cl * o->n_ops + op) * SS * SS + e];
          if (blk >= 0 && o->gb_dims[3 * blk] != want) {
            delete r1;
            ctx->err = "matrix-free plan: a Γ block's leading dimension differs from its "
                       "term's integrals";
            return FCG_EINVAL;
          }
        }
      }
  }
  fcg_plan *pl = new fcg_plan();
  pl->ctx = ctx;
  pl->sp = pl->ksp = sp;
  pl->r1 = r1;
  pl->r1_ham = h;
  pl->r1_ops = o;
  pl->precisions = precisions | (1 << FCG_FP64);
  pl->holds_blocks = true;  // can apply sigma (matrix-free)
  auto up = [&](auto **dst, const auto *src, int64_t cnt) -> int {
    using T = std::remove_reference_t<decltype(**dst)>;
    *dst = static_cast<T *>(fcg_dmalloc(ctx, sizeof(T) * std::max<int64_t>(cnt, 1)));
    if (!*dst) return FCG_ENOMEM;
    if (cnt > 0 &&
        hipMemcpyAsync(*dst, src, sizeof(T) * cnt, hipMemcpyHostToDevice, ctx->stream) !=
            hipSuccess)
      return FCG_EDEVICE;
    return FCG_OK;
  };
  int rc = up(&r1->d_foff, foff.data(), n_fock + 1);
  if (!rc) rc = up(&r1->d_meta, meta.data(), (int64_t)meta.size());
  if (!rc) rc = up(&r1->d_fock, sp->fock.data(), (int64_t)sp->fock.size());
  if (!rc) rc = up(&r1->d_tcs, h->tc_start.data(), (int64_t)h->tc_start.size());
  if (!rc) rc = up(&r1->d_terms, terms.data(), (int64_t)terms.size());
  if (!rc) rc = up(&r1->d_gblock, o->gblock.data(), (int64_t)o->gblock.size());
  if (!rc) rc = up(&r1->d_perm, perm.data(), n_var);
  if (!rc) {
    r1->d_err = static_cast<unsigned int *>(fcg_dmalloc(ctx, sizeof(unsigned int)));
    r1->d_nzb = static_cast<uint8_t *>(fcg_dmalloc(ctx, std::max<int64_t>(n_fock, 1)));
    rc = r1->d_err && r1->d_nzb ? FCG_OK : FCG_ENOMEM;
  }
  if (!rc && hipMemsetAsync(r1->d_err, 0, sizeof(unsigned int), ctx->stream) != hipSuccess)
    rc = FCG_EDEVICE;
  if (!rc) rc = fcg_device_fock_pairs(ctx, h, sp, nbody, S, &r1->d_fp_ptr, &r1->d_fp_fk,
                                      &r1->d_fp_g, &r1->n_pairs);
  if (!rc && (pl->precisions & (1 << FCG_FP32))) {
    const int64_t ng = o->n_gdata;
    int64_t ni = 0;
    for (int t = 0; t < h->n_terms; t++) {
      int64_t sz = 1;
      if (h->nbody[t] > 1)
        for (int q = 0; q < h->nbody[t]; q++) sz *= h->dims[4 * t + q];
      ni = std::max(ni, h->ioff[t] + sz);
    }
    r1->d_g32 = static_cast<float *>(fcg_dmalloc(ctx, sizeof(float) * std::max<int64_t>(ng, 1)));
    r1->d_i32 = static_cast<float *>(fcg_dmalloc(ctx, sizeof(float) * std::max<int64_t>(ni, 1)));
    if (!r1->d_g32 || !r1->d_i32) {
      rc = FCG_ENOMEM;
    } else {
      hipLaunchKernelGGL(k_to_float, dim3(1024), dim3(256), 0, ctx->stream, ng, o->d_gdata,
                         r1->d_g32);
      hipLaunchKernelGGL(k_to_float, dim3(1024), dim3(256), 0, ctx->stream, ni, h->d_ints,
                         r1->d_i32);
    }
  }
  if (!rc && hipStreamSynchronize(ctx->stream) != hipSuccess) rc = FCG_EDEVICE;
  if (rc) {
    if (ctx->err.empty()) ctx->err = "matrix-free plan: device allocation or upload failed";
    fcg_plan_destroy(pl);
    return rc;
  }
  pl->n_pair = r1->n_pairs;
  fcg_plan_register(pl);
  *out = pl;
  return FCG_OK;
}

// errors the kernels flagged (a missing or mis-shaped Γ block)
int fcg_rank1_check(fcg_ctx *ctx, fcg_plan *pl) {
  unsigned int e = 0;
  FCG_HIP(hipMemcpyAsync(&e, pl->r1->d_err, sizeof(e), hipMemcpyDeviceToHost, ctx->stream), ctx);
  FCG_HIP(hipStreamSynchronize(ctx->stream), ctx);
  if (e) {
    ctx->err = "matrix-free sigma: a term needs a Γ block that ClusterOps lacks or mis-shapes";
    return FCG_EMISSING_BLOCK;
  }
  return FCG_OK;
}
