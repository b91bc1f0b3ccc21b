// Kronecker form of the superblock Hamiltonian: the operator of the assembled CRS
// (GET_HAM_LLLRRRRL from the recorded term list) applied without assembling it.
//
// The superblock basis (GET_BASIS_SUPERBLOCK: states ordered by the LLLR quantum numbers,
// then LL, LR, RR, RL) falls into sectors of one LLLR quantum number, and a sector holds
// every (LL, LR) state of that number combined with every (RR, RL) state of the
// complementary one, LLLR-major.  A sector's part of a vector is therefore a dense row-major
// da x db matrix X (da LLLR states, db RRRL states).  A term of the list that acts only on
// LL and LR (kinds LL, LR, LLLR) keeps the sector and acts on the rows of X; one that acts
// only on RR and RL (RR, RL, RRRL) acts on its columns.  Summed per sector they are dense
// matrices M_L (da x da) and M_R (db x db), built once from the term list with the element
// makers' rules (operator rows of the row state, sign rules of the row's parities,
// contributions with |value| <= 1e-15 or outside the superblock basis dropped), and
//     (H x)_sector = M_L X + X M_R^T + (coupling terms)
// where the coupling terms (LLRL, LLRR, LRRL, LRRR: one operator on each half) are applied
// row by row from the term list through the superblock inverse, as the matrix-free product of
// dmrg/DMRG_MATRIX_VECTOR_PRODUCT_OBC.c:18-83 applies its M_LRRL.
//
// A product is one kernel (kron_tile.h): each workgroup computes an output tile of both dense
// products on the FP64 matrix cores, adds the coupling terms and runs the solver's epilogue.
// The sums are in an order of their own (the CRS sums every term's contributions to an
// entry first), so results agree with the CRS product to rounding.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>

#include "superblock.h"

#pragma clang fp contract(off)

namespace dmrgx {
namespace {


struct KronBuild {
  int32_t d, nstate_a, nstate_b;
  const int16_t *aLL, *aLR, *bRR, *bRL;   // flat state lists (sector order)
  const int32_t *asec, *bsec;             // sector of each flat state
  const int32_t *aidx, *bidx;             // (LL*d+LR) -> flat a-state, (RR*d+RL) -> flat b-state, -1 if none
  const KronSector *sec;
};

// One thread per LLLR state: its row of M_L, from the terms acting on LL and LR only, in
// term order (op1 row outer, op2 row inner, as DMRG_MAKE_ELEM_LLLR_LLLRRRRL.c:54-79).
__global__ __launch_bounds__(256) void k_kron_left(KronBuild kb, const DTerm *terms, const int32_t *ids, int nt,
                                                   const DOp *ops, const int32_t *const *eles, double *ML) {
  const int32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kb.nstate_a) return;
  const int s = kb.asec[i];
  const KronSector S = kb.sec[s];
  const int32_t ap = i - S.a0;
  double *M = ML + S.ml;
  const int q[4] = {kb.aLL[i], kb.aLR[i], 0, 0};
  for (int u = 0; u < nt; u++) {
    const DTerm t = terms[ids[u]];
    const DOp a = ops[t.op1];
    const double sc = (double)term_sign(t, eles, q) * t.coeff;
    const int64_t b1 = a.row[q[t.s1]], e1 = a.row[q[t.s1] + 1];
    for (int64_t i1 = b1; i1 < e1; i1++) {
      int qq[2] = {q[0], q[1]};
      qq[t.s1] = a.col[i1];
      const double p1 = sc * a.val[i1];
      if (t.s2 < 0) {
        const int32_t c = kb.aidx[qq[0] * kb.d + qq[1]];
        if (c >= 0 && kb.asec[c] == s && fabs(p1) > 1.0e-15) M[kron_at(ap, c - S.a0, S.da)] += p1;
        continue;
      }
      const DOp b = ops[t.op2];
      const int64_t b2 = b.row[q[t.s2]], e2 = b.row[q[t.s2] + 1];
      for (int64_t i2 = b2; i2 < e2; i2++) {
        qq[t.s2] = b.col[i2];
        const double p = p1 * b.val[i2];
        const int32_t c = kb.aidx[qq[0] * kb.d + qq[1]];
        if (c >= 0 && kb.asec[c] == s && fabs(p) > 1.0e-15) M[kron_at(ap, c - S.a0, S.da)] += p;
      }
    }
  }
}

// One thread per RRRL state: its row of M_R, from the terms acting on RR and RL only.
__global__ __launch_bounds__(256) void k_kron_right(KronBuild kb, const DTerm *terms, const int32_t *ids, int nt,
                                                    const DOp *ops, const int32_t *const *eles, double *MR) {
  const int32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kb.nstate_b) return;
  const int s = kb.bsec[i];
  const KronSector S = kb.sec[s];
  const int32_t bp = i - S.b0;
  double *M = MR + S.mr;
  const int q[4] = {0, 0, kb.bRR[i], kb.bRL[i]};
  for (int u = 0; u < nt; u++) {
    const DTerm t = terms[ids[u]];
    const DOp a = ops[t.op1];
    const double sc = (double)term_sign(t, eles, q) * t.coeff;
    const int64_t b1 = a.row[q[t.s1]], e1 = a.row[q[t.s1] + 1];
    for (int64_t i1 = b1; i1 < e1; i1++) {
      int qq[4] = {q[0], q[1], q[2], q[3]};
      qq[t.s1] = a.col[i1];
      const double p1 = sc * a.val[i1];
      if (t.s2 < 0) {
        const int32_t c = kb.bidx[qq[2] * kb.d + qq[3]];
        if (c >= 0 && kb.bsec[c] == s && fabs(p1) > 1.0e-15) M[kron_at(bp, c - S.b0, S.db)] += p1;
        continue;
      }
      const DOp b = ops[t.op2];
      const int64_t b2 = b.row[q[t.s2]], e2 = b.row[q[t.s2] + 1];
      for (int64_t i2 = b2; i2 < e2; i2++) {
        qq[t.s2] = b.col[i2];
        const double p = p1 * b.val[i2];
        const int32_t c = kb.bidx[qq[2] * kb.d + qq[3]];
        if (c >= 0 && kb.bsec[c] == s && fabs(p) > 1.0e-15) M[kron_at(bp, c - S.b0, S.db)] += p;
      }
    }
  }
}

// The same rows with one wavefront per state and the row in LDS, its lanes over the (op1 entry,
// op2 entry) products of a term.  Within a term no two products reach one state (the operators'
// rows hold a column once: dmrgx_superblock::ascending; otherwise, or for a row above
// kHalfRow states, the kernels above), and a wavefront's LDS accesses are in order, so
// every element sums the same products in the same order.  The kernels above wait for a chain of
// some thousand dependent loads: KLM m = 799 479 + 468 us, Hubbard m = 396 231 + 258; this one
// takes 41 + 38 and below 20 + 20.
constexpr int kHalfRow = 2048;
template <bool kLeft>
__global__ __launch_bounds__(256) void k_kron_half(KronBuild kb, const DTerm *terms, const int32_t *ids, int nt,
                                                   const DOp *ops, const int32_t *const *eles, double *M) {
  __shared__ double rows[4][kHalfRow];
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int32_t i = blockIdx.x * 4 + wave;
  if (i >= (kLeft ? kb.nstate_a : kb.nstate_b)) return;   // no barrier below
  const int32_t *sec = kLeft ? kb.asec : kb.bsec, *idx = kLeft ? kb.aidx : kb.bidx;
  const int s = sec[i];
  const KronSector S = kb.sec[s];
  const int32_t first = kLeft ? S.a0 : S.b0, dim = kLeft ? S.da : S.db;
  const int block = kLeft ? kb.aLL[i] : kb.bRR[i], site = kLeft ? kb.aLR[i] : kb.bRL[i];
  const int q[4] = {kLeft ? block : 0, kLeft ? site : 0, kLeft ? 0 : block, kLeft ? 0 : site};
  double *row = rows[wave];
  for (int32_t c = l; c < dim; c += 64) row[c] = 0.0;
  __builtin_amdgcn_wave_barrier();
  for (int u = 0; u < nt; u++) {
    const DTerm t = terms[ids[u]];
    const DOp a = ops[t.op1], b = t.s2 < 0 ? a : ops[t.op2];
    const double sc = (double)term_sign(t, eles, q) * t.coeff;
    const int64_t b1 = a.row[q[t.s1]], n1 = a.row[q[t.s1] + 1] - b1;
    const int64_t b2 = t.s2 < 0 ? 0 : b.row[q[t.s2]], n2 = t.s2 < 0 ? 1 : b.row[q[t.s2] + 1] - b2;
    for (int64_t e = l; e < n1 * n2; e += 64) {
      const int64_t i1 = e / n2, i2 = e - i1 * n2;
      int st[2] = {block, site};
      st[t.s1 & 1] = a.col[b1 + i1];
      double p = sc * a.val[b1 + i1];
      if (t.s2 >= 0) {
        st[t.s2 & 1] = b.col[b2 + i2];
        p = p * b.val[b2 + i2];
      }
      const int32_t c = idx[st[0] * kb.d + st[1]];
      if (c >= 0 && sec[c] == s && fabs(p) > 1.0e-15) row[c - first] += p;
    }
    __builtin_amdgcn_wave_barrier();
  }
  double *out = M + (kLeft ? S.ml : S.mr);
  for (int32_t c = l; c < dim; c += 64) out[kron_at(i - first, c, dim)] = row[c];
}

// zc = coupling terms applied to x, the general form (KronDev::general).  A coupling term has
// one operator on each half (op1 on LL or LR, op2 on RR or RL) and a sign that is a product of a
// factor of the row's LLLR state and one of its RRRL state, so per term the builder lists,
// for every LLLR state a', the states a it reaches with op1 and their coefficients (left parity
// sign x op1 value), and likewise for every RRRL state b' (right parity sign x op2 value);
// the term's own factor is its coefficient times the sign rule's constant.  One workgroup
// per LLLR state a' of the output, its threads over the sector's RRRL states b': for each
// term (in term order), op1 entry and op2 entry (in row order, as the element makers enumerate
// them) the contribution c_t c_l c_r x[a, b] is added when (a, b) is a superblock state (a and
// b in one sector) and |c_t c_l c_r| > 1e-15, as the element makers drop it.
struct KronCross {
  int nt, na, nb;
  const double *ct;                         // per term
  const int32_t *lptr, *lidx, *rptr, *ridx;  // term t: lptr[t (na + 1) + a'] ... into lidx / lval
  const double *lval, *rval;
  const int32_t *asec, *bsec;
  const KronSector *sec;
};
__device__ __forceinline__ void kron_cross_row(const KronCross &kc, int32_t i, const double *__restrict__ x,
                                               double *__restrict__ z) {
  const KronSector S = kc.sec[kc.asec[i]];   // i: flat LLLR state of the output rows
  double *zr = z + S.off + (int64_t)(i - S.a0) * S.db;
  for (int32_t bl = threadIdx.x; bl < S.db; bl += 256) {
    const int32_t bf = S.b0 + bl;
    double acc = 0.0;
    for (int t = 0; t < kc.nt; t++) {
      const double c = kc.ct[t];
      const int32_t *lp = kc.lptr + (int64_t)t * (kc.na + 1), *rp = kc.rptr + (int64_t)t * (kc.nb + 1);
      for (int32_t e = lp[i]; e < lp[i + 1]; e++) {
        const int32_t a = kc.lidx[e];
        const int sa = kc.asec[a];
        const double pl = c * kc.lval[e];
        for (int32_t f = rp[bf]; f < rp[bf + 1]; f++) {
          const int32_t b = kc.ridx[f];
          if (kc.bsec[b] != sa) continue;
          const double p = pl * kc.rval[f];
          if (!(fabs(p) > 1.0e-15)) continue;
          const KronSector T = kc.sec[sa];
          acc += p * x[T.off + (int64_t)(a - T.a0) * T.db + (b - T.b0)];
        }
      }
    }
    zr[bl] = acc;
  }
}

__global__ __launch_bounds__(256) void k_kron_cross(KronCross kc, const double *__restrict__ x, double *__restrict__ z) {
  kron_cross_row(kc, blockIdx.x, x, z);
}

__global__ __launch_bounds__(256) void k_zero(int64_t n, double *p) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0.0;
}

// Output tiles of t x t over all sectors, in launch order: the sectors cut into bands of whole
// tile rows, the bands dealt to the eight XCDs (workgroup i runs on XCD i mod 8) by their work, so
// that a band's operands are read into one L2 (KLM m = 799: L2 misses 1.8 M lines a product
// against 4.0 M with the tiles dealt by length alone, a solve 83 ms against 92); each XCD's
// bands longest k extent (da + db) first, so that the short tiles fill in behind the long ones.
std::vector<KronTile> kron_tiles(const std::vector<KronSector> &sec, int32_t t) {
  auto rows = [&](size_t s) { return (sec[s].da + t - 1) / t; };
  auto cols = [&](size_t s) { return (sec[s].db + t - 1) / t; };
  auto length = [&](size_t s) { return sec[s].da + sec[s].db; };
  double total = 0.0;
  for (size_t s = 0; s < sec.size(); s++) total += (double)rows(s) * cols(s) * length(s);
  struct Band {
    size_t sector;
    int32_t i0, i1;
    double work;
  };
  std::vector<Band> bands;
  for (size_t s = 0; s < sec.size(); s++) {
    const double row = (double)cols(s) * length(s);
    const int32_t n = rows(s), cut = std::min(n, (int32_t)std::ceil(row * n / (total / (4 * kXcds))));
    for (int32_t c = 0; c < cut; c++) {
      const int32_t i0 = (int32_t)((int64_t)n * c / cut), i1 = (int32_t)((int64_t)n * (c + 1) / cut);
      bands.push_back(Band{s, i0, i1, row * (i1 - i0)});
    }
  }
  std::stable_sort(bands.begin(), bands.end(), [](const Band &a, const Band &b) { return a.work > b.work; });
  double load[kXcds] = {};
  std::vector<Band> mine[kXcds];
  for (const Band &b : bands) {
    const int q = (int)(std::min_element(load, load + kXcds) - load);
    load[q] += b.work;
    mine[q].push_back(b);
  }
  std::vector<KronTile> queue[kXcds], out;
  for (int q = 0; q < kXcds; q++) {
    std::stable_sort(mine[q].begin(), mine[q].end(),
                     [&](const Band &a, const Band &b) { return length(a.sector) > length(b.sector); });
    for (const Band &b : mine[q])
      for (int32_t i = b.i0; i < b.i1; i++)
        for (int32_t j = 0; j < cols(b.sector); j++) queue[q].emplace_back(sec[b.sector], i * t, j * t);
  }
  size_t nt = 0, at[kXcds] = {};
  for (const auto &q : queue) nt += q.size();
  for (size_t p = 0; p < nt; p++) {
    int q = (int)(p % kXcds);
    if (at[q] == queue[q].size())   // used up: the one with most left
      for (int k = 0; k < kXcds; k++)
        if (queue[k].size() - at[k] > queue[q].size() - at[q]) q = k;
    out.push_back(queue[q][at[q]++]);
  }
  return out;
}

// 32 x 32 tiles once there are enough of them to keep the 256 CUs' four slots each busy
// through a good part of the launch; below, 16 x 16 tiles, whose chains are shorter and which
// are four times as many.  Solves, microseconds a step, 16 x 16 against 32 x 32: Hubbard m = 396
// (208 tiles of 32) 18.9 and 20.4, KLM m = 280 (313) 23.6 and 23.6, m = 400 (580) 41.1 and 35.5,
// m = 799 (2133) 196 and 107.
int kron_shape_rule(const KronDev &K) { return K.ntiles[1] >= 400 ? 1 : 0; }

// The short form of the coupling terms (KronMap) from their lists; false if some term has a
// state with several targets, or with targets in several sectors.
bool kron_maps(const KronDev &K, const std::vector<int32_t> &asec, const std::vector<int32_t> &bsec,
               const std::vector<double> &ct, const std::vector<int32_t> &lptr, const std::vector<int32_t> &lidx,
               const std::vector<double> &lval, const std::vector<int32_t> &rptr, const std::vector<int32_t> &ridx,
               const std::vector<double> &rval, std::vector<KronMap> &lmap, std::vector<KronMap> &rmap) {
  const int nt = (int)ct.size();
  lmap.assign((size_t)nt * K.na, KronMap{0.0, -1, 0});
  rmap.assign((size_t)nt * K.nb, KronMap{0.0, -1, 0});
  for (int t = 0; t < nt; t++) {
    const int32_t *lp = lptr.data() + (size_t)t * (K.na + 1), *rp = rptr.data() + (size_t)t * (K.nb + 1);
    for (const KronSector &S : K.hsec) {
      int32_t sa = -1, sb = -1;   // target sectors
      for (int32_t i = S.a0; i < S.a0 + S.da; i++) {
        if (lp[i + 1] - lp[i] > 1) return false;
        for (int32_t e = lp[i]; e < lp[i + 1]; e++) {
          const int32_t q = asec[lidx[e]];
          if (sa >= 0 && q != sa) return false;
          sa = q;
        }
      }
      for (int32_t i = S.b0; i < S.b0 + S.db; i++) {
        if (rp[i + 1] - rp[i] > 1) return false;
        for (int32_t e = rp[i]; e < rp[i + 1]; e++) {
          const int32_t q = bsec[ridx[e]];
          if (sb >= 0 && q != sb) return false;
          sb = q;
        }
      }
      if (sa < 0 || sa != sb) continue;
      const KronSector &T = K.hsec[sa];
      for (int32_t i = S.a0; i < S.a0 + S.da; i++)
        if (lp[i + 1] > lp[i]) {
          const int32_t e = lp[i];
          lmap[(size_t)t * K.na + i] = KronMap{ct[t] * lval[e], (int32_t)(T.off + (int64_t)(lidx[e] - T.a0) * T.db), 0};
        }
      for (int32_t i = S.b0; i < S.b0 + S.db; i++)
        if (rp[i + 1] > rp[i]) rmap[(size_t)t * K.nb + i] = KronMap{rval[rp[i]], ridx[rp[i]] - T.b0, 0};
    }
  }
  return true;
}

bool left_kind(int k) { return k == K_LL || k == K_LR || k == K_LLLR; }
bool right_kind(int k) { return k == K_RR || k == K_RL || k == K_RRRL; }

}  // namespace

int KronDev::shape() const { return variant == 0 ? 0 : variant == 2 ? 1 : rule; }

void KronDev::cross(const double *x, hipStream_t s) const {
  if (!general || na == 0) return;
  const KronCross kc{ncross, na, nb, ct.p, lptr.p, lidx.p, rptr.p, ridx.p, lval.p, rval.p, asec.p, bsec.p, sec.p};
  k_kron_cross<<<na, 256, 0, s>>>(kc, x, zc.p);
  HIPCHK(hipGetLastError());
}

}  // namespace dmrgx

using namespace dmrgx;

struct dmrgx_kron {
  KronDev K;
};

namespace dmrgx {
const KronDev &kron_dev(const dmrgx_kron *K) { return K->K; }
}  // namespace dmrgx

extern "C" {

int dmrgx_superblock_kron(const dmrgx_superblock *S, dmrgx_kron **out) {
  if (!S || !out) return DMRGX_ERR_ARG;
  *out = nullptr;
  return run_status([&] {
    auto H = std::make_unique<dmrgx_kron>();
    KronDev &K = H->K;
    const int32_t n = S->n, d = S->d;
    K.n = n;
    K.sb = S;
    hipStream_t st = ctx().stream;
    std::vector<int16_t> aLL, aLR, bRR, bRL;
    std::vector<int32_t> asec, bsec;
    if (!S->qn_sec.empty()) {
      // the sectors as the basis was built from them
      for (size_t s = 0; s < S->qn_sec.size(); s++) {
        const BasisSector &q = S->qn_sec[s];
        const bool end = s + 1 == S->qn_sec.size();
        KronSector sc{};
        sc.off = q.off;
        sc.db = q.dB;
        sc.da = (end ? (int32_t)(S->qn_a.size() / 2) : S->qn_sec[s + 1].a0) - q.a0;
        sc.a0 = (int32_t)aLL.size();
        sc.b0 = (int32_t)bRR.size();
        for (int32_t i = 0; i < sc.da; i++) {
          aLL.push_back(S->qn_a[2 * (q.a0 + i)]);
          aLR.push_back(S->qn_a[2 * (q.a0 + i) + 1]);
          asec.push_back(K.nsec);
        }
        for (int32_t j = 0; j < sc.db; j++) {
          bRR.push_back(S->qn_b[2 * (q.b0 + j)]);
          bRL.push_back(S->qn_b[2 * (q.b0 + j) + 1]);
          bsec.push_back(K.nsec);
        }
        K.hsec.push_back(sc);
        K.nsec++;
      }
    } else {   // the basis (host copy) and its sectors
      std::vector<int16_t> LL(n), LR(n), RR(n), RL(n);
      ctx().copy_out(LL.data(), S->LL.p, sizeof(int16_t) * n);
      ctx().copy_out(LR.data(), S->LR.p, sizeof(int16_t) * n);
      ctx().copy_out(RR.data(), S->RR.p, sizeof(int16_t) * n);
      ctx().copy_out(RL.data(), S->RL.p, sizeof(int16_t) * n);
      int64_t r = 0;
      while (r < n) {
        KronSector sc{};
        sc.off = r;
        // db: rows until (LL, LR) changes; da: runs of db rows with the same RRRL sequence
        int64_t e = r;
        while (e < n && LL[e] == LL[r] && LR[e] == LR[r]) e++;
        sc.db = (int32_t)(e - r);
        int64_t a = r;
        while (a < n && a + sc.db <= n && RR[a] == RR[r] && RL[a] == RL[r]) a += sc.db;
        sc.da = (int32_t)((a - r) / sc.db);
        // every row of the sector must be (LLLR state i, RRRL state j) at off + i db + j
        // the product check: every row run of the sector has one (LL, LR) and the first run's
        // RRRL sequence
        for (int32_t i = 0; i < sc.da; i++) {
          const int64_t q0 = r + (int64_t)i * sc.db;
          int same = std::memcmp(&RR[q0], &RR[r], sizeof(int16_t) * sc.db) == 0 &&
                     std::memcmp(&RL[q0], &RL[r], sizeof(int16_t) * sc.db) == 0;
          const int16_t ll = LL[q0], lr = LR[q0];
          for (int32_t j = 1; j < sc.db; j++) same &= (int)(LL[q0 + j] == ll) & (int)(LR[q0 + j] == lr);
          if (!same) throw Failure(DMRGX_ERR_ARG, "superblock basis is not a product of LLLR and RRRL states per sector");
        }
        sc.a0 = (int32_t)aLL.size();
        sc.b0 = (int32_t)bRR.size();
        for (int32_t i = 0; i < sc.da; i++) {
          aLL.push_back(LL[r + (int64_t)i * sc.db]);
          aLR.push_back(LR[r + (int64_t)i * sc.db]);
          asec.push_back(K.nsec);
        }
        for (int32_t j = 0; j < sc.db; j++) {
          bRR.push_back(RR[r + j]);
          bRL.push_back(RL[r + j]);
          bsec.push_back(K.nsec);
        }
        K.hsec.push_back(sc);
        K.nsec++;
        r += (int64_t)sc.da * sc.db;
      }
    }
    // state -> flat index maps (each LLLR / RRRL state belongs to one sector)
    std::vector<int32_t> aidx((size_t)S->dim_LL * d, -1), bidx((size_t)S->dim_RR * d, -1);
    for (size_t i = 0; i < aLL.size(); i++) {
      int32_t &m = aidx[(size_t)aLL[i] * d + aLR[i]];
      if (m >= 0) throw Failure(DMRGX_ERR_ARG, "an LLLR state appears in two sectors");
      m = (int32_t)i;
    }
    for (size_t i = 0; i < bRR.size(); i++) {
      int32_t &m = bidx[(size_t)bRR[i] * d + bRL[i]];
      if (m >= 0) throw Failure(DMRGX_ERR_ARG, "an RRRL state appears in two sectors");
      m = (int32_t)i;
    }
    K.na = (int32_t)aLL.size();
    K.nb = (int32_t)bRR.size();
    int64_t ml = 0, mr = 0;
    for (KronSector &sc : K.hsec) {
      const int64_t na16 = (sc.da + 15) / 16, nb16 = (sc.db + 15) / 16;
      sc.ml = ml;
      sc.mr = mr;
      ml += na16 * na16 * 256;
      mr += nb16 * nb16 * 256;
      K.flops += 2.0 * sc.da * sc.db * (double)(sc.da + sc.db);
    }
    std::vector<KronTile> tiles[kKronShapes];
    for (int sh = 0; sh < kKronShapes; sh++) {
      tiles[sh] = kron_tiles(K.hsec, kKronTile[sh]);
      K.ntiles[sh] = (int32_t)tiles[sh].size();
    }
    K.rule = kron_shape_rule(K);
    // the term list split by the halves it acts on
    std::vector<int32_t> left, right, cross;
    for (size_t i = 0; i < S->hterms.size(); i++) {
      const int k = S->hterms[i].kind;
      if (left_kind(k)) left.push_back((int32_t)i);
      else if (right_kind(k)) right.push_back((int32_t)i);
      else cross.push_back((int32_t)i);
    }
    K.ncross = (int32_t)cross.size();
    // the coupling terms' per-state lists (see k_kron_cross), from host copies of the operators
    std::vector<double> ct, lval, rval;
    std::vector<int32_t> lptr, lidx, rptr, ridx;
    std::vector<KronMap> lmap, rmap;
    Upload up;
    {
      for (int32_t ci : cross) {
        const DTerm &t = S->hterms[ci];
        const auto &r1 = S->hop[t.op1].row, &r2 = S->hop[t.op2].row;
        const auto &c1 = S->hop[t.op1].col, &c2 = S->hop[t.op2].col;
        const auto &v1 = S->hop[t.op1].val, &v2 = S->hop[t.op2].val;
        auto par = [&](int e, int state) { return S->hele[e][state]; };
        // parity of the row's LLLR part and of its RRRL part in the term's sign rule
        auto left_parity = [&](int ll, int lr) {
          if (t.sign_mode == 0) return 0;
          switch (t.kind) {
            case K_LLRL: return par(t.e0, ll) + par(t.e2, lr);
            case K_LLRR: return par(t.e0, ll) + par(t.e1, lr);
            case K_LRRL: return par(t.e1, lr);
            case K_LRRR: return par(t.e0, lr);
            default: return 0;
          }
        };
        auto right_parity = [&](int rr) {
          if (t.sign_mode == 0) return 0;
          switch (t.kind) {
            case K_LLRL: return par(t.e1, rr);
            case K_LRRL: return par(t.e0, rr);
            default: return 0;
          }
        };
        ct.push_back((t.sign_mode == 1 ? -1.0 : 1.0) * t.coeff);
        for (int32_t i = 0; i < K.na; i++) {
          lptr.push_back((int32_t)lidx.size());
          const int q[2] = {aLL[i], aLR[i]};
          const double sg = (left_parity(q[0], q[1]) % 2 == 0) ? 1.0 : -1.0;
          for (int64_t e = r1[q[t.s1]]; e < r1[q[t.s1] + 1]; e++) {
            int qq[2] = {q[0], q[1]};
            qq[t.s1] = c1[e];
            const int32_t a = aidx[(size_t)qq[0] * d + qq[1]];
            if (a < 0) continue;
            lidx.push_back(a);
            lval.push_back(sg * v1[e]);
          }
        }
        lptr.push_back((int32_t)lidx.size());
        for (int32_t i = 0; i < K.nb; i++) {
          rptr.push_back((int32_t)ridx.size());
          const int q[4] = {0, 0, bRR[i], bRL[i]};
          const double sg = (right_parity(q[2]) % 2 == 0) ? 1.0 : -1.0;
          for (int64_t e = r2[q[t.s2]]; e < r2[q[t.s2] + 1]; e++) {
            int qq[4] = {q[0], q[1], q[2], q[3]};
            qq[t.s2] = c2[e];
            const int32_t b = bidx[(size_t)qq[2] * d + qq[3]];
            if (b < 0) continue;
            ridx.push_back(b);
            rval.push_back(sg * v2[e]);
          }
        }
        rptr.push_back((int32_t)ridx.size());
      }
      if ((int64_t)lidx.size() > INT32_MAX / 2 || (int64_t)ridx.size() > INT32_MAX / 2)
        throw Failure(DMRGX_ERR_ARG, "coupling-term lists too long");
      // the short form: at most one target per state and term, and per term and sector one
      // target sector on each half (an operator of a site changes the quantum numbers by a
      // fixed amount); a term and sector whose target sectors differ contributes nothing
      K.general = !kron_maps(K, asec, bsec, ct, lptr, lidx, lval, rptr, ridx, rval, lmap, rmap);
      if (K.general) {
        up.add(K.ct, ct);
        up.add(K.lptr, lptr);
        up.add(K.lidx, lidx);
        up.add(K.lval, lval);
        up.add(K.rptr, rptr);
        up.add(K.ridx, ridx);
        up.add(K.rval, rval);
        K.zc.resize(n);
      } else {
        up.add(K.lmap, lmap);
        up.add(K.rmap, rmap);
      }
    }
    up.add(K.sec, K.hsec);
    for (int sh = 0; sh < kKronShapes; sh++) up.add(K.tiles[sh], tiles[sh]);
    DevView<int16_t> daLL, daLR, dbRR, dbRL;   // read by the kernels below only
    DevView<int32_t> dleft, dright;
    up.add(daLL, aLL);
    up.add(daLR, aLR);
    up.add(dbRR, bRR);
    up.add(dbRL, bRL);
    up.add(K.asec, asec);
    up.add(K.bsec, bsec);
    up.add(K.aidx, aidx);
    up.add(K.bidx, bidx);
    up.add(dleft, left);
    up.add(dright, right);
    up.place(K.pack);
    up.send();
    K.ML.resize(std::max<int64_t>(ml, 1));
    K.MR.resize(std::max<int64_t>(mr, 1));
    k_zero<<<1024, 256, 0, st>>>(ml, K.ML.p);
    k_zero<<<1024, 256, 0, st>>>(mr, K.MR.p);
    const KronBuild kb{d, K.na, K.nb, daLL.p, daLR.p, dbRR.p, dbRL.p, K.asec.p, K.bsec.p, K.aidx.p, K.bidx.p, K.sec.p};
    int32_t widest = 0;
    for (const KronSector &sc : K.hsec) widest = std::max({widest, sc.da, sc.db});
    const int nl = (int)left.size(), nr = (int)right.size();
#define HALF_ARGS(ids, n, M) kb, S->terms.p, ids.p, n, S->ops.p, S->ele_ptrs.p, M.p
    if (K.na > 0 && K.nb > 0) {
      if (S->ascending && widest <= kHalfRow) {
        k_kron_half<true><<<(K.na + 3) / 4, 256, 0, st>>>(HALF_ARGS(dleft, nl, K.ML));
        k_kron_half<false><<<(K.nb + 3) / 4, 256, 0, st>>>(HALF_ARGS(dright, nr, K.MR));
      } else {
        k_kron_left<<<(K.na + 255) / 256, 256, 0, st>>>(HALF_ARGS(dleft, nl, K.ML));
        k_kron_right<<<(K.nb + 255) / 256, 256, 0, st>>>(HALF_ARGS(dright, nr, K.MR));
      }
    }
#undef HALF_ARGS
    HIPCHK(hipGetLastError());
    *out = H.release();   // no wait: the host lists have been read, products queue behind the build
  });
}

int dmrgx_kron_info(const dmrgx_kron *K, int32_t *n, int32_t *sectors, int32_t *coupling_terms, double *flops) {
  if (!K) return DMRGX_ERR_ARG;
  if (n) *n = K->K.n;
  if (sectors) *sectors = K->K.nsec;
  if (coupling_terms) *coupling_terms = K->K.ncross;
  if (flops) *flops = K->K.flops;
  return DMRGX_OK;
}

int dmrgx_kron_set_kernel(dmrgx_kron *K, int32_t variant) {
  if (!K || variant < 0 || variant >= kKronVariants) return DMRGX_ERR_ARG;
  K->K.variant = variant;
  return DMRGX_OK;
}

int dmrgx_kron_autotune(dmrgx_kron *K, int32_t *variant_out, double *us_out) {
  if (!K) return DMRGX_ERR_ARG;
  return run_status([&] {
    KronDev &D = K->K;
    hipStream_t st = ctx().stream;
    DevBuf<double> x(std::max<int32_t>(D.n, 1)), y(std::max<int32_t>(D.n, 1));
    launch_start_vector(D.n, 7, x.p, st);
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    int best = kKronDefault;
    float best_ms = 1e30f, dflt_ms = 1e30f;
    for (int v : {kKronDefault, 0, 2}) {
      D.variant = v;
      launch_spmv(op_of(D), x.p, y.p, st);
      HIPCHK(hipEventRecord(e0, st));
      for (int r = 0; r < 5; r++) launch_spmv(op_of(D), x.p, y.p, st);
      HIPCHK(hipEventRecord(e1, st));
      HIPCHK(hipEventSynchronize(e1));
      float ms = 0;
      HIPCHK(hipEventElapsedTime(&ms, e0, e1));
      if (v == kKronDefault) dflt_ms = ms;
      if (ms < best_ms) {
        best_ms = ms;
        best = v;
      }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    // the default stays unless another is more than 2 % faster: the five products' timing
    // varies by about 1 %
    if (dflt_ms <= 1.02f * best_ms) {
      best_ms = dflt_ms;
      best = kKronDefault;
    }
    D.variant = best;
    if (variant_out) *variant_out = best;
    if (us_out) *us_out = best_ms * 1000.0 / 5;
  });
}

int dmrgx_kron_spmv(const dmrgx_kron *K, const double *x, double *y) {
  if (!K || !x || !y) return DMRGX_ERR_ARG;
  return run_status([&] {
    const int32_t n = K->K.n;
    DevBuf<double> dx(n), dy(n);
    ctx().copy_in(dx.p, x, sizeof(double) * n);
    launch_spmv(op_of(K->K), dx.p, dy.p, ctx().stream);
    ctx().copy_out(y, dy.p, sizeof(double) * n);
  });
}

void dmrgx_kron_free(dmrgx_kron *K) {
  if (!K) return;
  (void)hipStreamSynchronize(ctx().stream);
  delete K;
}

}  // extern "C"
