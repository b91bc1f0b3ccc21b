// The fused product kernel of the Kronecker form: one launch computes a solver step's
// H x with its epilogue.  Included by kernels.hip, which holds the epilogues.
#pragma once

#include <hip/hip_runtime.h>

#include "internal.h"
#include "reduce.h"

namespace dmrgx {
namespace {

typedef double kron_v4d __attribute__((ext_vector_type(4)));

// Loads from a scalar base plus the lane's byte offset, as buffer loads: written with pointers the
// compiler keeps a 64-bit address per load and lane and moves it on with vector adds.
__device__ __forceinline__ auto kron_rsrc(const double *base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(base), 0, -1, 0x00027000);
}
__device__ __forceinline__ double kron_load(const double *base, int32_t bytes) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(kron_rsrc(base), bytes, 0, 0));
}
__device__ __forceinline__ double2 kron_load2(const double *base, int32_t bytes) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(kron_rsrc(base), bytes, 0, 0));
}

// The 16 k of a slab are dealt to v_mfma_f64_16x16x4 (A fragment: lane l holds A[l % 16][l / 16];
// B fragment: B[l / 16][l % 16]; result register v of lane l: D[4 v + l / 16][l % 16], as a
// one-hot scan of the instruction on gfx950 shows) so that lane group g = l / 16 takes
// k = 4 g + t in the slab's t-th instruction: any assignment gives the same sum, and this one
// makes a lane's values of a row neighbours in memory.  A fragment holds the operands of half a
// slab, t = 2 h and 2 h + 1.
template <int B>
struct KronFrag {
  double a[B][2], b[B][2];
};

// One output tile of one sector per workgroup: H x on 16 B x 16 B elements, both dense products in
// one accumulator,
//     M_L[rows, :] X[:, cols] + X[rows, :] M_R[cols, :]^T,
// then the coupling terms and the solver's epilogue (Epi, as in k_apply: normalisation,
// shift, dot product) on the finished elements.  The four wavefronts split the k range (the
// slabs of the left product, then those of the right one) and add their parts through LDS: a
// tile's chain of products is then a quarter as long, which is what small superblocks wait for
// and what lets tiles of very different length fill the chip evenly in large ones.
//
// What bounds it is the vector cache: a load whose neighbouring lanes lie in different rows
// takes a cycle per lane.  M_L and M_R are therefore stored in fragment order (kron_at), so
// that their loads are contiguous; the left product's X fragment is contiguous as it is
// (neighbouring lanes hold neighbouring columns); the right product's is read along
// its rows and turned round in LDS, in a part of it that only the wavefront itself uses
// (16 x 16 tiles, which small superblocks take and which wait for latency, load it directly).
// So there is no barrier in the loop: wavefronts run independently, operands ahead of the
// matrix instructions by half a slab or more.  FP64 matrix and vector instructions share their
// issue, so the loop holds no vector arithmetic: every load is a scalar base, moved on by
// the slab, plus an offset of the lane that the loop does not change (hence the shifted last slab,
// kron_slab: no clamping at the edge).
//
// Measured (MI355X, KLM m = 799: 3.23 GFLOP a product, 2133 tiles of 32 x 32): 88 us with the Lanczos
// epilogue and 75 with CG's, of which the matrix cores are busy 46; 64 x 64 LDS-staged tiles took 86 us
// and the epilogue's own kernel 14 to 25 more, with the coupling terms on a side stream.  Whole
// solves by tile: 32 x 32 83 ms, 32 x 64 84 to 87 ms, 64 x 64 101 to 107 ms.  Hubbard m = 396
// (68 MFLOP, 641 tiles of 16 x 16): 9 us against 30, most of it latency.
//
// M_L and M_R are zero where a shifted last slab repeats a k or a sector is narrower than a slab
// (X's operand there is its last row or column again), and in rows beyond the sector.
template <int B, class Epi>
__global__ __launch_bounds__(256, 4) void k_kron(KronView kv, const double *__restrict__ x, Epi epi, double *partial) {
  if (epi.skip()) return;
  constexpr bool kStaged = B > 1;
  constexpr int kRow = 18;   // doubles per staged row: 16-byte aligned, few bank conflicts (1.5 cycles an access)
  constexpr int E = 4 * B * B, NE = B * B;   // a wavefront's elements per lane, this one's finished
  constexpr int kStage = kStaged ? 16 * B * kRow : 0;
  constexpr int kLds = 2 * kStage > E * 64 ? 2 * kStage : E * 64;
  __shared__ __align__(16) double lds[4][kLds];   // per wavefront: two staged slabs, then its partial sums
  [[maybe_unused]] typename PreOf<Epi>::type pf;
  if constexpr (LateBegin<Epi>::value) epi.prefetch(pf);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, li = l & 15, g = l >> 4;
  const KronTile S = kv.tiles[blockIdx.x];
  const int32_t r0 = S.r0, c0 = S.c0;
  const double *X = x + S.off;
  // This lane's finished elements: the wavefront's quarter of the E that a lane holds of the tile
  // (element e is register e mod 4 of block (e / 4 / B, e / 4 mod B), at row 4 (e mod 4) + g and
  // column li of the 16 x 16 block).
  auto row_of = [&](int q) { return r0 + 16 * ((wave * NE + q) / 4 / B) + 4 * ((wave * NE + q) & 3) + g; };
  auto col_of = [&](int q) { return c0 + 16 * ((wave * NE + q) / 4 % B) + li; };
  // They start as the coupling terms: c_t c_l(row) c_r(column) x[target], one target at most
  // per term.  Taken before the products, a few terms at a time, so that their two dependent
  // loads are in flight together with the first operands'.
  double h[NE];
#pragma unroll
  for (int q = 0; q < NE; q++) h[q] = 0.0;
  constexpr int kTerms = 4;
  for (int t0 = 0; t0 < kv.ncross; t0 += kTerms) {
    double p[kTerms][NE];
    int32_t at[kTerms][NE];
#pragma unroll
    for (int u = 0; u < kTerms; u++) {
      const int t = min(t0 + u, kv.ncross - 1);
      const KronMap *lm = kv.lmap + (int64_t)t * kv.na + S.a0, *rm = kv.rmap + (int64_t)t * kv.nb + S.b0;
#pragma unroll
      for (int q = 0; q < NE; q++) {
        const KronMap a = lm[min(row_of(q), S.da - 1)], b = rm[min(col_of(q), S.db - 1)];
        p[u][q] = a.c * b.c;
        const bool on = t0 + u < kv.ncross && a.at >= 0 && b.at >= 0 && fabs(p[u][q]) > 1.0e-15;
        at[u][q] = on ? a.at + b.at : -1;
      }
    }
    double v[kTerms][NE];   // always loaded (element 0 for a term without a target)
#pragma unroll
    for (int u = 0; u < kTerms; u++)
#pragma unroll
      for (int q = 0; q < NE; q++) v[u][q] = x[max(at[u][q], 0)];
#pragma unroll
    for (int u = 0; u < kTerms; u++)
#pragma unroll
      for (int q = 0; q < NE; q++) h[q] += at[u][q] >= 0 ? p[u][q] * v[u][q] : 0.0;
  }
  kron_v4d acc[B][B];
#pragma unroll
  for (int e = 0; e < E; e++) acc[e / 4 / B][e / 4 % B][e & 3] = wave == e / NE ? h[e % NE] : 0.0;
  {
    const int32_t SL = (S.da + 15) >> 4, SR = (S.db + 15) >> 4, T = SL + SR;
    const int32_t s0 = T * wave / 4, s1 = T * (wave + 1) / 4;
    using Frag = KronFrag<B>;
    auto mma = [&](const Frag &f) {
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int i = 0; i < B; i++)
#pragma unroll
          for (int j = 0; j < B; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[i][t], f.b[j][t], acc[i][j], 0, 0, 0);
    };
    // half h of slab s of block row ib of a matrix in fragment order (ns slabs a block row)
    const int32_t lane16 = 16 * l;
    auto matrix = [&](double (&f)[2], const double *m, int32_t ib, int32_t ns, int32_t s, int h) {
      const double2 v = kron_load2(m + ((int64_t)ib * ns + s) * 256 + 128 * h, lane16);
      f[0] = v.x;
      f[1] = v.y;
    };
    // slabs [b, e) of one product with D half slabs loaded ahead (past the end the last slab is
    // loaded again, so that the loop has no branch between loads)
    constexpr int D = 4;
    auto run = [&](auto load, int32_t b, int32_t e) {
      if (b >= e) return;
      Frag f[D];
#pragma unroll
      for (int d = 0; d < D; d++) load(f[d], min(b + d / 2, e - 1), d & 1);
      int32_t s = b;
      for (; s + D / 2 <= e; s += D / 2)
#pragma unroll
        for (int d = 0; d < D; d++) {
          mma(f[d]);
          load(f[d], min(s + (d + D) / 2, e - 1), d & 1);
        }
#pragma unroll
      for (int d = 0; d < D - 2; d += 2)
        if (s + d / 2 < e) {
          mma(f[d]);
          mma(f[d + 1]);
        }
    };
    {   // left: A = M_L, B = X
      const double *m = kv.ML + S.ml;
      int32_t ib[B];
      int32_t off[4][B];   // of X[4 g + t, column]
#pragma unroll
      for (int i = 0; i < B; i++) ib[i] = min((r0 >> 4) + i, SL - 1);
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int j = 0; j < B; j++)
          off[t][j] = 8 * (int32_t)((uint32_t)min(4 * g + t, S.da - 1) * (uint32_t)S.db + (uint32_t)min(c0 + 16 * j + li, S.db - 1));
      run(
          [&](Frag &f, int32_t s, int h) {
            const double *base = X + (int64_t)kron_slab(s, S.da) * S.db;
#pragma unroll
            for (int i = 0; i < B; i++) matrix(f.a[i], m, ib[i], SL, s, h);
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
              for (int j = 0; j < B; j++) f.b[j][t] = kron_load(base, off[2 * h + t][j]);
          },
          min(s0, SL), min(s1, SL));
    }
    {   // right: A = X, B = M_R^T
      const double *m = kv.MR + S.mr;
      const int32_t b = max(s0, SL) - SL, e = max(s1, SL) - SL;
      int32_t jb[B];
#pragma unroll
      for (int j = 0; j < B; j++) jb[j] = min((c0 >> 4) + j, SR - 1);
      if constexpr (!kStaged) {
        const double *Xr = X + (int64_t)r0 * S.db;
        int32_t off[4][B];   // of X[row, 4 g + t]
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
          for (int i = 0; i < B; i++)
            off[t][i] = 8 * (int32_t)((uint32_t)(min(r0 + 16 * i + li, S.da - 1) - r0) * (uint32_t)S.db +
                              (uint32_t)min(4 * g + t, S.db - 1));
        run(
            [&](Frag &f, int32_t s, int h) {
              const double *base = Xr + kron_slab(s, S.db);
#pragma unroll
              for (int j = 0; j < B; j++) matrix(f.b[j], m, jb[j], SR, s, h);
#pragma unroll
              for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < B; i++) f.a[i][t] = kron_load(base, off[2 * h + t][i]);
            },
            b, e);
      } else if (b < e) {
        double *stage = lds[wave];
        // staged elements of this lane: rows g + 4 u, column li of the slab
        const double *Xr = X + (int64_t)r0 * S.db;
        int32_t off[4 * B];
#pragma unroll
        for (int u = 0; u < 4 * B; u++)
          off[u] = 8 * (int32_t)((uint32_t)(min(r0 + g + 4 * u, S.da - 1) - r0) * (uint32_t)S.db + (uint32_t)min(li, S.db - 1));
        auto fetch = [&](double (&q)[4 * B], int32_t s) {
          const double *base = Xr + kron_slab(s, S.db);
#pragma unroll
          for (int u = 0; u < 4 * B; u++) q[u] = kron_load(base, off[u]);
        };
        auto put = [&](const double (&q)[4 * B], int buf) {
          __builtin_amdgcn_wave_barrier();   // LDS is in order per wavefront: only the compiler must keep it
#pragma unroll
          for (int u = 0; u < 4 * B; u++) stage[buf * kStage + (g + 4 * u) * kRow + li] = q[u];
          __builtin_amdgcn_wave_barrier();
        };
        auto load = [&](Frag &f, int32_t s, int h, int buf) {
#pragma unroll
          for (int j = 0; j < B; j++) matrix(f.b[j], m, jb[j], SR, s, h);
#pragma unroll
          for (int i = 0; i < B; i++) {
            const double2 v =
                *reinterpret_cast<const double2 *>(stage + buf * kStage + (16 * i + li) * kRow + 4 * g + 2 * h);
            f.a[i][0] = v.x;
            f.a[i][1] = v.y;
          }
        };
        Frag f0, f1;
        double q[4 * B];
        fetch(q, b);
        put(q, 0);
        fetch(q, min(b + 1, e - 1));
        load(f0, b, 0, 0);
        load(f1, b, 1, 0);
        auto step = [&](int32_t s, int buf) {   // slab s from f0, f1; s + 1 (staged in buf) into them
          put(q, buf);
          fetch(q, min(s + 2, e - 1));
          mma(f0);
          load(f0, min(s + 1, e - 1), 0, buf);
          mma(f1);
          load(f1, min(s + 1, e - 1), 1, buf);
        };
        int32_t s = b;
        for (; s + 1 < e; s += 2) {
          step(s, 1);
          step(s + 1, 0);
        }
        if (s < e) {
          mma(f0);
          mma(f1);
        }
      }
    }
  }
#pragma unroll
  for (int e = 0; e < E; e++) lds[wave][e * 64 + l] = acc[e / 4 / B][e / 4 % B][e & 3];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NE; q++) {
    const int at = (wave * NE + q) * 64 + l;
    h[q] = (lds[0][at] + lds[1][at]) + (lds[2][at] + lds[3][at]);
  }
  if constexpr (LateBegin<Epi>::value) epi.begin(pf);
  else epi.begin();
  double sum = 0.0;
#pragma unroll
  for (int q = 0; q < NE; q++) {
    const int32_t r = row_of(q), c = col_of(q);
    if (r < S.da && c < S.db) {
      const int32_t at = (int32_t)(S.off + (int64_t)r * S.db + c);
      sum += epi.row(at, kv.zc ? h[q] + kv.zc[at] : h[q]);
    }
  }
  if constexpr (Epi::kReduce) block_partial(sum, partial);
}

}  // namespace
}  // namespace dmrgx
