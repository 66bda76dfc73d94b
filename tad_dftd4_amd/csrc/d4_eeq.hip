// HIP kernels (gfx950) for the EEQ charges and their adjoint.
//
// Molecules whose packed Coulomb factor fits in LDS are solved by one
// work-group each (L D L^T by whole waves, FP64 matrix instructions); larger molecules use the tiled multi-work-group path.
// Every output element has one writer and every reduction a fixed order.

#include <map>
#include <mutex>
#include <utility>

#include "d4_device.h"

namespace d4 {
namespace {

// --------------------------------------------------------------------------
// EEQ charges: one work-group per molecule.
//
// The bordered system [[C, e], [e^T, 0]] [q; mu] = [b; Q] is solved with a
// symmetric factorisation of the Coulomb block C (in LDS when it fits) and the
// Schur complement of the border: q = y - mu z with y = C^-1 b, z = C^-1 e,
// mu = (e.y - Q) / (e.z). A non-positive pivot flags the molecule for the
// pivoted-LU kernel below.
// --------------------------------------------------------------------------

// ---- blocked Cholesky (16-column blocks) on a packed lower triangle -------
//
// Row i of the matrix starts at L + tri(i). For each block column kb:
//  1. wave 0 factorises the diagonal 16 x 16 block D in registers (lane r
//     holds row r; entries are broadcast with v_readlane, no LDS round trip)
//     and stores X = D^-1 (lower triangular) in its place;
//  2. every panel row below becomes a X^T (a = the row's block entries) and
//     the carried right-hand sides become X b: independent per thread;
//  3. the trailing triangle is updated in register tiles.
// The substitutions read X from the stored factor in the same way, so each
// solve step is a small parallel matrix-vector product between two barriers
// and no thread runs a serial dependent chain longer than 16 terms.
// All helpers are force-inlined so that pointers into LDS keep their
// address space (ds_* instructions rather than flat ones).

constexpr int kNB = 16;

__device__ __forceinline__ double lane_bcast(double v, int src) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), src);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), src);
  return __hiloint2double(hi, lo);
}

// Factor the diagonal block at kb (nb <= 16 rows) on wave 0 and overwrite it
// with the inverse of its Cholesky factor. Rows nb..15 are padded with the
// identity (their columns never mix with the real rows: their off-diagonal
// entries are zero and stay zero). Returns non-zero (uniform over the wave) if a pivot was not
// positive; the block is then left unspecified.
template <typename P>
__device__ __forceinline__ int chol_diag_block(P L, int kb, int nb) {
  const int lane = threadIdx.x & 63;
  double d[kNB];
#pragma unroll
  for (int c = 0; c < kNB; ++c) {
    double v = (c == lane) ? 1.0 : 0.0;
    if (lane < nb && c <= lane) v = L[tri(kb + lane) + kb + c];
    d[c] = v;
  }
  double invd[kNB];
  int bad = 0;
#pragma unroll
  for (int j = 0; j < kNB; ++j) {
    const double piv = lane_bcast(d[j], j);
    bad |= !(piv > 0.0);
    // 1 / sqrt(piv): hardware estimate and two Newton steps (the diagonal
    // of the factor itself is never needed, only its reciprocal)
    const double pv = piv > 0.0 ? piv : 1.0;
    double inv = __builtin_amdgcn_rsq(pv);
    inv = inv * fma(-0.5 * pv * inv, inv, 1.5);
    inv = inv * fma(-0.5 * pv * inv, inv, 1.5);
    const double s = pv * inv;
    invd[j] = inv;
    // Lanes above the diagonal (lane < j) carry junk from here on in d[j] and
    // in the columns they update; only lanes >= column are ever broadcast
    // (pivots and L[c][j] with c > j), so the junk is never read.
    d[j] = lane == j ? s : d[j] * inv;
#pragma unroll
    for (int c = j + 1; c < kNB; ++c) d[c] = fma(-d[j], lane_bcast(d[j], c), d[c]);
  }
  // lane r forms column r of X = D^-1 by forward substitution
  double x[kNB];
#pragma unroll
  for (int i = 0; i < kNB; ++i) {
    double s = (i == lane) ? 1.0 : 0.0;
#pragma unroll
    for (int k = 0; k < i; ++k) s = fma(-lane_bcast(d[k], i), x[k], s);
    x[i] = s * invd[i];
  }
  if (lane < nb) {
#pragma unroll
    for (int i = 0; i < kNB; ++i)
      if (i >= lane && i < nb) L[tri(kb + i) + kb + lane] = x[i];
  }
  return bad;
}

// Panel row i (full block, nb = 16): L[i][kb..kb+16) <- a X^T.
template <typename P>
__device__ __forceinline__ void panel_row(P L, int kb, int i) {
  P Li = L + tri(i) + kb;
  double a[kNB];
#pragma unroll
  for (int c = 0; c < kNB; ++c) a[c] = Li[c];
#pragma unroll
  for (int c = 0; c < kNB; ++c) {
    P Xc = L + tri(kb + c) + kb;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k <= c; ++k) s = fma(a[k], Xc[k], s);
    Li[c] = s;
  }
}

// Block forward step on a vector: v[kb..kb+nb) <- X v[kb..kb+nb), copied to y.
template <typename P, typename V>
__device__ __forceinline__ void block_lower(P L, int kb, int nb, V v, double* y) {
  double a[kNB];
#pragma unroll
  for (int c = 0; c < kNB; ++c) a[c] = c < nb ? v[kb + c] : 0.0;
#pragma unroll
  for (int c = 0; c < kNB; ++c) {
    if (c < nb) {
      P Xc = L + tri(kb + c) + kb;
      double s = 0.0;
#pragma unroll
      for (int k = 0; k <= c; ++k) s = fma(a[k], Xc[k], s);
      v[kb + c] = s;
      y[c] = s;
    }
  }
}

// Trailing update of one T x T tile: rows r0 + T ti + a, columns r0 + T tj + b
// (lower part only) lose the product of their panel rows.
template <int T, typename P>
__device__ __forceinline__ void trailing_tile(P L, int kb, int r0, int ti, int tj, int n) {
  const int i0 = r0 + T * ti, j0 = r0 + T * tj;
  P pi[T], pj[T];
#pragma unroll
  for (int a = 0; a < T; ++a) {
    pi[a] = L + tri(min(i0 + a, n - 1)) + kb;
    pj[a] = L + tri(min(j0 + a, n - 1)) + kb;
  }
  double acc[T][T];
#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int b = 0; b < T; ++b) acc[a][b] = 0.0;
#pragma unroll 1  // a rolled loop keeps only one chunk of rows in registers
  for (int c0 = 0; c0 < kNB; c0 += 4) {
    double xi[T][4], xj[T][4];
#pragma unroll
    for (int a = 0; a < T; ++a)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        xi[a][c] = pi[a][c0 + c];
        xj[a][c] = pj[a][c0 + c];
      }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int a = 0; a < T; ++a)
#pragma unroll
        for (int b = 0; b < T; ++b) acc[a][b] = fma(xi[a][c], xj[b][c], acc[a][b]);
  }
#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int b = 0; b < T; ++b) {
      const int i = i0 + a, j = j0 + b;
      if (i < n && j <= i) L[tri(i) + j] -= acc[a][b];
    }
}

__device__ __forceinline__ void tile_index(int e, int& ti, int& tj) {
  int r = (int)((sqrtf(8.0f * (float)e + 1.0f) - 1.0f) * 0.5f);
  while (r * (r + 1) / 2 > e) --r;
  while ((r + 1) * (r + 2) / 2 <= e) ++r;
  ti = r;
  tj = e - r * (r + 1) / 2;
}

// Trailing triangle (rows and columns r0..n-1) in T x T tiles, plus the
// update of the two carried right-hand sides by the block's solution y.
template <int T, bool RHS, typename P, typename V>
__device__ __forceinline__ void trailing_update(P L, int kb, int n, V rb, V re,
                                                const double* yblk) {
  const int r0 = kb + kNB;
  const int mr = n - r0;
  const int mt = (mr + T - 1) / T;
  const int ntl = mt * (mt + 1) / 2;
  // right-hand-side rows first, on the threads that the tiles leave idle last
  const int first = (256 - (ntl + mr) % 256) % 256;
  for (int e = threadIdx.x - first; RHS && e < mr; e += 256) {
    if (e < 0) continue;
    const int i = r0 + e;
    P Pi = L + tri(i) + kb;
    double sb = 0.0, se = 0.0;
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      sb = fma(Pi[c], yblk[c], sb);
      se = fma(Pi[c], yblk[kNB + c], se);
    }
    rb[i] -= sb;
    re[i] -= se;
  }
  for (int e = threadIdx.x; e < ntl; e += 256) {
    int ti, tj;
    tile_index(e, ti, tj);
    trailing_tile<T>(L, kb, r0, ti, tj, n);
  }
}

// Blocked right-looking Cholesky of the assembled n x n lower triangle; the
// diagonal blocks end up holding their inverses. With RHS, two right-hand
// sides are carried along (forward substitution fused): on return rb, re
// hold L^-1 b and L^-1 e. yblk: 2 * kNB doubles of LDS, flag: one double.
// Returns non-zero if a pivot was not positive.
template <bool RHS, typename P, typename V>
__device__ __forceinline__ int chol_factor(P L, int n, V rb, V re, double* yblk,
                                           double* flag) {
  const int tid = threadIdx.x;
  constexpr int nrhs = RHS ? 2 : 0;
  for (int kb = 0; kb < n; kb += kNB) {
    const int nb = min(kNB, n - kb);
    if (tid < 64) {
      const int bad = chol_diag_block(L, kb, nb);
      if (tid == 0) flag[0] = bad ? 1.0 : 0.0;
    }
    __syncthreads();
    if (flag[0] != 0.0) return 1;  // uniform
    const int mr = n - kb - nb;    // > 0 only for full blocks
    for (int t2 = tid; t2 < mr + nrhs; t2 += 256) {
      if (t2 < mr)
        panel_row(L, kb, kb + nb + t2);
      else if (RHS)
        block_lower(L, kb, nb, t2 == mr ? rb : re, yblk + (t2 - mr) * kNB);
    }
    __syncthreads();
    if (mr > 0) {
      if (mr >= 48)
        trailing_update<4, RHS>(L, kb, n, rb, re, yblk);
      else
        trailing_update<2, RHS>(L, kb, n, rb, re, yblk);
    }
    __syncthreads();
  }
  return 0;
}

// ---- L D L^T by whole waves (molecules held in LDS) ------------------------
//
// Row i of the matrix starts at L + tri(i); the border rows b and e live in
// registers (thread i holds entry i of both). On return the strict lower
// triangle holds L (unit diagonal), the diagonal the pivots D. Per 16-column
// block:
//  1. left-looking update: 16 x 16 tiles of the block column lose the product
//     of their finished rows, four v_mfma_f64_16x16x4 per earlier block. The
//     FP64 matrix rate equals the vector one here; what this saves is LDS
//     traffic: 6 to 10 wave reads per 16 x 16 x 16 product, against 14 for a
//     right-looking update with the same instructions and 48 with 4 x 4
//     register tiles.
//  2. panel: every 16-lane row of a wave holds the block's own 16 rows, and
//     the wave's 64 lanes another 64 rows below (the border rows last), one
//     row of 16 entries per lane. The broadcasts of the elimination are the
//     DPP operand of v_fmac_f64 (row_newbcast), so the diagonal block is
//     factored redundantly by every wave and the rows below are finished
//     beside it: no inverse block, no second pass over the panel, no barrier
//     in between. The chain from pivot to pivot is a broadcast, a reciprocal,
//     a multiply and an FMA, interleaved with the previous column's other
//     updates; no square root is taken.
// The substitutions keep the vector in one wave's registers (lane l holds
// elements l, l + 64, ..): a step is a broadcast and one FMA per 64 elements
// (the unit diagonal needs no scaling), with no barrier and the rows of the
// next steps in flight.
// What bounds it: instruction issue (one wave issues an FP64 instruction every
// 6 cycles) in the panels' few waves and in the assembly, then the chains.
// One 150-atom molecule takes 64 us (assembly 14, panels 17, updates 18,
// substitution 8, the rest loads and barriers); the blocked Cholesky with
// inverse diagonal blocks and 4 x 4 register tiles that was here before, by
// four waves with barriers in the substitutions, took 147 us. 1024 molecules
// of 20-120 atoms: 108 instead of 177 us.

typedef double d4_acc __attribute__((ext_vector_type(4)));

// Value of lane C of each 16-lane row.
template <int C>
__device__ __forceinline__ double row_bcast(double v) {
  double r;
  asm("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
      : "=v"(r)
      : "v"(v), "n"(C));
  return r;
}

// d += u t with u of lane C of each 16-lane row. (A DPP operand may not be
// written by the two instructions before: here t depends on u through the
// pivot chain, so u is always older than that.)
template <int C>
__device__ __forceinline__ void fmac_bcast(double& d, double u, double t) {
  asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+v"(d)
      : "v"(u), "v"(t), "n"(C));
}

// A panel: D holds row (lane & 15) of the block itself, d the lane's row below
// it, w the reciprocal pivots. Entries right of a row's diagonal in D are junk.
struct Panel {
  double D[kNB], d[kNB], w[kNB];
  unsigned long long good;  // non-zero lanes: every pivot so far is positive
};

// Column J of the elimination for columns C .. C1 - 1 of the block's rows and,
// with ROWS, of the rows below.
template <bool ROWS, int J, int C, int C1>
__device__ __forceinline__ void panel_columns(Panel& P, double t, double t2) {
  if constexpr (C < C1 && C < kNB) {
    fmac_bcast<C>(P.D[C], P.D[J], t);
    if (ROWS) fmac_bcast<C>(P.d[C], P.D[J], t2);
    panel_columns<ROWS, J, C + 1, C1>(P, t, t2);
  }
}

// Eliminate column J and go on with J + 1, whose pivot chain is spread between
// the updates of column J. The columns keep their values before the division
// by the pivot.
constexpr int kFcmpOgt = 2;  // ordered and greater than

template <bool ROWS, int J>
__device__ __forceinline__ void panel_step(Panel& P, int nb) {
  if constexpr (J + 1 < kNB) {
    P.w[J + 1] = 0.0;
    if (J + 1 < nb) {  // uniform (columns past nb are padding)
      const double t = -P.D[J] * P.w[J], t2 = ROWS ? -P.d[J] * P.w[J] : 0.0;
      panel_columns<ROWS, J, J + 1, J + 2>(P, t, t2);
      const double pv = row_bcast<J + 1>(P.D[J + 1]);
      const double r = __builtin_amdgcn_rcp(pv);  // relative error below 2^-23
      panel_columns<ROWS, J, J + 2, J + 5>(P, t, t2);
      const double e = fma(-pv, r, 1.0);
      panel_columns<ROWS, J, J + 5, J + 7>(P, t, t2);
      const double e2 = fma(e, e, e);
      panel_columns<ROWS, J, J + 7, J + 9>(P, t, t2);
      P.w[J + 1] = fma(r, e2, r);  // third-order step: 1 / pv
      P.good &= __builtin_amdgcn_fcmp(pv, 0.0, kFcmpOgt);
      panel_columns<ROWS, J, J + 9, kNB>(P, t, t2);
    }
    panel_step<ROWS, J + 1>(P, nb);
  }
}

template <bool ROWS>
__device__ __forceinline__ void panel_factor(Panel& P, int nb) {
  const double pv = row_bcast<0>(P.D[0]);
  P.good = __builtin_amdgcn_fcmp(pv, 0.0, kFcmpOgt);
  P.w[0] = rcp_nt(pv);
  panel_step<ROWS, 0>(P, nb);
}

// Left-looking update of the 16 x 16 tile (TWO: and a second one) of block
// column kb at rows i0 .. (i1 ..): minus sum_k L[i][k] D_k L[j][k], k < kb.
template <bool TWO>
__device__ __forceinline__ void mfma_block(double* L, int n, int kb, int i0, int i1) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const double* pb = L + tri(min(kb + l16, n - 1)) + 4 * g;
  const double* pa0 = L + tri(min(i0 + l16, n - 1)) + 4 * g;
  const double* pa1 = TWO ? L + tri(min(i1 + l16, n - 1)) + 4 * g : pa0;
  d4_acc c0 = {0.0, 0.0, 0.0, 0.0}, c1 = c0;
  // operands of block kk: four columns kk + 4 g + s of each row, and the
  // pivots of those columns at tri(k) + k
  int k4 = 4 * g, dk = tri(4 * g) + 4 * g;
  auto fetch = [&](int kk, double (&a0)[4], double (&a1)[4], double (&b)[4], double (&dd)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      b[s] = pb[kk + s];
      a0[s] = pa0[kk + s];
      if (TWO) a1[s] = pa1[kk + s];
      dd[s] = L[dk + s * k4 + (s * (s + 3)) / 2];
    }
    if (kk + 2 * kNB <= kb) {  // the last block is fetched again at the end
      dk += kNB * k4 + kNB * (kNB + 1) / 2 + kNB;
      k4 += kNB;
    }
  };
  auto product = [&](const double (&a0)[4], const double (&a1)[4], const double (&b)[4],
                     const double (&dd)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const double bs = -b[s] * dd[s];
      c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[s], bs, c0, 0, 0, 0);
      if (TWO) c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[s], bs, c1, 0, 0, 0);
    }
  };
  double a0[4], a1[4], b[4], dd[4], xa0[4], xa1[4], xb[4], xd[4];
  const int lastk = kb - kNB;
  fetch(0, a0, a1, b, dd);
  for (int kk = 0; kk < kb; kk += 2 * kNB) {  // two blocks, each fetched during the other
    fetch(min(kk + kNB, lastk), xa0, xa1, xb, xd);
    product(a0, a1, b, dd);
    if (kk + kNB < kb) {
      fetch(min(kk + 2 * kNB, lastk), a0, a1, b, dd);
      product(xa0, xa1, xb, xd);
    }
  }
  // entries (i, j) of the product: lane column j, rows i0 + 4 r + g
  const int j = kb + l16;
#pragma unroll
  for (int h = 0; h < (TWO ? 2 : 1); ++h) {
    int i = (h ? i1 : i0) + g, o = tri(i) + j;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (i < n && j <= i) L[o] += h ? c1[r] : c0[r];
      o += 4 * i + 10;  // tri(i + 4) - tri(i)
      i += 4;
    }
  }
}

// Small LDS arrays of a solve.
struct EeqSmall {
  double (*blk)[kNB];  // [2][kNB] border entries of a block before and after
  double (*y)[kNB];    // [2][kNB]   its elimination
  double* val;         // two per wave
  int* idx;            // one per wave
};

// Factor the assembled n x n matrix (n + 2 <= 208) with its border rows:
// thread i < n holds b_i and e_i, on return L^-1 b and L^-1 e. Three waves do
// the rows of the panels and a fourth the block itself, all NW >= 4 the
// updates (64 NW >= n). Returns non-zero (uniform
// over the work-group) if a pivot was not positive.
template <int NW>
__device__ __forceinline__ int ldl_factor_waves(double* L, int n, double& vb, double& ve,
                                                const EeqSmall& sm) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int kb = 0; kb < n; kb += kNB) {
    const int nb = min(kNB, n - kb);
    if (kb > 0) {
      // the border's share of the previous block
      if (tid >= kb && tid < n) {
        const double* Lr = L + tri(tid) + kb - kNB;
        double sb = 0.0, se = 0.0;
#pragma unroll
        for (int c = 0; c < kNB; ++c) {
          sb = fma(Lr[c], sm.y[0][c], sb);
          se = fma(Lr[c], sm.y[1][c], se);
        }
        vb -= sb;
        ve -= se;
      }
      // tiles from the last wave on (the first waves hold the border)
      const int nt = (n - kb + kNB - 1) / kNB;
      for (int t = NW - 1 - wave; t < nt; t += 2 * NW) {
        if (t + NW < nt)
          mfma_block<true>(L, n, kb, kb + kNB * t, kb + kNB * (t + NW));
        else
          mfma_block<false>(L, n, kb, kb + kNB * t, 0);
      }
    }
    if (tid >= kb && tid < kb + nb) {
      sm.blk[0][tid - kb] = vb;
      sm.blk[1][tid - kb] = ve;
    }
    __syncthreads();
    const int row = kb + kNB + 64 * wave + lane;
    const int border = nb < kNB ? row - kb - kNB : row - n;  // 0: b, 1: e
    const bool is_border = border == 0 || border == 1;
    const bool rows = wave == 0 || (wave < 3 && kb + kNB + 64 * wave <= n + 1);
    Panel P;
    if (rows || wave == 3) {
      const int rl = min(kb + (lane & 15), n - 1);
      const double* Dr = L + tri(rl) + kb;
      if (nb == kNB) {
        const double* Lr = is_border ? sm.blk[border] : L + tri(min(row, n - 1)) + kb;
#pragma unroll
        for (int c = 0; c < kNB; ++c) {
          P.D[c] = Dr[c];
          P.d[c] = Lr[c];
        }
      } else {
        const double* Lr = sm.blk[is_border ? border : 0];
#pragma unroll
        for (int c = 0; c < kNB; ++c) {
          const int cc = min(c, nb - 1);  // (columns past nb are never used)
          P.D[c] = Dr[cc];
          P.d[c] = Lr[cc];
        }
      }
    }
    __syncthreads();  // the block is read before wave 3 replaces it
    if (rows) {
      panel_factor<true>(P, nb);
      if (row < n) {  // (only below a full block)
        double* Lr = L + tri(row) + kb;
#pragma unroll
        for (int c = 0; c < kNB; ++c) Lr[c] = P.d[c] * P.w[c];
      }
      if (is_border) {  // L^-1 b and L^-1 e are not divided by the pivots
#pragma unroll
        for (int c = 0; c < kNB; ++c) sm.y[border][c] = P.d[c];
      }
    } else if (wave == 3) {
      panel_factor<false>(P, nb);
      if (lane == 0) sm.idx[0] = P.good != 0ull ? 0 : 1;
      if (lane < nb) {
        double* Dr = L + tri(kb + lane) + kb;
#pragma unroll
        for (int c = 0; c < kNB; ++c)
          if (c <= lane) Dr[c] = c < lane ? P.D[c] * P.w[c] : P.D[c];
      }
    }
    __syncthreads();
    if (sm.idx[0]) return 1;
    if (tid >= kb && tid < kb + nb) {
      vb = sm.y[0][tid - kb];
      ve = sm.y[1][tid - kb];
    }
  }
  return 0;
}

// Vector elements per lane in the substitutions, and steps whose rows are kept
// in flight: as many as fit about 64 registers, so that the adjoint's waves
// find room beside the three-body kernel's.
template <int NV>
struct SolveShape {
  static constexpr int kU = NV <= 2 ? 8 : 4;
};
inline int solve_regs(int64_t N) { return N <= 128 ? 2 : 4; }
// The substitutions read whole 64-entry pieces of a row: up to 63 doubles past
// the last row of the factor.
constexpr int kSolvePad = 64;

// Rows i, i - 1, .. i - U + 1 of L, the pieces of register blocks 0 .. Q.
template <int Q, int U>
__device__ __forceinline__ void backward_rows(const double* L, int i, double (&l)[U][Q + 1]) {
  const double* p = L + (threadIdx.x & 63);
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int q = 0; q <= Q; ++q) l[u][q] = p[tri(i - u) + 64 * q];
}

// U steps from row i = 64 Q + r on: x_i is final, columns left of the diagonal
// lose L[i][j] x_i.
template <int Q, int U, int NV>
__device__ __forceinline__ void backward_apply(int r, const double (&l)[U][Q + 1],
                                               double (&v)[NV]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const double x = -lane_bcast(v[Q], r - u);
    if (lane < r - u) v[Q] = fma(l[u][Q], x, v[Q]);
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = fma(l[u][q], x, v[q]);
  }
}

// Register block Q of L^T x = v (unit diagonal).
template <int Q, int NV>
__device__ __forceinline__ void backward_block(const double* L, int n, double (&v)[NV]) {
  constexpr int U = SolveShape<NV>::kU;
  int r = min(63, n - 1 - 64 * Q);
  for (; r >= 0 && (r + 1) % U; --r) {  // down to whole groups
    double l[1][Q + 1];
    backward_rows<Q, 1>(L, 64 * Q + r, l);
    backward_apply<Q, 1>(r, l, v);
  }
  if (r < 0) return;
  double l[U][Q + 1], ln[U][Q + 1];
  backward_rows<Q, U>(L, 64 * Q + r, l);
  for (; r >= 0; r -= U) {
    // the next group in flight during this one's chain (the last: its own rows)
    backward_rows<Q, U>(L, 64 * Q + (r >= U ? r - U : r), ln);
    backward_apply<Q, U>(r, l, v);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q <= Q; ++q) l[u][q] = ln[u][q];
  }
}

// L^T x = v in place for the vector of one wave (all 64 lanes active; lanes
// past n hold zeros).
template <int NV>
__device__ __forceinline__ void wave_backward(const double* L, int n, double (&v)[NV]) {
  if constexpr (NV > 3) backward_block<3>(L, n, v);
  if constexpr (NV > 2) backward_block<2>(L, n, v);
  backward_block<1>(L, n, v);
  backward_block<0>(L, n, v);
}

// Columns j .. j + U - 1 of L for the rows of register blocks Q ..; at[q]:
// start of the lane's row 64 q + lane (clamped to the last row).
template <int Q, int U, int NV>
__device__ __forceinline__ void forward_cols(const double* L, int j, const int (&at)[NV],
                                             double (&l)[U][NV]) {
#pragma unroll
  for (int q = Q; q < NV; ++q) {
    const double* p = L + at[q] + j;
#pragma unroll
    for (int u = 0; u < U; ++u) l[u][q] = p[u];
  }
}

template <int Q, int U, int NV>
__device__ __forceinline__ void forward_apply(int r, const double (&l)[U][NV], double (&v)[NV]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const double y = -lane_bcast(v[Q], r + u);
    if (lane > r + u) v[Q] = fma(l[u][Q], y, v[Q]);
#pragma unroll
    for (int q = Q + 1; q < NV; ++q) v[q] = fma(l[u][q], y, v[q]);
  }
}

// Register block Q of L y = v (unit diagonal).
template <int Q, int NV>
__device__ __forceinline__ void forward_block(const double* L, int n, const int (&at)[NV],
                                              double (&v)[NV]) {
  constexpr int U = SolveShape<NV>::kU;
  const int cnt = min(64, n - 64 * Q);
  if (cnt <= 0) return;
  int r = 0;
  if (cnt >= U) {
    double l[U][NV], ln[U][NV];
    forward_cols<Q, U>(L, 64 * Q, at, l);
    for (; r + U <= cnt; r += U) {
      // the next group in flight during this one's chain (the last: its own)
      forward_cols<Q, U>(L, 64 * Q + (r + 2 * U <= cnt ? r + U : r), at, ln);
      forward_apply<Q, U>(r, l, v);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = Q; q < NV; ++q) l[u][q] = ln[u][q];
    }
  }
  for (; r < cnt; ++r) {
    double l[1][NV];
    forward_cols<Q, 1>(L, 64 * Q + r, at, l);
    forward_apply<Q, 1>(r, l, v);
  }
}

// L y = v in place for the vector of one wave. (Lanes past n read the last row
// and return junk.)
template <int NV>
__device__ __forceinline__ void wave_forward(const double* L, int n, double (&v)[NV]) {
  const int lane = threadIdx.x & 63;
  int at[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) at[q] = tri(min(64 * q + lane, n - 1));
  forward_block<0>(L, n, at, v);
  forward_block<1>(L, n, at, v);
  if constexpr (NV > 2) forward_block<2>(L, n, at, v);
  if constexpr (NV > 3) forward_block<3>(L, n, at, v);
}

// LDS of the EEQ solve for a padded length N: the packed factor and behind it
// the staged atoms (x, y, z, radius; they also are the substitutions' pad).
// Where there is no room for those, the atoms are staged over the factor's
// last rows. kEeqMaxN: the longest in LDS.
constexpr size_t kLdsBytes = 160 * 1024 - 768;  // dynamic LDS budget per work-group
constexpr int kEeqStaged = 4;
constexpr int kEeqMaxN = 201;
static_assert(sizeof(double) * (kEeqMaxN * (kEeqMaxN + 1) / 2 + kSolvePad) <= kLdsBytes,
              "EEQ factor in LDS");

// doubles in front of (and with) the staged atoms' end
inline size_t eeq_doubles(int64_t N) {
  const size_t f = (size_t)tri((int)N), st = kEeqStaged * (size_t)N;
  const size_t both = f + (st > (size_t)kSolvePad ? st : (size_t)kSolvePad);
  return sizeof(double) * both <= kLdsBytes ? both : f + kSolvePad;
}

// Row of a strictly-lower packed index e: i (i - 1) / 2 <= e < i (i + 1) / 2.
__device__ __forceinline__ int strict_row(int e) {
  int i = (int)((sqrtf(8.0f * (float)e + 1.0f) + 1.0f) * 0.5f);
  while (i * (i - 1) / 2 > e) --i;
  while (i * (i + 1) / 2 <= e) ++i;
  return i;
}

__device__ void eeq_lu_molecule(const DevTables& t, const Inputs& in, const Work& w, int64_t m,
                                double* s_val, int* s_idx);

// Strictly-lower element e of the Coulomb block from the staged atoms.
__device__ __forceinline__ double eeq_element(const double* st, int N, int i, int j) {
  const double ri = st[3 * N + i], rj = st[3 * N + j];
  const double dx = st[i] - st[j], dy = st[N + i] - st[N + j], dz = st[2 * N + i] - st[2 * N + j];
  const double v = eeq_offdiag_r2(rsqrt_nt(ri * ri + rj * rj), dx * dx + dy * dy + dz * dz);
  return ri == 0.0 || rj == 0.0 ? 0.0 : v;  // (a padding atom)
}

// Charges of molecule m by one work-group of NW waves (L: the dynamic LDS of
// the launch, `doubles` long).
template <int NW, int NV>
__device__ __forceinline__ void eeq_chol_molecule(const DevTables& t, const Params& p,
                                                  const Inputs& in, const Work& w, int64_t m,
                                                  double* L, int doubles, const EeqSmall& sm) {
  constexpr int NT = 64 * NW;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t N = w.N;
  const int n = w.natom[m];
  const int64_t* Z = in.numbers + m * N;
  const double* R = in.positions + m * N * 3;
  double* q = w.q + m * N;

  if (in.q_in != nullptr) {  // charges supplied by the caller
    for (int i = tid; i < N; i += NT)
      q[i] = (i < n && Z[i] != 0) ? in.q_in[m * N + i] : 0.0;
    return;
  }
  for (int i = n + tid; i < N; i += NT) q[i] = 0.0;
  if (n == 0) return;
  if (p.force_lu) {
    if (tid == 0) w.status[m] |= kStatusLU;
    __syncthreads();
    eeq_lu_molecule(t, in, w, m, sm.val, sm.idx);
    return;
  }

  // assemble the lower triangle of C and the two right-hand sides: positions
  // and radii (0 marks a padding atom) are staged, then all threads fill the
  // triangle. Rows from r1 on overlap the staged atoms: their elements (at
  // most five rows) wait in registers until the staged atoms are read.
  const int base = doubles - kEeqStaged * (int)N;
  double* st = L + base;
  int r1 = n;
  while (r1 > 0 && tri(r1) > base) --r1;
  double vb = 0.0, ve = 0.0, diag = 1.0;
  if (tid < n) {
    const int zi = (int)Z[tid];
    st[tid] = R[3 * tid];
    st[N + tid] = R[3 * tid + 1];
    st[2 * N + tid] = R[3 * tid + 2];
    st[3 * N + tid] = zi != 0 ? t.rad[zi] : 0.0;
    if (zi != 0) {
      diag = eeq_diag(t, zi);
      vb = eeq_rhs(t, zi, w.cnq[m * N + tid]);
      ve = 1.0;
    }
  }
  __syncthreads();
  // 8 x 8 tiles (bx <= by) by waves, two at a time (the erf chains overlap)
  {
    const int nb8 = (r1 + 7) >> 3, tiles = nb8 * (nb8 + 1) / 2;
    const int tx = lane & 7, ty = lane >> 3;
    int by = 0, bx = wave;
    while (bx > by) bx -= ++by;
    for (int t0 = wave; t0 < tiles; t0 += 2 * NW) {
      int at[2];
      double v[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int j = 8 * bx + tx, i = 8 * by + ty;
        const bool on = j < i && i < r1;
        at[u] = on ? tri(i) + j : -1;
        v[u] = eeq_element(st, (int)N, on ? i : 0, on ? j : 0);
        bx += NW;
        while (bx > by) bx -= ++by;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (at[u] >= 0) L[at[u]] = v[u];
    }
  }
  const int e1 = r1 * (r1 - 1) / 2, ne = n * (n - 1) / 2;
  if (r1 < n) {  // uniform
    constexpr int kLate = (5 * kEeqMaxN + NT - 1) / NT;
    double late[kLate];
#pragma unroll
    for (int u = 0; u < kLate; ++u) {
      const int e = e1 + tid + NT * u;
      late[u] = 0.0;
      if (e < ne) {
        const int i = strict_row(e);
        late[u] = eeq_element(st, (int)N, i, e - i * (i - 1) / 2);
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kLate; ++u) {
      const int e = e1 + tid + NT * u;
      if (e < ne) {
        const int i = strict_row(e);
        L[tri(i) + e - i * (i - 1) / 2] = late[u];
      }
    }
  }
  if (tid < n) L[tri(tid) + tid] = diag;
  __syncthreads();

  if (ldl_factor_waves<NW>(L, n, vb, ve, sm)) {
    // a pivot <= 0: the pivoted LU of the bordered system in the workspace, by
    // this work-group (no separate launch behind this one)
    if (tid == 0) w.status[m] |= kStatusLU;
    __syncthreads();
    eeq_lu_molecule(t, in, w, m, sm.val, sm.idx);
    return;
  }
  // e^T C^-1 b = y_e D^-1 y_b and e^T C^-1 e = y_e D^-1 y_e, so one backward
  // substitution of D^-1 (y_b - mu y_e) gives q = C^-1 (b - mu e); the vector
  // moves to wave 0 through LDS, one wave's entries at a time
  const double dinv = tid < n ? rcp_nt(L[tri(tid) + tid]) : 0.0;
  const double ze = ve * dinv;  // D^-1 y_e, kept for the adjoint
  if (tid < n) w.ez[m * N + tid] = ze;
  const double sbe = wave_sum(ze * vb), see = wave_sum(ze * ve);
  __syncthreads();
  double* red = sm.val;  // [NW] and [NW] sums, then the moving entries
  if (lane == 0) {
    red[wave] = sbe;
    red[NW + wave] = see;
  }
  __syncthreads();
  double tbe = 0.0, tee = 0.0;
  for (int k = 0; k < NW; ++k) {
    tbe += red[k];
    tee += red[NW + k];
  }
  const double mu = (tbe - in.charge[m]) / tee;
  const double vi = tid < n ? fma(-mu, ze, vb * dinv) : 0.0;
  double v[NV] = {vi};
  double* move = &sm.blk[0][0];  // 64 doubles: blk and y
#pragma unroll
  for (int k = 1; k < NV; ++k) {
    if (64 * k < n) {  // uniform
      __syncthreads();
      if (wave == k) move[lane] = vi;
      __syncthreads();
      if (wave == 0) v[k] = move[lane];
    }
  }
  if (wave == 0) {
    wave_backward(L, n, v);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int i = 64 * k + lane;
      if (i < n) q[i] = Z[i] != 0 ? v[k] : 0.0;
    }
  } else {
    // the other waves keep the factor for the adjoint
    double* gL = w.chol + (size_t)m * (size_t)tri((int)N);
    const int nt = tri(n);
    for (int k = tid - 64; k < nt; k += NT - 64) gL[k] = L[k];
  }
}

// Waves of a solve: a molecule whose factor takes more than half of a CU's
// LDS (N > 140) has the CU to itself and gets eight waves; smaller ones share
// it, with four each.
inline int eeq_waves(int64_t N) { return N > 140 ? 8 : 4; }

// Two work-groups per CU fit the LDS of a 120-atom factor; keep the register
// use low enough for two waves per SIMD as well. With `paired` (factors that
// take a whole CU's LDS), work-group b solves the b-th largest and then the
// b-th smallest molecule: half the CUs hold the solve, and the others are
// free from the start for the three-body kernel on the companion stream.
template <int NW, int NV, bool PAIRED>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void k_eeq_chol(
    DevTables t, Params p, Inputs in, Work w, int doubles, int ordered) {
  extern __shared__ double smem[];
  __shared__ double s_blk[4][kNB];
  __shared__ double s_val[2 * NW];
  __shared__ int s_idx[NW];
  const EeqSmall sm = {s_blk, s_blk + 2, s_val, s_idx};
  const int64_t b = blockIdx.x;
  if (!PAIRED) {
    // smallest molecules first: their solves end early and leave their CUs
    // to the three-body side on the companion stream (the batch order and
    // largest first were both slower beside it)
    eeq_chol_molecule<NW, NV>(t, p, in, w, ordered ? w.eqord[w.B - 1 - b] : b, smem, doubles, sm);
    return;
  }
  const int64_t b2 = w.B - 1 - b;
  for (int k = 0; k < (b2 > b ? 2 : 1); ++k) {
    if (k) __syncthreads();  // the LDS is reused
    eeq_chol_molecule<NW, NV>(t, p, in, w, w.eqord[k ? b2 : b], smem, doubles, sm);
  }
}

// Pivoted LU of the full bordered matrix in HBM, for molecules whose
// Cholesky failed (or all molecules under D4_FLAG_FORCE_LU).
__device__ void lu_assemble(const DevTables& t, const Inputs& in, const Work& w,
                            int64_t m, int n, double* A, int ld, double* rhs) {
  const int64_t N = w.N;
  const int64_t* Z = in.numbers + m * N;
  const double* R = in.positions + m * N * 3;
  for (int e = threadIdx.x; e < (n + 1) * (n + 1); e += (int)blockDim.x) {
    const int i = e / (n + 1), j = e - i * (n + 1);
    double v;
    if (i == n && j == n) {
      v = 0.0;
    } else if (i == n || j == n) {
      const int k = i == n ? j : i;
      v = Z[k] != 0 ? 1.0 : 0.0;
    } else {
      const int zi = (int)Z[i], zj = (int)Z[j];
      if (i == j) {
        v = zi != 0 ? eeq_diag(t, zi) : 1.0;
      } else if (zi != 0 && zj != 0) {
        const double dx = R[3 * i] - R[3 * j], dy = R[3 * i + 1] - R[3 * j + 1],
                     dz = R[3 * i + 2] - R[3 * j + 2];
        v = eeq_offdiag(t, zi, zj, dx * dx + dy * dy + dz * dz);
      } else {
        v = 0.0;
      }
    }
    A[(size_t)i * ld + j] = v;
  }
  if (rhs != nullptr) {
    for (int i = threadIdx.x; i < n; i += (int)blockDim.x) {
      const int zi = (int)Z[i];
      rhs[i] = zi != 0 ? eeq_rhs(t, zi, w.cnq[m * N + i]) : 0.0;
    }
    if (threadIdx.x == 0) rhs[n] = in.charge[m];
  }
}

// Solve (P A = L U) x = b in place for b in HBM.
__device__ void lu_solve(const double* A, int ld, const int32_t* piv, int n1,
                         double* b) {
  const int tid = threadIdx.x, nthr = (int)blockDim.x;
  __syncthreads();
  if (tid == 0) {
    for (int k = 0; k < n1; ++k) {
      const int pk = piv[k];
      if (pk != k) {
        const double tmp = b[k];
        b[k] = b[pk];
        b[pk] = tmp;
      }
    }
  }
  for (int k = 0; k < n1; ++k) {  // unit lower
    __syncthreads();
    const double yk = b[k];
    for (int i = k + 1 + tid; i < n1; i += nthr) b[i] -= A[(size_t)i * ld + k] * yk;
  }
  for (int k = n1 - 1; k >= 0; --k) {  // upper
    __syncthreads();
    const double xk = b[k] / A[(size_t)k * ld + k];
    for (int i = tid; i < k; i += nthr) b[i] -= A[(size_t)i * ld + k] * xk;
  }
  __syncthreads();
  for (int i = tid; i < n1; i += nthr) b[i] /= A[(size_t)i * ld + i];
  __syncthreads();
}

// Largest |value| of the work-group and its index, the lowest index among
// equal values (the same pivot whatever the reduction order); s_val, s_idx:
// one entry of LDS per wave.
__device__ __forceinline__ void block_argmax(double& v, int& i, double* s_val, int* s_idx) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const double ov = __shfl_xor(v, off, 64);
    const int oi = __shfl_xor(i, off, 64);
    if (ov > v || (ov == v && oi < i)) {
      v = ov;
      i = oi;
    }
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    s_val[wave] = v;
    s_idx[wave] = i;
  }
  __syncthreads();
  v = s_val[0];
  i = s_idx[0];
  for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
    if (s_val[k] > v || (s_val[k] == v && s_idx[k] < i)) {
      v = s_val[k];
      i = s_idx[k];
    }
  }
  __syncthreads();
}

// Pivoted LU of the bordered system of molecule m (work-group wide);
// s_val, s_idx: one entry of LDS per wave.
__device__ void eeq_lu_molecule(const DevTables& t, const Inputs& in, const Work& w, int64_t m,
                                double* s_val, int* s_idx) {
  const int n = w.natom[m];
  const int n1 = n + 1;
  const int ld = (int)w.N + 1;
  const int tid = threadIdx.x, nthr = (int)blockDim.x;
  double* A = w.lu + (size_t)m * ld * ld;
  int32_t* piv = w.piv + m * ld;
  double* vec = w.vec + m * ld;
  lu_assemble(t, in, w, m, n, A, ld, vec);
  __syncthreads();
  int singular = 0;
  for (int k = 0; k < n1; ++k) {
    // pivot search in column k
    double best = -1.0;
    int bi = k;
    for (int i = k + tid; i < n1; i += nthr) {
      const double v = fabs(A[(size_t)i * ld + k]);
      if (v > best) {
        best = v;
        bi = i;
      }
    }
    block_argmax(best, bi, s_val, s_idx);
    const int pk = bi;
    const double pv = best;
    if (!(pv > 0.0)) {
      singular = 1;
      break;
    }
    if (tid == 0) piv[k] = pk;
    if (pk != k) {
      for (int j = tid; j < n1; j += nthr) {
        const double a = A[(size_t)k * ld + j];
        A[(size_t)k * ld + j] = A[(size_t)pk * ld + j];
        A[(size_t)pk * ld + j] = a;
      }
    }
    __syncthreads();
    const double inv = 1.0 / A[(size_t)k * ld + k];
    for (int i = k + 1 + tid; i < n1; i += nthr) A[(size_t)i * ld + k] *= inv;
    __syncthreads();
    const int rem = n1 - k - 1;
    for (int e = tid; e < rem * rem; e += nthr) {
      const int i = k + 1 + e / rem, j = k + 1 + e % rem;
      A[(size_t)i * ld + j] -= A[(size_t)i * ld + k] * A[(size_t)k * ld + j];
    }
    __syncthreads();
  }
  if (singular) {
    if (tid == 0) w.status[m] |= kStatusSingular;
    for (int i = tid; i < n; i += nthr) w.q[m * w.N + i] = NAN;
    return;
  }
  lu_solve(A, ld, piv, n1, vec);
  for (int i = tid; i < n; i += nthr)
    w.q[m * w.N + i] = in.numbers[m * w.N + i] != 0 ? vec[i] : 0.0;
}

// The molecules whose Cholesky pivot was <= 0 (or all, when forced): a few
// work-groups walk the batch, so the launch costs little when none needs it.
__global__ __launch_bounds__(256) void k_eeq_lu(DevTables t, Params p, Inputs in, Work w) {
  __shared__ double s_val[kWaves];
  __shared__ int s_idx[kWaves];
  if (in.q_in != nullptr) return;
  for (int64_t m = blockIdx.x; m < w.B; m += gridDim.x) {
    if (!(w.status[m] & kStatusLU)) continue;  // uniform over the work-group
    eeq_lu_molecule(t, in, w, m, s_val, s_idx);
    __syncthreads();
  }
}

// ==========================================================================
// Tiled EEQ for molecules whose packed factor does not fit in LDS.
//
// The matrix lives in HBM in the LU workspace as row-major rows of length N:
// rows 0..n-1 hold the lower triangle of C, row n holds b and row n+1 holds
// e. With the two border rows below the matrix, the forward substitution of
// b and e is just the panel and trailing steps applied to those rows. Per
// 64-column block step:
//   k_tf_diag   one work-group factors the 64 x 64 diagonal block in LDS
//               (16-column blocked Cholesky), forms X = D^-1 and stores it in
//               place of D;
//   k_tf_panel  64-row tiles below the block (and the border rows) become
//               A X^T;
//   k_tf_update 64 x 64 tiles of the trailing triangle lose P_I P_J^T.
// The substitutions then run one launch per block step: every work-group of
// a molecule recomputes the block's 64-entry solution from the same inputs
// and work-group 0 alone stores it, so no work-group reads what another
// writes within a launch.
// ==========================================================================

constexpr int kTB = 64;

// The tiled solve is a chain of a few hundred short launches that runs beside
// the screened three-body kernel's waves on the same SIMDs; its waves take
// issue priority over them, so the chain is not slowed to a third of its
// speed (the three-body waves use the cycles it leaves).
__device__ __forceinline__ void tf_priority() { __builtin_amdgcn_s_setprio(2); }

__device__ __forceinline__ double* tf_matrix(const Work& w, int64_t m) {
  return w.lu + (size_t)m * (size_t)(w.N + 1) * (size_t)(w.N + 1);
}

// Row r of an inclusive lower packed index: tri(r) <= e < tri(r + 1).
__device__ __forceinline__ int incl_row(int e) { return strict_row(e) - 1; }

// Molecule m still factorising at block kb (charges not given, no failure).
__device__ __forceinline__ bool tf_active(const Inputs& in, const Work& w, int64_t m,
                                          int kb) {
  return in.q_in == nullptr && kb < w.natom[m] && !(w.status[m] & kStatusLU);
}

// Assemble the lower triangle of C and the border rows b, e; one wave per row.
__global__ __launch_bounds__(256) void k_tf_assemble(DevTables t, Params p, Inputs in,
                                                     Work w) {
  const int lane = threadIdx.x & 63;
  const int64_t N = w.N, rows = N + 2;
  const int64_t g = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (g >= w.B * rows) return;
  const int64_t m = g / rows;
  const int i = (int)(g - m * rows);
  const int n = w.natom[m];
  if (in.q_in != nullptr || i >= n + 2) return;
  if (p.force_lu) {  // testing: every system goes to the pivoted-LU kernel
    if (i == 0 && lane == 0) w.status[m] |= kStatusLU;
    return;
  }
  const int64_t* Z = in.numbers + m * N;
  const double* R = in.positions + m * N * 3;
  double* Ai = tf_matrix(w, m) + (size_t)i * (size_t)N;
  if (i < n) {
    const int zi = (int)Z[i];
    const double xi = R[3 * i], yi = R[3 * i + 1], zzi = R[3 * i + 2];
    for (int j = lane; j <= i; j += 64) {
      const int zj = (int)Z[j];
      double v;
      if (j == i) {
        v = zi != 0 ? eeq_diag(t, zi) : 1.0;
      } else if (zi != 0 && zj != 0) {
        const double dx = xi - R[3 * j], dy = yi - R[3 * j + 1], dz = zzi - R[3 * j + 2];
        v = eeq_offdiag(t, zi, zj, dx * dx + dy * dy + dz * dz);
      } else {
        v = 0.0;
      }
      Ai[j] = v;
    }
  } else {
    const bool rhs = i == n;
    for (int j = lane; j < n; j += 64) {
      const int zj = (int)Z[j];
      Ai[j] = zj == 0 ? 0.0 : (rhs ? eeq_rhs(t, zj, w.cnq[m * N + j]) : 1.0);
    }
  }
}

// Factor the diagonal block at kb and replace it by the inverse of its factor.
// The tiled kernels take their LDS as dynamic shared memory and at most 64
// VGPRs (eight waves per SIMD as far as registers go): a work-group then fits
// beside the three-body kernel's waves (two per SIMD with 220 VGPRs) on any
// CU instead of waiting until one is nearly empty.
constexpr size_t kTfDiagLds = sizeof(double) * (kTB * (kTB + 1) / 2 + kTB * kTB + kNB * kTB +
                                                2 * kNB + 2);
constexpr size_t kTfTileLds = sizeof(double) * 2 * kTB * (kTB + 1);

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_tf_diag(
    Inputs in, Work w, int kb) {
  tf_priority();
  extern __shared__ double s_tf[];
  double* F = s_tf;                                             // [tri(kTB)]
  auto X = reinterpret_cast<double (*)[kTB]>(F + kTB * (kTB + 1) / 2);  // [kTB][kTB]
  auto T = reinterpret_cast<double (*)[kTB]>(&X[kTB][0]);      // [kNB][kTB]
  double* s_small = &T[kNB][0];                                 // [2 kNB + 2]
  const int64_t m = blockIdx.x;
  if (!tf_active(in, w, m, kb)) return;
  const int tid = threadIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  const int nb = min(kTB, n - kb);
  double* A = tf_matrix(w, m);
  for (int e = tid; e < tri(nb); e += 256) {
    const int r = incl_row(e), c = e - tri(r);
    F[e] = A[(size_t)(kb + r) * N + kb + c];
  }
  __syncthreads();
  if (chol_factor<false>(F, nb, (double*)nullptr, (double*)nullptr, s_small,
                         s_small + 2 * kNB)) {
    if (tid == 0) w.status[m] |= kStatusLU;
    return;
  }
  // X = F^-1 by block forward substitution over the 16-row sub-blocks, whose
  // own inverses the factorisation left on the diagonal of F:
  // X_s = X16_s (I_s - F_{s,<s} X_{<s})
  for (int r0 = 0; r0 < nb; r0 += kNB) {
    const int rn = min(kNB, nb - r0);
    const int ncol = r0 + rn;
    for (int e = tid; e < rn * ncol; e += 256) {
      const int r = e / ncol, c = e - r * ncol;
      const double* Fr = F + tri(r0 + r);
      double sacc = (r0 + r == c) ? 1.0 : 0.0;
      for (int k = c; k < r0; ++k) sacc = fma(-Fr[k], X[k][c], sacc);
      T[r][c] = sacc;
    }
    __syncthreads();
    for (int e = tid; e < rn * ncol; e += 256) {
      const int r = e / ncol, c = e - r * ncol;
      const double* Xr = F + tri(r0 + r) + r0;
      double sacc = 0.0;
      for (int rr = 0; rr <= r; ++rr) sacc = fma(Xr[rr], T[rr][c], sacc);
      X[r0 + r][c] = c <= r0 + r ? sacc : 0.0;
    }
    __syncthreads();
  }
  for (int e = tid; e < tri(nb); e += 256) {
    const int r = incl_row(e), c = e - tri(r);
    A[(size_t)(kb + r) * N + kb + c] = X[r][c];
  }
}

// Panel tile: rows kb + nb + 64 y ... of the matrix and border become A X^T.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_tf_panel(
    Inputs in, Work w, int kb) {
  tf_priority();
  extern __shared__ double s_tf[];
  auto Xs = reinterpret_cast<double (*)[kTB + 1]>(s_tf);  // [kTB][kTB + 1]
  auto As = Xs + kTB;                                      // [kTB][kTB + 1]
  const int64_t m = blockIdx.x;
  if (!tf_active(in, w, m, kb)) return;
  const int tid = threadIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  const int nb = min(kTB, n - kb);
  const int r0 = kb + nb + (int)blockIdx.y * kTB;
  const int rows = min(kTB, n + 2 - r0);
  if (rows <= 0) return;
  double* A = tf_matrix(w, m);
  for (int e = tid; e < kTB * kTB; e += 256) {
    const int r = e >> 6, c = e & (kTB - 1);
    Xs[r][c] = (r < nb && c <= r) ? A[(size_t)(kb + r) * N + kb + c] : 0.0;
    As[r][c] = (r < rows && c < nb) ? A[(size_t)(r0 + r) * N + kb + c] : 0.0;
  }
  __syncthreads();
  const int tr = tid >> 4, tc = tid & 15;
  double acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = 0.0;
  for (int k = 0; k < kTB; ++k) {
    double av[4], xv[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      av[a] = As[4 * tr + a][k];
      xv[a] = Xs[4 * tc + a][k];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = fma(av[a], xv[b], acc[a][b]);
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int r = 4 * tr + a, c = 4 * tc + b;
      if (r < rows && c < nb) A[(size_t)(r0 + r) * N + kb + c] = acc[a][b];
    }
}

// Trailing tile (I, J): rows r0 + 64 I.. (matrix and border), columns
// r0 + 64 J.. of the matrix, r0 = kb + 64, lose P_I P_J^T.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_tf_update(
    Inputs in, Work w, int kb) {
  tf_priority();
  extern __shared__ double s_tf[];
  auto Pi = reinterpret_cast<double (*)[kTB + 1]>(s_tf);  // [kTB][kTB + 1]
  auto Pj = Pi + kTB;                                      // [kTB][kTB + 1]
  const int64_t m = blockIdx.x;
  if (!tf_active(in, w, m, kb)) return;
  const int tid = threadIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  const int r0 = kb + kTB;
  if (r0 >= n) return;
  const int nI = (n + 2 - r0 + kTB - 1) / kTB, nJ = (n - r0 + kTB - 1) / kTB;
  const int e = (int)blockIdx.y;
  if (e >= nI * (nI + 1) / 2) return;
  const int I = incl_row(e), J = e - tri(I);
  if (J >= nJ) return;
  const int i0 = r0 + I * kTB, j0 = r0 + J * kTB;
  double* A = tf_matrix(w, m);
  for (int x = tid; x < kTB * kTB; x += 256) {
    const int r = x >> 6, c = x & (kTB - 1);
    Pi[r][c] = (i0 + r < n + 2) ? A[(size_t)(i0 + r) * N + kb + c] : 0.0;
    Pj[r][c] = (j0 + r < n) ? A[(size_t)(j0 + r) * N + kb + c] : 0.0;
  }
  __syncthreads();
  const int tr = tid >> 4, tc = tid & 15;
  double acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = 0.0;
  for (int k = 0; k < kTB; ++k) {
    double iv[4], jv[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      iv[a] = Pi[4 * tr + a][k];
      jv[a] = Pj[4 * tc + a][k];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = fma(iv[a], jv[b], acc[a][b]);
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int i = i0 + 4 * tr + a, j = j0 + 4 * tc + b;
      if (i < n + 2 && j < n && j <= i) A[(size_t)i * N + j] -= acc[a][b];
    }
}

// After the factorisation: charges given or padding, then mu and the
// right-hand side y_b - mu y_e of the backward substitution (in vec); y_e is
// kept for the adjoint.
__global__ __launch_bounds__(256) void k_tf_reduce(Inputs in, Work w) {
  tf_priority();
  __shared__ double red[2 * kWaves];
  const int64_t m = blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  const int64_t* Z = in.numbers + m * N;
  double* q = w.q + m * N;
  if (in.q_in != nullptr) {
    for (int i = tid; i < N; i += 256)
      q[i] = (i < n && Z[i] != 0) ? in.q_in[m * N + i] : 0.0;
    return;
  }
  for (int i = n + tid; i < N; i += 256) q[i] = 0.0;
  if (n == 0 || (w.status[m] & kStatusLU)) return;
  const double* A = tf_matrix(w, m);
  const double* yb = A + (size_t)n * N;
  const double* ye = A + (size_t)(n + 1) * N;
  double sbe = 0.0, see = 0.0;
  for (int i = tid; i < n; i += 256) {
    sbe = fma(ye[i], yb[i], sbe);
    see = fma(ye[i], ye[i], see);
  }
  sbe = block_sum(sbe, red);
  see = block_sum(see, red + kWaves);
  const double mu = (sbe - in.charge[m]) / see;
  double* v = w.vec + m * (N + 1);
  double* gz = w.ez + m * N;
  for (int i = tid; i < n; i += 256) {
    v[i] = fma(-mu, ye[i], yb[i]);
    gz[i] = ye[i];
  }
}

// One backward-substitution step L^T x = v at block kb (descending kb):
// x_kb = X^T v_kb is stored to dst (zero on padding atoms) by work-group 0;
// work-group y updates v[j] for j in [256 y, 256 y + 256) below kb.
__global__ __launch_bounds__(256) void k_tf_bsolve(Inputs in, Work w, int kb,
                                                   double* dst_base) {
  tf_priority();
  __shared__ double xs[kTB];
  const int64_t m = blockIdx.x;
  const int y = (int)blockIdx.y;
  const int tid = threadIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  if (in.q_in != nullptr || kb >= n || (w.status[m] & kStatusLU)) return;
  const int j = y * 256 + tid;
  if (y > 0 && y * 256 >= kb) return;
  const int nb = min(kTB, n - kb);
  const double* A = tf_matrix(w, m);
  double* v = w.vec + m * (N + 1);
  if (tid < nb) {
    double sacc = 0.0;
    for (int k = tid; k < nb; ++k) sacc = fma(A[(size_t)(kb + k) * N + kb + tid], v[kb + k], sacc);
    xs[tid] = sacc;
  }
  __syncthreads();
  if (y == 0 && tid < nb) {
    const int64_t* Z = in.numbers + m * N;
    dst_base[m * N + kb + tid] = Z[kb + tid] != 0 ? xs[tid] : 0.0;
  }
  if (j < kb) {
    double sacc = 0.0;
    for (int c = 0; c < nb; ++c) sacc = fma(A[(size_t)(kb + c) * N + j], xs[c], sacc);
    v[j] -= sacc;
  }
}

// One forward-substitution step L y = v at block kb (ascending kb): y_kb =
// X v_kb is stored to dst by work-group 0; work-group y updates the rows
// kb + nb + 256 y .. below the block.
__global__ __launch_bounds__(256) void k_tf_fsolve(Inputs in, Work w, int kb,
                                                   double* dst_base) {
  tf_priority();
  __shared__ double ys[kTB];
  const int64_t m = blockIdx.x;
  const int y = (int)blockIdx.y;
  const int tid = threadIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  if (in.q_in != nullptr || kb >= n || (w.status[m] & (kStatusLU | kStatusSingular))) return;
  const int nb = min(kTB, n - kb);
  const int j = kb + nb + y * 256 + tid;
  if (y > 0 && kb + nb + y * 256 >= n) return;
  const double* A = tf_matrix(w, m);
  double* v = w.vec + m * (N + 1);
  if (tid < nb) {
    const double* Xr = A + (size_t)(kb + tid) * N + kb;
    double sacc = 0.0;
    for (int k = 0; k <= tid; ++k) sacc = fma(Xr[k], v[kb + k], sacc);
    ys[tid] = sacc;
  }
  __syncthreads();
  if (y == 0 && tid < nb) dst_base[m * N + kb + tid] = ys[tid];
  if (j < n) {
    const double* Aj = A + (size_t)j * N + kb;
    double sacc = 0.0;
    for (int c = 0; c < nb; ++c) sacc = fma(Aj[c], ys[c], sacc);
    v[j] -= sacc;
  }
}

// Adjoint set-up for the tiled solve: v = dL/dq on real atoms.
__global__ __launch_bounds__(256) void k_tf_adj_init(Inputs in, Work w) {
  tf_priority();
  const int64_t m = blockIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  if (in.q_in != nullptr || (w.status[m] & (kStatusLU | kStatusSingular))) return;
  const int64_t* Z = in.numbers + m * N;
  double* v = w.vec + m * (N + 1);
  for (int i = threadIdx.x; i < n; i += 256) v[i] = Z[i] != 0 ? w.dldq[m * N + i] : 0.0;
}

// Between the two adjoint substitutions: w' = L^-1 g is in lam; v = w' - nu y_e
// with nu = y_e . w' / y_e . y_e.
__global__ __launch_bounds__(256) void k_tf_adj_mid(Inputs in, Work w) {
  tf_priority();
  __shared__ double red[2 * kWaves];
  const int64_t m = blockIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  if (in.q_in != nullptr || n == 0 || (w.status[m] & (kStatusLU | kStatusSingular))) return;
  const int tid = threadIdx.x;
  const double* wl = w.lam + m * N;
  const double* ye = w.ez + m * N;
  double sw = 0.0, sz = 0.0;
  for (int i = tid; i < n; i += 256) {
    sw = fma(ye[i], wl[i], sw);
    sz = fma(ye[i], ye[i], sz);
  }
  sw = block_sum(sw, red);
  sz = block_sum(sz, red + kWaves);
  const double nu = sw / sz;
  double* v = w.vec + m * (N + 1);
  for (int i = tid; i < n; i += 256) v[i] = fma(-nu, ye[i], wl[i]);
}

// --------------------------------------------------------------------------
// EEQ adjoint: lambda = A^-1 [dL/dq; 0] (A symmetric), then
// beta_i = lambda_i d b_i / d raw-CN_i. One work-group per molecule.
// --------------------------------------------------------------------------

template <bool TILED, int NV>
__global__ __launch_bounds__(256) void k_adjoint(DevTables t, Params p, Inputs in,
                                                 Work w, int ordered) {
  extern __shared__ double smem[];
  const int64_t m = ordered ? w.eqord[blockIdx.x] : blockIdx.x;  // largest molecules first
  const int64_t N = w.N;
  const int n = w.natom[m];
  const int tid = threadIdx.x;
  const int64_t* Z = in.numbers + m * N;
  double* lam = w.lam + m * N;
  double* beta = w.beta + m * N;
  if (in.q_in != nullptr || n == 0 || (w.status[m] & kStatusSingular)) {
    for (int i = tid; i < N; i += 256) {
      lam[i] = 0.0;
      beta[i] = 0.0;
    }
    return;
  }
  for (int i = n + tid; i < N; i += 256) {
    lam[i] = 0.0;
    beta[i] = 0.0;
  }
  const double* g = w.dldq + m * N;
  if (w.status[m] & kStatusLU) {
    const int ld = (int)N + 1;
    const double* A = w.lu + (size_t)m * ld * ld;
    const int32_t* piv = w.piv + m * ld;
    double* vec = w.vec + m * ld;
    for (int i = tid; i < n; i += 256) vec[i] = Z[i] != 0 ? g[i] : 0.0;
    if (tid == 0) vec[n] = 0.0;
    lu_solve(A, ld, piv, n + 1, vec);
    for (int i = tid; i < n; i += 256) lam[i] = Z[i] != 0 ? vec[i] : 0.0;
  } else if (!TILED) {
    const double* gL = w.chol + (size_t)m * (size_t)tri((int)N);
    double* L = smem;
    const int nt = tri(n);
    for (int k0 = tid; k0 < nt; k0 += 8 * 256) {  // eight loads in flight
      double c[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) c[u] = gL[min(k0 + 256 * u, nt - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k0 + 256 * u < nt) L[k0 + 256 * u] = c[u];
    }
    __syncthreads();
    if (tid < 64) {
      // lambda = C^-1 (g - nu e), nu = e^T C^-1 g / e^T C^-1 e, with z_e =
      // D^-1 L^-1 e kept by the charge kernel
      const double* ye = w.ez + m * N;
      double v[NV], z[NV];
      double sw = 0.0, sz = 0.0;
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const int i = 64 * k + tid;
        v[k] = i < n && Z[i] != 0 ? g[i] : 0.0;
        z[k] = i < n ? ye[i] : 0.0;
      }
      wave_forward(L, n, v);
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const int i = min(64 * k + tid, n - 1);
        const double d = L[tri(i) + i];
        v[k] = 64 * k + tid < n ? v[k] : 0.0;
        sw = fma(z[k], v[k], sw);
        sz = fma(z[k] * d, z[k], sz);
        v[k] *= rcp_nt(d);
      }
      sw = wave_sum(sw);
      sz = wave_sum(sz);
      const double nu = sw / sz;
#pragma unroll
      for (int k = 0; k < NV; ++k) v[k] = fma(-nu, z[k], v[k]);
      wave_backward(L, n, v);
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const int i = 64 * k + tid;
        if (i < n) lam[i] = Z[i] != 0 ? v[k] : 0.0;
      }
    }
  }
  __syncthreads();
  for (int i = tid; i < n; i += 256) {
    const int zi = (int)Z[i];
    double b = 0.0;
    if (zi != 0) {
      const double c = w.cnq[m * N + i];
      const double dsq = c > kEps ? 0.5 / sqrt(c) : 0.0;
      b = lam[i] * t.kcn[zi] * dsq * w.dcnq[m * N + i];
    }
    beta[i] = b;
  }
}

// Order of the molecules for the one-work-group-per-molecule adjoint kernel:
// by atom count, largest first (counting sort; atom counts above kOrdMax
// share the first bin), so that the longest solves start first and the short
// ones fill in behind them (the adjoint of the 1024 x 20-120 batch alone 67 ->
// 48 us). Which work-group solves which molecule does not change any result;
// the order within a bin is arbitrary. (The charge kernel keeps the batch
// order: taking the largest first there made it faster alone, 217 -> 153 us,
// but the two-stream step slower, 1.10 -> 1.13 ms, as it then crowds the
// three-body pair pass that runs beside it.)
constexpr int kOrdMax = 256;

__global__ __launch_bounds__(1024) void k_eeq_order(Work w) {
  __shared__ int hist[kOrdMax + 1];
  __shared__ int start[kOrdMax + 1];
  const int tid = threadIdx.x;
  for (int c = tid; c <= kOrdMax; c += 1024) hist[c] = 0;
  __syncthreads();
  for (int64_t m = tid; m < w.B; m += 1024) atomicAdd(&hist[min(w.natom[m], kOrdMax)], 1);
  __syncthreads();
  if (tid == 0) {
    int acc = 0;
    for (int c = kOrdMax; c >= 0; --c) {
      start[c] = acc;
      acc += hist[c];
    }
  }
  __syncthreads();
  for (int64_t m = tid; m < w.B; m += 1024) {
    const int r = atomicAdd(&start[min(w.natom[m], kOrdMax)], 1);
    w.eqord[r] = (int32_t)m;
  }
}

}  // namespace

hipError_t ensure_lds(const void* kernel, size_t bytes) {
  // the limit is a property of the kernel on one device: remember what each
  // (kernel, device) was given
  static std::mutex mu;
  static std::map<std::pair<const void*, int>, size_t> given;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mu);
  size_t& have = given[{kernel, dev}];
  if (bytes <= have) return hipSuccess;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) have = bytes;
  return e;
}

// Launch a per-molecule EEQ kernel with `shmem` bytes of dynamic LDS, raising
// the kernel's LDS limit first when needed.
template <typename... Args>
hipError_t launch_lds(void (*kernel)(Args...), unsigned grid, unsigned block, size_t shmem,
                      hipStream_t s, Args... args) {
  hipError_t e = ensure_lds((const void*)kernel, shmem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), shmem, s, args...);
  return hipGetLastError();
}

// Molecules of this padded length take the tiled path (or every size, for
// testing).
inline bool eeq_tiled(const Params& p, int64_t N) {
  return p.force_tiled || N > kEeqMaxN;
}

hipError_t launch_eeq_tiled(hipStream_t s, const DevTables& t, const Params& p,
                            const Inputs& in, const Work& w) {
  const int N = (int)w.N;
  const unsigned B = (unsigned)w.B;
  const unsigned rows = (unsigned)((w.B * (w.N + 2) + kWaves - 1) / kWaves);
  hipLaunchKernelGGL(k_tf_assemble, dim3(rows), dim3(256), 0, s, t, p, in, w);
  hipError_t e = ensure_lds((const void*)k_tf_diag, kTfDiagLds);
  if (e == hipSuccess) e = ensure_lds((const void*)k_tf_panel, kTfTileLds);
  if (e == hipSuccess) e = ensure_lds((const void*)k_tf_update, kTfTileLds);
  if (e != hipSuccess) return e;
  for (int kb = 0; kb < N; kb += kTB) {
    hipLaunchKernelGGL(k_tf_diag, dim3(B), dim3(256), kTfDiagLds, s, in, w, kb);
    const unsigned ptiles = (unsigned)((N - kb + 1 + kTB - 1) / kTB);
    hipLaunchKernelGGL(k_tf_panel, dim3(B, ptiles), dim3(256), kTfTileLds, s, in, w, kb);
    if (kb + kTB < N) {
      const int nI = (N + 2 - kb - kTB + kTB - 1) / kTB;
      hipLaunchKernelGGL(k_tf_update, dim3(B, (unsigned)(nI * (nI + 1) / 2)), dim3(256),
                         kTfTileLds, s, in, w, kb);
    }
  }
  hipLaunchKernelGGL(k_tf_reduce, dim3(B), dim3(256), 0, s, in, w);
  for (int kb = ((N - 1) / kTB) * kTB; kb >= 0; kb -= kTB) {
    const unsigned chunks = (unsigned)max(1, (kb + 255) / 256);
    hipLaunchKernelGGL(k_tf_bsolve, dim3(B, chunks), dim3(256), 0, s, in, w, kb, w.q);
  }
  return hipGetLastError();
}

constexpr unsigned kLuGroups = 64;  // work-groups of the LU fallback launch

// Batches that fit the chip in one round (one work-group per CU) take the
// molecules in batch order: there the order cannot save a round, and the
// sort is a launch on the chain of every evaluation (6 us of a single
// molecule's). The paired solve reads the order at any size.
inline bool eeq_ordered(const Work& w) { return w.B > 256; }

// Padded lengths from here on pair two molecules per work-group in
// energy-only evaluations.
constexpr int64_t kEeqPairedMinN = 196;

template <int NW, int NV, bool PAIRED>
hipError_t launch_chol(hipStream_t s, const DevTables& t, const Params& p, const Inputs& in,
                       const Work& w) {
  const unsigned grid = (unsigned)(PAIRED ? (w.B + 1) / 2 : w.B);
  const size_t doubles = eeq_doubles(w.N);
  return launch_lds(k_eeq_chol<NW, NV, PAIRED>, grid, 64 * NW, sizeof(double) * doubles, s, t, p, in,
                    w, (int)doubles, eeq_ordered(w) ? 1 : 0);
}

hipError_t launch_eeq(hipStream_t s, const DevTables& t, const Params& p,
                      const Inputs& in, const Work& w, bool paired) {
  const unsigned grid = (unsigned)w.B;
  if (grid == 0) return hipSuccess;
  const bool tiled = eeq_tiled(p, w.N);
  paired = paired && !tiled && w.N >= kEeqPairedMinN;
  // molecule order of the solve and the adjoint (the backward reads the order
  // the forward left in the workspace)
  if (paired || eeq_ordered(w)) hipLaunchKernelGGL(k_eeq_order, dim3(1), dim3(1024), 0, s, w);
  hipError_t e;
  if (tiled)
    e = launch_eeq_tiled(s, t, p, in, w);
  else if (paired)  // one work-group per CU: two molecules each (sizes from k_eeq_order)
    e = launch_chol<8, 4, true>(s, t, p, in, w);
  else if (eeq_waves(w.N) == 8)
    e = launch_chol<8, 4, false>(s, t, p, in, w);
  else if (solve_regs(w.N) > 2)
    e = launch_chol<4, 4, false>(s, t, p, in, w);
  else
    e = launch_chol<4, 2, false>(s, t, p, in, w);
  if (e != hipSuccess) return e;
  if (tiled)  // (the LDS kernels solve their failed systems themselves)
    hipLaunchKernelGGL(k_eeq_lu, dim3(grid < kLuGroups ? grid : kLuGroups), dim3(256), 0, s, t,
                       p, in, w);
  return hipGetLastError();
}

hipError_t launch_adjoint(hipStream_t s, const DevTables& t, const Params& p,
                          const Inputs& in, const Work& w) {
  const unsigned grid = (unsigned)w.B;
  const int ordered = eeq_ordered(w) ? 1 : 0;
  if (eeq_tiled(p, w.N)) {
    const int N = (int)w.N;
    hipLaunchKernelGGL(k_tf_adj_init, dim3(grid), dim3(256), 0, s, in, w);
    for (int kb = 0; kb < N; kb += kTB) {
      const unsigned chunks = (unsigned)max(1, (N - kb + 255) / 256);
      hipLaunchKernelGGL(k_tf_fsolve, dim3(grid, chunks), dim3(256), 0, s, in, w, kb, w.lam);
    }
    hipLaunchKernelGGL(k_tf_adj_mid, dim3(grid), dim3(256), 0, s, in, w);
    for (int kb = ((N - 1) / kTB) * kTB; kb >= 0; kb -= kTB) {
      const unsigned chunks = (unsigned)max(1, (kb + 255) / 256);
      hipLaunchKernelGGL(k_tf_bsolve, dim3(grid, chunks), dim3(256), 0, s, in, w, kb, w.lam);
    }
    hipLaunchKernelGGL((k_adjoint<true, 2>), dim3(grid), dim3(256), 0, s, t, p, in, w, ordered);
    return hipGetLastError();
  }
  const size_t shmem = sizeof(double) * ((size_t)tri((int)w.N) + kSolvePad);
  if (solve_regs(w.N) > 2)
    return launch_lds(k_adjoint<false, 4>, grid, 256, shmem, s, t, p, in, w, ordered);
  return launch_lds(k_adjoint<false, 2>, grid, 256, shmem, s, t, p, in, w, ordered);
}

}  // namespace d4
