// HIP kernels (gfx950) for the EEQ charges and their adjoint.
//
// Molecules whose packed Coulomb factor fits in LDS are solved by one
// work-group each (L D L^T by whole waves, FP64 matrix instructions); larger
// molecules use the tiled multi-work-group path.
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

constexpr int kNB = 16;  // columns of a block

__device__ __forceinline__ double lane_bcast(double v, int src) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), src);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), src);
  return __hiloint2double(hi, lo);
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
// One 150-atom molecule takes 63 us (assembly 14, panels 17, updates 18,
// substitution 8, the rest loads and barriers); the blocked Cholesky with
// inverse diagonal blocks and 4 x 4 register tiles that was here before, by
// four waves with barriers in the substitutions, took 147 us. 1024 molecules
// of 20-120 atoms alone: 86 instead of 177 us.

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

// A panel: D holds row (lane & 15) of the block itself, d the lane's row below
// it, w the reciprocal pivots. Entries right of a row's diagonal in D are junk.
struct Panel {
  double D[kNB], d[kNB], w[kNB];
  unsigned long long good;  // non-zero lanes: every pivot so far is positive
};

// Column J of the elimination, u = D[J], for other columns C: D[C] += u t and, with
// ROWS, d[C] += u t2, with u of lane C of each 16-lane row. A DPP operand may not
// be written by the two instructions before, and the compiler, which does not look
// into the assembly, could place a copy of u just there: each statement fills the
// two slots itself, with a link of the pivot chain and a wait. (Captured step of
// one 150-atom molecule: 151.8 us with the slots left open, 153.5 with two waits
// in each statement, 152.8 so.)
#define D4_FMAC(acc, t, c) \
  "v_fmac_f64_dpp %[" acc "], %[u], %[" t "] row_newbcast:%[" c "] row_mask:0xf bank_mask:0xf\n\t"
#define D4_COL(k) D4_FMAC("D" k, "t", "c" k)
#define D4_COL2(k) D4_FMAC("D" k, "t", "c" k) D4_FMAC("d" k, "t2", "c" k)

// The next column, with the products t = -u w and t2 = -d[J] w in the two slots,
// and its pivot for all lanes of a row.
template <bool ROWS, int J>
__device__ __forceinline__ double panel_next(Panel& P, double& t, double& t2) {
  double pv;
  if constexpr (ROWS)
    asm("v_mul_f64 %[t], -%[u], %[w]\n\t"
        "v_mul_f64 %[t2], -%[v], %[w]\n\t"
        D4_COL2("0")
        "s_nop 0\n\t"
        "v_mov_b64_dpp %[pv], %[D0] row_newbcast:%[c0] row_mask:0xf bank_mask:0xf"
        : [D0] "+&v"(P.D[J + 1]), [d0] "+&v"(P.d[J + 1]), [t] "=&v"(t), [t2] "=&v"(t2),
          [pv] "=&v"(pv)
        : [u] "v"(P.D[J]), [v] "v"(P.d[J]), [w] "v"(P.w[J]), [c0] "n"(J + 1));
  else
    asm("v_mul_f64 %[t], -%[u], %[w]\n\t"
        "s_nop 0\n\t"
        D4_COL("0")
        "s_nop 1\n\t"
        "v_mov_b64_dpp %[pv], %[D0] row_newbcast:%[c0] row_mask:0xf bank_mask:0xf"
        : [D0] "+&v"(P.D[J + 1]), [t] "=&v"(t), [pv] "=&v"(pv)
        : [u] "v"(P.D[J]), [w] "v"(P.w[J]), [c0] "n"(J + 1));
  return pv;
}

// Columns C .. C + K - 1 (K <= 4) behind x = the link of the chain that LEAD names.
enum { kLeadRcp, kLeadError, kLeadSquare, kLeadStep };
#define D4_COLUMNS(LEAD, ...)                                                              \
  if constexpr (K == 1 && ROWS)                                                            \
    asm(LEAD D4_COL2("0")                                                                  \
        : [x] "=&v"(x), [D0] "+&v"(P.D[C]), [d0] "+&v"(P.d[C])                             \
        : [u] "v"(P.D[J]), [t] "v"(t), [t2] "v"(t2), [c0] "n"(C), __VA_ARGS__);            \
  if constexpr (K == 1 && !ROWS)                                                           \
    asm(LEAD D4_COL("0")                                                                   \
        : [x] "=&v"(x), [D0] "+&v"(P.D[C])                                                 \
        : [u] "v"(P.D[J]), [t] "v"(t), [c0] "n"(C), __VA_ARGS__);                          \
  if constexpr (K == 2 && ROWS)                                                            \
    asm(LEAD D4_COL2("0") D4_COL2("1")                                                     \
        : [x] "=&v"(x), [D0] "+&v"(P.D[C]), [d0] "+&v"(P.d[C]), [D1] "+&v"(P.D[C + 1]),    \
          [d1] "+&v"(P.d[C + 1])                                                           \
        : [u] "v"(P.D[J]), [t] "v"(t), [t2] "v"(t2), [c0] "n"(C), [c1] "n"(C + 1),         \
          __VA_ARGS__);                                                                    \
  if constexpr (K == 2 && !ROWS)                                                           \
    asm(LEAD D4_COL("0") D4_COL("1")                                                       \
        : [x] "=&v"(x), [D0] "+&v"(P.D[C]), [D1] "+&v"(P.D[C + 1])                         \
        : [u] "v"(P.D[J]), [t] "v"(t), [c0] "n"(C), [c1] "n"(C + 1), __VA_ARGS__);         \
  if constexpr (K == 3 && ROWS)                                                            \
    asm(LEAD D4_COL2("0") D4_COL2("1") D4_COL2("2")                                        \
        : [x] "=&v"(x), [D0] "+&v"(P.D[C]), [d0] "+&v"(P.d[C]), [D1] "+&v"(P.D[C + 1]),    \
          [d1] "+&v"(P.d[C + 1]), [D2] "+&v"(P.D[C + 2]), [d2] "+&v"(P.d[C + 2])           \
        : [u] "v"(P.D[J]), [t] "v"(t), [t2] "v"(t2), [c0] "n"(C), [c1] "n"(C + 1),         \
          [c2] "n"(C + 2), __VA_ARGS__);                                                   \
  if constexpr (K == 3 && !ROWS)                                                           \
    asm(LEAD D4_COL("0") D4_COL("1") D4_COL("2")                                           \
        : [x] "=&v"(x), [D0] "+&v"(P.D[C]), [D1] "+&v"(P.D[C + 1]), [D2] "+&v"(P.D[C + 2]) \
        : [u] "v"(P.D[J]), [t] "v"(t), [c0] "n"(C), [c1] "n"(C + 1), [c2] "n"(C + 2),      \
          __VA_ARGS__);                                                                    \
  if constexpr (K == 4 && ROWS)                                                            \
    asm(LEAD D4_COL2("0") D4_COL2("1") D4_COL2("2") D4_COL2("3")                           \
        : [x] "=&v"(x), [D0] "+&v"(P.D[C]), [d0] "+&v"(P.d[C]), [D1] "+&v"(P.D[C + 1]),    \
          [d1] "+&v"(P.d[C + 1]), [D2] "+&v"(P.D[C + 2]), [d2] "+&v"(P.d[C + 2]),          \
          [D3] "+&v"(P.D[C + 3]), [d3] "+&v"(P.d[C + 3])                                   \
        : [u] "v"(P.D[J]), [t] "v"(t), [t2] "v"(t2), [c0] "n"(C), [c1] "n"(C + 1),         \
          [c2] "n"(C + 2), [c3] "n"(C + 3), __VA_ARGS__);                                  \
  if constexpr (K == 4 && !ROWS)                                                           \
    asm(LEAD D4_COL("0") D4_COL("1") D4_COL("2") D4_COL("3")                               \
        : [x] "=&v"(x), [D0] "+&v"(P.D[C]), [D1] "+&v"(P.D[C + 1]), [D2] "+&v"(P.D[C + 2]), \
          [D3] "+&v"(P.D[C + 3])                                                           \
        : [u] "v"(P.D[J]), [t] "v"(t), [c0] "n"(C), [c1] "n"(C + 1), [c2] "n"(C + 2),      \
          [c3] "n"(C + 3), __VA_ARGS__);

template <int LEAD, bool ROWS, int J, int C, int K>
__device__ __forceinline__ double panel_columns(Panel& P, double t, double t2, double a, double b) {
  double x;
  if constexpr (K == 0 && LEAD == kLeadRcp) x = __builtin_amdgcn_rcp(a);
  if constexpr (K == 0 && LEAD == kLeadError) x = fma(-a, b, 1.0);
  if constexpr (K == 0 && LEAD == kLeadSquare) x = fma(a, a, a);
  if constexpr (K == 0 && LEAD == kLeadStep) x = fma(b, a, b);
  if constexpr (LEAD == kLeadRcp) {
    D4_COLUMNS("v_rcp_f64 %[x], %[a]\n\ts_nop 0\n\t", [a] "v"(a))
  } else if constexpr (LEAD == kLeadError) {
    D4_COLUMNS("v_fma_f64 %[x], -%[a], %[b], 1.0\n\ts_nop 0\n\t", [a] "v"(a), [b] "v"(b))
  } else if constexpr (LEAD == kLeadSquare) {
    D4_COLUMNS("v_fma_f64 %[x], %[a], %[a], %[a]\n\ts_nop 0\n\t", [a] "v"(a))
  } else {
    D4_COLUMNS("v_fma_f64 %[x], %[b], %[a], %[b]\n\ts_nop 0\n\t", [a] "v"(a), [b] "v"(b))
  }
  return x;
}
#undef D4_COLUMNS
#undef D4_COL2
#undef D4_COL
#undef D4_FMAC

// Columns left of at most `most` from column C on.
constexpr int panel_part(int c, int most) {
  return kNB - c < 0 ? 0 : kNB - c < most ? kNB - c : most;
}

// Eliminate column J and go on with J + 1, whose pivot chain is spread between
// the updates of column J. The columns keep their values before the division
// by the pivot.
constexpr int kFcmpOgt = 2;  // ordered and greater than

template <bool ROWS, bool FULL, bool WLDS, int J>
__device__ __forceinline__ void panel_step(Panel& P, int nb, double* W) {
  if constexpr (J + 1 < kNB) {
    P.w[J + 1] = 0.0;
    if (FULL || J + 1 < nb) {  // uniform (columns past nb are padding)
      double t, t2 = 0.0;
      const double pv = panel_next<ROWS, J>(P, t, t2);
      // 1 / pv from the hardware estimate (relative error below 2^-23) by a
      // third-order step, its links between the other columns
      constexpr int C0 = J + 2, K0 = panel_part(C0, 4), C1 = C0 + K0, K1 = panel_part(C1, 3),
                    C2 = C1 + K1, K2 = panel_part(C2, 3), C3 = C2 + K2, K3 = panel_part(C3, 4);
      static_assert(C3 + K3 >= kNB, "all columns");
      const double r = panel_columns<kLeadRcp, ROWS, J, C0, K0>(P, t, t2, pv, pv);
      const double e = panel_columns<kLeadError, ROWS, J, C1, K1>(P, t, t2, pv, r);
      const double e2 = panel_columns<kLeadSquare, ROWS, J, C2, K2>(P, t, t2, e, e);
      P.w[J + 1] = panel_columns<kLeadStep, ROWS, J, C3, K3>(P, t, t2, e2, r);
      if (WLDS) W[J + 1] = P.w[J + 1];  // (every lane the same value)
      P.good &= __builtin_amdgcn_fcmp(pv, 0.0, kFcmpOgt);
      __builtin_amdgcn_sched_barrier(0);  // (hoisting across columns only costs registers)
    }
    panel_step<ROWS, FULL, WLDS, J + 1>(P, nb, W);
  }
}

// (whole panels have no branches between their columns: 2.1 k clocks for the
// block alone, 3.0 k with the rows below, against 4-5 k)
// WLDS: the reciprocal pivots also go to W in LDS, for a caller that has no
// registers to keep them.
template <bool ROWS, bool FULL, bool WLDS = false>
__device__ __forceinline__ void panel_factor(Panel& P, int nb, double* W = nullptr) {
  const double pv = row_bcast<0>(P.D[0]);
  P.good = __builtin_amdgcn_fcmp(pv, 0.0, kFcmpOgt);
  P.w[0] = rcp_nt(pv);
  if (WLDS) W[0] = P.w[0];
  panel_step<ROWS, FULL, WLDS, 0>(P, nb, W);
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

// A wave's share of a panel in LDS: its 64 rows below the block (`row`; a border
// row goes to `border`, not divided by the pivots).
template <bool FULL>
__device__ __forceinline__ void panel_rows(Panel& P, double* L, int n, int kb, int nb, int row,
                                           double* border) {
  panel_factor<true, FULL>(P, nb);
  if (FULL && row < n) {  // (there are rows below a full block only)
    double* Lr = L + tri(row) + kb;
#pragma unroll
    for (int c = 0; c < kNB; ++c) Lr[c] = P.d[c] * P.w[c];
  }
  if (border != nullptr) {
#pragma unroll
    for (int c = 0; c < kNB; ++c) border[c] = P.d[c];
  }
}

// The block itself, by one wave: L below the diagonal, the pivots on it.
template <bool FULL>
__device__ __forceinline__ void panel_block(Panel& P, double* L, int kb, int nb, int* flag) {
  const int lane = threadIdx.x & 63;
  panel_factor<false, FULL>(P, nb);
  if (lane == 0) *flag = P.good != 0ull ? 0 : 1;
  if (lane < nb) {
    double* Dr = L + tri(kb + lane) + kb;
#pragma unroll
    for (int c = 0; c < kNB; ++c)
      if (c <= lane) Dr[c] = c < lane ? P.D[c] * P.w[c] : P.D[c];
  }
}

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
      if (nb == kNB)
        panel_rows<true>(P, L, n, kb, nb, row, is_border ? sm.y[border] : nullptr);
      else
        panel_rows<false>(P, L, n, kb, nb, row, is_border ? sm.y[border] : nullptr);
    } else if (wave == 3) {
      if (nb == kNB)
        panel_block<true>(P, L, kb, nb, sm.idx);
      else
        panel_block<false>(P, L, kb, nb, sm.idx);
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
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 4 ? 3 : 2))) void k_eeq_chol(
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
#pragma unroll 1
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
// e (the forward substitution of b and e is the elimination of those rows).
// L D L^T in 64-column blocks, one launch per block (k_tl_step): the launch of
// block kb applies block kb - 64 to everything behind it, and factors its own.
//  - A work-group of panel row tile y updates the diagonal tile and its own
//    64-row tile (MFMA), factors the diagonal tile in LDS and finishes its own
//    rows beside it. Every one factors the same diagonal tile, so the rows
//    need no other launch; work-group 0 alone stores it.
//  - The other work-groups update the 64 x 64 tiles of the trailing triangle.
// The finished diagonal tile goes transposed into the upper triangle of A (the
// tile itself is still being read by the other work-groups), its pivots to
// w.dpiv; the rows below are finished in place. So a work-group only reads
// what earlier launches wrote or what it writes itself.
// The substitutions go by 256 entries: one work-group per molecule solves them
// (k_tl_solve, 64 at a time with the vector in LDS), then many work-groups take
// their share off the rest of the vector (k_tl_gemv).
// What bounds it: the panel chain (four 16-column panels a launch) and launch
// latency. One 701-atom molecule (11 blocks): 26 us a launch of k_tl_step
// (loads and update 6-12 us, panels 8) where the three launches per block
// that were here before took 115 (diagonal block 65, panel 23, update 27), and
// 22 us per 256 entries of a substitution against 60-100; its energy and
// forces through autograd 2.4 -> 1.3 ms.
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

// States of the factorisation of molecule m, non-zero where it goes to the
// pivoted LU: word 0 is written by the assembly, word b + 1 by work-group 0 of
// block b's launch, which reads word b. A launch so reads nothing that it
// writes: all waves of its work-groups leave together or stay together. (The
// words lie in the pivot rows, which the LU kernel fills later.)
__device__ __forceinline__ int32_t* tf_state(const Work& w, int64_t m) {
  return w.piv + m * (w.N + 1);
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
  // (testing: every system goes to the pivoted-LU kernel)
  if (i == 0 && lane == 0) tf_state(w, m)[0] = p.force_lu;
  if (p.force_lu) return;
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

// The tiled kernels take their LDS as dynamic shared memory and at most 80
// VGPRs (k_tl_step spills 31 of them, k_tl_solve 20): a work-group then fits
// beside the three-body kernel's waves with gradients (two per SIMD with 192
// VGPRs, 86 KB of LDS per CU) on any CU instead of waiting until one is nearly
// empty. Beside the energy kernel (108 VGPRs, four waves per SIMD) it waits for
// the first ones to end.
constexpr int kTS = kTB + 1;  // row stride of a tile in LDS
constexpr size_t kTlLds = sizeof(double) * (2 * kTB * kTS + kTB + 3 * kNB + 2);

// c0 (TWO: and c1) -= rows r0 .. of P times rows q0 .. (q1 ..) of Q over K
// columns, the columns weighted by piv[k * ps] (P, Q: tiles in LDS).
template <bool TWO>
__device__ __forceinline__ void tl_product(const double* P, int r0, const double* Q, int q0, int q1,
                                           const double* piv, int ps, int K, d4_acc& c0,
                                           d4_acc& c1) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const double* pa = P + (r0 + l16) * kTS + 4 * g;
  const double* pb = Q + (q0 + l16) * kTS + 4 * g;
  const double* pc = Q + (q1 + l16) * kTS + 4 * g;
  const double* pd = piv + 4 * g * ps;
#pragma unroll 1
  for (int k = 0; k < K; k += kNB) {
    double a[4], b[4], c[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      a[s] = -pa[k + s] * pd[(k + s) * ps];
      b[s] = pb[k + s];
      if (TWO) c[s] = pc[k + s];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[s], c0, 0, 0, 0);
      if (TWO) c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], c[s], c1, 0, 0, 0);
    }
  }
}

// Rows r0 .. r0 + 63 (below `rows`, else zero), columns c0 .. c0 + 63 (below
// `cols`, else zero) of A into a tile, eight loads in flight per thread. LOWER:
// a diagonal tile, whose upper triangle (which work-group 0 of the launch
// replaces) is neither read nor used.
template <bool LOWER = false>
__device__ __forceinline__ void tl_load(const double* A, int64_t N, int r0, int rows, int c0,
                                        int cols, double* T) {
  const int c = threadIdx.x & (kTB - 1), rr = threadIdx.x >> 6;
  const double* p = A + (size_t)r0 * N + c0 + min(c, cols - 1);
#pragma unroll 1
  for (int h = 0; h < 2; ++h) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int r = min(rr + 32 * h + 4 * u, rows - 1);
      v[u] = p[r * (int)N - (LOWER ? max(0, min(c, cols - 1) - r) : 0)];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int r = rr + 32 * h + 4 * u;
      T[r * kTS + c] = r < rows && c < cols ? v[u] : 0.0;
    }
  }
}

// A wave's share of a 16-column panel in the tiles (block of D at c0, nbs
// columns used): the block itself (ROWS = false: L below the diagonal, the
// pivots on it, junk that nothing reads right of it), or a row per lane
// (`row` null: none). All waves read the block before any writes it. W: 16
// doubles of LDS of the wave.
template <bool ROWS, bool FULL>
__device__ __forceinline__ void tl_panel(double* D, int c0, int nbs, double* row, double* W,
                                         int* flag) {
  const int lane = threadIdx.x & 63;
  Panel P;
  const double* Dl = D + (c0 + (lane & 15)) * kTS + c0;
  const double* rl = ROWS && row != nullptr ? row : Dl;
#pragma unroll
  for (int c = 0; c < kNB; ++c) {
    P.D[c] = Dl[FULL ? c : min(c, nbs - 1)];
    if (ROWS) P.d[c] = rl[FULL ? c : min(c, nbs - 1)];
  }
  __syncthreads();
  panel_factor<ROWS, FULL, true>(P, nbs, W);
  if (ROWS) {
    if (row != nullptr) {
#pragma unroll
      for (int c = 0; c < kNB; ++c)
        if (FULL || c < nbs) row[c] = P.d[c] * W[c];
    }
    return;
  }
  if (lane == 0) *flag = P.good != 0ull ? 0 : 1;
  if (lane < nbs) {
    double* Dr = D + (c0 + lane) * kTS + c0;
    double pivot = P.D[0];
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      pivot = lane == c ? P.D[c] : pivot;
      Dr[c] = P.D[c] * (FULL || c < nbs ? W[c] : 0.0);
    }
    Dr[lane] = pivot;
  }
}

template <bool FULL>
__device__ __forceinline__ void tl_panels(double* D, double* T, bool own, int dmax, int c0, int nbs,
                                          double* W, int* flag, int wave) {
  const int lane = threadIdx.x & 63;
  if (wave == 0 && own) {
    tl_panel<true, FULL>(D, c0, nbs, T + lane * kTS + c0, W, flag);
  } else if (wave == 1) {
    const int r = c0 + nbs + lane;
    tl_panel<true, FULL>(D, c0, nbs, r < dmax ? D + r * kTS + c0 : nullptr, W + kNB, flag);
  } else if (wave == 3) {
    tl_panel<false, FULL>(D, c0, nbs, nullptr, W + 2 * kNB, flag);
  } else {
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_tl_step(
    Inputs in, Work w, int kb, int npanel) {
  tf_priority();
  extern __shared__ double s_tl[];
  double* X = s_tl;               // [64][65]
  double* Y = X + kTB * kTS;      // [64][65]
  double* piv = Y + kTB * kTS;    // [64] pivots of block kb - 64
  double* W = piv + kTB;          // [3][16] reciprocal pivots
  int* flag = reinterpret_cast<int*>(W + 3 * kNB);
  const int64_t m = blockIdx.x;
  if (in.q_in != nullptr || kb >= w.natom[m]) return;
  int32_t* state = tf_state(w, m) + kb / kTB;
  if (state[0]) {
    if (blockIdx.y == 0 && threadIdx.x == 0) state[1] = 1;
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t N = w.N;
  const int n = w.natom[m], last = n + 2;  // rows with the border
  const int nb = min(kTB, n - kb), pk = kb - kTB;
  double* A = tf_matrix(w, m);
  double* dpiv = w.dpiv + m * N;
  const int y = (int)blockIdx.y;
  if (kb > 0 && tid < kTB) piv[tid] = dpiv[pk + tid];

  if (y >= npanel) {  // a trailing tile
    const int e = y - npanel, r0 = kb + kTB;
    if (r0 >= n) return;
    const int I = incl_row(e), J = e - tri(I);
    const int i0 = r0 + I * kTB, j0 = r0 + J * kTB;
    if (i0 >= last || j0 >= n) return;
    tl_load(A, N, i0, last - i0, pk, kTB, X);
    tl_load(A, N, j0, n - j0, pk, kTB, Y);
    __syncthreads();
#pragma unroll 1
    for (int ct = 0; ct < 4; ct += 2) {
      d4_acc c[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int j = j0 + kNB * (ct + h) + l16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = i0 + kNB * wave + 4 * r + g;
          c[h][r] = i < last && j < n && j <= i ? A[(size_t)i * N + j] : 0.0;
        }
      }
      tl_product<true>(X, kNB * wave, Y, kNB * ct, kNB * ct + kNB, piv, 1, kTB, c[0], c[1]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int j = j0 + kNB * (ct + h) + l16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = i0 + kNB * wave + 4 * r + g;
          if (i < last && j < n && j <= i) A[(size_t)i * N + j] = c[h][r];
        }
      }
    }
    return;
  }

  // a panel row tile: D the diagonal tile (its rows past nb: border rows), T
  // the work-group's own rows
  const int r0 = kb + y * kTB, rows = last - r0;
  if (rows <= 0) return;
  const bool own = y > 0;
  // (border rows in the diagonal tile are work-group 0's alone: it stores them
  // in place during this launch)
  const int drows = own ? nb : last - kb;
  double* D = Y;
  double* T = X;
  if (kb == 0) {
    tl_load<true>(A, N, 0, drows, 0, nb, D);
    if (own) tl_load(A, N, r0, rows, 0, nb, T);
    __syncthreads();
  } else {
    d4_acc o[4];
    if (own) {
      const double* Ao = A + (size_t)r0 * N + kb;
      tl_load(A, N, r0, rows, pk, kTB, Y);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        const int c = kNB * ct + l16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = kNB * wave + 4 * r + g;
          o[ct][r] = i < rows && c < nb ? Ao[i * (int)N + c] : 0.0;
        }
      }
    }
    tl_load(A, N, kb, drows, pk, kTB, X);
    __syncthreads();
    if (own) {
      tl_product<true>(Y, kNB * wave, X, 0, kNB, piv, 1, kTB, o[0], o[1]);
      tl_product<true>(Y, kNB * wave, X, 2 * kNB, 3 * kNB, piv, 1, kTB, o[2], o[3]);
      __syncthreads();  // Y is free
    }
    // the ten 16 x 16 tiles on and below the diagonal, as five pairs: wave q
    // row 3 columns (0, 1), row 3 columns (2, 3), row 2 columns (0, 1) and row
    // 1 columns (0, 1), then waves 0 and 1 the diagonal tiles (2, 2) and (0, 0)
#pragma unroll 1
    for (int q = wave; q < 6; q += 4) {
      const int rt = q < 2 ? 3 : q == 2 || q == 4 ? 2 : q == 3 ? 1 : 0;
      const int ct = q == 1 ? 2 : q == 4 ? 2 : 0;
      const bool two = q < 4;
      d4_acc v[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int c = kNB * (ct + h) + l16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = kNB * rt + 4 * r + g;
          v[h][r] = (h == 0 || two) && i < drows && c < nb && c <= i
                        ? A[(size_t)(kb + i) * N + kb + c] : 0.0;
        }
      }
      if (two)
        tl_product<true>(X, kNB * rt, X, kNB * ct, kNB * ct + kNB, piv, 1, kTB, v[0], v[1]);
      else
        tl_product<false>(X, kNB * rt, X, kNB * ct, 0, piv, 1, kTB, v[0], v[1]);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (h == 0 || two) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            D[(kNB * rt + 4 * r + g) * kTS + kNB * (ct + h) + l16] = v[h][r];
        }
    }
    __syncthreads();  // X is free
    if (own) {
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          T[(kNB * wave + 4 * r + g) * kTS + kNB * ct + l16] = o[ct][r];
    }
    __syncthreads();
  }

  const int dmax = min(kTB, drows);
  for (int c0 = 0; c0 < nb; c0 += kNB) {
    const int nbs = min(kNB, nb - c0);
    if (c0 > 0) {
      // left-looking update of the 16 columns in D's rows from c0 on and in T
      const int nd = 4 - c0 / kNB, total = nd + (own ? 4 : 0);
      for (int t = wave; t < total; t += 4) {
        double* M = t < nd ? D : T;
        const int rt = t < nd ? c0 + kNB * t : kNB * (t - nd);
        d4_acc c = {0.0, 0.0, 0.0, 0.0};
        tl_product<false>(M, rt, D, c0, 0, D, kTS + 1, c0, c, c);
#pragma unroll
        for (int r = 0; r < 4; ++r) M[(rt + 4 * r + g) * kTS + c0 + l16] += c[r];
      }
      __syncthreads();
    }
    if (nbs == kNB)
      tl_panels<true>(D, T, own, dmax, c0, nbs, W, flag, wave);
    else
      tl_panels<false>(D, T, own, dmax, c0, nbs, W, flag, wave);
    __syncthreads();
    if (*flag) {  // uniform
      if (y == 0 && tid == 0) state[1] = 1;
      return;
    }
  }

  if (own) {
    for (int e = tid; e < kTB * kTB; e += 256) {
      const int r = e >> 6, c = e & (kTB - 1);
      if (r < rows && c < nb) A[(size_t)(r0 + r) * N + kb + c] = T[r * kTS + c];
    }
    return;
  }
  for (int e = tid; e < kTB * kTB; e += 256) {
    const int c = e >> 6, r = e & (kTB - 1);
    if (c < r && r < nb) A[(size_t)(kb + c) * N + kb + r] = D[r * kTS + c];
  }
  if (tid == 0) state[1] = 0;
  if (tid < nb) dpiv[kb + tid] = D[tid * (kTS + 1)];
  for (int r = nb; r < dmax; ++r)  // border rows in the diagonal tile
    if (tid < nb) A[(size_t)(kb + r) * N + kb + tid] = D[r * kTS + tid];
}

// After the factorisation: charges given or padding, then mu and the
// right-hand side D^-1 L^-1 (b - mu e) of the backward substitution (in vec);
// D^-1 L^-1 e is kept for the adjoint.
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
  if (n == 0) return;
  if (tf_state(w, m)[(n - 1) / kTB + 1]) {
    if (tid == 0) w.status[m] |= kStatusLU;
    return;
  }
  // the border rows hold D^-1 L^-1 b and D^-1 L^-1 e
  const double* A = tf_matrix(w, m);
  const double* zb = A + (size_t)n * N;
  const double* ze = A + (size_t)(n + 1) * N;
  const double* dpiv = w.dpiv + m * N;
  double sbe = 0.0, see = 0.0;
  for (int i = tid; i < n; i += 256) {
    const double u = ze[i] * dpiv[i];
    sbe = fma(u, zb[i], sbe);
    see = fma(u, ze[i], see);
  }
  sbe = block_sum(sbe, red);
  see = block_sum(see, red + kWaves);
  const double mu = (sbe - in.charge[m]) / see;
  double* v = w.vec + m * (N + 1);
  double* gz = w.ez + m * N;
  for (int i = tid; i < n; i += 256) {
    v[i] = fma(-mu, ze[i], zb[i]);
    gz[i] = ze[i];
  }
}

// Vector entries of one k_tl_solve: one per thread of a work-group of four
// waves, which fits beside the three-body waves (a work-group of sixteen waits
// for a CU without any).
constexpr int kTV = 256;
constexpr int kTQ = kTB * kTB / kTV;  // tile entries per thread
constexpr size_t kTlSolveLds = sizeof(double) * (kTB * kTS + kTV + kTB);

// Whether the substitutions of molecule m run (charges solved by this factor).
__device__ __forceinline__ bool tl_solving(const Inputs& in, const Work& w, int64_t m) {
  return in.q_in == nullptr && !(w.status[m] & (kStatusLU | kStatusSingular));
}

// 64 steps of a substitution within a diagonal tile, lane r: entry r of the
// vector. BACK: x = L^-T v, else y = L^-1 v; T[c][r] = L[r][c], zero unless
// r > c.
template <bool BACK>
__device__ __forceinline__ double tl_tile_solve(const double* T, double v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 0; h < 8; ++h) {
    double l[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = BACK ? 63 - 8 * h - u : 8 * h + u;
      l[u] = BACK ? T[lane * kTS + k] : T[k * kTS + lane];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = BACK ? 63 - 8 * h - u : 8 * h + u;
      v = fma(-l[u], lane_bcast(v, k), v);
    }
  }
  return v;
}

// Entries s0 .. s0 + kTV - 1 of L^T x = v (BACK, their later entries already
// taken off) or L y = v; the result goes to w.vec and to dst (BACK: zero on
// padding atoms).
template <bool BACK>
__global__ __launch_bounds__(kTV) __attribute__((amdgpu_waves_per_eu(6))) void k_tl_solve(
    Inputs in, Work w, int s0, double* dst) {
  tf_priority();
  extern __shared__ double s_tl[];
  double* s_t = s_tl;              // [64][65]
  double* s_v = s_t + kTB * kTS;   // [kTV]
  double* s_x = s_v + kTV;         // [64]
  const int64_t m = blockIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  if (s0 >= n || !tl_solving(in, w, m)) return;
  const int tid = threadIdx.x;
  const int s1 = min(s0 + kTV, n), nblk = (s1 - s0 + kTB - 1) / kTB;
  const double* A = tf_matrix(w, m);
  double* v = w.vec + m * (N + 1);
  s_v[tid] = s0 + tid < s1 ? v[s0 + tid] : 0.0;
  double next[kTQ];  // the tile of the next block, transposed as it is stored
  auto fetch = [&](int b) {
    const int kb = s0 + kTB * b;
#pragma unroll
    for (int u = 0; u < kTQ; ++u) {
      const int e = tid + kTV * u, c = e >> 6, r = e & (kTB - 1);
      next[u] = c < r && kb + r < n ? A[(size_t)(kb + c) * N + kb + r] : 0.0;
    }
  };
  fetch(BACK ? nblk - 1 : 0);
  for (int q = 0; q < nblk; ++q) {
    const int b = BACK ? nblk - 1 - q : q;
    const int kb = s0 + kTB * b, nb = min(kTB, s1 - kb);
#pragma unroll
    for (int u = 0; u < kTQ; ++u) {
      const int e = tid + kTV * u;
      s_t[(e >> 6) * kTS + (e & (kTB - 1))] = next[u];
    }
    __syncthreads();
    if (tid < kTB) {
      const double x = tl_tile_solve<BACK>(s_t, s_v[kTB * b + tid]);
      s_x[tid] = x;
      s_v[kTB * b + tid] = x;
    }
    __syncthreads();
    if (q + 1 < nblk) {
      fetch(BACK ? b - 1 : b + 1);  // in flight during the update
      if (BACK) {
        // entries before the block, a thread each
        if (tid < kTB * b) {
          const double* p = A + (size_t)kb * N + s0 + tid;
          double acc = 0.0;
#pragma unroll 1
          for (int c = 0; c < nb; c += 8) {  // (s_x is zero past the last atom)
            double l[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) l[u] = p[min(c + u, nb - 1) * (int)N];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc = fma(l[u], s_x[c + u], acc);
          }
          s_v[tid] -= acc;
        }
      } else {
        // entries behind the block, a thread each
        if (tid >= kTB * (b + 1) && s0 + tid < s1) {
          const double* p = A + (size_t)(s0 + tid) * N + kb;
          double acc = 0.0;
#pragma unroll 1
          for (int c = 0; c < kTB; c += 8) {
            double l[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) l[u] = p[c + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc = fma(l[u], s_x[c + u], acc);
          }
          s_v[tid] -= acc;
        }
      }
    }
    __syncthreads();
  }
  const int64_t* Z = in.numbers + m * N;
  if (s0 + tid < s1) {
    const double x = s_v[tid];
    v[s0 + tid] = x;
    dst[m * N + s0 + tid] = BACK && Z[s0 + tid] == 0 ? 0.0 : x;
  }
}

// The share of the solved entries s0 .. s0 + kTV - 1 in the entries before them
// (BACK: 64 per work-group) or behind them (16 per work-group).
template <bool BACK>
__global__ __launch_bounds__(kTV) void k_tl_gemv(Inputs in, Work w, int s0) {
  tf_priority();
  __shared__ double s_x[kTV];
  __shared__ double s_p[4][kTB];
  const int64_t m = blockIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  if (s0 >= n || !tl_solving(in, w, m)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int s1 = min(s0 + kTV, n), len = s1 - s0;
  const double* A = tf_matrix(w, m);
  double* v = w.vec + m * (N + 1);
  if (!BACK && s1 + 16 * (int)blockIdx.y >= n) return;
  s_x[tid] = tid < len ? v[s0 + tid] : 0.0;
  __syncthreads();
  if (BACK) {
    const int j = kTB * (int)blockIdx.y + lane;  // < s0
    const double* p = A + (size_t)s0 * N + j;
    double acc = 0.0;
    for (int c = wave; c < len; c += 32) {  // every fourth row, eight in flight
      double l[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) l[u] = p[(size_t)min(c + 4 * u, len - 1) * N];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc = fma(l[u], c + 4 * u < len ? s_x[c + 4 * u] : 0.0, acc);
    }
    s_p[wave][lane] = acc;
    __syncthreads();
    if (wave == 0) v[j] -= (s_p[0][lane] + s_p[1][lane]) + (s_p[2][lane] + s_p[3][lane]);
  } else {
    // (len = kTV: there are entries behind)
    for (int k = 0; k < 4; ++k) {
      const int i = s1 + 16 * (int)blockIdx.y + 4 * k + wave;
      if (i >= n) break;  // uniform over the wave
      const double* p = A + (size_t)i * N + s0 + lane;
      double l[kTV / 64], acc = 0.0;
#pragma unroll
      for (int u = 0; u < kTV / 64; ++u) l[u] = p[64 * u];
#pragma unroll
      for (int u = 0; u < kTV / 64; ++u) acc = fma(l[u], s_x[64 * u + lane], acc);
      acc = wave_sum(acc);
      if (lane == 0) v[i] -= acc;
    }
  }
}

// Adjoint set-up for the tiled solve: v = dL/dq on real atoms.
__global__ __launch_bounds__(256) void k_tf_adj_init(Inputs in, Work w) {
  tf_priority();
  const int64_t m = blockIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  if (!tl_solving(in, w, m)) return;
  const int64_t* Z = in.numbers + m * N;
  double* v = w.vec + m * (N + 1);
  for (int i = threadIdx.x; i < n; i += 256) v[i] = Z[i] != 0 ? w.dldq[m * N + i] : 0.0;
}

// Between the two adjoint substitutions: w' = L^-1 g is in lam; v = D^-1 w' -
// nu z_e with z_e = D^-1 L^-1 e and nu = z_e . w' / z_e . D z_e.
__global__ __launch_bounds__(256) void k_tf_adj_mid(Inputs in, Work w) {
  tf_priority();
  __shared__ double red[2 * kWaves];
  const int64_t m = blockIdx.x;
  const int64_t N = w.N;
  const int n = w.natom[m];
  if (n == 0 || !tl_solving(in, w, m)) return;
  const int tid = threadIdx.x;
  const double* wl = w.lam + m * N;
  const double* ze = w.ez + m * N;
  const double* dpiv = w.dpiv + m * N;
  double sw = 0.0, sz = 0.0;
  for (int i = tid; i < n; i += 256) {
    sw = fma(ze[i], wl[i], sw);
    sz = fma(ze[i] * dpiv[i], ze[i], sz);
  }
  sw = block_sum(sw, red);
  sz = block_sum(sz, red + kWaves);
  const double nu = sw / sz;
  double* v = w.vec + m * (N + 1);
  for (int i = tid; i < n; i += 256) v[i] = fma(-nu, ze[i], wl[i] * rcp_nt(dpiv[i]));
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
// the order within a bin is arbitrary. (The charge kernel reads the order from
// its end, smallest first: with the largest first it is faster alone, but the
// two-stream step slower, 0.892 -> 0.921 ms, as it then crowds the three-body
// pair pass beside it; smallest first 0.890 -> 0.884 ms.)
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

// Substitution over all entries of the tiled factor, kTV at a time.
template <bool BACK>
void launch_tl_substitution(hipStream_t s, const Inputs& in, const Work& w, double* dst) {
  const int N = (int)w.N, blocks = (N + kTV - 1) / kTV;
  const unsigned B = (unsigned)w.B;
  for (int k = 0; k < blocks; ++k) {
    const int s0 = kTV * (BACK ? blocks - 1 - k : k);
    hipLaunchKernelGGL(k_tl_solve<BACK>, dim3(B), dim3(kTV), kTlSolveLds, s, in, w, s0, dst);
    if (k + 1 == blocks) break;
    const unsigned tiles = (unsigned)(BACK ? s0 / kTB : (N - s0 - kTV + 15) / 16);
    hipLaunchKernelGGL(k_tl_gemv<BACK>, dim3(B, tiles), dim3(kTV), 0, s, in, w, s0);
  }
}

hipError_t launch_eeq_tiled(hipStream_t s, const DevTables& t, const Params& p,
                            const Inputs& in, const Work& w) {
  const int N = (int)w.N;
  const unsigned B = (unsigned)w.B;
  const unsigned rows = (unsigned)((w.B * (w.N + 2) + kWaves - 1) / kWaves);
  hipLaunchKernelGGL(k_tf_assemble, dim3(rows), dim3(256), 0, s, t, p, in, w);
  hipError_t e = ensure_lds((const void*)k_tl_step, kTlLds);
  if (e != hipSuccess) return e;
  for (int kb = 0; kb < N; kb += kTB) {
    const int npanel = (N + 2 - kb + kTB - 1) / kTB;
    const int nI = kb > 0 ? npanel - 1 : 0;  // row tiles behind the panel
    hipLaunchKernelGGL(k_tl_step, dim3(B, (unsigned)(npanel + nI * (nI + 1) / 2)), dim3(256),
                       kTlLds, s, in, w, kb, npanel);
  }
  hipLaunchKernelGGL(k_tf_reduce, dim3(B), dim3(256), 0, s, in, w);
  launch_tl_substitution<true>(s, in, w, w.q);
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
    hipLaunchKernelGGL(k_tf_adj_init, dim3(grid), dim3(256), 0, s, in, w);
    launch_tl_substitution<false>(s, in, w, w.lam);
    hipLaunchKernelGGL(k_tf_adj_mid, dim3(grid), dim3(256), 0, s, in, w);
    launch_tl_substitution<true>(s, in, w, w.lam);
    hipLaunchKernelGGL((k_adjoint<true, 2>), dim3(grid), dim3(256), 0, s, t, p, in, w, ordered);
    return hipGetLastError();
  }
  const size_t shmem = sizeof(double) * ((size_t)tri((int)w.N) + kSolvePad);
  if (solve_regs(w.N) > 2)
    return launch_lds(k_adjoint<false, 4>, grid, 256, shmem, s, t, p, in, w, ordered);
  return launch_lds(k_adjoint<false, 2>, grid, 256, shmem, s, t, p, in, w, ordered);
}

}  // namespace d4
