// 64 x 64 FP64 tiles of the dense factorisation: the factor of a diagonal tile
// with its inverse, and the fragment layouts in which tiles meet the matrix
// instructions.  Used by k_chol.hip.
//
// Fragments.  v_mfma_f64_16x16x4 takes A[row = l % 16][k = l / 16] and
// B[k = l / 16][col = l % 16] from lane l and leaves C[4 r + l / 16][l % 16] in
// register r.  A product over 16 columns is four such steps; which of the 16
// columns a step takes is free as long as both operands agree:
//   operand fragments (tiles read as they lie): step s has column 4 (l / 16) + s,
//     so a lane's four values are neighbours in a row;
//   result fragments (a product used as the next one's operand): step r has
//     column 4 r + l / 16, because the transposed product X^T = M A^T leaves
//     X[l % 16][4 r + l / 16] in register r, which is that operand already.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "context.hpp"

namespace psba {

constexpr int NB = kNB;     // 64
constexpr int TS = NB + 2;  // LDS row length of a tile: rows 16-byte aligned, and sixteen lanes'
                            // 16-byte accesses to sixteen rows cover all banks
constexpr int kInvFrag = 10 * 256;  // values of a lower triangular tile's fragments (10 blocks of 16 x 16)

typedef double dvec4 __attribute__((ext_vector_type(4)));
typedef double dvec2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) double lds_dbl;
typedef __attribute__((address_space(3))) dvec2 lds_dvec2;

// this thread's wave, as the uniform value that it is
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

__device__ __forceinline__ dvec4 mfma(double a, double b, dvec4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// workgroup barrier for data handed over through LDS only (global accesses stay in flight)
__device__ __forceinline__ void lds_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// value of v on lane N of each 16-lane row (DPP row_newbcast)
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
  return __builtin_amdgcn_mov_dpp(v, 0x150 + N, 0xF, 0xF, true);
}

// 1/x: the hardware estimate and one cubic step (the estimate's error e becomes e^3)
__device__ __forceinline__ double fast_rcp(double x) {
  const double r = __builtin_amdgcn_rcp(x), e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// 1/sqrt(x), likewise
__device__ __forceinline__ double fast_rsq(double x) {
  const double y = __builtin_amdgcn_rsq(x), e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// Elimination step C of a 16-column block: a is row l % 16 of the diagonal
// block (the same in each 16-lane row of the wave), x this lane's row below it;
// r = 1 / pivot.  Both lose column C times their multiplier (x[q] -= x[C] a_q[C] / pivot,
// with a_q[C] / pivot from the lane of row q); the next pivot's reciprocal is
// taken between the updates, so that its chain (broadcast, estimate, cubic
// step) runs in their shadow.
template <int C, bool X = true>
struct ElimStep {
  // updates that are not on the chain: x[C + 2], a[C + 3], x[C + 3], a[C + 4], ..
  template <int I, int END>
  static __device__ __forceinline__ void bulk(double (&a)[16], double (&x)[16], double u) {
    constexpr int N = 27 - 2 * C;
    if constexpr (I < END && I < N) {
      if constexpr (I % 2 == 1) fmac_bcast<C + 3 + I / 2>(a[C + 3 + I / 2], a[C], u);
      else if constexpr (X) fmac_bcast<C + 2 + I / 2>(x[C + 2 + I / 2], u, x[C]);
      bulk<I + 1, END>(a, x, u);
    }
  }
  // returns 1 / (pivot C + 1)
  static __device__ __forceinline__ double run(double (&a)[16], double (&x)[16], double r, bool& ok) {
    if constexpr (C < 15) {
      double u, p, r0, e, t;
      __asm__ volatile("v_mul_f64 %0, -%1, %2" : "=v"(u) : "v"(a[C]), "v"(r));
      fmac_bcast<C + 1>(a[C + 1], a[C], u);
      if constexpr (C < 14) fmac_bcast<C + 2>(a[C + 2], a[C], u);
      else __asm__ volatile("s_nop 0");
      if constexpr (X) fmac_bcast<C + 1>(x[C + 1], u, x[C]);  // (u written three instructions ago)
      bulk<0, 2>(a, x, u);
      __asm__ volatile("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
                       : "=v"(p)
                       : "v"(a[C + 1]), "n"(C + 1));
      bulk<2, 4>(a, x, u);
      __asm__ volatile("v_rcp_f64 %0, %1" : "=v"(r0) : "v"(p));
      bulk<4, 8>(a, x, u);
      __asm__ volatile("s_nop 0\n\tv_fma_f64 %0, -%1, %2, 1.0" : "=v"(e) : "v"(p), "v"(r0));
      bulk<8, 10>(a, x, u);
      __asm__ volatile("v_fma_f64 %0, %1, %1, %1" : "=v"(t) : "v"(e));
      bulk<10, 12>(a, x, u);
      __asm__ volatile("v_fma_f64 %0, %1, %2, %1" : "=v"(r) : "v"(r0), "v"(t));
      bulk<12, 99>(a, x, u);
      ok = ok && p > 0.0;
    }
    return r;
  }
};

// What the factor of a tile (factor_pivots, factor_blocks, factor_last) works on (LDS).  Y: in, the tile (lower part); out, the
// factor L~ with its columns not yet scaled (L = L~ / sqrt(d)) below the 16 x 16
// diagonal blocks, which keep what they held before their own elimination
// (L's own diagonal blocks: factor_block).  W: out, the rows of L~^-T (row i
// from column i on); in, the identity in its four diagonal blocks.  r: 1 / d.
// prog: progress words, which only grow from one tile's `base` to the next
// (base + 16 at most is written).
typedef __attribute__((address_space(3))) volatile int lds_flag;
struct FactorLds {
  lds_dbl *Y, *W;  // NB x TS each
  lds_dbl* r;      // NB
  lds_flag* prog;
};

// prog's words: wave 0's pivots (base + 4 b + g + 1 after four columns g of block
// b), waves 1, 2, 3 and 7's blocks (base + b + 1), waves 5 and 6's last block
// column (base + 1), and word 8: base + 1 if a pivot of this tile was not positive.
enum { kProgPivot = 0, kProgBad = 8 };

// Progress within the workgroup goes through LDS words rather than barriers, so
// that no wave waits for one that does not feed it.  A wave's LDS accesses are
// carried out in order, so data written before the word are there when the word is.
__device__ __forceinline__ void progress(lds_flag* f, int v) {
  __asm__ volatile("" ::: "memory");
  *f = v;
}
__device__ __forceinline__ void await(lds_flag* f, int v) {
  while (*f < v) {
  }
  __asm__ volatile("" ::: "memory");
}
// words i of f[0..7] in `mask`
__device__ __forceinline__ void await_all(lds_flag* f, unsigned mask, int v) {
  const int i = threadIdx.x & 7;
  while (!__all(!(mask >> i & 1) || f[i] >= v)) {
  }
  __asm__ volatile("" ::: "memory");
}

// Cholesky factor of a 64 x 64 tile and the inverse of the factor, by waves 0-3
// and 5-7 (factor_pivots, factor_blocks, factor_last).  Bound by the chain of
// 64 pivots and by the issue of the updates around it (2 (15 - c) FMAs at pivot
// c of a block, 130 cycles a pivot on average): everything else is kept off
// wave 0.  Per 16-column block, wave 0 eliminates with lane = row: the lanes
// take the rows below the block and, since there are always 64 rows in all, the
// rows of the identity that has been eliminated along (L^-T appears in its
// place, at no extra step).  Every four columns go to LDS, and waves 1, 2, 3
// and 7 (a 16 x 16 block each) take them into the next block column at once
// (MFMA, one step of four columns), so that only the last four columns' product
// lies between two blocks; block columns further right take a panel one block
// later (the last one the first panel: waves 5 and 6).
// Only the first nkb 16-column blocks are eliminated; the rows from 16 nkb on
// must be padding (identity), and their part of Y and W is not touched.

// wave 0; block column b of Y, W and r is complete at base + 4 b + 4
__device__ __forceinline__ void factor_pivots(const FactorLds& m, int nkb, int base) {
  const int lane = threadIdx.x & 63, li = lane & 15;
#pragma unroll 1
  for (int b = 0; b < nkb; ++b) {
    const int b0 = 16 * b, np = 48 - b0;  // rows below the block
    if (b > 0) await_all(m.prog, 0x8e, base + b);  // this block column's blocks
    double a[16], x[16], r[17];
    const lds_dvec2* const ar = (const lds_dvec2*)(m.Y + (b0 + li) * TS + b0);
    // rows of L~^-T: lane np + i holds row i, the last sixteen the identity's
    lds_dvec2* const xr = (lds_dvec2*)(lane < np ? m.Y + (b0 + 16 + lane) * TS + b0 : m.W + (lane - np) * TS + b0);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const dvec2 t = ar[q];
      a[2 * q] = t[0];
      a[2 * q + 1] = t[1];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const dvec2 t = xr[q];
      x[2 * q] = t[0];
      x[2 * q + 1] = t[1];
    }
    const double p0 = row_bcast<0>(a[0]);
    bool ok = p0 > 0.0;
    r[0] = fast_rcp(p0);
    auto put = [&](auto g) {
      constexpr int G = decltype(g)::value;
      xr[2 * G] = dvec2{x[4 * G], x[4 * G + 1]};
      xr[2 * G + 1] = dvec2{x[4 * G + 2], x[4 * G + 3]};
      const double r01 = lane & 1 ? r[4 * G + 1] : r[4 * G], r23 = lane & 1 ? r[4 * G + 3] : r[4 * G + 2];
      if (lane < 4) m.r[b0 + 4 * G + lane] = lane & 2 ? r23 : r01;
      progress(m.prog + kProgPivot, base + 4 * b + G + 1);
    };
#define PSBA_ELIM(C) r[C + 1] = ElimStep<C>::run(a, x, r[C], ok)
    PSBA_ELIM(0); PSBA_ELIM(1); PSBA_ELIM(2); PSBA_ELIM(3);
    put(std::integral_constant<int, 0>());
    PSBA_ELIM(4); PSBA_ELIM(5); PSBA_ELIM(6); PSBA_ELIM(7);
    put(std::integral_constant<int, 1>());
    PSBA_ELIM(8); PSBA_ELIM(9); PSBA_ELIM(10); PSBA_ELIM(11);
    put(std::integral_constant<int, 2>());
    PSBA_ELIM(12); PSBA_ELIM(13); PSBA_ELIM(14); PSBA_ELIM(15);
    if (!ok) progress(m.prog + kProgBad, base + 1);
    put(std::integral_constant<int, 3>());
#undef PSBA_ELIM
  }
}

// one step of a block's update: columns k0 + 4 g .. + 3 of its rows and, over -d,
// of Y's rows of block column jb
__device__ __forceinline__ void factor_step(const FactorLds& m, dvec4& c, const lds_dbl* row, int jb, int k0, int g) {
  const int lane = threadIdx.x & 63, li = lane & 15, k = k0 + 4 * g + (lane >> 4);
  const double av = row[li * TS + k];
  const double bv = m.Y[(16 * jb + li) * TS + k] * -m.r[k];
  c = mfma(av, bv, c);
}

__device__ __forceinline__ void block_load(dvec4& c, const lds_dbl* M, int jb) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int q = 0; q < 4; ++q) c[q] = M[(4 * q + lk) * TS + 16 * jb + li];
}
__device__ __forceinline__ void block_store(lds_dbl* M, int jb, const dvec4& c) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int q = 0; q < 4; ++q) M[(4 * q + lk) * TS + 16 * jb + li] = c[q];
}

// waves 1, 2, 3 and 7: block t of block column b + 1, Y's from the diagonal down,
// then W's rows 0 .. b
__device__ __forceinline__ void factor_blocks(const FactorLds& m, int nkb, int base) {
  const int w = wave_id(), t = w == 7 ? 3 : w - 1;
#pragma unroll 1
  for (int b = 0; b + 1 < nkb; ++b) {
    const int ny = 3 - b, i = t - ny;
    lds_dbl* const M = i < 0 ? m.Y + 16 * (b + 1 + t) * TS : m.W + 16 * i * TS;
    dvec4 c = {0.0, 0.0, 0.0, 0.0};  // W's rows have no entry here before block row i's panel
    if (b == 2) await_all(m.prog, 0x60, base + 1);
    if (i < 0 || i < b - 1) block_load(c, M, b + 1);
    if (b >= 1 && i != b) {
#pragma unroll
      for (int g = 0; g < 4; ++g) factor_step(m, c, M, b + 1, 16 * (b - 1), g);
    }
#pragma unroll 1
    for (int g = 0; g < 4; ++g) {
      await(m.prog + kProgPivot, base + 4 * b + g + 1);
      factor_step(m, c, M, b + 1, 16 * b, g);
    }
    block_store(M, b + 1, c);
    progress(m.prog + w, base + b + 1);
  }
}

// waves 5 and 6: block column 3 takes block column 0 (Y's last block, W's first)
__device__ __forceinline__ void factor_last(const FactorLds& m, int nkb, int base) {
  const int w = wave_id();
  if (nkb < 4) return;
  lds_dbl* const M = w == 5 ? m.Y + 48 * TS : m.W;
  dvec4 c = {0.0, 0.0, 0.0, 0.0};
  await(m.prog + kProgPivot, base + 4);
  if (w == 5) block_load(c, M, 3);
#pragma unroll
  for (int g = 0; g < 4; ++g) factor_step(m, c, M, 3, 0, g);
  block_store(M, 3, c);
  progress(m.prog + w, base + 1);
}

// block (mb, kb <= mb) of a lower triangular tile's fragments
__device__ __forceinline__ int inv_block(int mb, int kb) { return mb * (mb + 1) / 2 + kb; }

// Block (mb, kb) of M = L^-1 from the factor's W and r, by one wave: as operand
// fragments (M[16 mb + l % 16][16 kb + 4 (l / 16) + s], values s, s + 1 of lane l as a pair
// at block * 128 + (s / 2) * 64 + l) in LDS and in global memory, and row-major
// (64 x 64, nothing above the diagonal blocks) in global memory.
__device__ __forceinline__ void inv_fragments(lds_dbl* frag, double* Mg, double* Mr, const lds_dbl* r,
                                              const lds_dbl* W, int mb, int kb, int nkb) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const double rd = r[16 * mb + li], rs = mb < nkb ? rd * fast_rsq(rd) : 1.0;
  const int at = inv_block(mb, kb) * 128 + lane;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    dvec2 v;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int row = 4 * lk + 2 * h + q;
      v[q] = W[(16 * kb + row) * TS + 16 * mb + li] * rs;
      if (mb >= nkb) v[q] = (kb == mb && row == li) ? 1.0 : 0.0;
      if (kb == mb && row > li) v[q] = 0.0;
    }
    if (frag) ((lds_dvec2*)frag)[at + 64 * h] = v;
    if (Mg) ((dvec2*)Mg)[at + 64 * h] = v;
    if (Mr) *(dvec2*)(Mr + (16 * mb + li) * NB + 16 * kb + 4 * lk + 2 * h) = v;
  }
}

// L's rows below the diagonal block of block column cb, by one wave
__device__ __forceinline__ void store_panel(const lds_dbl* Y, const lds_dbl* r, int cb, double* L, int ld) {
  const int lane = threadIdx.x & 63, c = 16 * cb + (lane & 15);
  const double rd = r[c], rs = rd * fast_rsq(rd);
  for (int row = 16 * cb + 16 + (lane >> 4); row < NB; row += 4) L[(size_t)row * ld + c] = Y[row * TS + c] * rs;
}

template <int C>
__device__ __forceinline__ void factor_block_steps(double (&a)[16], double (&r)[16], bool& ok) {
  if constexpr (C < 15) {
    double none[16];
    r[C + 1] = ElimStep<C, false>::run(a, none, r[C], ok);
    factor_block_steps<C + 1>(a, r, ok);
  }
}

// L's diagonal block b, by one wave: the elimination again, from what Y still
// holds there (wave 0 has no time to write its rows during the factorisation)
__device__ __forceinline__ void factor_block(const lds_dbl* Y, int b, double* L, int ld) {
  const int lane = threadIdx.x & 63, li = lane & 15;
  const lds_dvec2* const ar = (const lds_dvec2*)(Y + (16 * b + li) * TS + 16 * b);
  double a[16], r[16];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const dvec2 t = ar[q];
    a[2 * q] = t[0];
    a[2 * q + 1] = t[1];
  }
  bool ok = true;
  r[0] = fast_rcp(row_bcast<0>(a[0]));
  factor_block_steps<0>(a, r, ok);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const double sd = fast_rsq(r[q]);  // sqrt(d_q)
    if (lane < 16 && q <= li) L[(size_t)(16 * b + li) * ld + 16 * b + q] = q == li ? sd : a[q] * (r[q] * sd);
  }
}

// X^T = M A^T for sixteen rows of A given as operand fragments av[4 kb + s];
// out: result fragments of X, xt[mb][r] = X[l % 16][16 mb + 4 r + l / 16]
__device__ __forceinline__ void solve_rows(dvec4 (&xt)[4], const double (&av)[16], const lds_dbl* frag) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) xt[mb] = dvec4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      dvec2 f[4];
#pragma unroll
      for (int mb = kb; mb < 4; ++mb) f[mb] = ((const lds_dvec2*)frag)[inv_block(mb, kb) * 128 + s2 * 64 + lane];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int mb = kb; mb < 4; ++mb) xt[mb] = mfma(f[mb][q], av[4 * kb + 2 * s2 + q], xt[mb]);
    }
  }
}

// its 16-column block MB alone
template <int MB>
__device__ __forceinline__ void solve_block(dvec4& xt, const double (&av)[16], const lds_dbl* frag) {
  const int lane = threadIdx.x & 63;
  xt = dvec4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kb = 0; kb <= MB; ++kb)
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const dvec2 f = ((const lds_dvec2*)frag)[inv_block(MB, kb) * 128 + s2 * 64 + lane];
      xt = mfma(f[0], av[4 * kb + 2 * s2], xt);
      xt = mfma(f[1], av[4 * kb + 2 * s2 + 1], xt);
    }
}

// A tile from global memory straight to LDS as operand fragments (no registers,
// in flight until vmcnt says otherwise): pairs at ((rb * 4 + kb) * 2 + s / 2) * 64 + l
// for rows 16 rb + l % 16.  Chunks c0, c0 + step, .. of the 32, one wave each.
__device__ __forceinline__ void rows_to_lds(lds_dbl* dst, const double* A, int ld, int c0, int step) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  for (int c = c0; c < 32; c += step) {
    const int rb = c >> 3, kb = (c >> 1) & 3, h = c & 1;
    const double* src = A + (size_t)(16 * rb + li) * ld + 16 * kb + 4 * lk + 2 * h;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)(dst + 128 * c), 16, 0, 0);
  }
}

// row block rb of those
__device__ __forceinline__ void rows_from_lds(double (&av)[16], const lds_dbl* src, int rb) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const dvec2 t = ((const lds_dvec2*)src)[(rb * 8 + c) * 64 + lane];
    av[2 * c] = t[0];
    av[2 * c + 1] = t[1];
  }
}

// sixteen rows of a tile in global memory as operand fragments (row: the first
// row of the sixteen)
__device__ __forceinline__ void load_rows(double (&av)[16], const double* row, int ld) {
  const int lane = threadIdx.x & 63;
  const dvec2* p = (const dvec2*)(row + (size_t)(lane & 15) * ld + 4 * (lane >> 4));
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const dvec2 t = p[8 * kb + s2];
      av[4 * kb + 2 * s2] = t[0];
      av[4 * kb + 2 * s2 + 1] = t[1];
    }
}

// result fragments of sixteen rows (row block rb of a tile) in LDS:
// xf[((rb * 8 + mb * 2 + r / 2) * 64 + l) * 2 + r % 2]
__device__ __forceinline__ void put_result(lds_dbl* xf, int rb, const dvec4 (&xt)[4]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      ((lds_dvec2*)xf)[(rb * 8 + mb * 2 + h) * 64 + lane] = dvec2{xt[mb][2 * h], xt[mb][2 * h + 1]};
}

}  // namespace psba
