// Cholesky factor of the reduced camera matrix and the solve S dpa = e_a in one
// launch (replaces the reference's explicit inverse, PSBA/CL_files/SPD_inv.cl:
// kern_cholesky/_s2 + kern_trigMat_inv/_mul + kern_fill_rest, and
// matVec_mul.cl).  S is n_pad x n_pad, row-major, lower triangle, its rows from
// n on the identity; T = n_pad / 64 tiles a side.
//
// Tiles flow between workgroups instead of the workgroups meeting at a barrier:
//   workgroup 0    the diagonal chain: factors tile (k, k) with its inverse M_k,
//                  publishes M_k, forms L_{k+1,k} = A_{k+1,k} M_k^T for itself and
//                  takes it into A_{k+1,k+1}, which it factors next;
//   workgroup 1    the triangular solves: y_k = M_k b_k and b_i -= L_ik y_k behind
//                  the factorisation, then x_k = M_k^T r_k;
//   the others     own the remaining tiles (i, j): for k < j they form
//                  L_ik = A_ik M_k^T and L_jk and take L_ik L_jk^T off A_ij as soon
//                  as M_k is there, publish A_ij when it is complete, and then
//                  store L_ij.  Afterwards they sum the terms of the back
//                  substitution that workgroup 1 does not take itself.
// A solve with M_k is a matrix product, so a tile's whole work is on the matrix
// units, and its latency (about 6 us from M_k to the next complete tile) is short
// enough that workgroup 0 rarely waits.
//
// Bound by workgroup 0's chain, not by arithmetic or memory: 11.6 us a tile
// (factor 7.0, the rest of M_k 0.8, L_{k+1,k} 1.5, its product 2.2), then 1.8 us
// a tile back.  Workgroups that met at a barrier after each phase, with solves
// by substitution, took 14.5 us a phase and more: 117 us at n = 300, 230 at 594,
// 323 at 828, 1916 at 2700; this kernel takes 69, 138, 183 and 700.
//
// With more tiles than workgroups (T > 22 on 256 compute units) an owner has
// several tiles: then the solves are not repeated per tile, but go through memory
// once, and kForward workgroups share the forward substitution.  With one tile
// each, repeating the solves saves a hop between workgroups: 14.1 us a tile at
// T = 22, 15.1 at T = 24.
//
// Every wait is for one flag (a word that only grows: done is the launch's epoch
// plus one, so nothing is reset between launches), set by its producer behind a
// release fence and read behind an acquire fence.  The grid is at most one
// workgroup per CU, so that on the context's in-order stream every workgroup is
// resident.  Beside another stream's launches they may not all be: up to T = 22 a
// tile waits only for lower-numbered workgroups, and all but the last T - 4 owners
// leave when their tile is done, so that the others find room (two contexts of 16
// tiles together have 272 workgroups); from T = 23 on a launch needs the
// whole device, and one that does not get it ends after the bounded waits (give_up).
// d_scal[SC_FACTOR_OK] becomes 1 on success, 0 when a pivot is not positive
// and -1 when a wait timed out.
#include <algorithm>

#include "context.hpp"
#include "dense_tile.hpp"

namespace psba {

namespace {

typedef unsigned long long ull;

// Words of the sync array: epoch, x and y flags, M flags (T), r and s flags (T each),
// then A and L flags of the lower tiles, row by row.
struct Sync {
  ull* w;
  int T;
  __device__ __forceinline__ ull* epoch() const { return w; }
  __device__ __forceinline__ ull* x() const { return w + 1; }
  __device__ __forceinline__ ull* y() const { return w + 2; }
  __device__ __forceinline__ ull* m(int k) const { return w + 3 + k; }
  __device__ __forceinline__ ull* r(int k) const { return w + 3 + T + k; }
  __device__ __forceinline__ ull* s(int k) const { return w + 3 + 2 * T + k; }
  __device__ __forceinline__ ull* a(int i, int j) const { return w + 3 + 3 * T + i * (i + 1) / 2 + j; }
  __device__ __forceinline__ ull* l(int i, int j) const { return a(i, j) + T * (T + 1) / 2; }
};

__device__ __forceinline__ ull peek(ull* f) { return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// one thread: wait until *f reaches v (bounded)
__device__ __forceinline__ void poll(ull* f, ull v, int* fail) {
  for (unsigned polls = 1; peek(f) < v; ++polls) {
    __builtin_amdgcn_s_sleep(1);
    if (give_up(polls, fail)) break;
  }
}

// The workgroup waits for one or two flags, a thread each, and may then read
// what was published before them.
__device__ __forceinline__ void wait_flags(ull v, int* fail, ull* f0, ull* f1 = nullptr) {
  const int t = threadIdx.x;
  if (t < 64) {
    ull* f = t == 0 ? f0 : t == 1 ? f1 : nullptr;
    if (f) poll(f, v, fail);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
}

// After the workgroup's stores: make them visible and set the flag.
__device__ __forceinline__ void publish(ull* f, ull v) {
  drain_stores();
  __syncthreads();  // every wave's stores are in L2
  if (threadIdx.x == 0) {
    release_stores();
    __hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Workgroup 0's progress words beyond the factorisation's, in groups of eight
// that one wait can cover: what L_{k+1,k} needs (k + 1 when there for tile k),
// what its product needs, what the next factorisation needs.
enum {
  kProgFrag = 16,   // 4 waves: M_k's last block row in F
  kProgRows = 20,   // A_{k+1,k} in AX
  kProgInv = 21,    // M_k's other block rows in F
  kProgX = 24,      // 4 waves: L_{k+1,k} in AX
  kProgOut = 28,    // k + 2: tile k is stored, its Y free
  kProgNext = 32,   // 4 waves: the next tile in Y
  kProgUnit = 36,   // the identity in W again
  kChainWords = 40
};

// workgroup 1's, in the back substitution (x_k is step T - k)
enum {
  kProgPx = 0,   // 4 waves: their part of x_k
  kProgXk = 4,   // x_k
  kProgPn = 8,   // 4 waves: their parts of the terms of x_k
  kProgHelp = 12,  // the helper's sum of row k - 1
  kSolveWords = 16
};

struct SolveLds {
  // workgroup 0: the tile being factored and the next one; 1: the right-hand
  // side; owners: a row-major copy of their tile
  double Y[2][NB * TS];
  double W[NB * TS];   // L~^-T while factoring; owners: result fragments of a tile
  double F[kInvFrag];  // fragments of M_k
  union {
    double AX[NB * NB];  // workgroup 0: A_{k+1,k}, then L_{k+1,k}, as fragments
    struct {
      double part[4][4][NB];
      double v[NB], h[4][NB];
    };
  };
  double r[2][NB];
  int prog[kChainWords];
};
static_assert(2 * NB * TS >= kMaxSolveN, "the right-hand side must fit");

constexpr int kInvLen = kInvFrag + NB * NB;  // what is stored of M_k: fragments, then row-major
constexpr int kNear = 3;  // the terms of row k's three neighbours are workgroup 1's
// With more tiles than workgroups, so many workgroups take the far terms of the
// forward substitution: one workgroup reads tiles at about 60 GB/s, which left it
// behind the factorisation by 100 of 965 us at T = 43
constexpr int kForward = 8;
constexpr int kHeld = 4;  // and so many tiles an owner keeps in registers

// the tile's accumulators: wave w has rows 16 w .. + 15, acc[c] columns 16 c .. + 15
__device__ __forceinline__ void acc_load(dvec4 (&acc)[4], const double* A, int ld, int w) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[c][r] = A[(size_t)(16 * w + 4 * r + lk) * ld + 16 * c + li];
}

__device__ __forceinline__ void acc_store(const dvec4 (&acc)[4], double* A, int ld, int w) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) A[(size_t)(16 * w + 4 * r + lk) * ld + 16 * c + li] = acc[c][r];
}

// acc -= X Y^T, X the wave's sixteen rows, Y's fragments of all four row blocks in
// LDS (both in the same fragment form)
__device__ __forceinline__ void acc_update(dvec4 (&acc)[4], const dvec4 (&x)[4], const lds_dbl* yf) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      dvec2 f[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) f[c] = ((const lds_dvec2*)yf)[(c * 8 + mb * 2 + h) * 64 + lane];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = mfma(-x[mb][2 * h + q], f[c][q], acc[c]);
    }
}

// fragments of M_k from global memory into LDS, by the workgroup's first 256 threads
__device__ __forceinline__ void load_inv(lds_dbl* F, const double* M) {
  dvec2 t[5];
  if (threadIdx.x >= 256) return;
#pragma unroll
  for (int q = 0; q < 5; ++q) t[q] = ((const dvec2*)M)[threadIdx.x + 256 * q];
#pragma unroll
  for (int q = 0; q < 5; ++q) ((lds_dvec2*)F)[threadIdx.x + 256 * q] = t[q];
}

// L_ij of the wave's sixteen rows, from its result fragments
__device__ __forceinline__ void store_rows(const dvec4 (&xt)[4], double* L, int ld, int w) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) L[(size_t)(16 * w + li) * ld + 16 * mb + 4 * r + lk] = xt[mb][r];
}

// the identity in W's diagonal blocks, by one wave
__device__ __forceinline__ void init_inverse(lds_dbl* W) {
  const int row = threadIdx.x & 63, b = row & 48;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int c = b + 2 * q;
    *(lds_dvec2*)(W + row * TS + c) = dvec2{row == c ? 1.0 : 0.0, row == c + 1 ? 1.0 : 0.0};
  }
}

// A 64 x 64 tile in the registers of NW waves, for products with a vector: the
// thread has columns 2 c, 2 c + 1 (c = lane % 32) of rows 2 w + lane / 32 + 2 NW q.
template <int NW>
struct TileRegs {
  dvec2 t[32 / NW];
  __device__ __forceinline__ static int row(int q) { return 2 * wave_id() + ((threadIdx.x >> 5) & 1) + 2 * NW * q; }
  __device__ __forceinline__ void load(const double* A, int ld) {
#pragma unroll
    for (int q = 0; q < 32 / NW; ++q) t[q] = *(const dvec2*)(A + (size_t)row(q) * ld + 2 * (threadIdx.x & 31));
  }
  // out[row] = sum over the columns, each row by one wave
  __device__ __forceinline__ void rows(const lds_dbl* x, lds_dbl* out) const {
    const dvec2 xv = ((const lds_dvec2*)x)[threadIdx.x & 31];
#pragma unroll
    for (int q = 0; q < 32 / NW; ++q) {
      double s = fma(t[q][1], xv[1], t[q][0] * xv[0]);
      s += dpp_perm<0xB1>(s);   // quad: lanes 1, 0, 3, 2
      s += dpp_perm<0x4E>(s);   // 2, 3, 0, 1
      s += dpp_perm<0x141>(s);  // half row mirrored
      s += dpp_perm<0x140>(s);  // row mirrored
      s += __shfl_xor(s, 16, 64);
      if ((threadIdx.x & 31) == 0) out[row(q)] = s;
    }
  }
  // this wave's part of the sums over the rows, into part[w][64]
  __device__ __forceinline__ void cols(const lds_dbl* x, lds_dbl* part) const {
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int q = 0; q < 32 / NW; ++q) {
      const double xr = x[row(q)];
      s0 = fma(t[q][0], xr, s0);
      s1 = fma(t[q][1], xr, s1);
    }
    s0 += __shfl_xor(s0, 32, 64);
    s1 += __shfl_xor(s1, 32, 64);
    if ((threadIdx.x & 63) < 32) ((lds_dvec2*)(part + wave_id() * NB))[threadIdx.x & 31] = dvec2{s0, s1};
  }
  template <int CTRL>
  __device__ __forceinline__ static double dpp_perm(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  }
};

// part[0..3][lane] summed, in the waves' order
__device__ __forceinline__ double part_sum(const lds_dbl* part) {
  const int l = threadIdx.x & 63;
  return ((part[l] + part[NB + l]) + part[2 * NB + l]) + part[3 * NB + l];
}

// owner number o -> tile: column by column, (j, j) for j >= 2 and (i, j), i > j
__device__ __forceinline__ void owner_tile(int o, int T, int* i, int* j) {
  int c = 0;
  for (;; ++c) {
    const int cnt = T - 1 - c + (c >= 2 ? 1 : 0);
    if (o < cnt) break;
    o -= cnt;
  }
  *j = c;
  *i = c >= 2 ? c + o : c + 1 + o;
}

}  // namespace

__global__ __launch_bounds__(512) void k_chol_solve(double* __restrict__ S, int ld, int T, double* __restrict__ Lf,
                                                    double* __restrict__ Mg, const double* __restrict__ ea,
                                                    double* __restrict__ yv, double* __restrict__ xs,
                                                    double* __restrict__ dp, int n, double* __restrict__ okp, ull* sync,
                                                    int* __restrict__ fail, const unsigned char* __restrict__ gate) {
  __shared__ __attribute__((aligned(16))) SolveLds sm;
  // with gate (device-side LM control): the trial queued behind the one that
  // stopped the solve ends before anything is written
  const bool run = !gate || *gate;
  const int G = gridDim.x, tid = threadIdx.x, lane = tid & 63, w = wave_id(), li = lane & 15, lk = lane >> 4;
  const Sync sy{sync, T};
  // (workgroup 1 advances it at its end, after every other workgroup's last wait)
  const ull epoch = peek(sy.epoch()), done = epoch + 1;
  if (!run) return;
  auto tile = [&](double* base, int i, int j) { return base + (size_t)i * NB * ld + (size_t)j * NB; };
  auto rows_of = [&](int i) { return min(NB, n - i * NB); };
  lds_dbl* const F = (lds_dbl*)sm.F;
  lds_dbl* const XF = (lds_dbl*)sm.W;

  if (blockIdx.x == 0) {
    // ---- the diagonal chain: every wave its part of every tile, in step by the
    // progress words
    lds_flag* const prog = (lds_flag*)sm.prog;
    lds_dbl* const W = (lds_dbl*)sm.W;
    lds_dbl* const AX = (lds_dbl*)sm.AX;
    {
      double v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = S[(size_t)(w + 8 * q) * ld + lane];
#pragma unroll
      for (int q = 0; q < 8; ++q) sm.Y[0][(w + 8 * q) * TS + lane] = v[q];
      if (tid < kChainWords) prog[tid] = tid == kProgOut ? 1 : 0;
      if (w == 7) init_inverse(W);
      __syncthreads();
    }
#pragma unroll 1
    for (int k = 0; k < T; ++k) {
      lds_dbl* const Y = (lds_dbl*)sm.Y[k & 1];
      lds_dbl* const rd = (lds_dbl*)sm.r[k & 1];
      const FactorLds m{Y, W, rd, prog};
      const int nkb = (rows_of(k) + 15) >> 4, base = 16 * k;
      const bool more = k + 1 < T;
      if (w < 4 || w == 7) {
        await_all(prog + kProgNext, 0x1f, k);
        if (w == 0) {
          factor_pivots(m, nkb, base);
        } else {
          factor_blocks(m, nkb, base);
        }
        if (!more) break;
        if (w == 7) {
          await_all(prog + kProgFrag, 0x2f, k + 1);  // W has been read
          init_inverse(W);
          progress(prog + kProgUnit, k + 1);
          continue;
        }
        await(prog + kProgPivot, base + 16);
        inv_fragments(F, nullptr, nullptr, rd, W, 3, w, 4);
        progress(prog + kProgFrag + w, k + 1);
        // the lower 16 x 16 blocks of A_{k+1,k+1}: wave 0 (3,0) (3,1) (3,2), wave 1
        // (2,0) (2,1) (2,2), wave 2 (1,0) (1,1), wave 3 (3,3) (0,0); the last two
        // form a third product that goes nowhere, so that all run one code
        // without branches (the time is that of three blocks)
        const int nb = w < 2 ? 3 : 2;
        auto row_of = [&](int u) { return w == 3 ? (u == 0 ? 3 : 0) : 3 - w; };
        auto col_of = [&](int u) { return w == 3 ? (u == 0 ? 3 : 0) : w == 2 && u == 2 ? 0 : u; };
        await_all(prog + kProgFrag, 0x3f, k + 1);
        const double* An = tile(S, k + 1, k + 1);
        dvec4 acc[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[u][r] = An[(size_t)(16 * row_of(u) + 4 * r + lk) * ld + 16 * col_of(u) + li];
          }
        {
          double av[16];
          rows_from_lds(av, AX, w);
          dvec4 xt[4];
          solve_rows(xt, av, F);
          put_result(AX, w, xt);  // over the wave's own rows of A
        }
        progress(prog + kProgX + w, k + 1);
        await_all(prog + kProgX, 0x1f, k + 1);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const lds_dvec2* const x = (const lds_dvec2*)AX + (mb * 2 + h) * 64 + lane;
#pragma unroll
            for (int u = 0; u < 3; ++u) {
              const dvec2 xa = x[row_of(u) * 512], xb = x[col_of(u) * 512];
              acc[u] = mfma(-xa[0], xb[0], acc[u]);
              acc[u] = mfma(-xa[1], xb[1], acc[u]);
            }
          }
        double* const Yn = sm.Y[(k + 1) & 1];
#pragma unroll
        for (int u = 0; u < 3; ++u)
          if (u < nb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) Yn[(16 * row_of(u) + 4 * r + lk) * TS + 16 * col_of(u) + li] = acc[u][r];
          }
        progress(prog + kProgNext + w, k + 1);
      } else if (w == 4) {
        // A_{k+1,k} into LDS once its owner has completed it
        if (!more) break;
        await_all(prog + kProgNext, 0x0f, k);
        if (k >= 1) {
          if (lane < 2) poll(lane == 0 ? sy.a(k + 1, k) : sy.a(k + 1, k + 1), done, fail);
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        rows_to_lds(AX, tile(S, k + 1, k), ld, 0, 1);
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        progress(prog + kProgRows, k + 1);
      } else if (w == 5) {
        // M_k out, and its first three block rows into F
        double* const Mk = Mg + (size_t)k * kInvLen;
        double* const Mr = Mk + kInvFrag;
        factor_last(m, nkb, base);
#pragma unroll 1
        for (int mb = 0; mb < (more ? 3 : 4); ++mb) {
          await(prog + kProgPivot, base + min(4 * mb + 4, 4 * nkb));
#pragma unroll 1
          for (int kb = 0; kb <= mb; ++kb) inv_fragments(F, Mk, Mr, rd, W, mb, kb, nkb);
        }
        if (more) {
          progress(prog + kProgInv, k + 1);
          await_all(prog + kProgFrag, 0x0f, k + 1);
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const dvec2 v = ((const lds_dvec2*)F)[6 * 128 + 64 * q + lane];
            ((dvec2*)Mk)[6 * 128 + 64 * q + lane] = v;
            *(dvec2*)(Mr + (48 + li) * NB + 16 * (q >> 1) + 4 * lk + 2 * (q & 1)) = v;
          }
        }
        if (lane == 0 && prog[kProgBad] == base + 1)
          __hip_atomic_fetch_or(fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        release_stores();
        if (lane == 0) __hip_atomic_store(sy.m(k), done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        // L_kk out
        double* const Lkk = tile(Lf, k, k);
        factor_last(m, nkb, base);
#pragma unroll 1
        for (int c = 0; c < nkb; ++c) {
          await(prog + kProgPivot, base + 4 * c + 4);
          factor_block(Y, c, Lkk, ld);
          store_panel(Y, rd, c, Lkk, ld);
        }
        if (nkb < 4) {
          // padding: the identity, and the zeros that its panels are
          for (int row = 16 * nkb; row < NB; ++row)
            if (lane <= row) Lkk[(size_t)row * ld + lane] = row == lane ? 1.0 : 0.0;
        }
        progress(prog + kProgOut, k + 2);
      }
    }
    if (G > 1) return;
    if (w == 5) progress(prog + kProgInv, 1);  // (M_0 is in memory: the fence above)
    if (w >= 4) return;
    // one tile: both solves here, as soon as M_0 is there (L_00 may still be on its
    // way out: n = 60 19.3 -> 17.8 us against waiting for every wave)
    lds_dbl* const v = (lds_dbl*)sm.part[0][0];
    lds_dbl* const y = (lds_dbl*)sm.part[1][0];
    lds_dbl* const part = (lds_dbl*)sm.part[2][0];
    v[lane] = ea[lane];  // (every wave the same values)
    await(prog + kProgInv, 1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    TileRegs<4> t;
    t.load(Mg + kInvFrag, NB);
    t.rows(v, y);
    progress(prog + kProgFrag + w, 1);
    await_all(prog + kProgFrag, 0x0f, 1);
    t.cols(y, part);
    progress(prog + kProgFrag + w, 2);
    if (w > 0) return;
    await_all(prog + kProgFrag, 0x0f, 2);
    const double x = part_sum(part);
    xs[lane] = x;
    if (lane < n) dp[lane] = x;
    if (tid == 0) {
      const int f = __hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *okp = f ? 0.0 : 1.0;  // (there is nothing to wait for)
      __hip_atomic_store(fail, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return;
  }

  const int ntiles = T * (T - 1) / 2 + max(0, T - 2);
  const bool many = ntiles > G - 2;  // more tiles than workgroups
  // eight waves: row i's share of b (rows i0, i0 + step, .. below i1; row i
  // lies at place i / step) -= L_ik y, with the next two tiles'
  // loads in flight.  At most 64 rows, a lane each for their flags: all 21 with a
  // workgroup per tile (T <= 22), kNear or an eighth of 128 with several tiles each.
  auto forward = [&](lds_dbl* b, lds_dbl* y, int k, int i0, int step, int i1) {
    if (i0 >= i1) return;
    if (w == 0) {
      if (i0 + lane * step < i1) poll(sy.l(i0 + lane * step, k), done, fail);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    TileRegs<8> t[2][2];
    auto load = [&](int s, int i) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (i + u * step < i1) t[s][u].load(tile(Lf, i + u * step, k), ld);
    };
    auto take = [&](int s, int i) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (i + u * step < i1) t[s][u].rows(y, (lds_dbl*)sm.part[s][u]);
      __syncthreads();
      if (w < 2 && i + w * step < i1) b[(i + w * step) / step * NB + lane] -= sm.part[s][w][lane];
    };
    load(0, i0);
    for (int i = i0; i < i1; i += 4 * step) {
      load(1, i + 2 * step);
      take(0, i);
      load(0, i + 4 * step);
      take(1, i + 2 * step);
    }
  };

  if (blockIdx.x == 1) {
    // ---- the triangular solves.  b holds b_i, then y_i, then x_i.
    lds_dbl* const b = (lds_dbl*)&sm.Y[0][0];
    lds_dbl* const y = (lds_dbl*)sm.W;
    lds_flag* const prog = (lds_flag*)sm.prog;
    for (int q = tid; q < T * NB; q += 512) b[q] = ea[q];
    if (tid < kSolveWords) prog[tid] = 0;
    __syncthreads();
    // forward, eight waves
    for (int k = 0; k < T; ++k) {
      wait_flags(done, fail, sy.m(k));
      {
        TileRegs<8> t;
        t.load(Mg + (size_t)k * kInvLen + kInvFrag, NB);
        t.rows(b + k * NB, y);
      }
      __syncthreads();
      if (w == 0) b[k * NB + lane] = y[lane];
      if (many) {
        if (w == 0) {
          xs[(size_t)k * NB + lane] = y[lane];
          release_stores();
          if (lane == 0) __hip_atomic_store(sy.y(), epoch + (ull)(k + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        forward(b, y, k, k + 1, 1, min(T, k + 1 + kNear));
        const int i = k + 1;  // the helper's sum of row k + 1
        if (i < T && i > kNear) {
          wait_flags(done, fail, sy.s(i));
          if (w == 0) b[i * NB + lane] += yv[(size_t)i * NB + lane];
        }
      } else {
        forward(b, y, k, k + 1, 1, T);
      }
      __syncthreads();
    }
    // back substitution: r_k = y_k - sum_{j > k} L_jk^T x_j, x_k = M_k^T r_k.  Waves 0-3
    // take x_j into rows j - 1 .. j - kNear, with a step's tiles loaded one step
    // ahead; wave 4 publishes x_j to the rows' helpers, which sum the other
    // terms; wave 5 fetches those sums.
    if (w < 4) {
      lds_dbl* const v = (lds_dbl*)sm.v;
      lds_dbl* const px = (lds_dbl*)sm.part[3][0];
      TileRegs<4> m, l[kNear];
      m.load(Mg + (size_t)(T - 1) * kInvLen + kInvFrag, NB);
#pragma unroll
      for (int u = 0; u < kNear; ++u)
        if (T - 2 - u >= 0) l[u].load(tile(Lf, T - 1, T - 2 - u), ld);
      v[lane] = b[(T - 1) * NB + lane];  // (every wave the same values, here and below)
      for (int k = T - 1; k >= 0; --k) {
        const int s = T - k;
        m.cols(v, px);
        progress(prog + kProgPx + w, s);
        if (k >= 1) m.load(Mg + (size_t)(k - 1) * kInvLen + kInvFrag, NB);
        await_all(prog + kProgPx, 0x0f, s);
        lds_dbl* const x = b + k * NB;
        x[lane] = part_sum(px);
        if (w == 0) progress(prog + kProgXk, s);
        if (k == 0) break;
#pragma unroll
        for (int u = 0; u < kNear; ++u)
          if (k - 1 - u >= 0) {
            l[u].cols(x, (lds_dbl*)sm.part[u][0]);
            if (k - 2 - u >= 0) l[u].load(tile(Lf, k - 1, k - 2 - u), ld);
          }
        progress(prog + kProgPn + w, s);
        const bool helped = k - 1 + kNear + 1 < T;
        await_all(prog + kProgPn, helped ? 0x1f : 0x0f, s);
        double r = b[(k - 1) * NB + lane] - part_sum((lds_dbl*)sm.part[0][0]);
        if (helped) r += sm.h[(k - 1) & 3][lane];
        v[lane] = r;
        if (w >= 1 && w < kNear && k - 1 - w >= 0) b[(k - 1 - w) * NB + lane] -= part_sum((lds_dbl*)sm.part[w][0]);
      }
    } else if (w == 4) {
      for (int k = T - 1; k >= 0; --k) {
        await(prog + kProgXk, T - k);
        const double x = b[k * NB + lane];
        if (k * NB + lane < n) dp[k * NB + lane] = x;
        xs[(size_t)k * NB + lane] = x;
        release_stores();
        if (lane == 0) __hip_atomic_store(sy.x(), epoch + (ull)(T - k), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    } else if (w == 5) {
      // the helpers' sums, row i needed in step k = i + 1 (the ring's slot of row i + 4
      // has been read by then: row i is complete only after x_{i+4})
      for (int i = T - 2 - kNear; i >= 0; --i) {
        if (lane == 0) poll(sy.r(i), done, fail);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        sm.h[i & 3][lane] = yv[(size_t)i * NB + lane];
        progress(prog + kProgHelp, T - 1 - i);
      }
    }
    __syncthreads();
    if (tid == 0) {
      const int f = __hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *okp = (f & 2) ? -1.0 : (f ? 0.0 : 1.0);
      if (!(f & 2)) {
        __hip_atomic_store(fail, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(sy.epoch(), epoch + (ull)(T + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    return;
  }

  // ---- owners of tiles
  const int o = (int)blockIdx.x - 2;
  if (many && o >= G - 2 - kForward) {
    // the far terms of rows i = h, h + kForward, .. : L_ik y_k for k < i - kNear
    const int h = o - (G - 2 - kForward);
    lds_dbl* const b = (lds_dbl*)&sm.Y[0][0];
    lds_dbl* const y = (lds_dbl*)sm.W;
    for (int q = tid; q < (T + kForward - 1) / kForward * NB; q += 512) b[q] = 0.0;
    for (int k = 0; k + kNear + 1 < T; ++k) {
      const int lo = k + kNear + 1, i0 = lo + (h - lo % kForward + kForward) % kForward;
      if (i0 >= T) break;
      wait_flags(epoch + (ull)(k + 1), fail, sy.y());
      if (tid < NB) y[tid] = xs[(size_t)k * NB + tid];
      __syncthreads();
      forward(b, y, k, i0, kForward, T);
      __syncthreads();
      if (i0 == lo) {  // its last
        if (tid < NB) yv[(size_t)lo * NB + tid] = b[lo / kForward * NB + tid];
        publish(sy.s(lo), done);
      }
    }
    if (w >= 4) return;
  } else if (many) {
    // more tiles than workgroups: tiles o, o + H, .. each, column by column, all eight
    // waves on one tile at a time (wave w: rows 16 (w % 4) .., columns 32 (w / 4) ..).
    // L_ik is formed once, by its owner, and the products read it from memory.  The
    // tiles' chain from column to column (complete -> L -> flag -> product ->
    // complete) has to keep up with workgroup 0's, so the next column's tile goes
    // first, from the accumulators straight into its solve, with M_{k+1} fetched
    // ahead of the product if it is there; the other products run while L is on
    // its way.  The last kHeld tiles, which live longest, stay in registers: behind
    // the acquire fences nothing stays in an L2, and reading and writing every
    // tile in every phase (128 KB a product, 5.5 TB/s over the device) was what
    // bound the first phases.  T = 43: 868 us without either and with four waves a
    // tile, 834 with pairs of tiles a workgroup, 700 so.
    const int H = G - 2 - kForward, half = w >> 2, wt = w & 3;
    const int nown = o < ntiles ? (ntiles - o + H - 1) / H : 0, nmem = max(0, nown - kHeld);
    auto own = [&](int q) {
      int2 t;
      owner_tile(o + q * H, T, &t.x, &t.y);
      return t;
    };
    // 0: no product in phase k (the diagonal's last is workgroup 0's), 2: the last
    auto product = [&](const int2& t, int k) {
      const int last = t.x == t.y ? t.y - 2 : t.y - 1;
      return k > last ? 0 : k == last ? 2 : 1;
    };
    int turn = 0;
    auto buffer = [&](int n) { return n & 1 ? (lds_dbl*)sm.Y[0] : XF; };
    auto multiply = [&](const int2& t, int k, dvec4 (&acc)[2], bool from_memory) {
      double* const A = tile(S, t.x, t.y) + (size_t)16 * wt * ld + 32 * half;
      double av[16];
      dvec2 y[4];
      const dvec2* const yp = (const dvec2*)(tile(Lf, t.y, k) + (size_t)(16 * wt + li) * ld + 32 * half + 4 * lk);
#pragma unroll
      for (int q = 0; q < 4; ++q) y[q] = yp[8 * (q >> 1) + (q & 1)];
      load_rows(av, tile(Lf, t.x, k) + (size_t)16 * wt * ld, ld);
      if (from_memory) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[c][r] = A[(size_t)(4 * r + lk) * ld + 16 * c + li];
      }
      lds_dbl* const xt = buffer(turn++);
#pragma unroll
      for (int q = 0; q < 4; ++q) ((lds_dvec2*)xt)[(8 * wt + 4 * half + q) * 64 + lane] = y[q];
      lds_barrier();
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        dvec2 f[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) f[c] = ((const lds_dvec2*)xt)[((2 * half + c) * 8 + m) * 64 + lane];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[c] = mfma(-av[2 * m + q], f[c][q], acc[c]);
      }
      const bool last = product(t, k) == 2;
      if (from_memory || last) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) A[(size_t)(4 * r + lk) * ld + 16 * c + li] = acc[c][r];
      }
      if (last) publish(sy.a(t.x, t.y), done);
    };
    auto load_m = [&](dvec2 (&mf)[3], int j) {
      const dvec2* const M = (const dvec2*)(Mg + (size_t)j * kInvLen);
#pragma unroll
      for (int q = 0; q < 3; ++q) mf[q] = M[min(tid + 512 * q, kInvFrag / 2 - 1)];
    };
    // L_ij of the complete tile in acc; mf: M_j's fragments if they are here already
    auto solve = [&](const int2& t, dvec4 (&acc)[2], dvec2 (&mf)[3], bool have) {
      lds_dbl* const rows = (lds_dbl*)sm.Y[1];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) rows[(16 * wt + 4 * r + lk) * TS + 32 * half + 16 * c + li] = acc[c][r];
      if (!have) {
        wait_flags(done, fail, sy.m(t.y));
        load_m(mf, t.y);
      }
#pragma unroll
      for (int q = 0; q < 3; ++q)
        if (tid + 512 * q < kInvFrag / 2) ((lds_dvec2*)F)[tid + 512 * q] = mf[q];
      lds_barrier();
      // (the halves take column blocks 0, 3 and 1, 2: the same work)
      double av[16];
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const dvec2 v = *(const lds_dvec2*)(rows + (16 * wt + li) * TS + 16 * (m >> 1) + 4 * lk + 2 * (m & 1));
        av[2 * m] = v[0];
        av[2 * m + 1] = v[1];
      }
      double* const L = tile(Lf, t.x, t.y);
      auto blocks = [&](auto m0, auto m1) {
        dvec4 xt;
        solve_block<decltype(m0)::value>(xt, av, F);
        dvec4 xu;
        solve_block<decltype(m1)::value>(xu, av, F);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          L[(size_t)(16 * wt + li) * ld + 16 * decltype(m0)::value + 4 * r + lk] = xt[r];
          L[(size_t)(16 * wt + li) * ld + 16 * decltype(m1)::value + 4 * r + lk] = xu[r];
        }
      };
      if (half) blocks(std::integral_constant<int, 2>(), std::integral_constant<int, 1>());
      else blocks(std::integral_constant<int, 3>(), std::integral_constant<int, 0>());
      publish(sy.l(t.x, t.y), done);
    };
    // wave 0: the flags of phase k's products of own tiles q0 .. q1 - 1, a lane each
    auto await_products = [&](int q0, int q1, int k) {
      if (tid < 64) {
        for (int q = q0 + (tid >> 1); q < q1; q += 32) {
          const int2 t = own(q);
          if (product(t, k)) poll(sy.l(tid & 1 ? t.y : t.x, k), done, fail);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      }
      __syncthreads();
    };
    auto load_tile = [&](const int2& t, dvec4 (&acc)[2]) {
      const double* const A = tile(S, t.x, t.y) + (size_t)16 * wt * ld + 32 * half;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[c][r] = A[(size_t)(4 * r + lk) * ld + 16 * c + li];
    };
    int2 held[kHeld];
    dvec4 acc[kHeld][2];
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
      held[u] = nmem + u < nown ? own(nmem + u) : make_int2(0, 0);
      load_tile(held[u], acc[u]);
    }
    int cur = 0;  // own tiles of columns up to k
    for (; cur < nown; ++cur) {
      const int2 t = own(cur);
      if (t.y != 0) break;
      dvec2 mf[3];
      dvec4 a0[2];
      load_tile(t, a0);
      solve(t, a0, mf, false);
    }
    auto column = [&](const int2& t, int k, dvec4 (&acc)[2], bool from_memory) {
      dvec2 mf[3];
      const bool have = *(lds_flag*)sm.prog != 0;
      if (have) load_m(mf, k + 1);
      multiply(t, k, acc, from_memory);
      solve(t, acc, mf, have);
    };
    for (int k = 0; k + 1 < T; ++k) {
      for (; cur < nown; ++cur) {
        const int2 t = own(cur);
        if (t.y != k + 1) break;
        if (t.x == t.y) continue;
        if (tid == 0) *(lds_flag*)sm.prog = peek(sy.m(k + 1)) >= done;
        await_products(cur, cur + 1, k);
        if (cur < nmem) {
          dvec4 am[2];
          column(t, k, am, true);
        }
#pragma unroll
        for (int u = 0; u < kHeld; ++u)
          if (cur == nmem + u) column(t, k, acc[u], false);
      }
      await_products(cur, nown, k);
      for (int q = cur; q < nmem; ++q) {
        dvec4 am[2];
        const int2 t = own(q);
        if (product(t, k)) multiply(t, k, am, true);
      }
#pragma unroll
      for (int u = 0; u < kHeld; ++u)
        if (nmem + u >= cur && nmem + u < nown && product(held[u], k)) multiply(held[u], k, acc[u], false);
      __syncthreads();
    }
    if (w >= 4) return;
  } else {
    if (w >= 4) return;  // one tile is four waves' work
    int i, j;
    owner_tile(o, T, &i, &j);
    double* const Aij = tile(S, i, j);
    const bool diag = i == j;
    dvec4 acc[4];
    acc_load(acc, Aij, ld, w);
    const int steps = diag ? j - 1 : j;
    for (int k = 0; k < steps; ++k) {
      double av[16], bv[16];
      if (k >= 1) wait_flags(done, fail, sy.a(i, k), diag ? nullptr : sy.a(j, k));
      load_rows(av, tile(S, i, k) + (size_t)16 * w * ld, ld);
      if (!diag) load_rows(bv, tile(S, j, k) + (size_t)16 * w * ld, ld);
      wait_flags(done, fail, sy.m(k));
      load_inv(F, Mg + (size_t)k * kInvLen);
      lds_barrier();
      dvec4 xt[4], yt[4];
      solve_rows(xt, av, F);
      if (!diag) {
        solve_rows(yt, bv, F);
        put_result(XF, w, yt);
      } else {
        put_result(XF, w, xt);
      }
      lds_barrier();
      acc_update(acc, xt, XF);
      lds_barrier();
    }
    if (j > 0 && !(diag && steps == 0)) {
      acc_store(acc, Aij, ld, w);
      publish(sy.a(i, j), done);
    }
    if (!diag) {
      // L_ij = A_ij M_j^T: the accumulators as operand rows through LDS (each
      // wave its own sixteen rows)
      double av[16];
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) sm.Y[0][(16 * w + 4 * r + lk) * TS + 16 * c + li] = acc[c][r];
      wait_flags(done, fail, sy.m(j));
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const dvec2 t = *(const lds_dvec2*)((lds_dbl*)sm.Y[0] + (16 * w + li) * TS + 16 * kb + 4 * lk + 2 * h);
          av[4 * kb + 2 * h] = t[0];
          av[4 * kb + 2 * h + 1] = t[1];
        }
      load_inv(F, Mg + (size_t)j * kInvLen);
      lds_barrier();
      dvec4 xt[4];
      solve_rows(xt, av, F);
      store_rows(xt, tile(Lf, i, j), ld, w);
      publish(sy.l(i, j), done);
    }
  }
  // ---- helpers of the back substitution: row i's terms x_j, j = T - 1 .. i + kNear + 1
  // (x_{T-1} is published after every L_ik, so the tiles can be loaded ahead of the
  // x that they wait for).  With a workgroup per tile the last owners do it, and
  // the others leave with their tile.
  for (int i = many ? o : G - 3 - o; i + kNear + 1 < T; i += G - 2) {
    double s = 0.0;
    TileRegs<4> l;
    for (int j = T - 1; j >= i + kNear + 1; --j) {
      wait_flags(epoch + (ull)(T - j), fail, sy.x());
      if (j == T - 1) l.load(tile(Lf, j, i), ld);
      if (tid < NB) sm.v[tid] = xs[(size_t)j * NB + tid];
      __syncthreads();
      l.cols((lds_dbl*)sm.v, (lds_dbl*)sm.part[0][0]);
      if (j > i + kNear + 1) l.load(tile(Lf, j - 1, i), ld);
      __syncthreads();
      s -= part_sum((lds_dbl*)sm.part[0][0]);
    }
    if (tid < NB) yv[(size_t)i * NB + tid] = s;
    publish(sy.r(i), done);
  }
}

int launch_chol(psba_ctx* c) {
  const int T = c->n_pad / NB;
  if (c->chol_grid <= 0) {
    int per_cu = 0, ncu = 0;
    PSBA_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_chol_solve, 512, 0));
    PSBA_HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
    // at most one workgroup per CU (the LDS use allows no more), so that every
    // workgroup of a launch is resident at once on the stream's device
    const int resident = std::min(per_cu, 1) * ncu;
    // the diagonal chain, the triangular solves and, up to what is resident, a
    // workgroup for every other tile
    const int want = T == 1 ? 1 : 2 + T * (T - 1) / 2 + std::max(0, T - 2);
    if (resident < std::min(want, 3 + kForward)) return PSBA_ERR_UNSUPPORTED;
    c->chol_grid = std::min(want, resident);
  }
  probe_begin(c, PSBA_PROBE_FACTOR);
  hipLaunchKernelGGL(k_chol_solve, dim3(c->chol_grid), dim3(512), 0, c->stream, c->S, c->n_pad, T, c->Lf, c->Minv,
                     c->ea, c->yv, c->xsol, c->dp, c->n, c->d_scal + SC_FACTOR_OK, c->sync, c->chol_fail,
                     gate_of(c, kGateActive));
  probe_end(c, PSBA_PROBE_FACTOR);
  c->L_cur = c->Lf;
  PSBA_LAUNCH_TRY();
  return PSBA_OK;
}

long chol_sync_words(int T) { return 3 + 3L * T + (long)T * (T + 1); }
long chol_inv_len(int T) { return (long)T * kInvLen; }

}  // namespace psba
