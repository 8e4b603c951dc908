// FP32 LU factorisation with partial pivoting, in place and row-major: the
// factorisation inside the reference's FP32 solve (jnp.linalg.solve(A32, .),
// ozaki_jax/solve.py:159).  Right-looking and blocked by panels of 32
// columns; each panel step is three kernels:
//  1. lu_panel_kernel (one workgroup): factors the panel's rows c .. n-1 in
//     registers, 16 columns at a time (each column: a pivot search and the
//     rank-1 update of the rows not yet pivots; rows stay where they were
//     read and their final positions are composed after the panel), and
//     writes the permutation the panel's swaps make of the rows;
//  2. lu_rowfix_trsm_kernel (64 columns outside the panel per workgroup):
//     applies that permutation to its columns (and to the permutation
//     vector) and, right of the panel, solves the unit-lower 32 x 32
//     diagonal block for its rows c .. c+31 (the U12 block);
//  3. lu_update_kernel: trailing A22 -= L21 U12, 64 x 64 tiles, K = 32.
// The panel step is the critical path: 32 pivot searches, one workgroup
// barrier each (about 0.9 us).
#include <cfloat>

#include "common.h"

namespace ozk {

constexpr int kLuThreads = 512;                  // panel workgroup
constexpr int kLuRpt = 8;                        // rows per thread
constexpr int kLuSub = 16;                       // sub-panel columns, in registers
constexpr int kLuPanel = 2 * kLuSub;             // panel width
constexpr int kLuMaxRows = kLuThreads * kLuRpt;  // panel height the registers hold
constexpr int kLuPairs = 2 * kLuPanel;           // rows a panel's swaps can move
constexpr int kLuWaves = kLuThreads / 64;
constexpr int kLuMapInts = 4 + 2 * kLuPairs;  // (the L block behind them 16-byte aligned)

// ---------------------------------------------------------------- waves
template <int CTRL>
__device__ __forceinline__ uint32_t lu_dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}

// Wave-uniform maximum (MAX) or minimum of u: quad, half-row and row
// mirrors, then the two permlane swaps across rows of 16 and 32 lanes.
template <bool MAX>
__device__ __forceinline__ uint32_t lu_wave_reduce(uint32_t u) {
  auto op = [](uint32_t x, uint32_t y) { return MAX ? max(x, y) : min(x, y); };
  u = op(u, lu_dpp<0xB1>(u));   // quad_perm [1, 0, 3, 2]
  u = op(u, lu_dpp<0x4E>(u));   // quad_perm [2, 3, 0, 1]
  u = op(u, lu_dpp<0x141>(u));  // half-row mirror
  u = op(u, lu_dpp<0x140>(u));  // row mirror
  {
    const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    u = op((uint32_t)s[0], (uint32_t)s[1]);
  }
  {
    const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    u = op((uint32_t)s[0], (uint32_t)s[1]);
  }
  return __builtin_amdgcn_readfirstlane(u);
}

// ---------------------------------------------------------------- panel
// The panel's rows stay where they were read: thread t holds physical rows
// t + i * kLuThreads (relative to row c), i < S.  A pivot is not moved in
// registers; the kernel keeps what became of each row and stores it at its
// final position.
//
// What bounds it: one workgroup on one CU, 32 dependent column steps.  Each
// step is a chain of a pivot search, an LDS exchange with one barrier and
// the rank-1 update: 0.9 us at one row slot, 28.8 a panel.  What taller panels
// take beyond that (34.9 us at 2 slots, 42.4 at 4, 51.9 at 6, 76.2 at 8) is the
// vector work and the loads of one CU, and at 7 and 8 slots, and from 5 on
// without 16-byte rows, registers spilled to scratch.  The steps run as a rolled
// loop: unrolled over the 32 columns the kernel was 28000 instructions, and
// fetching that much straight-line code (200 KB, over the 64 KB instruction
// cache) cost about a sixth of every short step and more of the tall ones.  The
// loop needs the active column in a fixed register, so each step rotates a row's
// registers by one: the updated columns move down and the finished L entry
// enters at the end.
// Measured with the row slots a compile-time count, the loads and stores
// four lanes a row and the permutation composed in parallel (us a panel,
// unrolled -> rolled): 4096 rows 108 -> 83, 2048 71 -> 45, 512 46 -> 30; n =
// 4096 factored in 9.1 ms (12.7; 8.7 with the update below).  Four waves (one
// a SIMD) instead of eight were slower (55 at 2048 rows), reading the pivot row
// back from LDS instead of by readlane too (50).
struct LuPanelShared {
  // per-wave candidates: the bits of |value| (0: none), and the physical row
  // with kLuTied if another row of the wave may equal it
  uint2 ckey[2][kLuWaves];
  float crow[2][kLuWaves][kLuSub];      //   and those rows' sub-panel registers
  float prow[kLuPanel][kLuSub];         // pivot rows: their own sub-panel's columns
  float b0[kLuSub][kLuSub];             // first sub-panel's pivots: the second's columns
  float l10[kLuSub][kLuSub];            // second sub-panel's pivots: the first's columns
  float u01[kLuSub][kLuSub];            // U block right of the first sub-panel
  int prow_of[kLuPanel];                // physical pivot row of column j
  int pos[kLuWaves][64];
  float4 stage[kLuWaves][64 * kLuSub / 4];
};

// Column `col` of a sub-panel after lu_factor_sub sits in register
// lu_reg(col): its two rotations (16 wide, then 8 wide) leave the halves
// swapped.
constexpr int lu_reg(int col) { return (col + kLuSub / 2) % kLuSub; }

// One dword per lane from global memory into LDS at lds_addr + 4 lane, for
// the active lanes (as dma16; the reader waits with wait_vm).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lu_dma4(uint32_t lds_addr, const void* gbase, uint32_t voff) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %1, %2"
      :
      : "s"(lds_addr), "v"(voff), "s"(gbase)
      : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ __forceinline__ float lu_readlane(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Where the first `cols` columns' swaps leave physical row x, which must not be
// a pivot of theirs (lanes with none: kLuNoRow): a row below `cols` went where its
// column's pivot row was; if that is a row below `cols` too, where that row's
// column's pivot was, and so on.  (Pivot rows differ, so the walk from a row
// that is none never comes back to a row: it ends.)
constexpr uint32_t kLuNoRow = ~0u, kLuTied = 1u << 31;
__device__ __forceinline__ uint32_t lu_position(uint32_t x, uint32_t cols, const int* prow_of) {
#pragma unroll 1
  for (int k = 0; k < kLuPanel && x < cols; ++k) x = (uint32_t)prow_of[x];
  return x;
}

// `steps` columns (panel columns dj0 ..) of a sub-panel over the rotating
// registers 0 .. WD - 1: register 0 holds the active column, registers
// WD - s .. WD - 1 the L entries of the s columns finished here.  lm[i]: all
// ones while row slot i can still become a pivot, 0 for a pivot or no row;
// 6-bit field i of pcode receives 1 + the panel column a row becomes the pivot
// of.  The pivot is the candidate with the largest |value| (bit patterns: a NaN
// wins); of equal ones the lowest in LAPACK's row order, its swaps so far
// applied (lu_position): where several tie, the search is repeated among them
// by position.  That path is almost never taken, but its presence costs random
// matrices 0.5% (n = 4096: 8.66 -> 8.71 ms) to 1.6% (2048: 3.25 -> 3.30);
// ordering inside the first search, before or behind its stores, cost 3 to 10%.
// Where every candidate is zero the lowest row is taken, the column left as
// it is and OZK_FLAG_SINGULAR raised.  fetch(pr, dj) starts the copy of pivot
// row pr's other sub-panel into LDS (one wave).
template <int S, int WD, class Fetch>
__device__ __forceinline__ void lu_columns(float (&r)[S][kLuSub], uint32_t (&lm)[S],
                                           uint64_t& pcode, int dj0, int steps,
                                           LuPanelShared& sh, uint32_t* status, Fetch fetch) {
  const int t = threadIdx.x, lane = t % 64;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int k0 = 2 * (lane % kLuWaves);  // the lane's registers of record lane / kLuWaves
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    const int dj = dj0 + s, par = dj & 1;
    uint32_t u[S];
#pragma unroll
    for (int i = 0; i < S; ++i) u[i] = __float_as_uint(r[i][0]) & lm[i] & 0x7fffffffu;
    bool by_row = false;  // the candidates are those of equal magnitude, by position
    uint2 kv;
    float2 rv;
    float pvl, rl;
    int qw, pr;
#pragma unroll 1
    for (;;) {
      uint32_t m1 = S > 1 ? u[S - 1] : 0u;  // of the slots above the first
#pragma unroll
      for (int i = 1; i < S - 1; ++i) m1 = max(m1, u[i]);
      const uint32_t mx = max(u[0], m1);
      // the lane's slot (lowest of equals), while the wave's maximum forms
      int sel = S - 1;
#pragma unroll
      for (int i = S - 2; i >= 0; --i) sel = u[i] == mx ? i : sel;
      const uint32_t wb = lu_wave_reduce<true>(mx);
      // several lanes' candidates; or one lane's, whose first slot alone may
      // hold a displaced row
      const uint64_t tie = __ballot(mx == wb), both = S > 1 ? __ballot(u[0] == m1) : 0u;
      const uint32_t tied = (tie & ((tie - 1u) | both)) != 0u ? kLuTied : 0u;
      const int hl = (int)__builtin_ctzll(tie);
      const int slot = S > 1 ? __builtin_amdgcn_readlane(sel, hl) : 0;
      if (lane == hl) {
        sh.ckey[par][wave] = make_uint2(wb, (uint32_t)(slot * kLuThreads + t) | tied);
        static_for<0, S>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          if (i == slot) {
            float4* const d = (float4*)sh.crow[par][wave];
#pragma unroll
            for (int q = 0; q < kLuSub / 4; ++q)
              d[q] = make_float4(r[i][4 * q], r[i][4 * q + 1], r[i][4 * q + 2], r[i][4 * q + 3]);
            // (distinct per case: keeps the compiler from merging the cases
            // into one store of a run-time-indexed row)
            asm volatile("; lu candidate row %0" ::"n"(i));
          }
        });
      }
      __syncthreads();
      // Lane l reads key l % 8 and two values of candidate row l / 8, so the
      // winner's row is there without a second LDS round trip.
      kv = sh.ckey[par][lane % kLuWaves];
      pvl = sh.crow[par][lane % kLuWaves][0];
      rv = *(const float2*)&sh.crow[par][lane / kLuWaves][k0];
      uint32_t best = kv.x;
      best = max(best, lu_dpp<0xB1>(best));   // quad_perm [1, 0, 3, 2]
      best = max(best, lu_dpp<0x4E>(best));   // quad_perm [2, 3, 0, 1]
      best = max(best, lu_dpp<0x141>(best));  // half-row mirror: 8 lanes
      best = __builtin_amdgcn_readfirstlane(best);
      // LAPACK's getf2 scales by the pivot's reciprocal.  Every lane inverts
      // its candidate while the maximum forms (the empty asm keeps the
      // compiler from doing it after the choice instead).
      rl = 1.0f / pvl;
      asm volatile("" : "+v"(rl));
      const uint64_t won = __ballot(kv.x == best);
      qw = (int)__builtin_ctzll(won);
      pr = __builtin_amdgcn_readlane((int)kv.y, qw);
      // one wave's only candidate (8 lanes read its key): uniform over the workgroup
      if (__builtin_expect(
              (__builtin_popcountll(won) == 64 / kLuWaves && pr >= 0) || by_row, 1))
        break;
      by_row = true;
      const uint32_t at = lu_position(lm[0] ? (uint32_t)t : kLuNoRow, (uint32_t)dj, sh.prow_of);
#pragma unroll
      for (int i = 0; i < S; ++i)
        u[i] = u[i] == best
                   ? ((uint32_t)INT_MAX - (i ? (uint32_t)(t + kLuThreads * i) : at)) & lm[i]
                   : 0u;
      __syncthreads();
    }
    const float pv = lu_readlane(pvl, qw);
    float rinv = lu_readlane(rl, qw);
    // the pivot row's columns right of the active one (0 for finished ones)
    const float px = k0 < WD - s ? rv.x : 0.0f, py = k0 + 1 < WD - s ? rv.y : 0.0f;
    float p[WD];
#pragma unroll
    for (int k = 1; k < WD; ++k) p[k] = lu_readlane(k & 1 ? py : px, qw * kLuWaves + k / 2);
    if (wave == dj % kLuWaves && lane / kLuWaves == qw) {
      // the lane's registers of the pivot row, at their columns
      constexpr int H = kLuSub / 2;
      const int c0 = WD == kLuSub ? (k0 + s) % kLuSub : (k0 < H ? H + (k0 + s) % H : k0 - H);
      const int c1 = WD == kLuSub ? (k0 + 1 + s) % kLuSub
                                  : (k0 < H ? H + (k0 + 1 + s) % H : k0 + 1 - H);
      sh.prow[dj][c0] = rv.x;
      sh.prow[dj][c1] = rv.y;
      if (k0 == 0) sh.prow_of[dj] = pr;
    }
    fetch(pr, dj);
    if (wave == (int)((uint32_t)pr / 64u % kLuWaves)) {  // uniform: the wave of the pivot's owner
      if (lane == (int)((uint32_t)pr % 64u))
        pcode |= (uint64_t)(dj + 1) << (6 * ((uint32_t)pr / kLuThreads));
#pragma unroll
      for (int i = 0; i < S; ++i) lm[i] = t + i * kLuThreads == pr ? 0u : lm[i];
    }
    if (fabsf(pv) < FLT_MIN) {  // uniform
      if (pv == 0.0f) {
        // no update: 0 * p would carry an infinity of its row to all others
        rinv = 0.0f;
#pragma unroll
        for (int k = 1; k < WD; ++k) p[k] = 0.0f;
        if (t == 0) atomicOr(status, OZK_FLAG_SINGULAR);
      } else {
        // the reciprocal can overflow: getf2 divides here, one rounding a
        // multiplier (the pivot row itself is out of lm by now)
        rinv = 1.0f;
#pragma unroll
        for (int i = 0; i < S; ++i) r[i][0] = lm[i] ? r[i][0] / pv : r[i][0];
      }
    }
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const uint32_t q = __float_as_uint(r[i][0] * rinv);
      const float l = __uint_as_float(q & lm[i]);
      const float keep = __uint_as_float((q & lm[i]) | (__float_as_uint(r[i][0]) & ~lm[i]));
#pragma unroll
      for (int k = 1; k < WD; ++k) r[i][k - 1] = fmaf(-l, p[k], r[i][k]);
      r[i][WD - 1] = keep;
    }
  }
}

// Rotates registers 0 .. WD - 1 by `steps` columns that a narrow sub-panel
// does not have.
template <int S, int WD>
__device__ __forceinline__ void lu_rotate(float (&r)[S][kLuSub], int steps) {
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const float f = r[i][0];
#pragma unroll
      for (int k = 1; k < WD; ++k) r[i][k - 1] = r[i][k];
      r[i][WD - 1] = f;
    }
  }
}

// Partial pivoting on one sub-panel of ncols columns (panel columns off ..)
// in registers: r[i][k] comes in as column k and leaves as column c in
// register lu_reg(c).  The first 8 columns rotate all 16 registers, the last
// 8 only the upper columns' (11 FMAs a row and column instead of 15).
template <int S, class Fetch>
__device__ __forceinline__ void lu_factor_sub(float (&r)[S][kLuSub], uint32_t (&lm)[S],
                                              uint64_t& pcode, int off, int ncols,
                                              LuPanelShared& sh, uint32_t* status,
                                              Fetch fetch) {
  constexpr int H = kLuSub / 2;
  const int n0 = ncols < H ? ncols : H, n1 = ncols - n0;
  lu_columns<S, kLuSub>(r, lm, pcode, off, n0, sh, status, fetch);
  if (n0 < H) lu_rotate<S, kLuSub>(r, H - n0);
  lu_columns<S, H>(r, lm, pcode, off + H, n1, sh, status, fetch);
  if (n1 < H) lu_rotate<S, H>(r, H - n1);
}

// Row slots [I0, I1) of a sub-panel from global memory: r[i][k] = P[ph * lda
// + col0 + k].  VEC (16-byte aligned rows, full panels) reads 16 rows of 64 bytes per
// load, four lanes a row (one row per lane would touch 64 cache lines a
// load); lu_load_finish then turns the rows into one per lane through the
// wave's LDS.  Rows past m are zero.
template <bool VEC, int I0, int I1, int S>
__device__ __forceinline__ void lu_load_issue(float (&r)[S][kLuSub], const float* P, int64_t lda,
                                              int col0, int ncols, int m) {
  const int t = threadIdx.x, lane = t % 64;
#pragma unroll
  for (int i = I0; i < I1; ++i) {
    if constexpr (VEC) {
#pragma unroll
      for (int q = 0; q < kLuSub / 4; ++q) {
        const int ph = i * kLuThreads + (t - lane) + 16 * q + lane / 4;
        const float4 v = *(const float4*)(P + (int64_t)(ph < m ? ph : 0) * lda + col0 +
                                          4 * (lane % 4));
        r[i][4 * q] = v.x;
        r[i][4 * q + 1] = v.y;
        r[i][4 * q + 2] = v.z;
        r[i][4 * q + 3] = v.w;
      }
    } else {
      const int ph = t + i * kLuThreads;
      const float* const row = P + (int64_t)(ph < m ? ph : 0) * lda + col0;
#pragma unroll
      for (int k = 0; k < kLuSub; ++k) r[i][k] = (ph < m && k < ncols) ? row[k] : 0.0f;
    }
  }
}

// 16-byte unit of (row, quarter of its 64 bytes) in a wave's stage: the
// quarters rotate with row / 4, which spreads both access patterns over the
// banks.
__device__ __forceinline__ int lu_stage(int row, int q) { return 4 * row + (q ^ ((row / 4) % 4)); }

template <bool VEC, int I0, int I1, int S>
__device__ __forceinline__ void lu_load_finish(float (&r)[S][kLuSub], int ncols, int m,
                                               LuPanelShared& sh) {
  if (!VEC) return;
  const int t = threadIdx.x, lane = t % 64;
  float4* const st = sh.stage[t / 64];
#pragma unroll
  for (int i = I0; i < I1; ++i) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int q = 0; q < 4; ++q)
      st[lu_stage(16 * q + lane / 4, lane % 4)] =
          make_float4(r[i][4 * q], r[i][4 * q + 1], r[i][4 * q + 2], r[i][4 * q + 3]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const bool live = t + i * kLuThreads < m;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = st[lu_stage(lane, q)];
      r[i][4 * q] = live ? v.x : 0.0f;
      r[i][4 * q + 1] = live ? v.y : 0.0f;
      r[i][4 * q + 2] = live ? v.z : 0.0f;
      r[i][4 * q + 3] = live ? v.w : 0.0f;
    }
  }
}

// Stores a factored sub-panel's rows, row slot i of this lane at position
// pos(i) (negative: not stored), through the wave's LDS as the loads.
template <bool VEC, int S, class Pos>
__device__ __forceinline__ void lu_store_rows(const float (&r)[S][kLuSub], float* P, int64_t lda,
                                              int col0, int ncols, LuPanelShared& sh, Pos pos) {
  const int t = threadIdx.x, lane = t % 64;
  float4* const st = sh.stage[t / 64];
  int* const ps = sh.pos[t / 64];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int at = pos(i);
    if constexpr (VEC) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      ps[lane] = at;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = lu_reg(4 * q);
        st[lu_stage(lane, q)] = make_float4(r[i][k], r[i][k + 1], r[i][k + 2], r[i][k + 3]);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 16 * q + lane / 4, to = ps[row];
        const float4 v = st[lu_stage(row, lane % 4)];
        if (to >= 0) *(float4*)(P + (int64_t)to * lda + col0 + 4 * (lane % 4)) = v;
      }
    } else if (at >= 0) {
      float* const row = P + (int64_t)at * lda + col0;
#pragma unroll
      for (int k = 0; k < kLuSub; ++k)
        if (k < ncols) row[k] = r[i][lu_reg(k)];
    }
  }
}

// b[i] -= a[i] U01 for the rows that are not pivots of the first sub-panel,
// i in [I0, I1).
template <int I0, int I1, int S>
__device__ __forceinline__ void lu_update_rows(float (&b)[S][kLuSub], const float (&a)[S][kLuSub],
                                               const uint32_t (&lm)[S], const LuPanelShared& sh) {
#pragma unroll
  for (int q = 0; q < kLuSub; ++q) {
    asm volatile("" ::: "memory");  // one row of U01 at a time in registers
    float u[kLuSub];
#pragma unroll
    for (int k = 0; k < kLuSub; ++k) u[k] = sh.u01[q][k];
#pragma unroll
    for (int i = I0; i < I1; ++i) {
      const float l = __uint_as_float(__float_as_uint(a[i][lu_reg(q)]) & lm[i]);
#pragma unroll
      for (int k = 0; k < kLuSub; ++k) b[i][k] = fmaf(-l, u[k], b[i][k]);
    }
  }
}

// Factors panel columns [c, c + w) over rows [c, n) (m = n - c <= S *
// kLuThreads rows, w <= kLuPanel) and writes to maps the row permutation its
// swaps make: maps[0] = w, then kLuPairs destination rows (absolute, -1 =
// unused) and kLuPairs source rows.  Entries e < w are the diagonal
// positions c + e; entry kLuPanel + x puts row c + x, x < w, if it is no
// pivot, where the swaps moved it.  Behind them lies the panel's L block (rows
// c .. c + w - 1, kLuPanel x kLuPanel, zero on and above the diagonal).  The
// first sub-panel's columns are stored with their rows where they were; the
// row fix moves them with the columns left of the panel.
//
// Up to S = kLuPreload row slots the second sub-panel's loads are issued
// before the first is factored; above, the registers hold them in two halves
// after it.
constexpr int kLuPreload = 4;

template <bool VEC, int S>
__global__ __launch_bounds__(kLuThreads) void lu_panel_kernel(float* __restrict__ A,
                                                              int64_t lda, int n, int c, int cols,
                                                              int* __restrict__ maps,
                                                              uint32_t* __restrict__ status) {
  __shared__ LuPanelShared sh;
  const int w = VEC ? kLuPanel : cols;
  const int t = threadIdx.x, lane = t % 64;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int m = n - c;
  const int w0 = w < kLuSub ? w : kLuSub, w1 = w - w0;
  float* const P = A + (int64_t)c * lda + c;
  uint64_t pcode = 0u;
  uint32_t lm[S];
#pragma unroll
  for (int i = 0; i < S; ++i) lm[i] = t + i * kLuThreads < m ? ~0u : 0u;

  float a[S][kLuSub], b[S][kLuSub];
  lu_load_issue<VEC, 0, S>(a, P, lda, 0, w0, m);
  if (S <= kLuPreload && w1 > 0) lu_load_issue<VEC, 0, S>(b, P, lda, kLuSub, w1, m);
  lu_load_finish<VEC, 0, S>(a, w0, m, sh);
  // wave 7 copies each pivot row's second sub-panel columns (still as they
  // came) into b0 for the U01 block
  const uint32_t lds_b0 = lds_offset(sh.b0), lds_l10 = lds_offset(sh.l10);
  lu_factor_sub<S>(a, lm, pcode, 0, w0, sh, status, [&](int pr, int dj) {
    if (wave == kLuWaves - 1 && lane < w1)
      lu_dma4(__builtin_amdgcn_readfirstlane(lds_b0 + dj * kLuSub * 4),
              P + (int64_t)pr * lda + kLuSub, 4u * (uint32_t)lane);
  });
  lu_store_rows<VEC>(a, P, lda, 0, w0, sh, [&](int i) {
    return t + i * kLuThreads < m ? t + i * kLuThreads : -1;
  });

  if (w1 > 0) {
    if (wave == kLuWaves - 1) wait_vm<0>();
    __syncthreads();  // b0 and the first sub-panel's pivot rows in LDS
    if (t < kLuSub) {
      // U01 = L00^-1 B0; lane k holds column k (zeros past w1)
      float u[kLuSub];
#pragma unroll
      for (int q = 0; q < kLuSub; ++q) u[q] = t < w1 ? sh.b0[q][t] : 0.0f;
#pragma unroll
      for (int q = 0; q < kLuSub; ++q) {
#pragma unroll
        for (int k = q + 1; k < kLuSub; ++k) u[k] = fmaf(-sh.prow[k][q], u[q], u[k]);
      }
#pragma unroll
      for (int q = 0; q < kLuSub; ++q) {
        sh.u01[q][t] = u[q];
      }
    }
    __syncthreads();  // U01 in LDS
    if constexpr (S <= kLuPreload) {
      lu_load_finish<VEC, 0, S>(b, w1, m, sh);
      lu_update_rows<0, S>(b, a, lm, sh);
    } else {
      // Half of the rows at a time, so that a and b do not both fill the
      // registers.
      lu_load_issue<VEC, 0, S / 2>(b, P, lda, kLuSub, w1, m);
      lu_load_finish<VEC, 0, S / 2>(b, w1, m, sh);
      lu_update_rows<0, S / 2>(b, a, lm, sh);
      asm volatile("" ::: "memory");  // the first half's registers of a are free now
      lu_load_issue<VEC, S / 2, S>(b, P, lda, kLuSub, w1, m);
      lu_load_finish<VEC, S / 2, S>(b, w1, m, sh);
      lu_update_rows<S / 2, S>(b, a, lm, sh);
    }
    // wave 7 copies each pivot row's L entries of the first sub-panel, as
    // stored above, into l10
    lu_factor_sub<S>(b, lm, pcode, kLuSub, w1, sh, status, [&](int pr, int dj) {
      if (wave == kLuWaves - 1 && lane < kLuSub)
        lu_dma4(__builtin_amdgcn_readfirstlane(lds_l10 + (dj - kLuSub) * kLuSub * 4),
                P + (int64_t)pr * lda, 4u * (uint32_t)lane);
    });
    if (t < kLuSub) {  // positions 0 .. 15 hold the first sub-panel's pivots
#pragma unroll
      for (int q = 0; q < kLuSub; ++q)
        if (t < w1) P[(int64_t)q * lda + kLuSub + t] = sh.u01[q][t];
    }
    if (wave == kLuWaves - 1) wait_vm<0>();
  }
  __syncthreads();  // prow_of, prow and l10 final
  // The permutation: position j takes pivot row j, and a row below w that is
  // no pivot goes where the swaps left it.
  const bool moves = t < w && (pcode & 63u) == 0u;
  const int top = (int)lu_position(moves ? (uint32_t)t : kLuNoRow, (uint32_t)w, sh.prow_of);
  if (t < kLuPanel) {
    const bool col = t < w;
    maps[1 + t] = col ? c + t : -1;
    maps[1 + kLuPairs + t] = c + (col ? sh.prow_of[t] : 0);
    maps[1 + kLuPanel + t] = moves ? c + top : -1;
    maps[1 + kLuPairs + kLuPanel + t] = c + (moves ? t : 0);
    if (t == 0) maps[0] = w;
  }
  float* const L = (float*)(maps + kLuMapInts);
#pragma unroll
  for (int e = t; e < kLuPanel * kLuPanel; e += kLuThreads) {
    const int rr = e / kLuPanel, cc = e % kLuPanel;
    float v = 0.0f;
    if (cc < rr && rr < w)
      v = rr < kLuSub ? sh.prow[rr][cc]
                      : (cc < kLuSub ? sh.l10[rr - kLuSub][cc] : sh.prow[rr][cc - kLuSub]);
    L[e] = v;
  }
  if (w1 > 0) {
    lu_store_rows<VEC>(b, P, lda, kLuSub, w1, sh, [&](int i) {
      const int ph = t + i * kLuThreads, code = (int)((pcode >> (6 * i)) & 63u);
      if (ph >= m || (code > 0 && code <= kLuSub)) return -1;  // U01's rows are stored above
      if (code > 0) return code - 1;
      return ph < w ? top : ph;
    });
  }
}

// The columns outside the panel [c, c + w), 64 per workgroup (lane = column,
// wave = a sixteenth of the permutation's entries), and the permutation
// vector (the last workgroup): applies the panel's row permutation, every
// source value read before any is written.  Right of the panel, wave 0 then
// solves the unit-lower diagonal block for its 64 columns (rows c .. c+w-1
// become U12) from the values staged in LDS.
constexpr int kLuFixCols = 64;
constexpr int kLuFixThreads = 1024;  // 16 waves, 4 entries each

__global__ __launch_bounds__(kLuFixThreads) void lu_rowfix_trsm_kernel(
    float* __restrict__ A, int64_t lda, int n, int c, const int* __restrict__ maps,
    int32_t* __restrict__ perm) {
  __shared__ float L[kLuPanel][kLuPanel + 1];
  __shared__ float buf[kLuPairs][kLuFixCols + 1];
  const int t = threadIdx.x, lane = t % 64, wv = t / 64;
  const int w = maps[0];
  const int right = n - c - w;
  const int left = c + (w < kLuSub ? w : kLuSub);  // and the first sub-panel's columns
  const int nleft = (left + kLuFixCols - 1) / kLuFixCols;
  const int nright = (right + kLuFixCols - 1) / kLuFixCols;
  constexpr int kPer = kLuPairs / (kLuFixThreads / 64);  // entries per wave

  if ((int)blockIdx.x == nleft + nright) {  // the permutation vector
    int v = 0;
    const int dst = t < kLuPairs ? maps[1 + t] : -1;
    if (dst >= 0) v = perm[maps[1 + kLuPairs + t]];
    __syncthreads();
    if (dst >= 0) perm[dst] = v;
    return;
  }
  const bool is_right = (int)blockIdx.x >= nleft;
  const int64_t x = is_right ? (int64_t)c + w + ((int)blockIdx.x - nleft) * kLuFixCols + lane
                             : (int64_t)blockIdx.x * kLuFixCols + lane;
  const bool live = is_right ? x < n : x < left;
  if (is_right) {
    const float* const Lg = (const float*)(maps + kLuMapInts);
    for (int q = t; q < kLuPanel * kLuPanel; q += kLuFixThreads)
      L[q / kLuPanel][q % kLuPanel] = Lg[q];
  }
  float v[kPer];
  int dst[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int e = wv * kPer + k;
    dst[k] = maps[1 + e];
    v[k] = (live && dst[k] >= 0) ? A[(int64_t)maps[1 + kLuPairs + e] * lda + x] : 0.0f;
  }
  __syncthreads();  // every load before any store: rows move between waves
  if (is_right) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) buf[wv * kPer + k][lane] = v[k];
    __syncthreads();
    if (wv == 0) {  // entries j < w are the diagonal rows c + j, in order
      // column-oriented: once u[q] is final it updates every later row, so
      // the dependent chain is 32 steps, not 496
      float u[kLuPanel];
#pragma unroll
      for (int j = 0; j < kLuPanel; ++j) u[j] = buf[j][lane];
#pragma unroll
      for (int q = 0; q < kLuPanel - 1; ++q) {
#pragma unroll
        for (int j = q + 1; j < kLuPanel; ++j) u[j] = fmaf(-L[j][q], u[q], u[j]);
      }
#pragma unroll
      for (int j = 0; j < kLuPanel; ++j) buf[j][lane] = u[j];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k) v[k] = buf[wv * kPer + k][lane];
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k)
    if (live && dst[k] >= 0) A[(int64_t)dst[k] * lda + x] = v[k];
}

// Trailing update A[r][x] -= sum_q A[r][c + q] A[c + q][x] over rows and
// columns [c + kLuPanel, n): one 64 x 64 tile per workgroup, 4 x 4 outputs per
// thread.  K = 32 makes it bound by the read and write of A22 and, in tiles of one
// round, by the latency of its loads: the tile's own values are therefore loaded
// together with its operands and not after the products, and L is kept
// transposed in LDS, so that a step of q reads two float4.
// n = 4096: 14.9 -> 12.6 us a step on average; 28.8 at 4064 rows, the rate of a
// large copy (4.7 TB/s).
template <bool VEC>
__device__ __forceinline__ float4 lu_load4(const float* src, int64_t left) {
  if (VEC && left >= 4) return *(const float4*)src;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (left > 0) v.x = src[0];
  if (left > 1) v.y = src[1];
  if (left > 2) v.z = src[2];
  if (left > 3) v.w = src[3];
  return v;
}

template <bool VEC>
__global__ __launch_bounds__(256) void lu_update_kernel(float* __restrict__ A, int64_t lda,
                                                        int n, int c) {
  constexpr int kLd = 68;  // float4 rows whose transposing stores meet 2 to a bank
  __shared__ __align__(16) float As[kLuPanel][kLd];
  __shared__ float4 Bs[kLuPanel][16];
  const int t = threadIdx.x;
  const int s = c + kLuPanel;
  const int64_t r0 = s + (int64_t)blockIdx.y * 64, x0 = s + (int64_t)blockIdx.x * 64;
  const int ty = t / 16, tx = t % 16;
  const int64_t x = x0 + 4 * tx;
  float4 l[2], u[2], old[4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t r = r0 + t / 8 + 32 * h;
    l[h] = lu_load4<VEC>(A + r * lda + c + 4 * (t % 8), r < n ? 4 : 0);
    u[h] = lu_load4<VEC>(A + (int64_t)(c + ty + 16 * h) * lda + x, n - x);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t r = r0 + ty * 4 + i;
    old[i] = lu_load4<VEC>(A + r * lda + x, r < n ? n - x : 0);
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int rr = t / 8 + 32 * h, kk = 4 * (t % 8);
    As[kk][rr] = l[h].x;
    As[kk + 1][rr] = l[h].y;
    As[kk + 2][rr] = l[h].z;
    As[kk + 3][rr] = l[h].w;
    Bs[ty + 16 * h][tx] = u[h];
  }
  __syncthreads();
  float acc[4][4] = {};
#pragma unroll 8
  for (int kk = 0; kk < kLuPanel; ++kk) {
    const float4 a = *(const float4*)&As[kk][ty * 4], b = Bs[kk][tx];
    const float av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i][0] = fmaf(av[i], b.x, acc[i][0]);
      acc[i][1] = fmaf(av[i], b.y, acc[i][1]);
      acc[i][2] = fmaf(av[i], b.z, acc[i][2]);
      acc[i][3] = fmaf(av[i], b.w, acc[i][3]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t r = r0 + ty * 4 + i;
    if (r >= n) continue;
    float* const dst = A + r * lda + x;
    const float v[4] = {old[i].x - acc[i][0], old[i].y - acc[i][1], old[i].z - acc[i][2],
                        old[i].w - acc[i][3]};
    if (VEC && x + 4 <= n) {
      *(float4*)dst = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (x + j < n) dst[j] = v[j];
    }
  }
}

__global__ void lu_iota_kernel(int32_t* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

int64_t lu_factor_max_n() { return kLuMaxRows; }
size_t lu_factor_workspace_bytes() {
  return kLuMapInts * sizeof(int) + kLuPanel * kLuPanel * sizeof(float);
}

// The panel kernel with as many row slots per thread as the rows need.
template <bool VEC, int S>
static void launch_lu_panel(float* A, int64_t lda, int n, int c, int w, int* maps,
                            uint32_t* status, hipStream_t st) {
  if constexpr (S > 1) {
    if (n - c <= (S - 1) * kLuThreads) {
      launch_lu_panel<VEC, S - 1>(A, lda, n, c, w, maps, status, st);
      return;
    }
  }
  hipLaunchKernelGGL((lu_panel_kernel<VEC, S>), dim3(1), dim3(kLuThreads), 0, st, A, lda, n, c,
                     w, maps, status);
}

template <bool VEC>
static int lu_factor_steps(float* A, int64_t lda, int n, int32_t* perm, int* maps,
                           uint32_t* status, hipStream_t st) {
  for (int c = 0; c < n; c += kLuPanel) {
    const int w = n - c < kLuPanel ? n - c : kLuPanel;
    if (VEC && w == kLuPanel)
      launch_lu_panel<true, kLuRpt>(A, lda, n, c, w, maps, status, st);
    else
      launch_lu_panel<false, kLuRpt>(A, lda, n, c, w, maps, status, st);
    OZK_LAUNCH_CHECK();
    const int right = n - c - w;
    const int left = c + (w < kLuSub ? w : kLuSub);
    const int groups =
        (left + kLuFixCols - 1) / kLuFixCols + (right + kLuFixCols - 1) / kLuFixCols;
    hipLaunchKernelGGL(lu_rowfix_trsm_kernel, dim3(groups + 1), dim3(kLuFixThreads), 0, st, A,
                       lda, n, c, maps, perm);
    OZK_LAUNCH_CHECK();
    if (right > 0) {
      const unsigned tiles = (unsigned)((right + 63) / 64);
      hipLaunchKernelGGL(lu_update_kernel<VEC>, dim3(tiles, tiles), dim3(256), 0, st, A, lda,
                         n, c);
      OZK_LAUNCH_CHECK();
    }
  }
  return OZK_OK;
}

int launch_lu_factor(float* A, int64_t lda, int64_t n, int32_t* perm, void* ws,
                     uint32_t* status, hipStream_t st) {
  hipLaunchKernelGGL(lu_iota_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, perm,
                     (int)n);
  OZK_LAUNCH_CHECK();
  const bool vec = ((uintptr_t)A % 16 == 0) && (lda % 4 == 0);
  return vec ? lu_factor_steps<true>(A, lda, (int)n, perm, (int*)ws, status, st)
             : lu_factor_steps<false>(A, lda, (int)n, perm, (int*)ws, status, st);
}

}  // namespace ozk
