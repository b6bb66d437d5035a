// k_tri.hip -- twisted plane solves: both planes of a factor slot from one half
// of its symmetric block inverses, complex64 and complex128.
//
// Planes k and nz - k share a factor slot, and a slot's chain is eliminated
// from both ends (block j < m: top-down inverse G_j, j = m: T_m, j > m:
// bottom-up inverse B_j; sig_j = cm_y(j) cp_y(j-1)).  Phase 0 (forward):
//   top:    t_0 = f_0, t_j = f_j - cm_y(j) G_{j-1} t_{j-1} (0 < j < m), y_top = G_{m-1} t_{m-1}
//   bottom: b_{ny-1} = f_{ny-1}, b_j = f_j - cp_y(j) B_{j+1} b_{j+1} (m < j < ny-1), y_bot = B_{m+1} b_{m+1}
// Phase 1 (backward):
//   x_m = T_m (f_m - cm_y(m) y_top - cp_y(m) y_bot),
//   top x_j = G_j (t_j - cp_y(j) x_{j+1}) down to j = 0, bottom x_j = B_j (b_j - cm_y(j) x_{j-1}) up to ny-1.
// One workgroup per (slot, half) carries both planes: 2 nslot workgroups walk
// about ny/2 dependent block products each and every stored value is read once
// for two planes.  y_top, y_bot and f_m pass between the phases in scr.
//
// Adjoint: with D = diag(dx(i) dy(j)) the plane operator satisfies M^T =
// D^-1 M D, so M^H x = b is the forward solve M z = D conj(b), x =
// conj(D^-1 z); the scalings are folded into the line loads and stores.
//
// K_j = X_j D_j is symmetric, and y = X_j v = K_j v' with v' = D_j^-1 v held in
// LDS as the four real columns of the two planes.  K_j is kept as one half of
// its 16 x 16 tiles, taken round the diagonals: tile row R holds the tile
// columns R, R + 1, ... (mod NT), NT/2 + 1 of them (even NT: NT/2 where R >=
// NT/2), so every pair of tiles (R, C), (C, R) is kept once and every wave gets
// the same static program: rows w and w + NW, or row w alone.  Tiles go straight from memory
// into registers: lane 4 b + i holds row 4 (b & 3) + i and the four columns
// 4 (b >> 2) .. + 3 (two 16-byte units), so a load instruction reads 1 KB in
// order.  Each value serves both products on the matrix cores
// (v_mfma_f32_4x4x1f32, 16 blocks of 4 x 4: D(4b+j, reg i) += A(4b+i) B(4b+j),
// no idle column):
//   direct, y_r += K(r, c) v'_c: A = K, B = the components of v'_c; the rows'
//     sums stay in registers over the whole tile row;
//   transposed, y_c += K(r, c) v'_r: A = the components of v'_r, B = K
//     transposed within its 4 x 4 block (quad permutes); summed over the tile's
//     four row groups by row rotations and stored as the tile's partial sum.
// complex128 takes the 4x4x4 products (v_mfma_f64_4x4x4f64: four blocks, A lane
// (i = l & 3, block (l >> 2) & 3, k = l >> 4), B lane j for i, D lane (j, block,
// i)): register p of a lane holds row 4 p + i, column 4 block + k.  The direct
// products keep one sum per p and add the blocks at the row's end; a product
// with the identity moves a 4 x 4 block from the A to the B layout exactly, and
// the transposed products then sum over all rows in the accumulator.
// The complex64 adjoint sums in FP64 wherever the sweep before it did (solve_tri's
// wide): the same 4x4x4 products on the complex64 tiles, whose layout is the A
// operand of block b & 3 with k = b >> 2, so that a row's direct sum is complete
// in the accumulator and the transposed ones are summed over the row groups by
// row rotations.
// No value is added to by two waves: the thread of (plane, row) adds the row's
// direct sum and its transposed partials in a fixed order.
//
// What bounds it: the chain of dependent blocks per workgroup, and the issue of
// about 60 instructions a tile.  A slot's registers are refilled with the next
// block's tile as soon as they are read, so a whole block (186 KB at 200
// columns) is in flight per CU across the two barriers of a step; the loads do
// not depend on the vector.  Small grids are bound by a step's two barriers, its
// sums and its update, some 0.6 us, so the update's coefficients are fetched and
// its scaling is formed before the products.  At 200^3 a solve takes 1.50 to 1.57
// ms, its 7.84 GB at the rate of a large device copy (the products and barriers
// alone, without the loads: 1.00 ms); at 64^3 0.093 ms, 1.2 us a step.
// complex128 at 200^3 2.87 ms (15.0 GB, 5.2 TB/s), at 140 x 140 x 150 0.92 ms.
// Measured against it: the kernel it replaced at 128, 160, 192 and 200 columns
// (tiles through an LDS ring per wave) 0.55, 0.81, 1.33 and 1.60 ms against
// 0.34, 0.71, 1.23 and 1.55.  Registers: complex64 past 240 columns spills 6, its
// adjoint past 208 columns 2 to 26, nothing else does.
#include <type_traits>

#include "hz_internal.h"
#include "k_plane.h"

namespace hz {
namespace {

constexpr int TRI_MAX_NT = 16;  // up to 256 columns

template <int CTRL>
__device__ __forceinline__ float tri_dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
// a's sum over the lane pairs that CTRL joins where !hi, b's where hi
template <int CTRL>
__device__ __forceinline__ float tri_pair(float a, float b, bool hi) {
  return (hi ? b : a) + tri_dpp<CTRL>(hi ? a : b);
}
template <int CTRL>
__device__ __forceinline__ double tri_dpp(double x) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
template <int CTRL>
__device__ __forceinline__ double tri_pair(double a, double b, bool hi) {
  return (hi ? b : a) + tri_dpp<CTRL>(hi ? a : b);
}
// sum over lane bit 4 (5): a's where the bit is 0, b's where it is 1
__device__ __forceinline__ float tri_sum16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned x = r[0], y = r[1];
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
__device__ __forceinline__ float tri_sum32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned x = r[0], y = r[1];
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
// 4 x 4 transposes within each quad of two matrices: k[c] of lane i becomes
// k[i] of lane c.  One select with a permuted operand per value and stage
// (written out: the compiler takes a move and a select for each); vcc is the
// lanes that keep their own value, first those of even and odd index, then
// those of the quad's lower and upper half.
__device__ __forceinline__ void tri_quad_transpose(float* k, float* l) {
  float a0, a1, a2, a3, b0, b1, b2, b3, c0, c1, c2, c3, d0, d1, d2, d3;
  const unsigned long long even = 0x5555555555555555ull, low = 0x3333333333333333ull;
  asm("s_mov_b64 vcc, %16\n\ts_nop 1\n\t"
      "v_cndmask_b32_dpp %0, %9, %8, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %2, %11, %10, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %4, %13, %12, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %6, %15, %14, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "s_not_b64 vcc, vcc\n\t"
      "v_cndmask_b32_dpp %1, %8, %9, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %3, %10, %11, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %5, %12, %13, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %7, %14, %15, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
      : "=&v"(a0), "=&v"(a1), "=&v"(a2), "=&v"(a3), "=&v"(b0), "=&v"(b1), "=&v"(b2), "=&v"(b3)
      : "v"(k[0]), "v"(k[1]), "v"(k[2]), "v"(k[3]), "v"(l[0]), "v"(l[1]), "v"(l[2]), "v"(l[3]), "s"(even)
      : "vcc", "scc");
  asm("s_mov_b64 vcc, %16\n\ts_nop 1\n\t"
      "v_cndmask_b32_dpp %0, %10, %8, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %1, %11, %9, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %4, %14, %12, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %5, %15, %13, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "s_not_b64 vcc, vcc\n\t"
      "v_cndmask_b32_dpp %2, %8, %10, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %3, %9, %11, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %6, %12, %14, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %7, %13, %15, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf"
      : "=&v"(c0), "=&v"(c1), "=&v"(c2), "=&v"(c3), "=&v"(d0), "=&v"(d1), "=&v"(d2), "=&v"(d3)
      : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "v"(b0), "v"(b1), "v"(b2), "v"(b3), "s"(low)
      : "vcc", "scc");
  k[0] = c0; k[1] = c1; k[2] = c2; k[3] = c3;
  l[0] = d0; l[1] = d1; l[2] = d2; l[3] = d3;
}

// T: the stored factors and vectors, A: the arithmetic
template <typename T, typename A, int NT>
struct TriShape {
  static constexpr int NW = (NT + 1) / 2;  // waves: tile rows w and w + NW (the last wave of an odd NT: one row)
  static constexpr int NA = NT / 2 + 1;    // tiles of row w
  static constexpr int NB = NT - NT / 2;   // tiles of row w + NW
  static constexpr int NS = NA + NB;       // NT + 1
  // up to 4 tile rows: a wave for each row, NA tiles each (a row of NB < NA: its
  // last one is dead), so that the four SIMDs of a compute unit share them.
  // 48^3 0.081 -> 0.063 ms, 64^3 0.114 -> 0.094, x 7 0.172 -> 0.133; complex128
  // 64^3 0.145 -> 0.109.  Past 4 the SIMDs have no fewer tiles each: one vector
  // gained (96^3 0.206 -> 0.195, 112^3 0.274 -> 0.229), but several on a compute
  // unit lost (96^3 x 4 0.32 -> 0.38, 128^3 x 4 0.74 -> 0.86).
  static constexpr bool SPLIT = NT <= 4;
  static constexpr int WAVES = SPLIT ? NT : NW;
  static constexpr int NSW = SPLIT ? NA : NS;  // tiles a wave
  static constexpr int THREADS = 64 * WAVES;   // >= 2 * 16 NT: one thread per (plane, row) in the update
  static constexpr int NP = 64 * ((16 * NT - 16 + 63) / 64) + 16;  // values a component: 16 mod 64, the four
                                                                   // components' reads fall in distinct banks
  // tiles in flight a wave: a whole block's, or (complex128, whose tiles take
  // 16 registers) a half or a third of them where they would not fit
  static constexpr int RD = sizeof(T) == 4 || NS <= 9 ? NSW : NS <= 10 ? (NS + 1) / 2 : (NS + 2) / 3;
  static constexpr int NSR = (NSW + RD - 1) / RD * RD;  // slots of a block, the last possibly empty
  static constexpr size_t lds = sizeof(A) * (8 * (size_t)NP + 64 * ((size_t)(NT + 1) * NA + NT + 1));
};

template <typename T, typename A, int NT, int PH, bool ADJ>
__global__ __launch_bounds__((TriShape<T, A, NT>::THREADS)) void k_solve_tri(
    const typename Cx<T>::t* __restrict__ P, typename Cx<T>::t* __restrict__ X, const double2* __restrict__ cmy,
    const double2* __restrict__ cpy, const double2* __restrict__ symd, int n, int ny, int m, int nz, int64_t n2,
    int64_t N, const int2* __restrict__ slotp, int nslot, int nrhs, typename Cx<T>::t* __restrict__ scr) {
  typedef typename Cx<T>::t C;
  typedef typename Cx<A>::t CA;
  typedef TriShape<T, A, NT> S;
  constexpr bool F32 = sizeof(T) == 4, A32 = sizeof(A) == 4;
  constexpr int NP = S::NP;
  constexpr int BS = NT * (NT + 1) / 2 * 256;  // complex values of a packed block
  extern __shared__ __align__(16) unsigned char smem_raw[];
  A* const vq = reinterpret_cast<A*>(smem_raw);  // [4][NP] components of v'
  A* const vr = vq + 4 * NP;                     // [4][NP] rotated: (-Im A, Re A, -Im B, Re B)
  A* const dsum = vr + 4 * NP;                   // [NT + 1][2][16][2] direct sums (plane, row, re/im)
  A* const tsum = dsum + 64 * (NT + 1);          // [C][d][2][16][2] transposed sums of tile (C - d, C)
                                                 // (the last of either: sums nobody reads)

  // Workgroups go to the 8 XCDs in turn: the right-hand sides of one (slot,
  // half) take every eighth place, so they run side by side on one XCD and
  // share its L2's copy of the blocks.
  const int place = blockIdx.x >> 3, pair = place / nrhs * 8 + (blockIdx.x & 7);
  const int slot = pair >> 1, half = pair & 1;
  if (slot >= nslot) return;
  const int2 sp = slotp[slot];
  const bool twoB = sp.y >= 0;
  const int64_t rhs = place % nrhs;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bi = lane >> 2, qi = lane & 3, rg = bi & 3, cg = bi >> 2;
  const bool b2 = lane & 4, b3 = lane & 8;
  const C* const Pk = P + (size_t)slot * ny * BS;
  const double2 *dx = symd, *dy = symd + n, *dxi = symd + n + ny, *dyi = symd + 2 * n + ny;
  const int nsteps = PH == 0 ? (half == 0 ? m : ny - 1 - m) : (half == 0 ? m + 1 : ny - m);
  auto blk_of = [&](int st) {
    if (PH == 0) return half == 0 ? st : ny - 1 - st;
    return half == 0 ? m - st : m + st;
  };
  // block whose vector the update after step st forms (-1: none; -2: y goes to scr)
  auto next_of = [&](int st) {
    const int jb = blk_of(st);
    if (PH == 0) {
      if (half == 0) return jb + 1 < m ? jb + 1 : -2;
      return jb - 1 > m ? jb - 1 : -2;
    }
    if (half == 0) return jb > 0 ? jb - 1 : -1;
    return jb < ny - 1 ? jb + 1 : -1;
  };
  // ---- the thread's (plane, row) of the updates
  const bool row_ok = tid < 2 * n;
  const int ps = tid >= n ? 1 : 0, pr = row_ok ? tid - ps * n : 0;
  const int pl = ps && twoB ? sp.y : sp.x;
  const bool wr = row_ok && (ps == 0 || twoB);
  C* const xs = X + rhs * N + (int64_t)pl * n2 + pr;
  // scr: [what][rhs][plane][n], what = 0 y_top, 1 y_bot, 2 f_m
  auto scr_at = [&](int what) { return scr + (((int64_t)what * nrhs + rhs) * nz + pl) * n + pr; };
  const double2 dxr = dx[pr], dxir = dxi[pr];
  auto cmul_d = [](double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); };
  // Values of the lines' tables are fetched a step ahead by vector loads: scalar
  // loads would be waited for with the step's first LDS reads.
  int vz;
  asm("v_mov_b32 %0, 0" : "=v"(vz));
  // a line value of the right-hand side: f, or D conj(f) for the adjoint
  auto load_f = [&](C f, double2 dyj) {
    if (!ADJ) return f;
    const double2 d = cmul_d(dxr, dyj);
    const double2 v = cmul_d(make_double2(f.x, -(double)f.y), d);
    return mk<C>(v.x, v.y);
  };

  if (PH == 0 && half == 0 && wr) *scr_at(2) = load_f(xs[(int64_t)m * n], dy[m]);
  if (nsteps <= 0) return;

  // ---- this wave's tiles: NA of row ra, NB of row rb.  (The last wave of an
  // odd NT has no second row: it computes some row's first tiles once more,
  // into sums that nobody reads.)
  const int ra = w, rb = w + S::NW < NT ? w + S::NW : w;
  const bool spare = S::SPLIT ? w >= S::NW && S::NB < S::NA : w + S::NW >= NT;
  // the first slot of a wave that holds no tile of its own, where spare
  constexpr int SP0 = S::SPLIT ? S::NB : S::NA;
  constexpr int UL = F32 ? 2 : 1, UQ = F32 ? 2 : 4;  // complex values a unit, units a lane and tile
  const C* const tiles =
      Pk + (S::SPLIT && w >= S::NW ? (size_t)(w - S::NW) * S::NS + S::NA : (size_t)w * S::NS) * 256 + UL * lane;
  struct alignas(16) Unit { C c[UL]; };
  Unit q[S::RD][UQ];
  // (no branch around a load: with one, the compiler cannot count the younger
  // loads in flight and waits for all of them before each tile)
  auto load_slot = [&](int t, const C* blk) {
    const C* const a = blk + (spare && t >= SP0 ? t - SP0 : t) * 256;
#pragma unroll
    for (int u = 0; u < UQ; ++u) q[t % S::RD][u] = *reinterpret_cast<const Unit*>(a + u * 64 * UL);
  };
  {
    const C* const blk = tiles + (size_t)blk_of(0) * BS;
#pragma unroll
    for (int t = 0; t < S::RD; ++t) {
      load_slot(t, blk);
      __builtin_amdgcn_sched_barrier(0);  // in the order of use, as in the steps: the waits count on it
    }
  }

  // ---- v' of the first block
  for (int e = tid; e < 8 * NP; e += S::THREADS) vq[e] = (A)0;
  __syncthreads();
  auto put_v = [&](double2 v) {  // v' = D^-1 v of this thread's row
    const A a = (A)v.x, b = (A)v.y;
    vq[(2 * ps) * NP + pr] = a;
    vq[(2 * ps + 1) * NP + pr] = b;
    vr[(2 * ps) * NP + pr] = -b;
    vr[(2 * ps + 1) * NP + pr] = a;
  };
  if (row_ok) {
    const int j0 = blk_of(0);
    double2 f;
    if (PH == 0) {
      const C v = load_f(xs[(int64_t)j0 * n], dy[j0]);
      if (ADJ && wr) xs[(int64_t)j0 * n] = v;
      f = make_double2(v.x, v.y);
    } else {
      const C v = *scr_at(2);
      f = make_double2(v.x, v.y);
      if (m > 0) {
        const C y = *scr_at(0);
        const double2 t = cmul_d(cmy[m], make_double2(y.x, y.y));
        f.x -= t.x;
        f.y -= t.y;
      }
      if (m < ny - 1) {
        const C y = *scr_at(1);
        const double2 t = cmul_d(cpy[m], make_double2(y.x, y.y));
        f.x -= t.x;
        f.y -= t.y;
      }
    }
    put_v(cmul_d(f, cmul_d(dxir, dyi[j0])));
  }
  __syncthreads();

  // what the update after step st takes of its next line jn: the line's value,
  // its coefficient, 1 / dy(jn) and (adjoint, first phase) dy(jn)
  struct Line { C f; double2 cf, di, d; };
  const bool lower = PH == 0 ? half == 0 : half != 0;
  auto fetch = [&](int st) {
    const int jn = next_of(st), j = jn >= 0 ? jn : blk_of(st);
    Line l;
    l.f = xs[(int64_t)j * n];
    l.cf = (lower ? cmy : cpy)[j + vz];
    l.di = dyi[j + vz];
    if (ADJ && PH == 0) l.d = dy[j + vz];
    return l;
  };
  Line line = fetch(0);
  double2 sb = cmul_d(dxir, dyi[blk_of(0)]);  // D^-1 of this row, block jb

  for (int st = 0; st < nsteps; ++st) {
    const int jb = blk_of(st), jn = next_of(st);
    const C* const cblk = tiles + (size_t)jb * BS;
    const C* const nblk = tiles + (size_t)blk_of(st + 1 < nsteps ? st + 1 : st) * BS;
    // the slot that takes tile t's registers (past the empty slots of a block,
    // the next block's)
    auto reload = [&](int t) {
      int u = t + S::RD;
      if (u < S::NSW) {
        load_slot(u, cblk);
      } else {
        if (u < S::NSR) u += S::RD;
        load_slot(u - S::NSR, nblk);
      }
    };
    auto col_of = [&](int t) {
      // a dead tile: the vector's zeros past the last column
      if (S::SPLIT && spare && t >= SP0) return NP / 16 - 1;
      const int c = t < S::NA ? ra + t : rb + t - S::NA;
      return c < NT ? c : c - NT;
    };
    // v' = D^-1 (f - cf y), all but y known before the products.  (The difference
    // first, as it is stored: with D^-1 f and D^-1 cf formed ahead both sides of
    // it round, and v' is not D^-1 of the stored line.)
    const C f = PH == 0 ? load_f(line.f, line.d) : line.f;
    const double2 cf = line.cf, sn = cmul_d(dxir, line.di);
    line = fetch(st + 1 < nsteps ? st + 1 : st);

    if constexpr (A32) {
      // Software pipeline over the tiles, one scheduling region each: tile t's
      // direct products, transposes and reload, tile t - 1's transposed products
      // and tile t - 2's sum over the row groups.  (Without the fences the
      // compiler moves the reloads to the end of the step.)
      const hz_v4f z4 = {0.f, 0.f, 0.f, 0.f};
      hz_v4f da0 = z4, da1 = z4, db0 = z4, db1 = z4;  // direct sums of rows ra, rb
      // components of the rows' v' (A operands of the transposed products)
      const float4 va = *reinterpret_cast<const float4*>(vq + qi * NP + 16 * ra + 4 * rg);
      const float4 vb = *reinterpret_cast<const float4*>(vr + qi * NP + 16 * ra + 4 * rg);
      const float4 wa = *reinterpret_cast<const float4*>(vq + qi * NP + 16 * rb + 4 * rg);
      const float4 wb = *reinterpret_cast<const float4*>(vr + qi * NP + 16 * rb + 4 * rg);
      float tk[2][8];
      hz_v4f ts[2];
      float4 cv[2], cr[2];  // components of the tile column's v', one tile ahead
      auto load_col = [&](int t) {
        const int at = qi * NP + 16 * col_of(t) + 4 * cg;
        cv[t & 1] = *reinterpret_cast<const float4*>(vq + at);
        cr[t & 1] = *reinterpret_cast<const float4*>(vr + at);
      };
      load_col(0);
  #pragma unroll
      for (int t = 0; t < S::NSW + 2; ++t) {
        if (t + 1 < S::NSW) load_col(t + 1);
        if (t < S::NSW) {
          float kr[4], ki[4];
  #pragma unroll
          for (int i = 0; i < 4; ++i) {
            kr[i] = q[t][i / 2].c[i % UL].x;
            ki[i] = q[t][i / 2].c[i % UL].y;
          }
          const float4 u = cv[t & 1], v = cr[t & 1];
          hz_v4f& d0 = t < S::NA ? da0 : db0;
          hz_v4f& d1 = t < S::NA ? da1 : db1;
          d0 = __builtin_amdgcn_mfma_f32_4x4x1f32(kr[0], u.x, d0, 0, 0, 0);
          d1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ki[0], v.x, d1, 0, 0, 0);
          d0 = __builtin_amdgcn_mfma_f32_4x4x1f32(kr[1], u.y, d0, 0, 0, 0);
          d1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ki[1], v.y, d1, 0, 0, 0);
          d0 = __builtin_amdgcn_mfma_f32_4x4x1f32(kr[2], u.z, d0, 0, 0, 0);
          d1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ki[2], v.z, d1, 0, 0, 0);
          d0 = __builtin_amdgcn_mfma_f32_4x4x1f32(kr[3], u.w, d0, 0, 0, 0);
          d1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ki[3], v.w, d1, 0, 0, 0);
          tri_quad_transpose(kr, ki);
  #pragma unroll
          for (int i = 0; i < 4; ++i) {
            tk[t & 1][i] = kr[i];
            tk[t & 1][4 + i] = ki[i];
          }
          reload(t);
        }
        if (t >= 1 && t <= S::NSW) {
          const int u = t - 1;
          const float4 a = u < S::NA ? va : wa, b = u < S::NA ? vb : wb;
          // the diagonal tiles' own 4 x 4 blocks have no transposed product
          // (their lower blocks are stored as zeros)
          const bool off = (u != 0 && u != S::NA) || cg > rg;
          const float av[4] = {off ? a.x : 0.f, off ? a.y : 0.f, off ? a.z : 0.f, off ? a.w : 0.f};
          const float bv[4] = {off ? b.x : 0.f, off ? b.y : 0.f, off ? b.z : 0.f, off ? b.w : 0.f};
          hz_v4f x = z4;
  #pragma unroll
          for (int i = 0; i < 4; ++i) {
            x = __builtin_amdgcn_mfma_f32_4x4x1f32(av[i], tk[u & 1][i], x, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_4x4x1f32(bv[i], tk[u & 1][4 + i], x, 0, 0, 0);
          }
          ts[u & 1] = x;
        }
        if (t >= 2) {
          // lane (rg, cg, j) gets component rg of column 4 cg + j
          const int u = t - 2;
          const hz_v4f x = ts[u & 1];
          const float s = tri_pair<0x128>(tri_pair<0x124>(x[0], x[1], b2), tri_pair<0x124>(x[2], x[3], b2), b3);
          const int d = u < S::NA ? u : u - S::NA, at = u < SP0 || !spare ? col_of(u) : NT;
          tsum[64 * (at * S::NA + d) + (rg >> 1) * 32 + (4 * cg + qi) * 2 + (rg & 1)] = s;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // the direct sums over the column groups (lane bits 4, 5)
      {
        const hz_v4f a = da0 + da1, b = db0 + db1;
        const int at = (qi >> 1) * 32 + (4 * rg + cg) * 2 + (qi & 1);
        dsum[64 * ra + at] = tri_sum32(tri_sum16(a[0], a[1]), tri_sum16(a[2], a[3]));
        if (!S::SPLIT) dsum[64 * (spare ? NT : rb) + at] = tri_sum32(tri_sum16(b[0], b[1]), tri_sum16(b[2], b[3]));
      }
    } else if constexpr (F32) {
      // complex64 tiles, sums in FP64: register e of a lane holds column 4 cg + e
      // of row 4 rg + qi, the A operand of block rg (k = cg) as it lies.
      const int i4 = lane >> 4;                  // k of an operand, i of a result
      const double one = i4 == qi ? 1.0 : 0.0;  // the identity, as B operand
      double va, vb, dp;
      auto row_operands = [&](int R) {
        va = vq[qi * NP + 16 * R + 4 * rg + i4];
        vb = vr[qi * NP + 16 * R + 4 * rg + i4];
        dp = 0.0;
      };
      auto flush_row = [&](int out) { dsum[64 * out + (qi >> 1) * 32 + (4 * rg + i4) * 2 + (qi & 1)] = dp; };
      row_operands(ra);
#pragma unroll
      for (int t = 0; t < S::NSW; ++t) {
        if (t == S::NA) {
          flush_row(ra);
          row_operands(rb);
        }
        const int cc = col_of(t), d = t < S::NA ? t : t - S::NA;
        const int at0 = qi * NP + 16 * cc + 4 * cg;
        const double2 u0 = *reinterpret_cast<const double2*>(vq + at0), u1 = *reinterpret_cast<const double2*>(vq + at0 + 2);
        const double2 w0 = *reinterpret_cast<const double2*>(vr + at0), w1 = *reinterpret_cast<const double2*>(vr + at0 + 2);
        const double u[4] = {u0.x, u0.y, u1.x, u1.y}, v[4] = {w0.x, w0.y, w1.x, w1.y};
        double kr[4], ki[4], x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const C k = q[t % S::RD][e / UL].c[e % UL];
          dp = __builtin_amdgcn_mfma_f64_4x4x4f64((double)k.x, u[e], dp, 0, 0, 0);
          kr[e] = __builtin_amdgcn_mfma_f64_4x4x4f64((double)k.x, one, 0.0, 0, 0, 0);
          dp = __builtin_amdgcn_mfma_f64_4x4x4f64((double)k.y, v[e], dp, 0, 0, 0);
          ki[e] = __builtin_amdgcn_mfma_f64_4x4x4f64((double)k.y, one, 0.0, 0, 0, 0);
        }
        reload(t);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] = __builtin_amdgcn_mfma_f64_4x4x4f64(va, kr[e], 0.0, 0, 0, 0);
          x[e] = __builtin_amdgcn_mfma_f64_4x4x4f64(vb, ki[e], x[e], 0, 0, 0);
          // the diagonal tile's own 4 x 4 blocks have no transposed product
          // (its lower blocks are stored as zeros)
          if (d == 0) x[e] = qi > rg ? x[e] : 0.0;
        }
        // sum over the row groups (lane bits 2, 3): group b gets the columns 4 j + b
        const double xs4 = tri_pair<0x128>(tri_pair<0x124>(x[0], x[1], b2), tri_pair<0x124>(x[2], x[3], b2), b3);
        const int at = t < SP0 || !spare ? cc : NT;
        tsum[64 * (at * S::NA + d) + (i4 >> 1) * 32 + (4 * qi + rg) * 2 + (i4 & 1)] = xs4;
        __builtin_amdgcn_sched_barrier(0);  // the reloads stay in order
      }
      flush_row(S::SPLIT ? ra : spare ? NT : rb);
    } else {
      const int i4 = lane >> 4;  // k of an operand, i of a result
      const double one = i4 == qi ? 1.0 : 0.0;  // the identity, as B operand
      double va[4], vb[4], dp[4];
      auto row_operands = [&](int R) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          va[p] = vq[qi * NP + 16 * R + 4 * p + i4];
          vb[p] = vr[qi * NP + 16 * R + 4 * p + i4];
          dp[p] = 0.0;
        }
      };
      // sum over the blocks (lane bits 2, 3): block b gets the rows 4 b ..
      auto flush_row = [&](int out) {
        const double s = tri_pair<0x128>(tri_pair<0x124>(dp[0], dp[1], b2), tri_pair<0x124>(dp[2], dp[3], b2), b3);
        dsum[64 * out + (qi >> 1) * 32 + (4 * rg + i4) * 2 + (qi & 1)] = s;
      };
      row_operands(ra);
#pragma unroll
      for (int t = 0; t < S::NSW; ++t) {
        if (t == S::NA) {
          flush_row(ra);
          row_operands(rb);
        }
        const int cc = col_of(t), d = t < S::NA ? t : t - S::NA;
        const double u = vq[qi * NP + 16 * cc + 4 * rg + i4], v = vr[qi * NP + 16 * cc + 4 * rg + i4];
        double kr[4], ki[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const C k = q[t % S::RD][p].c[0];
          dp[p] = __builtin_amdgcn_mfma_f64_4x4x4f64(k.x, u, dp[p], 0, 0, 0);
          kr[p] = __builtin_amdgcn_mfma_f64_4x4x4f64(k.x, one, 0.0, 0, 0, 0);
          dp[p] = __builtin_amdgcn_mfma_f64_4x4x4f64(k.y, v, dp[p], 0, 0, 0);
          ki[p] = __builtin_amdgcn_mfma_f64_4x4x4f64(k.y, one, 0.0, 0, 0, 0);
        }
        reload(t);
        double x = 0.0;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          // the diagonal tile's own 4 x 4 blocks have no transposed product
          // (its lower blocks are stored as zeros)
          const bool off = d > 0 || rg > p;
          x = __builtin_amdgcn_mfma_f64_4x4x4f64(off ? va[p] : 0.0, kr[p], x, 0, 0, 0);
          x = __builtin_amdgcn_mfma_f64_4x4x4f64(off ? vb[p] : 0.0, ki[p], x, 0, 0, 0);
        }
        const int at = t < SP0 || !spare ? cc : NT;
        tsum[64 * (at * S::NA + d) + (i4 >> 1) * 32 + (4 * rg + qi) * 2 + (i4 & 1)] = x;
        __builtin_amdgcn_sched_barrier(0);  // the reloads stay in order
      }
      flush_row(S::SPLIT ? ra : spare ? NT : rb);
    }
    __syncthreads();

    if (row_ok) {
      const int rt = pr >> 4, at = ps * 32 + (pr & 15) * 2;
      CA y = *reinterpret_cast<const CA*>(dsum + 64 * rt + at);
#pragma unroll
      for (int d = 0; d < S::NA; ++d) {
        const CA u = *reinterpret_cast<const CA*>(tsum + 64 * (rt * S::NA + d) + at);
        // even NT: tile (C - NT/2, C) is kept where C - NT/2 is below NT/2
        const bool kept = NT % 2 != 0 || d < NT / 2 || rt >= NT / 2;
        y.x += kept ? u.x : (A)0;
        y.y += kept ? u.y : (A)0;
      }
      const double2 v = make_double2(f.x - (cf.x * y.x - cf.y * y.y), f.y - (cf.x * y.y + cf.y * y.x));
      if (jn >= 0) put_v(cmul_d(v, sn));
      if (wr && PH == 1 && (half == 0 || st > 0)) {  // x_jb
        C o = mk<C>(y.x, y.y);
        if (ADJ) {
          const double2 z = cmul_d(make_double2(y.x, y.y), sb);
          o = mk<C>(z.x, -z.y);
        }
        xs[(int64_t)jb * n] = o;
      }
      if (wr && jn == -2) *scr_at(half) = mk<C>(y.x, y.y);                 // y_top / y_bot
      if (wr && PH == 0 && jn >= 0) xs[(int64_t)jn * n] = mk<C>(v.x, v.y);  // t_jn / b_jn
    }
    sb = sn;
    __syncthreads();
  }
}

// Packed blocks of the slots' twisted chains: tile blockIdx.x of block
// blockIdx.y = slot ny + j, X_j from G (j < m) or Gb (j >= m), times D_j.
template <typename T>
__global__ __launch_bounds__(256) void k_pack_tri(const typename Cx<T>::t* __restrict__ G,
                                                  const typename Cx<T>::t* __restrict__ Gb,
                                                  typename Cx<T>::t* __restrict__ P, const double2* __restrict__ dx,
                                                  const double2* __restrict__ dy, int n, int ny, int m, int nt) {
  typedef typename Cx<T>::t C;
  __shared__ C v[16][17];
  const int j = blockIdx.y % ny, slot = blockIdx.y / ny, tid = threadIdx.x;
  const size_t nn = (size_t)n * n;
  const C* const B = j >= m ? Gb + ((size_t)slot * (ny - m) + (j - m)) * nn : G + ((size_t)slot * ny + j) * nn;
  // slot t of wave w: tile row w, then tile row w + nw
  const int nw = (nt + 1) / 2, na = nt / 2 + 1;
  const int w = blockIdx.x / (nt + 1), t = blockIdx.x - w * (nt + 1);
  const int R = t < na ? w : w + nw, d = t < na ? t : t - na, c0 = R + d < nt ? R + d : R + d - nt;
  {
    const int r = tid & 15, c = tid >> 4, gr = 16 * R + r, gc = 16 * c0 + c;
    C o = mk<C>(0.0, 0.0);
    if (gr < n && gc < n && (R != c0 || r / 4 <= c / 4)) {
      // K(r, c) = K(c, r) from the lower triangle: the elimination leaves more
      // error in the upper one where the layers are thick (64 x 12 x 12 with four
      // layer points a side, numpy: error of a solve from the whole K, its lower
      // and its upper triangle 2.1e-6, 2.1e-6 and 3.5e-6 complex64, 5.5e-15,
      // 5.5e-15 and 7.2e-15 complex128)
      const int ur = max(gr, gc), uc = min(gr, gc);
      const C g = B[ur + (size_t)n * uc];
      const double2 a = dx[uc], b = dy[j];
      const double sx = a.x * b.x - a.y * b.y, sy = a.x * b.y + a.y * b.x;
      o = mk<C>((double)g.x * sx - (double)g.y * sy, (double)g.x * sy + (double)g.y * sx);
    }
    v[c][r] = o;
  }
  __syncthreads();
  int r, c;
  if (sizeof(T) == 4) {
    const int h = tid >> 7, l = (tid >> 1) & 63, e = tid & 1;
    r = 4 * ((l >> 2) & 3) + (l & 3);
    c = 4 * (l >> 4) + 2 * h + e;
  } else {
    const int p = tid >> 6, l = tid & 63;
    r = 4 * p + (l & 3);
    c = 4 * ((l >> 2) & 3) + (l >> 4);
  }
  P[((size_t)blockIdx.y * (nt * (nt + 1) / 2) + blockIdx.x) * 256 + tid] = v[c][r];
}

template <typename T>
void pack_tri_t(hz_problem* p, int prec, hipStream_t s) {
  typedef typename Cx<T>::t C;
  Factors& f = p->fac[prec];
  const int nt = ((int)p->nx + 15) / 16, tiles = nt * (nt + 1) / 2;
  const double2* dx = p->d_symd.as<double2>();
  // at most 65535 blocks a launch in the second grid dimension
  const int per = 32768 / (int)p->ny > 0 ? 32768 / (int)p->ny : 1;
  for (int s0 = 0; s0 < p->nslot; s0 += per) {
    const int ns = std::min(per, p->nslot - s0);
    hipLaunchKernelGGL(k_pack_tri<T>, dim3((unsigned)tiles, (unsigned)(ns * p->ny)), dim3(256), 0, s,
                       f.G.as<C>() + (size_t)s0 * p->ny * p->nx * p->nx,
                       f.Gb.as<C>() + (size_t)s0 * (p->ny - f.tw_m) * p->nx * p->nx,
                       f.Gtw.as<C>() + (size_t)s0 * p->ny * tiles * 256, dx, dx + p->nx, (int)p->nx, (int)p->ny,
                       f.tw_m, nt);
    HZ_HIP(hipGetLastError());
  }
}

template <typename T, typename A, int NT, bool ADJ>
void launch_tri(hz_problem* p, int prec, int nrhs, void* xv, hipStream_t s) {
  typedef typename Cx<T>::t C;
  const Factors& f = p->fac[prec];
  C* const x = (C*)xv;
  constexpr size_t lds = TriShape<T, A, NT>::lds;
  static_assert(lds <= 160 * 1024, "LDS");
  set_max_lds((const void*)&k_solve_tri<T, A, NT, 0, ADJ>, lds);
  set_max_lds((const void*)&k_solve_tri<T, A, NT, 1, ADJ>, lds);
  for (int r0 = 0; r0 < nrhs; r0 += TW_RHS) {
    const int nr = std::min(TW_RHS, nrhs - r0);
    const dim3 grid((unsigned)((2 * p->nslot + 7) / 8 * 8 * nr)), block(TriShape<T, A, NT>::THREADS);
    C* const xr = x + (size_t)r0 * p->N;
    hipLaunchKernelGGL((k_solve_tri<T, A, NT, 0, ADJ>), grid, block, lds, s, f.Gtw.as<C>(), xr, p->tab(1, 0),
                       p->tab(1, 1), p->d_symd.as<double2>(), (int)p->nx, (int)p->ny, f.tw_m, (int)p->nz, p->n2, p->N,
                       p->d_slotp.as<int2>(), p->nslot, nr, f.tw_scr.as<C>());
    hipLaunchKernelGGL((k_solve_tri<T, A, NT, 1, ADJ>), grid, block, lds, s, f.Gtw.as<C>(), xr, p->tab(1, 0),
                       p->tab(1, 1), p->d_symd.as<double2>(), (int)p->nx, (int)p->ny, f.tw_m, (int)p->nz, p->n2, p->N,
                       p->d_slotp.as<int2>(), p->nslot, nr, f.tw_scr.as<C>());
    HZ_HIP(hipGetLastError());
  }
}

template <typename T, typename A, bool ADJ>
void solve_tri_t(hz_problem* p, int prec, int nrhs, void* x, hipStream_t s) {
  const int nt = ((int)p->nx + 15) / 16;
#define HZ_TRI(NT) \
  if (nt == NT) return launch_tri<T, A, NT, ADJ>(p, prec, nrhs, x, s);
  // complex64 adjoint: FP64 sums to TRI_WIDE_MAX columns, FP32 sums past them and
  // at 64, 96 and 128
  constexpr bool WIDE = ADJ && sizeof(T) != sizeof(A), C64ADJ = ADJ && sizeof(T) == 4;
  HZ_TRI(4) HZ_TRI(6) HZ_TRI(8)
  if constexpr (!C64ADJ || WIDE) {
    HZ_TRI(1) HZ_TRI(2) HZ_TRI(3) HZ_TRI(5) HZ_TRI(7) HZ_TRI(9)
  }
  if constexpr (!WIDE) {
    static_assert(TRI_WIDE_MAX == 16 * 9, "");
    HZ_TRI(10) HZ_TRI(11) HZ_TRI(12) HZ_TRI(13) HZ_TRI(14) HZ_TRI(15) HZ_TRI(16)
  }
#undef HZ_TRI
  HZ_CHECK(false, HZ_ERR_ARG, "nx=%d", (int)p->nx);
}

}  // namespace

bool tri_available(int nx) { return nx <= 16 * TRI_MAX_NT; }

size_t tri_bytes(const hz_problem* p, size_t elem) {
  const size_t nt = ((size_t)p->nx + 15) / 16;
  return (size_t)p->nslot * p->ny * (nt * (nt + 1) / 2) * 256 * elem;
}

void pack_tri(hz_problem* p, int prec, hipStream_t s) {
  if (prec == HZ_PREC_FP64) pack_tri_t<double>(p, prec, s);
  else pack_tri_t<float>(p, prec, s);
}

void solve_tri(hz_problem* p, int prec, int nrhs, void* x, bool adjoint, bool wide, hipStream_t s) {
  if (prec == HZ_PREC_FP64) {
    if (adjoint) solve_tri_t<double, double, true>(p, prec, nrhs, x, s);
    else solve_tri_t<double, double, false>(p, prec, nrhs, x, s);
  } else if (adjoint) {
    if (wide) solve_tri_t<float, double, true>(p, prec, nrhs, x, s);
    else solve_tri_t<float, float, true>(p, prec, nrhs, x, s);
  } else {
    solve_tri_t<float, float, false>(p, prec, nrhs, x, s);
  }
}

}  // namespace hz
