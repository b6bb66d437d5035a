// k_rows.hip -- complex64 plane solves of groups of 8 right-hand sides, blocks
// read from memory straight into the matrix products.
//
// One-directional: the sweep of the other such kernels (t_{j+1} = b_{j+1} -
// cm_y(j+1) G_j t_j up, x_j = G_j (t_j - cp_y(j) x_{j+1}) down, 2 ny - 1 block
// products), one workgroup per plane and group.  Twisted: the two phases of
// k_tri.hip on the dense blocks, a workgroup per plane, end and group, ny / 2
// products a phase.  Adjoint: with D = diag(dx(i) dy(j)), M^H x = b is the forward
// solve M z = D conj(b), x = conj(D^-1 z).
//
// Wave w computes the tile rows w and w + 8 of every product.  A 16 x 16 tile of
// the column-major block is loaded once, by the one wave that needs it, in the
// operand order of v_mfma_f32_16x16x4f32: lane l holds row l & 15 and the
// columns 4 (l >> 4) .. + 3, 8 bytes a load along the rows.  The 16 result
// columns are the real and imaginary parts of the 8 vectors:
//   [Re Y | Im Y] += Re(G) [Re V | Im V] + Im(G) [-Im V | Re V].
// A wave's rows are complete in its own accumulators, so the update of the next
// vector needs no sums between waves: it is written to the other of two LDS
// buffers and a step has one barrier.  The adjoint to TRI_WIDE_MAX columns
// multiplies and sums in FP64 (A = double: v_mfma_f64_16x16x4f64, the same
// operand order; a lane's result rows are four apart instead of neighbours).
//
// What bounds it: the chain of steps, and below them the matrix products and the
// blocks' bytes.  The two planes of a factor slot and the groups of right-hand
// sides run side by side on one XCD and share its L2's copy of a block.  A wave
// keeps 12 tiles (24 KB) in flight; their registers are refilled as soon as they
// are read, and the loads do not depend on the vector.  A lane finishes two whole
// entries of the next vector after one exchange with the lane 8 away; with one
// component of four rows a lane a step took 0.25 us more (4.45 -> 4.2 at 128
// columns, 9.7 -> 9.0 at 192).  Measured, in ms, one-directional, blocks staged
// through LDS before -> now: 128^3 x 8 1.08 -> 1.07, x 16 1.24 -> 1.14, 160^3 x 8
// 3.37 -> 2.05, 192^3 x 8 5.03 -> 3.46, 200^3 x 8 6.16 -> 4.65.  Twisted, with half
// the steps, against one-directional at 60 lines: 96 x 64 planes x 16 0.166 / 0.275,
// 112 x 64 x 8 0.187 / 0.316, 140 x 96 x 8 0.361 / 0.616, 208 x 64 x 8 0.669 / 1.17;
// up to 112 columns two workgroups fit a compute unit.  Where the planes and
// groups of one end just fill the chip (256 workgroups; 140 x 96 x 16 0.690 /
// 0.614) the second end waits for a place and the full chain would be 3 to 11%
// faster.  FP64 sums take 1.3 to 1.65 times as long (140 x 96 x 8 0.515).
#include <algorithm>
#include <type_traits>

#include "hz_internal.h"
#include "k_plane.h"

namespace hz {
namespace {

constexpr int ROWS_MAX_NT = 16;  // up to 256 columns

// lane n ^ 8 within 16
__device__ __forceinline__ int rows_ror8(int x) { return __builtin_amdgcn_update_dpp(x, x, 0x128, 0xF, 0xF, false); }
__device__ __forceinline__ float rows_ror8(float x) { return __builtin_bit_cast(float, rows_ror8(__builtin_bit_cast(int, x))); }
__device__ __forceinline__ double rows_ror8(double x) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = rows_ror8((int)b), hi = rows_ror8((int)(b >> 32));
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

// the products' arithmetic: result type, and the tile row of a lane's result i
template <typename A> struct RowsMath;
template <> struct RowsMath<float> {
  typedef hz_v4f V;
  __device__ static __forceinline__ V mfma(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int kg, int i) { return 4 * kg + i; }
};
template <> struct RowsMath<double> {
  typedef hz_v4d V;
  __device__ static __forceinline__ V mfma(float a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64((double)a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int kg, int i) { return 4 * i + kg; }
};

template <typename A, int NT>
struct RowsShape {
  static constexpr int NWV = NT < 8 ? NT : 8;
  static constexpr int VB = 16 * NT * 16;  // values of one vector buffer (plain or rotated)
  static constexpr size_t lds(bool adj) { return sizeof(A) * 4 * VB + (adj ? sizeof(double2) * 32 * NT : 0); }
};

// PH -1: one-directional, blocks G ([slot][j]).  PH 0, 1: the phases of a twisted
// solve (k_tri.hip), blocks j < m from G, j >= m from Gb ([slot][j - m]); y_top,
// y_bot and f_m pass between them in scr.
template <typename A, int NT, int PH, bool ADJ>
__global__ __launch_bounds__(64 * (NT < 8 ? NT : 8)) void k_solve_rows(
    const float2* __restrict__ G, const float2* __restrict__ Gb, float2* __restrict__ X,
    const double2* __restrict__ cmy, const double2* __restrict__ cpy, const double2* __restrict__ symd, int n, int ny,
    int m, int nz, int64_t n2, int64_t N, const int2* __restrict__ two, int ntwo, const int* __restrict__ fmap,
    int nrhs, int ngroups, float2* __restrict__ scr) {
  typedef float2 C;
  typedef RowsShape<A, NT> S;
  typedef RowsMath<A> M;
  typedef typename M::V V;
  constexpr bool TW = PH >= 0;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  // vector buffers [2][plain, rotated][c / 4][16 columns][c % 4]
  A* const vb = reinterpret_cast<A*>(smem_raw);
  double2* const sdx = reinterpret_cast<double2*>(vb + 4 * S::VB);  // adjoint: dx, 1 / dx
  double2* const sdxi = sdx + 16 * NT;

  // Workgroups go to the 8 XCDs in turn: the planes and groups of one slot take
  // every eighth place.  No place is left empty between others: the workgroups
  // of an XCD go to its parts in turn, full ones too, and an early end of some
  // leaves compute units idle while others hold two (128^3, 16 right-hand
  // sides: 2.18 ms with each plane that has a slot alone beside an empty place,
  // 1.20 with the two side by side).
  const int per = (TW ? 4 : 2) * ngroups, place = blockIdx.x >> 3;
  const int unit = place / per * 8 + (blockIdx.x & 7), member = place % per;
  if (unit >= ntwo) return;
  const int2 sp = two[unit];
  const int pl = member & 1 ? sp.y : sp.x;
  if (pl < 0) return;
  const int slot = fmap[pl];
  const int end = TW ? member / (2 * ngroups) : 0;  // 0: from the top, 1: from the bottom
  const int q0 = 8 * ((member >> 1) % ngroups), nq = min(8, nrhs - q0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kg = lane >> 4;  // operand row / result column, and k group / result row group
  const int q = col & 7;                      // the lane's vector in the epilogue
  const int half = col >> 3;                  // ... and which two of its group's four rows
  const bool live = q < nq;
  C* const xq = X + (int64_t)(q0 + (live ? q : 0)) * N + (int64_t)pl * n2;
  const size_t nn = (size_t)n * n;
  const C* const Gs = G + (size_t)slot * ny * nn;
  const C* const Bs = TW ? Gb + (size_t)slot * (ny - m) * nn : nullptr;
  const int nsteps = !TW ? 2 * ny - 1 : PH == 0 ? (end == 0 ? m : ny - 1 - m) : (end == 0 ? m + 1 : ny - m);
  auto blk_of = [&](int s) {
    if (!TW) return s <= ny - 1 ? s : 2 * ny - 2 - s;
    if (PH == 0) return end == 0 ? s : ny - 1 - s;
    return end == 0 ? m - s : m + s;
  };
  auto block = [&](int j) { return TW && j >= m ? Bs + (size_t)(j - m) * nn : Gs + (size_t)j * nn; };
  // line whose vector the update after step s forms (-1: none; -2: the product goes to scr)
  auto next_of = [&](int s) {
    const int j = blk_of(s);
    if (!TW) return s < ny - 1 ? j + 1 : j - 1;
    if (PH == 0) return end == 0 ? (j + 1 < m ? j + 1 : -2) : (j - 1 > m ? j - 1 : -2);
    return end == 0 ? j - 1 : (j < ny - 1 ? j + 1 : -1);
  };
  // whether the line's coefficient is cm_y (its product comes from the line below)
  auto from_below = [&](int s) { return !TW ? s < ny - 1 : (PH == 0) == (end == 0); };
  // whether the products are the solution's lines (else those of the first sweep)
  auto solving = [&](int s) { return !TW ? s >= ny - 1 : PH == 1; };
  // scr: [what][rhs][plane][n], what = 0 y_top, 1 y_bot, 2 f_m
  auto scr_at = [&](int what) { return scr + (((int64_t)what * nrhs + q0 + (live ? q : 0)) * nz + pl) * n; };
  const double2 *dx = symd, *dy = symd + n, *dxi = symd + n + ny, *dyi = symd + 2 * n + ny;
  auto cmul_d = [](double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); };

  if (ADJ)
    for (int e = tid; e < 16 * NT; e += 64 * S::NWV) {
      sdx[e] = e < n ? dx[e] : make_double2(0, 0);
      sdxi[e] = e < n ? dxi[e] : make_double2(0, 0);
    }
  for (int e = tid; e < 4 * S::VB; e += 64 * S::NWV) vb[e] = (A)0;
  __syncthreads();
  // a line value of the right-hand side: f, or D conj(f) for the adjoint
  auto load_f = [&](C f, int r, int j) {
    if (!ADJ) return f;
    const double2 v = cmul_d(make_double2(f.x, -(double)f.y), cmul_d(sdx[r], dy[j]));
    return make_float2((float)v.x, (float)v.y);
  };

  // f_m is kept for the second phase before its top half writes x_m there
  if (PH == 0 && end == 0 && live)
    for (int r = tid >> 4; r < n; r += 4 * S::NWV)
      if (half == 0) scr_at(2)[r] = load_f(xq[(int64_t)m * n + r], r, m);
  if (nsteps <= 0) return;

  auto run = [&](auto rows_tag) {
    constexpr int RPW = decltype(rows_tag)::value;
    constexpr int NSL = RPW * NT, RD = NSL < 12 ? NSL : 12, NSR = (NSL + RD - 1) / RD * RD;
    // Loads of tile t: rows clamped (rows past n give results nobody reads), and
    // in the last tile column the columns (past n they meet zeros of the
    // vector).  Byte offsets per lane; the tile's place goes into the scalar base.
    unsigned off[RPW], last[RPW][4];
#pragma unroll
    for (int a = 0; a < RPW; ++a) {
      const int r = min(16 * (w + 8 * a) + col, n - 1);
      off[a] = 8u * (unsigned)(r + n * 4 * kg);
#pragma unroll
      for (int s = 0; s < 4; ++s) last[a][s] = 8u * (unsigned)(r + n * min(4 * kg + s, n - 1 - 16 * (NT - 1)));
    }
    C ring[RD][4];
    auto load_tile = [&](int t, const C* blk) {
      const int c = t / RPW, a = t % RPW;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const char* const at = reinterpret_cast<const char*>(blk) + 8 * (unsigned)n * (unsigned)(16 * c + (c < NT - 1 ? s : 0));
        ring[t % RD][s] = *reinterpret_cast<const C*>(at + (c < NT - 1 ? off[a] : last[a][s]));
      }
    };
    {
      const C* const blk = block(blk_of(0));
#pragma unroll
      for (int t = 0; t < RD; ++t) {
        load_tile(t, blk);
        __builtin_amdgcn_sched_barrier(0);  // in the order of use, as in the steps: the waits count on it
      }
    }
    // row of the lane's result i of tile row R (it keeps i = 2 half, 2 half + 1)
    auto row_of = [&](int R, int i) { return 16 * R + M::row(kg, 2 * half + i); };
    // this lane's two rows of its vector, into vector buffer b
    auto put_v = [&](int b, int R, double2 v0, double2 v1) {
      A* const at = vb + 2 * b * S::VB + q * 4;
      if (sizeof(A) == 4) {  // neighbours
        float* const t = reinterpret_cast<float*>(at) + (4 * R + kg) * 64 + 2 * half;
        *reinterpret_cast<C*>(t) = make_float2((float)v0.x, (float)v1.x);
        *reinterpret_cast<C*>(t + 32) = make_float2((float)v0.y, (float)v1.y);
        *reinterpret_cast<C*>(t + S::VB) = make_float2((float)-v0.y, (float)-v1.y);
        *reinterpret_cast<C*>(t + S::VB + 32) = make_float2((float)v0.x, (float)v1.x);
      } else {  // four rows apart
        A* const t = at + (4 * R + 2 * half) * 64 + kg;
        t[0] = (A)v0.x;
        t[64] = (A)v1.x;
        t[32] = (A)v0.y;
        t[96] = (A)v1.y;
        t[S::VB] = (A)-v0.y;
        t[S::VB + 64] = (A)-v1.y;
        t[S::VB + 32] = (A)v0.x;
        t[S::VB + 96] = (A)v1.x;
      }
    };
    // ---- the first vector
#pragma unroll
    for (int a = 0; a < RPW; ++a) {
      const int R = w + 8 * a, j0 = blk_of(0);
      double2 v[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = row_of(R, i), rc = min(r, n - 1);
        if (PH == 1) {
          const C f = scr_at(2)[rc];
          v[i] = make_double2(f.x, f.y);
          if (m > 0) {
            const C y = scr_at(0)[rc];
            const double2 t = cmul_d(cmy[m], make_double2(y.x, y.y));
            v[i].x -= t.x;
            v[i].y -= t.y;
          }
          if (m < ny - 1) {
            const C y = scr_at(1)[rc];
            const double2 t = cmul_d(cpy[m], make_double2(y.x, y.y));
            v[i].x -= t.x;
            v[i].y -= t.y;
          }
        } else {
          const C f = load_f(xq[(int64_t)j0 * n + rc], rc, j0);
          v[i] = make_double2(f.x, f.y);
          if (live && r < n && ADJ && (TW || ny > 1)) xq[(int64_t)j0 * n + r] = f;  // the scaled line, for the sweep back
        }
        if (!live || r >= n) v[i] = make_double2(0, 0);
      }
      put_v(0, R, v[0], v[1]);
    }
    __syncthreads();

    for (int st = 0; st < nsteps; ++st) {
      const int jb = blk_of(st), jn = next_of(st);
      const C* const cblk = block(jb);
      const C* const nblk = block(blk_of(st + 1 < nsteps ? st + 1 : st));
      const A* const vin = vb + (st & 1) * 2 * S::VB;
      auto reload = [&](int t) {
        int u = t + RD;
        if (u < NSL) {
          load_tile(u, cblk);
        } else {
          if (u < NSR) u += RD;
          load_tile(u - NSR, nblk);
        }
      };
      C pre[RPW][2];
#pragma unroll
      for (int a = 0; a < RPW; ++a)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          pre[a][i] = xq[(int64_t)(jn >= 0 ? jn : jb) * n + min(row_of(w + 8 * a, i), n - 1)];
      V y0[RPW], y1[RPW];
#pragma unroll
      for (int a = 0; a < RPW; ++a) y0[a] = y1[a] = V{(A)0, (A)0, (A)0, (A)0};
      struct alignas(16) Four { A v[4]; };
      Four bp[2], br[2];  // operands of the tile column, one ahead
      auto load_col = [&](int c) {
        const int at = ((4 * c + kg) * 16 + col) * 4;
        bp[c & 1] = *reinterpret_cast<const Four*>(vin + at);
        br[c & 1] = *reinterpret_cast<const Four*>(vin + at + S::VB);
      };
      load_col(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        if (c + 1 < NT) load_col(c + 1);
        const Four u = bp[c & 1], v = br[c & 1];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int a = 0; a < RPW; ++a) {
            const C g = ring[(c * RPW + a) % RD][s];
            y0[a] = M::mfma(g.x, u.v[s], y0[a]);
            y1[a] = M::mfma(g.y, v.v[s], y1[a]);
          }
#pragma unroll
        for (int a = 0; a < RPW; ++a) {
          reload(c * RPW + a);
          __builtin_amdgcn_sched_barrier(0);  // the reloads stay in order
        }
      }
      // ---- the update.  The product leaves a lane one component of four rows; it
      // takes the other of its two rows from the lane 8 away.
      const int jf = jn >= 0 ? jn : jb;
      const double2 cf = from_below(st) ? cmy[jf] : cpy[jf];
      const bool sol = solving(st);
#pragma unroll
      for (int a = 0; a < RPW; ++a) {
        const int R = w + 8 * a;
        const V y = y0[a] + y1[a];
        const A ya = y[0], yb = y[1], yc = y[2], yd = y[3];
        const A g0 = rows_ror8(half ? ya : yc), g1 = rows_ror8(half ? yb : yd);
        const A zx[2] = {half ? g0 : ya, half ? g1 : yb}, zy[2] = {half ? yc : g0, half ? yd : g1};
        double2 v[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = row_of(R, i), rc = min(r, n - 1);
          const double2 z = make_double2(zx[i], zy[i]);
          const C f = sol ? pre[a][i] : load_f(pre[a][i], rc, jf);
          v[i] = make_double2(f.x - (cf.x * z.x - cf.y * z.y), f.y - (cf.x * z.y + cf.y * z.x));
          if (live && r < n) {
            if (sol) {  // x_jb (both ends have x_m)
              const double2 o = ADJ ? cmul_d(cmul_d(sdxi[rc], dyi[jb]), z) : z;
              if (PH != 1 || end == 0 || st > 0)
                xq[(int64_t)jb * n + r] = make_float2((float)o.x, (float)(ADJ ? -o.y : o.y));
            } else if (TW && jn == -2) {  // y_top / y_bot
              scr_at(end)[r] = make_float2((float)z.x, (float)z.y);
            } else {  // t_jn
              xq[(int64_t)jn * n + r] = make_float2((float)v[i].x, (float)v[i].y);
            }
          }
          if (!live || r >= n) v[i] = make_double2(0, 0);
        }
        put_v((st + 1) & 1, R, v[0], v[1]);
      }
      __syncthreads();
    }
  };
  if (NT <= 8 || w + 8 >= NT) run(std::integral_constant<int, 1>{});
  else run(std::integral_constant<int, 2>{});
}

template <typename A, int NT, int PH, bool ADJ>
void launch_rows(hz_problem* p, int nrhs, float2* x, hipStream_t s) {
  constexpr size_t lds = RowsShape<A, NT>::lds(ADJ);
  static_assert(lds <= 160 * 1024, "LDS");
  const Factors& f = p->fac[HZ_PREC_C64];
  set_max_lds((const void*)&k_solve_rows<A, NT, PH, ADJ>, lds);
  const int ng = (nrhs + 7) / 8;
  hipLaunchKernelGGL((k_solve_rows<A, NT, PH, ADJ>), dim3((unsigned)((p->ntwo + 7) / 8 * 8 * (PH < 0 ? 2 : 4) * ng)),
                     dim3(64 * RowsShape<A, NT>::NWV), lds, s, f.G.as<float2>(), f.Gb.as<float2>(), x, p->tab(1, 0),
                     p->tab(1, 1), p->d_symd.as<double2>(), (int)p->nx, (int)p->ny, f.tw_m, (int)p->nz, p->n2, p->N,
                     p->d_two.as<int2>(), p->ntwo, p->d_fmap.as<int>(), nrhs, ng, f.tw_scr.as<float2>());
  HZ_HIP(hipGetLastError());
}

// both phases of a twisted solve, the vectors that one workspace serves at a time
template <typename A, int NT, bool ADJ>
void launch_twisted(hz_problem* p, int nrhs, float2* x, hipStream_t s) {
  for (int r0 = 0; r0 < nrhs; r0 += TW_RHS) {
    const int nr = std::min(TW_RHS, nrhs - r0);
    launch_rows<A, NT, 0, ADJ>(p, nr, x + (size_t)r0 * p->N, s);
    launch_rows<A, NT, 1, ADJ>(p, nr, x + (size_t)r0 * p->N, s);
  }
}

}  // namespace

bool rows_available(const hz_problem* p) { return p->slot_pairs && p->nx <= 16 * ROWS_MAX_NT; }

void solve_rows(hz_problem* p, int nrhs, void* x, bool adjoint, hipStream_t s) {
  switch (((int)p->nx + 15) / 16) {
#define HZ_ROWS(NT)                                                        \
  case NT:                                                                 \
    if (adjoint) launch_rows<float, NT, -1, true>(p, nrhs, (float2*)x, s); \
    else launch_rows<float, NT, -1, false>(p, nrhs, (float2*)x, s);        \
    break;
    HZ_ROWS(1) HZ_ROWS(2) HZ_ROWS(3) HZ_ROWS(4) HZ_ROWS(5) HZ_ROWS(6) HZ_ROWS(7) HZ_ROWS(8)
    HZ_ROWS(9) HZ_ROWS(10) HZ_ROWS(11) HZ_ROWS(12) HZ_ROWS(13) HZ_ROWS(14) HZ_ROWS(15) HZ_ROWS(16)
#undef HZ_ROWS
    default: HZ_CHECK(false, HZ_ERR_ARG, "nx=%d", (int)p->nx);
  }
}

void solve_rows_twisted(hz_problem* p, int nrhs, void* x, bool adjoint, bool wide, hipStream_t s) {
  const int nt = ((int)p->nx + 15) / 16;
#define HZ_ROWS(NT)                                                               \
  if (nt == NT) {                                                                 \
    if (!adjoint) return launch_twisted<float, NT, false>(p, nrhs, (float2*)x, s); \
    if (!wide) return launch_twisted<float, NT, true>(p, nrhs, (float2*)x, s);     \
    if constexpr (16 * NT <= TRI_WIDE_MAX) return launch_twisted<double, NT, true>(p, nrhs, (float2*)x, s); \
  }
  HZ_ROWS(1) HZ_ROWS(2) HZ_ROWS(3) HZ_ROWS(4) HZ_ROWS(5) HZ_ROWS(6) HZ_ROWS(7) HZ_ROWS(8)
  HZ_ROWS(9) HZ_ROWS(10) HZ_ROWS(11) HZ_ROWS(12) HZ_ROWS(13)
#undef HZ_ROWS
  HZ_CHECK(false, HZ_ERR_ARG, "nx=%d", (int)p->nx);
}

}  // namespace hz
