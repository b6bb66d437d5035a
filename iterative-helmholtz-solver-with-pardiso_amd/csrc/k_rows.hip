// k_rows.hip -- complex64 plane solves of groups of 8 right-hand sides on the
// one-directional factors, blocks read from memory straight into the matrix
// products.
//
// The sweep is that of the other one-directional kernels (t_{j+1} = b_{j+1} -
// cm_y(j+1) G_j t_j up, x_j = G_j (t_j - cp_y(j) x_{j+1}) down, 2 ny - 1 block
// products), one workgroup per plane and group.  Adjoint: with D = diag(dx(i)
// dy(j)), M^H x = b is the forward solve M z = D conj(b), x = conj(D^-1 z).
//
// Wave w computes the tile rows w and w + 8 of every product.  A 16 x 16 tile of
// the column-major block is loaded once, by the one wave that needs it, in the
// operand order of v_mfma_f32_16x16x4f32: lane l holds row l & 15 and the
// columns 4 (l >> 4) .. + 3, 8 bytes a load along the rows.  The 16 result
// columns are the real and imaginary parts of the 8 vectors:
//   [Re Y | Im Y] += Re(G) [Re V | Im V] + Im(G) [-Im V | Re V].
// A wave's rows are complete in its own accumulators, so the update of the next
// vector needs no sums between waves: it is written to the other of two LDS
// buffers and a step has one barrier.
//
// What bounds it: the blocks' bytes from memory, and below them the matrix
// products.  The two planes of a factor slot and the groups of right-hand sides
// run side by side on one XCD and share its L2's copy of a block.  A wave keeps
// 12 tiles (24 KB) in flight; their registers are refilled as soon as they are
// read, and the loads do not depend on the vector.  A lane finishes two whole
// entries of the next vector (8-byte loads and stores) after one exchange with
// the lane 8 away; with one component of four rows a lane a step took 0.25 us
// more (4.45 -> 4.2 at 128 columns, 9.7 -> 9.0 at 192).  Measured, in ms, blocks
// staged through LDS before -> now: 128^3 x 8 1.08 -> 1.07, x 16 1.24 -> 1.14,
// 160^3 x 8 3.37 -> 2.05, 192^3 x 8 5.03 -> 3.46, 200^3 x 8 6.16 -> 4.65; 104^3
// x 8 (vector units before) 2.54 -> 0.66.
#include <algorithm>
#include <type_traits>

#include "hz_internal.h"
#include "k_plane.h"

namespace hz {
namespace {

constexpr int ROWS_MAX_NT = 16;  // up to 256 columns

__device__ __forceinline__ float rows_ror8(float x) {  // lane n ^ 8 within 16
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x),
                                                               0x128, 0xF, 0xF, false));
}

template <int NT>
struct RowsShape {
  static constexpr int NWV = NT < 8 ? NT : 8;
  static constexpr int VB = 16 * NT * 16;  // floats of one vector buffer (plain or rotated)
  static constexpr size_t lds(bool adj) { return sizeof(float) * 4 * VB + (adj ? sizeof(double2) * 32 * NT : 0); }
};

template <int NT, bool ADJ>
__global__ __launch_bounds__(64 * (NT < 8 ? NT : 8)) void k_solve_rows(
    const float2* __restrict__ G, float2* __restrict__ X, const double2* __restrict__ cmy,
    const double2* __restrict__ cpy, const double2* __restrict__ symd, int n, int ny, int64_t n2, int64_t N,
    const int2* __restrict__ two, int ntwo, const int* __restrict__ fmap, int nrhs, int ngroups) {
  typedef float2 C;
  typedef RowsShape<NT> S;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  // vector buffers [2][plain, rotated][c / 4][16 columns][c % 4]
  float* const vb = reinterpret_cast<float*>(smem_raw);
  double2* const sdx = reinterpret_cast<double2*>(vb + 4 * S::VB);  // adjoint: dx, 1 / dx
  double2* const sdxi = sdx + 16 * NT;

  // Workgroups go to the 8 XCDs in turn: the planes and groups of one slot take
  // every eighth place.  No place is left empty between others: the workgroups
  // of an XCD go to its parts in turn, full ones too, and an early end of some
  // leaves compute units idle while others hold two (128^3, 16 right-hand
  // sides: 2.18 ms with each plane that has a slot alone beside an empty place,
  // 1.20 with the two side by side).
  const int per = 2 * ngroups, place = blockIdx.x >> 3;
  const int unit = place / per * 8 + (blockIdx.x & 7), member = place % per;
  if (unit >= ntwo) return;
  const int2 sp = two[unit];
  const int pl = member & 1 ? sp.y : sp.x;
  if (pl < 0) return;
  const int slot = fmap[pl];
  const int q0 = 8 * (member >> 1), nq = min(8, nrhs - q0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kg = lane >> 4;  // operand row / result column, and k group / result row group
  const int q = col & 7;                      // the lane's vector in the epilogue
  const int half = col >> 3;                  // ... and which two of its group's four rows
  const bool live = q < nq;
  C* const xq = X + (int64_t)(q0 + (live ? q : 0)) * N + (int64_t)pl * n2;
  const size_t nn = (size_t)n * n;
  const C* const Gs = G + (size_t)slot * ny * nn;
  const int nsteps = 2 * ny - 1;
  auto blk_of = [&](int s) { return s <= ny - 1 ? s : 2 * ny - 2 - s; };
  const double2 *dx = symd, *dy = symd + n, *dxi = symd + n + ny, *dyi = symd + 2 * n + ny;
  auto cmul_d = [](double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); };

  if (ADJ)
    for (int e = tid; e < 16 * NT; e += 64 * S::NWV) {
      sdx[e] = e < n ? dx[e] : make_double2(0, 0);
      sdxi[e] = e < n ? dxi[e] : make_double2(0, 0);
    }
  for (int e = tid; e < 4 * S::VB; e += 64 * S::NWV) vb[e] = 0.f;
  __syncthreads();
  // a line value of the right-hand side: f, or D conj(f) for the adjoint
  auto load_f = [&](C f, int r, int j) {
    if (!ADJ) return f;
    const double2 v = cmul_d(make_double2(f.x, -(double)f.y), cmul_d(sdx[r], dy[j]));
    return make_float2((float)v.x, (float)v.y);
  };

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
      const C* const blk = Gs;
#pragma unroll
      for (int t = 0; t < RD; ++t) {
        load_tile(t, blk);
        __builtin_amdgcn_sched_barrier(0);  // in the order of use, as in the steps: the waits count on it
      }
    }
    // this lane's two rows of its vector, into vector buffer b
    auto put_v = [&](int b, int R, C v0, C v1) {
      float* const at = vb + 2 * b * S::VB + ((4 * R + kg) * 16 + q) * 4 + 2 * half;
      *reinterpret_cast<C*>(at) = make_float2(v0.x, v1.x);
      *reinterpret_cast<C*>(at + 32) = make_float2(v0.y, v1.y);
      *reinterpret_cast<C*>(at + S::VB) = make_float2(-v0.y, -v1.y);
      *reinterpret_cast<C*>(at + S::VB + 32) = make_float2(v0.x, v1.x);
    };
    // ---- t_0
#pragma unroll
    for (int a = 0; a < RPW; ++a) {
      const int R = w + 8 * a;
      C v[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 16 * R + 4 * kg + 2 * half + i, rc = min(r, n - 1);
        v[i] = load_f(xq[rc], rc, 0);
        if (!live || r >= n) v[i] = make_float2(0.f, 0.f);
        else if (ADJ && ny > 1) xq[r] = v[i];  // the scaled line, for the sweep back
      }
      put_v(0, R, v[0], v[1]);
    }
    __syncthreads();

    for (int st = 0; st < nsteps; ++st) {
      const int jb = blk_of(st), jn = st < ny - 1 ? st + 1 : jb - 1;  // jn = -1: the last block
      const C* const cblk = Gs + (size_t)jb * nn;
      const C* const nblk = Gs + (size_t)blk_of(st + 1 < nsteps ? st + 1 : st) * nn;
      const float* const vin = vb + (st & 1) * 2 * S::VB;
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
          pre[a][i] = xq[(int64_t)max(jn, 0) * n + min(16 * (w + 8 * a) + 4 * kg + 2 * half + i, n - 1)];
      hz_v4f y0[RPW], y1[RPW];
#pragma unroll
      for (int a = 0; a < RPW; ++a) y0[a] = y1[a] = hz_v4f{0.f, 0.f, 0.f, 0.f};
      float4 bp[2], br[2];  // operands of the tile column, one ahead
      auto load_col = [&](int c) {
        const int at = ((4 * c + kg) * 16 + col) * 4;
        bp[c & 1] = *reinterpret_cast<const float4*>(vin + at);
        br[c & 1] = *reinterpret_cast<const float4*>(vin + at + S::VB);
      };
      load_col(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        if (c + 1 < NT) load_col(c + 1);
        const float4 u = bp[c & 1], v = br[c & 1];
        const float up[4] = {u.x, u.y, u.z, u.w}, vp[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int a = 0; a < RPW; ++a) {
            const C g = ring[(c * RPW + a) % RD][s];
            y0[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.x, up[s], y0[a], 0, 0, 0);
            y1[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.y, vp[s], y1[a], 0, 0, 0);
          }
#pragma unroll
        for (int a = 0; a < RPW; ++a) {
          reload(c * RPW + a);
          __builtin_amdgcn_sched_barrier(0);  // the reloads stay in order
        }
      }
      // ---- the update.  The product leaves a lane one component of rows 4 kg ..
      // + 3; it takes the other of its two rows from the lane 8 away.
      const double2 cf = st < ny - 1 ? cmy[jn] : cpy[max(jn, 0)];
#pragma unroll
      for (int a = 0; a < RPW; ++a) {
        const int R = w + 8 * a;
        const hz_v4f y = y0[a] + y1[a];
        const float ya = y[0], yb = y[1], yc = y[2], yd = y[3];
        const float g0 = rows_ror8(half ? ya : yc), g1 = rows_ror8(half ? yb : yd);
        const C z[2] = {half ? make_float2(g0, yc) : make_float2(ya, g0), half ? make_float2(g1, yd) : make_float2(yb, g1)};
        C v[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = 16 * R + 4 * kg + 2 * half + i, rc = min(r, n - 1);
          const C f = st < ny - 1 ? load_f(pre[a][i], rc, max(jn, 0)) : pre[a][i];
          v[i] = make_float2(f.x - (float)(cf.x * z[i].x - cf.y * z[i].y), f.y - (float)(cf.x * z[i].y + cf.y * z[i].x));
          C o = v[i];  // t_jn on the way up, x_jb on the way down
          if (st >= ny - 1) {
            o = z[i];
            if (ADJ) {
              const double2 d = cmul_d(sdxi[rc], dyi[jb]);
              o = make_float2((float)(d.x * o.x - d.y * o.y), -(float)(d.x * o.y + d.y * o.x));
            }
          }
          if (!live || r >= n) v[i] = make_float2(0.f, 0.f);
          else xq[(int64_t)(st < ny - 1 ? jn : jb) * n + r] = o;
        }
        put_v((st + 1) & 1, R, v[0], v[1]);
      }
      __syncthreads();
    }
  };
  if (NT <= 8 || w + 8 >= NT) run(std::integral_constant<int, 1>{});
  else run(std::integral_constant<int, 2>{});
}

template <int NT, bool ADJ>
void launch_rows(hz_problem* p, int nrhs, float2* x, hipStream_t s) {
  constexpr size_t lds = RowsShape<NT>::lds(ADJ);
  static_assert(lds <= 160 * 1024, "LDS");
  set_max_lds((const void*)&k_solve_rows<NT, ADJ>, lds);
  const int ng = (nrhs + 7) / 8;
  hipLaunchKernelGGL((k_solve_rows<NT, ADJ>), dim3((unsigned)((p->ntwo + 7) / 8 * 8 * 2 * ng)),
                     dim3(64 * RowsShape<NT>::NWV), lds, s, p->fac[HZ_PREC_C64].G.as<float2>(), x, p->tab(1, 0),
                     p->tab(1, 1), p->d_symd.as<double2>(), (int)p->nx, (int)p->ny, p->n2, p->N,
                     p->d_two.as<int2>(), p->ntwo, p->d_fmap.as<int>(), nrhs, ng);
  HZ_HIP(hipGetLastError());
}

}  // namespace

bool rows_available(const hz_problem* p) { return p->slot_pairs && p->nx <= 16 * ROWS_MAX_NT; }

void solve_rows(hz_problem* p, int nrhs, void* x, bool adjoint, hipStream_t s) {
  switch (((int)p->nx + 15) / 16) {
#define HZ_ROWS(NT)                                             \
  case NT:                                                      \
    if (adjoint) launch_rows<NT, true>(p, nrhs, (float2*)x, s); \
    else launch_rows<NT, false>(p, nrhs, (float2*)x, s);        \
    break;
    HZ_ROWS(1) HZ_ROWS(2) HZ_ROWS(3) HZ_ROWS(4) HZ_ROWS(5) HZ_ROWS(6) HZ_ROWS(7) HZ_ROWS(8)
    HZ_ROWS(9) HZ_ROWS(10) HZ_ROWS(11) HZ_ROWS(12) HZ_ROWS(13) HZ_ROWS(14) HZ_ROWS(15) HZ_ROWS(16)
#undef HZ_ROWS
    default: HZ_CHECK(false, HZ_ERR_ARG, "nx=%d", (int)p->nx);
  }
}

}  // namespace hz
