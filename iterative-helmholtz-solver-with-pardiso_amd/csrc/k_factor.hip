// k_factor.hip -- block Schur recursion of the plane systems with every block
// inverted in registers.
//
// Same recursion, modes and pivots as k_factor (k_blocktri.hip): one workgroup
// walks a chain of blocks S_j = D_j - sig G_{j-1} and inverts each by blocked
// Gauss-Jordan with partial pivoting.  What bounds that work is one CU per
// chain: the chain is sequential and there are at most 2 nslot chains.  The
// matrix therefore stays in the CU's registers for a whole inversion (200 x 200
// complex64: 313 of 512 KB): 16 x 16 tiles in the accumulator layout of the
// 16x16x4 matrix instructions, dealt round robin to the 8 waves, so the
// trailing update of a 16-column panel is the matrix products alone, with no
// load or store of the matrix.
//
// Tiles hold the transpose of what they cover: lane l has row 16 rt + (l & 15)
// and columns 16 ct + 4 (l >> 4) + i (complex128: 4 i + (l >> 4)), so the
// global loads and stores of the column-major block run along lanes.
//
// Rows are never interchanged.  Step k takes as pivot the row p_k of largest
// |re| + |im| in column k among the rows not used yet (the rows partial
// pivoting would see below the diagonal) and exchanges the roles of y_{p_k}
// and x_k; afterwards tile element (r, l) is the inverse's element
// (kof[r], piv[l]) with piv[k] = p_k, kof[p_k] = k, which the store applies.
//
// Wave 0 eliminates the panels (16 columns), waves 1 .. 7 hold the tiles.  The
// tile waves update the next panel's column first and hand it over, so the
// elimination of one panel runs beside the matrix products of the one before.
// In the panel wave lane l has rows l, l + 64, ... in registers: no barrier and
// no memory access inside a panel.  Its columns move one place to the left with
// every step's update (the destination of the multiply-add), so the current
// column is always the first and the 16 steps are one short loop.  Panel and
// pivot rows pass to the matrix products through LDS in 16-byte units,
// swizzled by row against bank conflicts of the operand reads.
#include <type_traits>

#include "hz_internal.h"
#include "k_plane.h"

namespace hz {
namespace {

constexpr int FR_THREADS = 512;
constexpr int FR_TWAVES = FR_THREADS / 64 - 1;  // waves with tiles
constexpr int FR_AHEAD = 4;                     // tiles whose loads are in flight

template <typename T> struct FR;
template <> struct FR<float> {
  typedef hz_v4f V;
  static constexpr int CU = 2;  // complex values per 16-byte unit
  __device__ static __forceinline__ int col(int lg, int i) { return 4 * lg + i; }
  __device__ static __forceinline__ V mfma(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};
template <> struct FR<double> {
  typedef hz_v4d V;
  static constexpr int CU = 1;
  __device__ static __forceinline__ int col(int lg, int i) { return 4 * i + lg; }
  __device__ static __forceinline__ V mfma(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};

// largest value over the wave, in every lane
template <int CTRL>
__device__ __forceinline__ unsigned fr_dpp_max(unsigned x) {
  return max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ unsigned fr_wave_max(unsigned x) {
  x = fr_dpp_max<0xB1>(x);   // quad xor 1
  x = fr_dpp_max<0x4E>(x);   // quad xor 2
  x = fr_dpp_max<0x141>(x);  // row half mirror
  x = fr_dpp_max<0x140>(x);  // row mirror
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  x = max(r0, r1);
  const auto q = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  const unsigned q0 = q[0], q1 = q[1];
  return max(q0, q1);
}

// Rank of a column entry: |re| + |im| as the leading 32 bits of its (never
// negative) floating value, plus one; 0 is left for rows that are no
// candidates, 1 is an exact zero.  complex128 ranks by 20 bits of mantissa:
// the pivot is within 1e-6 of the largest.
__device__ __forceinline__ unsigned fr_rank(float2 a) {
  return __builtin_bit_cast(unsigned, fabsf(a.x) + fabsf(a.y)) + 1u;
}
__device__ __forceinline__ unsigned fr_rank(double2 a) {
  const double v = fabs(a.x) + fabs(a.y);
  const unsigned hi = (unsigned)(__builtin_bit_cast(unsigned long long, v) >> 32);
  return v == 0.0 ? 1u : hi + 2u;
}

// 1 / d for d in the normal range, by Newton's iteration from the hardware's
// approximation
__device__ __forceinline__ double fr_recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  r = fma(fma(-d, r, 1.0), r, r);
  return r;
}

// 1 / a.  complex64: |a|^2 of two floats neither overflows nor underflows in
// double, so the quotients are formed there and rounded once.
__device__ __forceinline__ float2 fr_inv(float2 a) {
  const double x = a.x, y = a.y;
  const double r = fr_recip(fma(x, x, y * y));
  return make_float2((float)(x * r), (float)(-y * r));
}
// complex128: |a|^2 scaled by a power of two (exact) against overflow
__device__ __forceinline__ double2 fr_inv(double2 a) {
  const int e = -__builtin_amdgcn_frexp_exp(fmax(fabs(a.x), fabs(a.y)));
  const double x = __builtin_amdgcn_ldexp(a.x, e), y = __builtin_amdgcn_ldexp(a.y, e);
  const double r = fr_recip(fma(x, x, y * y));
  return make_double2(__builtin_amdgcn_ldexp(x * r, e), __builtin_amdgcn_ldexp(-y * r, e));
}

struct alignas(16) FrUnit { unsigned w[4]; };

// The value, hidden from the compiler: what is derived from it is formed where
// it is used.  (Left visible, the addresses and masks of every tile are loop
// invariants, and keeping them costs more registers than the tiles have.)
__device__ __forceinline__ int fr_fresh_s(int x) {
  x = __builtin_amdgcn_readfirstlane(x);
  asm volatile("" : "+s"(x));
  return x;
}
__device__ __forceinline__ int fr_fresh_v(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// lane `l`'s value, in every lane (uniform)
__device__ __forceinline__ float fr_lane(float x, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
}
__device__ __forceinline__ double fr_lane(double x, int l) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

// TPW: tiles per tile wave, NQ: rows per lane of the panel wave
template <typename T, int TPW, int NQ>
__global__ __launch_bounds__(FR_THREADS) void k_factor_reg(typename Cx<T>::t* __restrict__ G, PlaneTabs tb, int n,
                                                           int ny, int nt, int* __restrict__ status,
                                                           const int* __restrict__ splane, int mode, int m,
                                                           typename Cx<T>::t* __restrict__ Gb, int jbeg, int jend) {
  typedef typename Cx<T>::t C;
  typedef FR<T> F;
  typedef typename F::V V;
  constexpr int CU = F::CU, UN = 16 / CU;  // units per 16-column row
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np = 16 * nt;
  FrUnit* const Pb = reinterpret_cast<FrUnit*>(smem_raw);  // [2][np][UN] panels
  FrUnit* const AK = Pb + (size_t)2 * np * UN;             // [np][UN] pivot rows by column
  int* const piv = reinterpret_cast<int*>(AK + (size_t)np * UN);  // [np] row of column
  int* const kof = piv + np;    // [np] column of row
  int* const pslot = kof + np;  // [np] the row's step within the panel, -1: not a pivot
  int* const prows = pslot + np;  // bit rt: row tile rt holds a pivot of the panel

  const int nsl = mode == 1 ? (int)gridDim.x / 2 : (int)gridDim.x;
  const bool up = mode == 1 && (int)blockIdx.x >= nsl;
  const int slot = up ? (int)blockIdx.x - nsl : (int)blockIdx.x;
  const bool rev = up || mode == 2;
  const int k = splane[slot];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t nn = (size_t)n * n;
  const double lam = tb.lamz[k];

  auto unit = [&](int row, int u) { return row * UN + (u ^ (row & 7)); };
  const int nblk = mode == 2 ? 1 : (up ? ny - 1 - m : jend - jbeg);

  if (wave == 0) {
    // ================================================== the panel wave
    bool singular = false;
    for (int jj = 0; jj < nblk; ++jj) {
      unsigned used = 0;  // bit q: row lane + 64 q has been a pivot (or is none)
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        if (lane + 64 * q >= n) used |= 1u << q;
      __syncthreads();
      for (int pc = 0; pc < nt; ++pc) {
        FrUnit* const P = Pb + (size_t)(pc & 1) * np * UN;
        const int kb = min(16, n - 16 * pc);
        C a[NQ][16];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const int r = lane + 64 * q, rr = r < np ? r : 0;  // rows past np copy row 0 and are never used
#pragma unroll
          for (int u = 0; u < UN; ++u) {
            const FrUnit w = P[unit(rr, u)];
#pragma unroll
            for (int e = 0; e < CU; ++e) a[q][u * CU + e] = reinterpret_cast<const C*>(&w)[e];
          }
        }
        int myslot[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) myslot[q] = -1;
#pragma unroll 1
        for (int kk = 0; kk < 16; ++kk) {
          unsigned rank[NQ], top = 0;
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            rank[q] = used >> q & 1 ? 0u : fr_rank(a[q][0]);
            top = max(top, rank[q]);
          }
          // steps past the last column only move the columns on
          const bool step = kk < kb;
          top = fr_wave_max(top);
          C pv[16], fp[NQ];
          int first = 0;
          bool done = !step;
#pragma unroll
          for (int c = 0; c < 16; ++c) pv[c].x = pv[c].y = (T)0;
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            const unsigned long long hit = __ballot(rank[q] == top);
            if (!done && hit) {
              done = true;
              first = __builtin_ctzll(hit);
#pragma unroll
              for (int c = 0; c < 16; ++c) {
                pv[c].x = fr_lane(a[q][c].x, first);
                pv[c].y = fr_lane(a[q][c].y, first);
              }
              if (lane == first) {
                used |= 1u << q;
                myslot[q] = kk;
                const int r = lane + 64 * q;
                piv[16 * pc + kk] = r;
                kof[r] = 16 * pc + kk;
#pragma unroll
                for (int c = 0; c < 16; ++c) a[q][c].x = a[q][c].y = (T)0;
              }
            }
          }
          if (step && top <= 1u) singular = true;
          const C pinv = fr_inv(pv[0]);
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            fp[q] = cmul(a[q][0], pinv);
            if (myslot[q] == kk) {
              fp[q].x = -pinv.x;
              fp[q].y = -pinv.y;
            }
            if (!step) fp[q].x = fp[q].y = (T)0;
          }
#pragma unroll
          for (int c = 1; c < 16; ++c)
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
              const C o = a[q][c];
              // the product, then the difference: one rounding at o's size a step
              // (the two products summed onto o in turn rounded twice: 1.7 times
              // the error of a chain of 16-column blocks)
              a[q][c - 1].x = o.x + fma(-fp[q].x, pv[c].x, fp[q].y * pv[c].y);
              a[q][c - 1].y = o.y - fma(fp[q].x, pv[c].y, fp[q].y * pv[c].x);
            }
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            a[q][15].x = -fp[q].x;
            a[q][15].y = -fp[q].y;
          }
        }
        int rows = 0;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const int r = lane + 64 * q;
          if (r < np) {
            pslot[r] = myslot[q];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
              FrUnit w;
#pragma unroll
              for (int e = 0; e < CU; ++e) reinterpret_cast<C*>(&w)[e] = a[q][u * CU + e];
              P[unit(r, u)] = w;
            }
          }
          const unsigned long long hit = __ballot(r < np && myslot[q] >= 0);
#pragma unroll
          for (int g = 0; g < 4; ++g)
            if (hit >> (16 * g) & 0xFFFF) rows |= 1 << (4 * q + g);
        }
        if (lane == 0) *prows = rows;
        __syncthreads();  // the panel is there
        __syncthreads();  // its pivot rows are there
        __syncthreads();  // the next panel's column is there
      }
      __syncthreads();  // the inverse is stored
    }
    if (lane == 0 && singular) atomicOr(status, 1);
    return;
  }

  // ==================================================== the tile waves
  // The wave's tiles: every seventh of the column-major tile order.  HZ_FR_TILES
  // runs its body for each, with the tile's row and column rt, ct and the lane's
  // li, lg; ct is nt or more past the last tile.
  const int mg = 65536 / nt + 1;  // id / nt = id mg >> 16 (id < 256)
#define HZ_FR_TILES(...)                                        \
  {                                                             \
    const int w_ = fr_fresh_s(wave) - 1, l_ = fr_fresh_v(lane); \
    const int li = l_ & 15, lg = l_ >> 4;                       \
    (void)lg;                                                   \
    _Pragma("unroll") for (int t = 0; t < TPW; ++t) {           \
      const int id_ = w_ + FR_TWAVES * t;                       \
      const int ct = (id_ * mg) >> 16, rt = id_ - ct * nt;      \
      __VA_ARGS__                                               \
    }                                                           \
  }
  // pivot rows past the last column of a short panel multiply zero columns of
  // P: they have to be numbers, also where no earlier panel left any (nt = 2)
  for (int q = tid - 64; q < np * UN; q += FR_THREADS - 64) AK[q] = FrUnit{};
  C* const Gs = rev ? Gb + (size_t)slot * (ny - m) * nn : G + (size_t)slot * ny * nn;
  for (int jj = 0; jj < nblk; ++jj) {
    const int j = mode == 2 ? m : (up ? ny - 1 - jj : jbeg + jj);
    C* const Gj = Gs + (size_t)(rev ? j - m : j) * nn;
    const bool hasp = rev ? j + 1 < ny : j > 0;
    const C* const Gp = rev ? Gj + nn : Gj - nn;
    const double2 sg = hasp ? tb.sig[rev ? j + 1 : j] : make_double2(0, 0);
    const bool mid = mode == 2 && m > 0;
    const C* const Gm = mid ? G + ((size_t)slot * ny + (m - 1)) * nn : nullptr;
    const double2 sgm = mid ? tb.sig[m] : make_double2(0, 0);
    const double2 cdy = tb.cdy[j];

    // ---- S_j into the tiles, the loads of the previous inverse FR_AHEAD tiles
    // ahead.  (Sums without branches and a fence per tile: the compiler would
    // otherwise keep every tile's loads apart from the tiles' registers.)
    V re[TPW], im[TPW];
    auto form = [&](auto hp, auto md) {
      constexpr bool HP = decltype(hp)::value, MID = decltype(md)::value;
      const int w_ = fr_fresh_s(wave) - 1, l_ = fr_fresh_v(lane);
      const int li = l_ & 15, lg = l_ >> 4;
      C g[FR_AHEAD][4], h[FR_AHEAD][4];
#pragma unroll
      for (int x = 0; x < TPW + FR_AHEAD; ++x) {
        if (x >= FR_AHEAD) {
          const int t = x - FR_AHEAD, b = t % FR_AHEAD;
          const int id = w_ + FR_TWAVES * t, ct = (id * mg) >> 16, rt = id - ct * nt;
          const int r = 16 * rt + li, rr = min(r, n - 1);
          const double2 lo = tb.cmx[rr], hi = tb.cpx[rr], dg = tb.cdx[rr];
          const double2 kp = tb.kappa[rr + (size_t)n * j];
          const double dx = dg.x + cdy.x + kp.x - lam, dy = dg.y + cdy.y + kp.y;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            double sx = 0.0, sy = 0.0;
            if (HP) {
              sx = -(sg.x * (double)g[b][i].x - sg.y * (double)g[b][i].y);
              sy = -(sg.x * (double)g[b][i].y + sg.y * (double)g[b][i].x);
            }
            if (MID) {
              sx -= sgm.x * (double)h[b][i].x - sgm.y * (double)h[b][i].y;
              sy -= sgm.x * (double)h[b][i].y + sgm.y * (double)h[b][i].x;
            }
            const int c = 16 * ct + F::col(lg, i), o = c - r;
            sx += o == 0 ? dx : o == -1 ? lo.x : o == 1 ? hi.x : 0.0;
            sy += o == 0 ? dy : o == -1 ? lo.y : o == 1 ? hi.y : 0.0;
            const bool in = r < n && c < n;
            re[t][i] = in ? (T)sx : (T)0;
            im[t][i] = in ? (T)sy : (T)0;
          }
        }
        if (x < TPW) {
          const int id = w_ + FR_TWAVES * x, ct = (id * mg) >> 16, rt = id - ct * nt, b = x % FR_AHEAD;
          const int rr = min(16 * rt + li, n - 1);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const size_t at = rr + (size_t)n * min(16 * ct + F::col(lg, i), n - 1);
            if (HP) g[b][i] = Gp[at];
            if (MID) h[b][i] = Gm[at];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (mid && hasp) form(std::true_type{}, std::true_type{});
    else if (mid) form(std::false_type{}, std::true_type{});
    else if (hasp) form(std::true_type{}, std::false_type{});
    else form(std::false_type{}, std::false_type{});

    // tiles of column pn to the panel buffer
    auto hand_over = [&](int pn) {
      C* const row = reinterpret_cast<C*>(Pb + (size_t)(pn & 1) * np * UN);
      HZ_FR_TILES(if (ct == pn) {
        const int r = 16 * rt + li;
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {
          const int c = F::col(lg, i);
          C v;
          v.x = re[t][i];
          v.y = im[t][i];
          row[unit(r, c / CU) * CU + c % CU] = v;
        }
      })
    };
    hand_over(0);
    __syncthreads();

    for (int pc = 0; pc < nt; ++pc) {
      const FrUnit* const P = Pb + (size_t)(pc & 1) * np * UN;
      __syncthreads();  // the panel is there
      // ---- pivot rows of the other columns to LDS (and out of the tiles);
      // the panel's own tiles take the eliminated panel
      const int rows = __builtin_amdgcn_readfirstlane(*prows);
      HZ_FR_TILES(if (ct == pc) {
        const int r = 16 * rt + li;
        const C* const row = reinterpret_cast<const C*>(P);
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {
          const int c = F::col(lg, i);
          const C v = row[unit(r, c / CU) * CU + c % CU];
          re[t][i] = v.x;
          im[t][i] = v.y;
        }
      } else if (ct < nt && (rows >> rt & 1)) {
        const int ps = pslot[16 * rt + li];
        if (ps >= 0) {
          C* const row = reinterpret_cast<C*>(AK);
          _Pragma("unroll") for (int i = 0; i < 4; ++i) {
            const int c = 16 * ct + F::col(lg, i);
            C v;
            v.x = re[t][i];
            v.y = im[t][i];
            row[unit(c, ps / CU) * CU + ps % CU] = v;
            re[t][i] = (T)0;
            im[t][i] = (T)0;
          }
        }
      })
      __syncthreads();  // its pivot rows are there

      // ---- A(:, c) += P A(pivot rows, c) on the matrix cores: tile
      // (transposed) += AK^T P^T, lane group lg holding steps 4 lg .. 4 lg + 3.
      // The products are summed from zero and added once: summed onto the tile,
      // each of the 32 would round at the tile's magnitude (up to 3.4 times the
      // error of the inverse).
#define HZ_FR_UPDATE()                                                         \
  {                                                                            \
    const int r = 16 * rt + li, c = 16 * ct + li;                              \
    C p[4], q[4];                                                              \
    _Pragma("unroll") for (int u = 0; u < 4 / CU; ++u) {                       \
      const FrUnit pu = P[unit(r, lg * (4 / CU) + u)];                         \
      const FrUnit qu = AK[unit(c, lg * (4 / CU) + u)];                        \
      _Pragma("unroll") for (int e = 0; e < CU; ++e) {                         \
        p[u * CU + e] = reinterpret_cast<const C*>(&pu)[e];                    \
        q[u * CU + e] = reinterpret_cast<const C*>(&qu)[e];                    \
      }                                                                        \
    }                                                                          \
    V tr = {}, ti = {};                                                        \
    _Pragma("unroll") for (int s = 0; s < 4; ++s) {                            \
      tr = F::mfma(q[s].x, p[s].x, tr);                                        \
      ti = F::mfma(q[s].x, p[s].y, ti);                                        \
      tr = F::mfma(-q[s].y, p[s].y, tr);                                       \
      ti = F::mfma(q[s].y, p[s].x, ti);                                        \
    }                                                                          \
    re[t] += tr;                                                               \
    im[t] += ti;                                                               \
  }
      if (pc + 1 < nt) {
        HZ_FR_TILES(if (ct == pc + 1) HZ_FR_UPDATE())
        hand_over(pc + 1);
      }
      __syncthreads();  // the next panel's column is there
      HZ_FR_TILES(if (ct < nt && ct != pc && ct != pc + 1) HZ_FR_UPDATE())
#undef HZ_FR_UPDATE
    }

    // ---- the inverse: element (r, l) goes to (kof[r], piv[l])
    HZ_FR_TILES({
      const int r = 16 * rt + li;
      if (ct < nt && r < n) {
        const int ro = kof[r];
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {
          const int c = 16 * ct + F::col(lg, i);
          if (c < n) {
            C v;
            v.x = re[t][i];
            v.y = im[t][i];
            Gj[ro + (size_t)n * piv[c]] = v;
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    })
    __syncthreads();  // the inverse is stored
  }
#undef HZ_FR_TILES
}

template <typename T, int TPW, int NQ>
void launch_reg(hz_problem* p, typename Cx<T>::t* G, const PlaneTabs& tb, int blocks, int nt, int* st, int mode, int m,
                typename Cx<T>::t* Gb, int jbeg, int jend, hipStream_t s) {
  const size_t np = 16 * (size_t)nt, lds = 3 * np * 16 * sizeof(typename Cx<T>::t) + (3 * np + 4) * sizeof(int);
  set_max_lds((const void*)&k_factor_reg<T, TPW, NQ>, lds);
  hipLaunchKernelGGL((k_factor_reg<T, TPW, NQ>), dim3((unsigned)blocks), dim3(FR_THREADS), lds, s, G, tb, (int)p->nx,
                     (int)p->ny, nt, st, p->d_splane.as<int>(), mode, m, Gb, jbeg, jend);
  HZ_HIP(hipGetLastError());
}

}  // namespace

bool launch_factor_reg(hz_problem* p, int prec, const PlaneTabs& tb, int blocks, int* st, int mode, int m, void* G,
                       void* Gb, int jbeg, int jend, hipStream_t s) {
  const int nt = ((int)p->nx + 15) / 16, tiles = (nt * nt + FR_TWAVES - 1) / FR_TWAVES;
#define HZ_FR(T, TPW, NQ)                                                         \
  if (tiles <= TPW) {                                                             \
    typedef Cx<T>::t C;                                                           \
    launch_reg<T, TPW, NQ>(p, (C*)G, tb, blocks, nt, st, mode, m, (C*)Gb, jbeg, jend, s); \
    return true;                                                                  \
  }
  // Tiles a wave, rows a panel lane: nx up to 64, 96, 128, 160, 192, 208
  // (complex128: 64, 96, 128, 144).  The line lies where a wave's tiles no longer
  // fit its 256 registers; below it the registers win at every width.  Whole
  // factorisations, panel by panel in memory -> here: complex64 24 x 22 x 28
  // 0.96 -> 0.54 ms; half chains, whole before: 64^3 10.8 -> 1.55, 112^3 46.0 ->
  // 7.5, 140^3 88.5 -> 15.1, complex128 64^3 11.3 -> 2.4, 128^3 78.0 -> 13.3; half
  // chains before and now: 200^3 136.8 -> 42.8.  The errors of a plane solve are those of before or smaller
  // (one-directional sweeps against 64 bits: complex64 64^3 3.4e-7 -> 2.8e-7, 200 x
  // 30 x 12 3.9e-5 -> 2.7e-5; complex128 64^3 1.11e-15 -> 0.91e-15).  What bounds
  // it: one compute unit a chain and, in it, the panel wave; at 200 columns the
  // matrix units are busy 2.1e10 of 3.8e10 wave cycles, half of which are waits.
  if (prec == HZ_PREC_C64) {
    HZ_FR(float, 3, 1)
    HZ_FR(float, 6, 2)
    HZ_FR(float, 10, 2)
    HZ_FR(float, 15, 3)
    HZ_FR(float, 21, 3)
    HZ_FR(float, 25, 4)
  } else {
    HZ_FR(double, 3, 1)
    HZ_FR(double, 6, 2)
    HZ_FR(double, 10, 2)
    HZ_FR(double, 12, 3)
  }
#undef HZ_FR
  return false;
}

}  // namespace hz
