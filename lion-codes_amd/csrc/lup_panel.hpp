// lup_panel.hpp -- panel LUP determinant kernels for gfx950 (CDNA4), n = 17..64.
//
// The same factorisation as lup_kernel.hpp in fused arithmetic, element for
// element and bit for bit, blocked by panels of four columns:
//
//   tile layout   The whole matrix stays in registers in the result layout of
//                 v_mfma_f64_4x4x4_4b: lane = col + 4*block + 16*i.  A wave
//                 holds G = 2 matrices (n <= 32, in batches that fill the
//                 device) or one; a matrix has 16/G lane-rows by 4
//                 lane-columns, R row slots and C column slots, and the real
//                 and imaginary parts are separate registers.  Column slot p
//                 is panel p.
//   panel layout  A panel (four columns of every row) goes through LDS into
//                 one row per lane.  Its four steps -- pivot search, pivot row
//                 to every lane, reciprocal, multipliers, update of the
//                 panel's later columns -- then cost one instruction per
//                 operation for all rows, and the row's position, scale and
//                 criterion are held once.
//
// After a panel its four raw pivot rows go to LDS, each lane takes one column
// of them and applies the panel's earlier steps to its four elements, and the
// trailing slots are updated with two MFMAs (four of the eight real products
// a panel adds to an element in each) per slot, row slot and part.
//
// The bits.  v_mfma_f64_4x4x4 adds its four products to each element as a
// chain of FMAs in ascending k (measured against that chain on 10^6 random
// tiles, subnormal, overflowing and non-finite ones included), so operands
// ordered (-lx, ly) and (ux, uy) for the real part, (-lx, ly) and (uy, -ux)
// for the imaginary part give every element the rounding steps of
// update_slots, in its order.  The pivot is searched in the upper words of
// the criteria first, which decides all columns but ties (PivotSearch).
//
// What bounds it.  MFMA and vector instructions share one FP64 pipe (they do
// not overlap, and alternating them is slower than running them in runs), so
// a step costs its issue: an n = 32 wave (two matrices) issues 3814
// instructions, 312 of them MFMAs of 16 cycles, where lup_det_kernel issued
// 6167; at two waves per SIMD they fill 73% of the cycles and LDS is busy for
// 45%.  The rest is the latency of the serial search, pivot row and
// reciprocal.  65536 x n = 32: 482 -> 398 us; above n = 56 the tile leaves
// room for one wave per SIMD only (n = 64: 82 -> 49 ns per determinant).
//
// H = 2 (one matrix, two waves) is for batches with fewer matrices than CUs,
// where a wave has a SIMD to itself and the trailing update is most of its
// time: both waves take the panel's steps, each holds and updates every other
// column slot, and a raw panel goes to the other wave through one of two
// shared buffers, with one barrier per panel.
#pragma once

#include "lup_kernel.hpp"

namespace lufqhe {

// Matrices per wave: the panel layout gives every row a lane.
constexpr int panel_groups(int n) { return n <= 32 ? 2 : 1; }

// LDS of one wave in double2.  Strides keep the accesses on distinct banks:
// rows of a panel 5 apart (tile rows of 16 lanes, and one row per lane), the
// pivot rows 4 modulo 16 apart, the two matrices of a wave 4 (a quarter of the
// banks: with 8, 20% of the LDS cycles of n = 32 were conflicts, now 8%; 0.9%
// of its time).
constexpr int kPanelStride = 5;
constexpr int panel_row_stride(int n) { return ((4 * ((n + 3) / 4) + 11) / 16) * 16 + 4; }
constexpr int panel_area(int g) { return 64 / g * kPanelStride + (g > 1 ? 4 : 0); }
constexpr int panel_pivot_area(int n) { return 4 * panel_row_stride(n) + 4; }
// One wave's own areas, and a workgroup's of h waves per matrix: with two
// also the raw panels they hand each other (two, in turn) and their row maxima.
constexpr int panel_wave_lds(int n, int g) {
  return g * (panel_area(g) + panel_pivot_area(n)) + 16;
}
constexpr int panel_lds(int n, int g, int h) {
  return h * panel_wave_lds(n, g) + (h > 1 ? 2 * panel_area(1) + 64 : 0);
}

// Row slots a matrix still needs when panel p is searched (p = 0: all).  Once
// the rows left fit in one slot less and at least kMinPanelsLeft panels
// follow, the rows of the last slot move into the places of finished rows:
// their trailing columns through the panel's LDS area (one slot is written,
// only the places that take a row read), the row's state by ds_bpermute.  All
// later panels then update, write and read one slot less.  Measured with and
// without, ns per determinant: n = 32 6.55 / 6.88 (with pivot rows still passed
// through LDS; now 6.23), n = 40 13.4 / 14.6, n = 48 18.5 / 19.7, n = 52
// 24.1 / 30.8 (one slot less after the first panel, and so no spills at two
// waves per SIMD), n = 64 48.7 / 50.4.  kMinPanelsLeft = 1, 3 and 4 are within
// 1% at n = 26..64.
constexpr int kMinPanelsLeft = 2;
constexpr int panel_slots(int n, int g, int p) {
  const int rg = 16 / g, c = (n + 3) / 4;
  int r = (n + rg - 1) / rg;
  for (int q = 0; q < p; ++q)
    if (r > 1 && n - 4 * (q + 1) <= (r - 1) * rg && c - 1 - q >= kMinPanelsLeft) --r;
  return r;
}

struct PanelSlots {
  int at[17];
};
constexpr PanelSlots panel_slot_table(int n, int g) {
  PanelSlots t{};
  for (int p = 0; p <= 16; ++p) t.at[p] = panel_slots(n, g, p);
  return t;
}

template <int N, int G, int H>
struct PanelTile {
  static constexpr PanelSlots slots = panel_slot_table(N, G);
  static_assert(H == 1 || (H == 2 && G == 1), "waves per matrix");
  static_assert(G == 1 || G == 2, "matrices per wave");
  static constexpr int L = 64 / G;             // panel layout: lanes (rows) per matrix
  static constexpr int RG = 16 / G;            // tile layout: lane-rows per matrix
  static constexpr int R = (N + RG - 1) / RG;  // row slots
  static constexpr int C = (N + 3) / 4;        // column slots = panels
  static constexpr int CL = (C + H - 1) / H;   // column slots of one wave
  static_assert(N <= L && R * RG <= L, "one lane per row");
  static_assert(panel_row_stride(N) >= 4 * C, "a pivot row");
};

__device__ __forceinline__ double mfma_4x4x4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ double readlane_d(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double neg_if(double v, unsigned mask) {
  return __hiloint2double(__double2hiint(v) ^ (int)mask, __double2loint(v));
}

// Bits of group g in a wave ballot.
template <int G>
__device__ __forceinline__ auto group_bits(uint64_t m, int g) {
  if constexpr (G == 1) {
    return m;
  } else {
    return g == 0 ? (uint32_t)m : (uint32_t)(m >> 32);
  }
}
template <int G>
__device__ __forceinline__ int group_first(uint64_t m, int g) {  // m has a bit in the group
  if constexpr (G == 1) return __builtin_ctzll(m);
  else return __builtin_ctz(group_bits<G>(m, g));
}

// The lanes `bits` (of one group) in every group.
template <int G>
constexpr uint64_t group_lanes(uint64_t bits) {
  uint64_t r = 0;
  for (int g = 0; g < G; ++g) r |= bits << (g * (64 / G));
  return r;
}

// Bits of `m` below this lane, in its group.
template <int G>
__device__ __forceinline__ int group_rank(uint64_t m, int lane) {
  const int lo = __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0);
  if constexpr (G == 1) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), lo);
  } else {
    const int hi = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), 0);
    return lane < 32 ? lo : hi;
  }
}

__device__ __forceinline__ double bpermute_d(int addr, double v) {
  const int lo = __builtin_amdgcn_ds_bpermute(addr, __double2loint(v));
  const int hi = __builtin_amdgcn_ds_bpermute(addr, __double2hiint(v));
  return __hiloint2double(hi, lo);
}

// RN(1/d) for d in [0.25, 2); any finite value for d == 0.
__device__ __forceinline__ double recip_pivot(double d) {
  double dd;
  asm("v_max_f64 %0, %1, %2" : "=v"(dd) : "v"(d), "s"(0.125));
  double r = __builtin_amdgcn_rcp(dd);
  double e = fma(-dd, r, 1.0);
  r = fma(r, e, r);
  e = fma(-dd, r, 1.0);
  r = fma(r, e, r);
  const double rem = fma(-dd, r, 1.0);
  return fma(rem, r, r);
}

// One pivot search over the column (x, y) of every matrix of the wave.
// `fast` names one lane per group from the upper words of the criteria,
// clamped to the range in which quot_rn's corrected quotient is exact: a
// criterion outside it wins only if it is the single one there, or ties with
// the others at the bound.  `settle` decides the columns where upper words
// tie (`slow`).
constexpr unsigned kKeyLo = 0x08F00000u;  // upper word of 2^-880
constexpr unsigned kKeyHi = 0x7BF00000u;  // upper word of 2^960

template <int G, int POLICY>
struct PivotSearch {
  static constexpr int L = 64 / G;

  static __device__ __forceinline__ uint64_t fast(double x, double y, double sc, double rs,
                                                  uint64_t am) {
    double c;
    unsigned lo = kKeyLo, hi = kKeyHi;
    if constexpr (POLICY == POLICY_CROUT_REF) {
      const double q0 = fabs(x) * rs;
      const double r = fma(-q0, sc, fabs(x));
      c = fma(r, rs, q0);
    } else {
      c = fabs(x) + fabs(y);
      lo = 0u;
      hi = 0x7FEFFFFFu;
    }
    const int k = (int)min(max((unsigned)__double2hiint(c), lo), hi);
    const int key = __builtin_amdgcn_inverse_ballot_w64(am) ? k : -1;
    return __builtin_amdgcn_ballot_w64(key == group_max_i<L>(key));
  }

  // `want` is G, or more to have every column settled
  static __device__ __forceinline__ bool slow(uint64_t m, int want) {
    return __builtin_popcountll(m) != want;
  }

  static __device__ __forceinline__ uint64_t settle(double x, double y, double sc, double rs,
                                                    uint64_t am, int pos) {
    const bool act = __builtin_amdgcn_inverse_ballot_w64(am);
    double c;
    if constexpr (POLICY == POLICY_CROUT_REF)
      c = quot_rn(fabs(x), sc, rs, act);
    else
      c = fabs(x) + fabs(y);
    c = vmin_f64(c, kDblMax);
    // every lane takes part in each maximum
    const int k1 = act ? __double2hiint(c) : -1;
    const int m1 = group_max_i<L>(k1);
    bool in = k1 == m1;
    const int k2 = in ? (__double2loint(c) ^ (int)0x80000000) : (int)0x80000000;
    const int m2 = group_max_i<L>(k2);
    in = in && k2 == m2;
    const int k3 = in ? tie_key<POLICY>(pos) : -1;
    const int m3 = group_max_i<L>(k3);
    return __builtin_amdgcn_ballot_w64(in && k3 == m3);
  }
};

template <int G>
__device__ __forceinline__ int select_group(const int (&v)[G], int g) {
  int r = v[0];
#pragma unroll
  for (int i = 1; i < G; ++i) r = g == i ? v[i] : r;
  return r;
}

template <int N, int G, int H, int POLICY>
__device__ __forceinline__ void panel_task(const BatchArgs& args, int64_t task,
                                           double2* __restrict__ lds_all, int lane, int wave) {
  using T = PanelTile<N, G, H>;
  constexpr int L = T::L, RG = T::RG, R = T::R, C = T::C, CL = T::CL;
  constexpr int PS = kPanelStride, PG = panel_area(G);
  constexpr int US = panel_row_stride(N), GS = panel_pivot_area(N);
  double2* lds = lds_all + (H > 1 ? wave * panel_wave_lds(N, G) : 0);
  double2* shared = lds_all + H * panel_wave_lds(N, G);  // H > 1
  double2* pan = lds;               // the panel, then its multipliers
  double2* ub = pan + G * PG;       // its pivot rows
  int* pjv = reinterpret_cast<int*>(ub + G * GS);  // step each row was pivot of

  // tile layout (MFMA 4x4x4 result): lane = col + 4*block + 16*i
  const int jc = lane & 3, blk = (lane >> 2) & 3, ti = lane >> 4;
  const int gt = G == 1 ? 0 : blk >> 1;
  const int rb = 4 * (blk & (4 / G - 1)) + ti;
  // A operand layout: lane = i + 4*block + 16*k
  const int rba = 4 * (blk & (4 / G - 1)) + jc;
  // panel layout: one row (or column) per lane
  const int gp = lane / L, row = lane % L;
  double2* mine = pan + gp * PG + row * PS;           // this row of the panel
  // this lane's element of row slot 0 and this row in raw panel p
  auto raw_tile = [&](int p) {
    return (H > 1 ? shared + (p & 1) * PG : pan + gt * PG) + rb * PS + jc;
  };
  auto raw_row = [&](int p) { return H > 1 ? shared + (p & 1) * PG + row * PS : mine; };
  auto raw_sync = [&]() {
    if constexpr (H > 1)
      __syncthreads();
    else
      wave_lds_sync();
  };

  const int64_t i_t = task * G + gt;
  const int64_t i_p = task * G + gp;
  const bool ok_t = i_t < args.count, ok_p = i_p < args.count;

  double ax[R][CL], ay[R][CL];  // slot q holds columns 4 * (q * H + wave) ..
  int bad_perm = 0;
  if (args.src == SRC_FQHE) {
    double2 z = make_double2(0.0, 0.0);
    double g = 0.0;
    if (ok_p && row < N) {
      const double2* __restrict__ base = args.offs ? args.A + args.offs[i_p] : args.A + i_p * args.stride;
      int src = row;
      if (args.row_perm) {
        const uint8_t* __restrict__ perm =
            args.row_perm + (args.perm_offs ? args.perm_offs[i_p] : i_p * N);
        src = perm[row];
        if (src >= N) bad_perm = 1;
        src = min(src, N - 1);
      }
      z = base[src];
      g = fqhe_gauss(z);
    }
    double2 pw = make_double2(1.0, 0.0);
#pragma unroll
    for (int s = 0; s < C; ++s) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (4 * s + c < N) {
          mine[c] = make_double2(pw.x * g, pw.y * g);
          pw = cmul_ref(pw, z);
        } else {
          mine[c] = make_double2(0.0, 0.0);
        }
      }
      wave_lds_sync();
#pragma unroll
      for (int t = 0; t < R; ++t) {
        if (H > 1 && s % H != wave) continue;
        const double2 v = pan[gt * PG + (rb + RG * t) * PS + jc];
        ax[t][s / H] = v.x;
        ay[t][s / H] = v.y;
      }
      wave_lds_sync();
    }
  } else {
    const double2* __restrict__ base = nullptr;
    if (ok_t) base = args.offs ? args.A + args.offs[i_t] : args.A + i_t * args.stride;
    const int64_t ld = args.offs ? (int64_t)N : args.ld;
    const uint8_t* __restrict__ perm = nullptr;
    if (ok_t && args.row_perm)
      perm = args.row_perm + (args.perm_offs ? args.perm_offs[i_t] : i_t * N);
#pragma unroll
    for (int t = 0; t < R; ++t) {
      const int r = rb + RG * t;
      if (ok_t && r < N) {
        int src = r;
        if (perm) src = min((int)perm[r], N - 1);
        const double2* __restrict__ rp = base + (int64_t)src * ld;
#pragma unroll
        for (int q = 0; q < CL; ++q) {
          const int col = jc + 4 * (q * H + wave);
          const double2 v = (col < N) ? rp[col] : make_double2(0.0, 0.0);
          ax[t][q] = v.x;
          ay[t][q] = v.y;
        }
      } else {
#pragma unroll
        for (int q = 0; q < CL; ++q) ax[t][q] = ay[t][q] = 0.0;
      }
    }
    if (args.row_perm && ok_p && row < N) {
      const uint8_t* pp = args.row_perm + (args.perm_offs ? args.perm_offs[i_p] : i_p * N);
      if (pp[row] >= N) bad_perm = 1;
    }
  }

  int pos = row;
  const uint64_t rows_mask = group_lanes<G>((1ull << (N - 1) << 1) - 1ull);
  uint64_t am = rows_mask;  // active rows
  double sc = 1.0, rs = 1.0;
  int rej = -1;
  int want = G;
  if constexpr (POLICY == POLICY_CROUT_REF) {
    double* scd = reinterpret_cast<double*>(H > 1 ? shared + 2 * PG : pan);
#pragma unroll
    for (int t = 0; t < R; ++t) {
      double m = fabs(ax[t][0]);
#pragma unroll
      for (int q = 1; q < CL; ++q)
        if (jc + 4 * (q * H + wave) < N) m = vmax_f64(m, fabs(ax[t][q]));
      m = lanerow_max<4>(m);
      if (jc == 0) scd[wave * 64 + gt * L + rb + RG * t] = m;
    }
    raw_sync();
    double m = scd[lane];
    if constexpr (H > 1) m = vmax_f64(m, scd[64 + lane]);
    wave_lds_sync();
    const bool bad = row < N && m < kRowScaleMin;
    sc = (row < N && !bad) ? m : 1.0;
    rs = sc <= 0x1p960 ? 1.0 / sc : __builtin_nan("");
    // a row scale without a reciprocal: its criteria need divisions
    if (__builtin_amdgcn_ballot_w64(!(sc <= 0x1p960)) != 0) want = 255;
    const int first_bad = group_max_i<L>(bad ? 255 - row : -1);
    if (first_bad >= 0) rej = 255 - first_bad;
  }

  double dx = 1.0, dy = 0.0;
  int de = 0, prec = row;
  int zk[G];
#pragma unroll
  for (int g = 0; g < G; ++g) zk[g] = 255;

  const double* pd = reinterpret_cast<const double*>(pan);
  const double* ud = reinterpret_cast<const double*>(ub);
  const unsigned odd = (ti & 1) ? 0x80000000u : 0u;  // operand lanes with k odd
  const int ubase = (gt * GS + (ti >> 1) * US + 4 * wave + jc) * 2 + (ti & 1);
  const int ubase_y = (gt * GS + (ti >> 1) * US + 4 * wave + jc) * 2 + ((ti & 1) ^ 1);

  // panel 0 to LDS
  if (H == 1 || wave == 0) {
    double2* tile = raw_tile(0);
#pragma unroll
    for (int t = 0; t < R; ++t) tile[RG * t * PS] = make_double2(ax[t][0], ay[t][0]);
  }
  raw_sync();

#pragma unroll
  for (int p = 0; p < C; ++p) {
    constexpr int W = 4;
    const int nb = N - 4 * p < W ? N - 4 * p : W;
    const int R1 = T::slots.at[p], R2 = T::slots.at[p + 1];
    const bool trail = p + 1 < C;
    const int q0 = (p + 1) / H;  // the first of a wave's slots that may lie beyond the panel
    double px[W], py[W];
    int pa[W];  // LDS row of each pivot (double2)
    int pj = -1, tj[R];
    double Ax[R][2];
    double2 uc[W];
    double2 u[W][W], lp[W][W];  // G > 1: pivot rows after their steps, their multipliers
#pragma unroll
    for (int c = 0; c < W; ++c) {
      if (c >= nb) continue;
      const double2 v = raw_row(p)[c];
      px[c] = v.x;
      py[c] = v.y;
    }
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < W; ++j) {
      if (j >= nb) continue;
      const int k = 4 * p + j;
      using Search = PivotSearch<G, POLICY>;
      uint64_t m = Search::fast(px[j], py[j], sc, rs, am);
      double ux[W], uy[W];
      int ppos;
      // the pivot row of the panel to every lane of its group
      auto publish = [&]() {
        if constexpr (G == 1) {
          const int pl = __builtin_ctzll(m);
          ux[j] = readlane_d(px[j], pl);
          uy[j] = readlane_d(py[j], pl);
          ppos = __builtin_amdgcn_readlane(pos, pl);
          pa[j] = pl * PS;
#pragma unroll
          for (int cc = 0; cc < W; ++cc)
            if (cc > j && cc < nb) {
              ux[cc] = readlane_d(px[cc], pl);
              uy[cc] = readlane_d(py[cc], pl);
            }
        } else {
          wave_lds_sync();
          // The row as the panel began it and its multipliers are in LDS: every
          // lane reads those and takes the row's earlier steps itself (64 more
          // instructions per panel, but no write that a read then waits for:
          // LDS moves 64 B per clock and CU on writes and was busy for 70% of
          // n = 32; 6.59 -> 6.33 ns per determinant there, 5.06 -> 4.90 at
          // n = 26; 45% now, with the areas' spacing too).  With one matrix per wave v_readlane is as fast (n = 40)
          // or faster (n = 64, 4%).
          int pl[G];
#pragma unroll
          for (int g = 0; g < G; ++g) pl[g] = group_first<G>(m, g);
          int pp[G], at[G];
#pragma unroll
          for (int g = 0; g < G; ++g) {
            pp[g] = __builtin_amdgcn_readlane(pos, g * L + pl[g]);
            at[g] = g * PG + pl[g] * PS;
          }
          ppos = select_group<G>(pp, gp);
          pa[j] = select_group<G>(at, gp);
          const double2* r = pan + pa[j];
          double2 v[W];
#pragma unroll
          for (int cc = 0; cc < W; ++cc)
            if (cc < nb) v[cc] = r[cc];
#pragma unroll
          for (int q = 0; q < W; ++q)
            if (q < j) {
              lp[j][q] = v[q];
#pragma unroll
              for (int cc = 0; cc < W; ++cc)
                if (cc >= j && cc < nb) {
                  v[cc].x = fma(v[q].x, u[q][cc].x, v[cc].x);
                  v[cc].y = fma(v[q].x, u[q][cc].y, v[cc].y);
                  v[cc].x = fma(v[q].y, u[q][cc].y, v[cc].x);
                  v[cc].y = fma(-v[q].y, u[q][cc].x, v[cc].y);
                }
            }
#pragma unroll
          for (int cc = 0; cc < W; ++cc)
            if (cc >= j && cc < nb) {
              ux[cc] = v[cc].x;
              uy[cc] = v[cc].y;
              u[j][cc] = v[cc];
            }
          wave_lds_sync();
        }
      };
      publish();
      if (__builtin_expect(Search::slow(m, want), 0)) {
        m = Search::settle(px[j], py[j], sc, rs, am, pos);
        publish();
      }
      am &= ~m;
      const bool is_piv = __builtin_amdgcn_inverse_ballot_w64(m);

      if (trail && j < W - 1) pj = is_piv ? j : pj;
      if (trail && j == W - 2) {
        // each row's step so far, for the tile lanes
        pjv[lane] = pj;
        wave_lds_sync();
#pragma unroll
        for (int t = 0; t < R; ++t)
          if (t < R1) tj[t] = pjv[gt * L + rb + RG * t];
      }
      if (trail && j == W - 1) {
        // raw pivot rows to LDS
        int pl[G];
#pragma unroll
        for (int g = 0; g < G; ++g) pl[g] = group_first<G>(m, g);
        const int pt = select_group<G>(pl, gt);
#pragma unroll
        for (int t = 0; t < R; ++t) {
          if (t >= R1) continue;
          const int q = rb + RG * t == pt ? j : tj[t];
          if (q >= 0) {
            double2* dst = ub + gt * GS + q * US + 4 * wave + jc;
#pragma unroll
            for (int c = 0; c < CL; ++c)
              if (c >= q0) dst[4 * H * c] = make_double2(ax[t][c], ay[t][c]);
          }
        }
        wave_lds_sync();
        // pivot rows: the steps of this panel before each row's own
        double2* up = ub + gp * GS + (4 * C >= L ? row : min(row, 4 * C - 1));
        double2 l[W][W];
#pragma unroll
        for (int i = 0; i < W; ++i) uc[i] = up[i * US];
#pragma unroll
        for (int i = 1; i < W; ++i)
#pragma unroll
          for (int q = 0; q < W; ++q)
            if (q < i) l[i][q] = G > 1 ? lp[i][q] : pan[pa[i] + q];
#pragma unroll
        for (int q = 0; q < W; ++q)
#pragma unroll
          for (int i = 1; i < W; ++i)
            if (q < i) {
              uc[i].x = fma(l[i][q].x, uc[q].x, uc[i].x);
              uc[i].y = fma(l[i][q].x, uc[q].y, uc[i].y);
              uc[i].x = fma(l[i][q].y, uc[q].y, uc[i].x);
              uc[i].y = fma(-l[i][q].y, uc[q].x, uc[i].y);
            }
#pragma unroll
        for (int i = 1; i < W; ++i) up[i * US] = uc[i];
        wave_lds_sync();
      }

      const int kp = __builtin_amdgcn_frexp_exp(vmax_abs_f64(ux[j], uy[j]));
      const double psx = ldexp(ux[j], -kp);
      const double psy = ldexp(uy[j], -kp);
      const double den = fma(psx, psx, psy * psy);
      const uint64_t zb = __builtin_amdgcn_ballot_w64(den == 0.0);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int z = group_bits<G>(zb, g) != 0 ? k + 1 : 255;
        zk[g] = min(zk[g], z);
        asm volatile("" : "+s"(zk[g]));
      }
      const double nx = fma(dx, psx, -(dy * psy));
      const double ny = fma(dx, psy, dy * psx);
      dx = nx;
      dy = ny;
      de += kp;
      asm volatile("" : "+v"(de), "+v"(dx), "+v"(dy));
      prec = __builtin_amdgcn_inverse_ballot_w64(group_lanes<G>(1ull << k)) ? ppos : prec;

      if (k + 1 < N) {
        const double rden = recip_pivot(den);
        const double ir = ldexp(psx * rden, -kp);
        const double ii = ldexp(-(psy * rden), -kp);
        const double lx = fma(px[j], ir, -(py[j] * ii));
        const double ly = fma(py[j], ir, px[j] * ii);
        double nl = -lx;
        asm("" : "+v"(nl));
        if (trail || (G > 1 && j + 1 < nb)) mine[j] = make_double2(nl, ly);
#pragma unroll
        for (int cc = 0; cc < W; ++cc)
          if (cc > j && cc < nb) {
            px[cc] = fma(nl, ux[cc], px[cc]);
            py[cc] = fma(nl, uy[cc], py[cc]);
            px[cc] = fma(ly, uy[cc], px[cc]);
            py[cc] = fma(-ly, ux[cc], py[cc]);
          }
        pos = pos == k ? ppos : pos;
        pos = is_piv ? k : pos;
      }
    }
    if (!trail) continue;

    wave_lds_sync();
    int sa[R], st[R];  // place each row slot's row comes from (operand and tile lanes)
#pragma unroll
    for (int t = 0; t < R; ++t) {
      sa[t] = rba + RG * t;
      st[t] = rb + RG * t;
    }
    if (R2 < R1) {
      // finished places below R2 row slots take the active rows above, in order
      const int low = R2 * RG;
      const uint64_t lowm = group_lanes<G>((1ull << low) - 1ull);
      const uint64_t up = am & ~lowm, dead = ~am & lowm;
      const int ru = group_rank<G>(up, lane), rd = group_rank<G>(dead, lane);
      int nu[G];
#pragma unroll
      for (int g = 0; g < G; ++g) nu[g] = __builtin_popcountll(group_bits<G>(up, g));
      if (__builtin_amdgcn_inverse_ballot_w64(up)) pjv[gp * L + ru] = row;
      wave_lds_sync();
      const uint64_t take =
          dead & __builtin_amdgcn_ballot_w64(rd < select_group<G>(nu, gp));
      int from = row;
      if (__builtin_amdgcn_inverse_ballot_w64(take)) from = pjv[gp * L + rd];
      wave_lds_sync();
      pjv[lane] = from;
      const int fl = (gp * L + from) * 4;
      pos = __builtin_amdgcn_ds_bpermute(fl, pos);
      if constexpr (POLICY == POLICY_CROUT_REF) {
        sc = bpermute_d(fl, sc);
        rs = bpermute_d(fl, rs);
      }
      am = (am & lowm) | take;
      wave_lds_sync();
#pragma unroll
      for (int t = 0; t < R; ++t) {
        if (t >= R2) continue;
        sa[t] = pjv[gt * L + rba + RG * t];
        st[t] = pjv[gt * L + rb + RG * t];
      }
    }
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (t < R2) Ax[t][h] = pd[(gt * PG + sa[t] * PS) * 2 + 4 * h + ti];
    if (R2 < R1) {
      // the moved rows' trailing columns, through the panel's area
      wave_lds_sync();
      constexpr int SW = 4;  // column slots a round moves
      static_assert(RG * (4 * SW + 1) <= L * PS, "staging area");
      double2* stage = pan + gt * PG;
#pragma unroll
      for (int s0 = 0; s0 < CL; s0 += SW) {
        if (s0 + SW <= q0) continue;
#pragma unroll
        for (int c = 0; c < SW; ++c)
          if (s0 + c >= q0 && s0 + c < CL)
            stage[rb * (4 * SW + 1) + 4 * c + jc] =
                make_double2(ax[R1 - 1][s0 + c], ay[R1 - 1][s0 + c]);
        wave_lds_sync();
#pragma unroll
        for (int t = 0; t < R; ++t) {
          if (t >= R2) continue;
          // by value, so that no address into the tile is ever selected
          double2 v[SW];
#pragma unroll
          for (int c = 0; c < SW; ++c)
            if (s0 + c >= q0 && s0 + c < CL) v[c] = make_double2(ax[t][s0 + c], ay[t][s0 + c]);
          if (st[t] >= R2 * RG) {
            const double2* row_t = stage + (st[t] - R2 * RG) * (4 * SW + 1) + jc;
#pragma unroll
            for (int c = 0; c < SW; ++c)
              if (s0 + c >= q0 && s0 + c < CL) v[c] = row_t[4 * c];
          }
#pragma unroll
          for (int c = 0; c < SW; ++c)
            if (s0 + c >= q0 && s0 + c < CL) {
              ax[t][s0 + c] = v[c].x;
              ay[t][s0 + c] = v[c].y;
            }
        }
        wave_lds_sync();
      }
    }
    // trailing update, the next panel first
#pragma unroll
    for (int q = 0; q < CL; ++q) {
      if (q < q0) continue;
      if (H == 1 || q > q0 || q * H + wave > p) {
        double Bx[2], By[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          Bx[h] = ud[ubase + (2 * h * US + 4 * H * q) * 2];
          By[h] = neg_if(ud[ubase_y + (2 * h * US + 4 * H * q) * 2], odd);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 0; t < R; ++t) {
            if (t >= R2) continue;
            ax[t][q] = mfma_4x4x4(Ax[t][h], Bx[h], ax[t][q]);
            ay[t][q] = mfma_4x4x4(Ax[t][h], By[h], ay[t][q]);
          }
      }
      if (q == q0) {
        if (H == 1 || (p + 1) % H == wave) {
          double2* tile = raw_tile(p + 1);
#pragma unroll
          for (int t = 0; t < R; ++t)
            if (t < R2) tile[RG * t * PS] = make_double2(ax[t][q], ay[t][q]);
        }
        if (H == 1) wave_lds_sync();
      }
    }
    if (H > 1) raw_sync();
  }

  // sign of the row permutation: one per step whose pivot was not in place
  const uint64_t swaps = __builtin_amdgcn_ballot_w64(prec != row) & rows_mask;
  int par[G];
#pragma unroll
  for (int g = 0; g < G; ++g) par[g] = __builtin_popcountll(group_bits<G>(swaps, g)) & 1;
  const double sg = select_group<G>(par, gp) ? -1.0 : 1.0;
  const int zfirst = select_group<G>(zk, gp);

  renorm(dx, dy, de);
  GroupResult res;
  res.mx = sg * dx;
  res.my = sg * dy;
  res.e = de;
  res.info = (rej >= 0) ? -(rej + 1) : zfirst == 255 ? 0 : zfirst;
  if (args.row_perm && group_max_i<L>(bad_perm) > 0) res.info = kInfoBadPerm;
  if (ok_p && (H == 1 || wave == 0)) {
    const int64_t o = args.out_idx ? args.out_idx[i_p] : i_p;
    if (args.out.piv && row < N)
      args.out.piv[o * args.piv_stride + row] = (int8_t)(res.info < 0 ? -1 : prec);
    if (row == 0) write_result(args.out, o, res);
  }
}

template <int N, int G, int H, int POLICY, int OCC>
__global__ void __launch_bounds__(64 * H, OCC) lup_panel_kernel(BatchArgs args) {
  __shared__ double2 lds[panel_lds(N, G, H)];
  const int64_t task = blockIdx.x;
  if (task * G >= args.count) return;  // the whole workgroup
  const int wave = H > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  panel_task<N, G, H, POLICY>(args, task, lds, (int)(threadIdx.x & 63), wave);
}

}  // namespace lufqhe
