// Compact-derivative line solves split into segments, one wavefront per
// segment: 64 lines per block, K segments of ~32 rows per line.
//
// The pentalu-factored solve (class_derivatives.f90:425-466) is two
// second-order linear recurrences per line:
//   forward   y_i = r_i - p_i y_{i-2} - f_i y_{i-1}   (- beta y_{n-4} on row n-1)
//   backward  x_i = (y_i - e_i x_{i+2} - d_i x_{i+1}) / c_i   (- alpha x_3 on row 0)
// On a segment [s, e) the forward values are affine in the two incoming
// values: y_i = P_i + A_i y_{s-2} + B_i y_{s-1}, with P the recurrence run from
// zero and A, B its homogeneous responses to unit incoming values, which
// depend on the coefficients only and are tabulated at set-up (likewise
// x_i = Q_i + C_i x_e + D_i x_{e+1} backward).  Each wave loads its
// segment's inputs at once, runs P in registers, publishes its boundary
// values in LDS, chains the maps of the segments before it to get its
// incoming values, and corrects P inside the backward sweep; then the same
// backward, corrected as it is stored.  The result is the sequential solve
// re-associated (rounding-level differences only), with K times the
// wavefronts of one-lane-per-line and every load of a segment in flight
// together.
//
// What bounds it: HBM (16 B per point) when the chip is full, the chain of
// the wave's own latencies when it is not.  The coefficients are the same for
// every lane; they sit in the wave's vector registers, one per lane (a
// segment's 14 x 32 doubles are 7 register pairs, loaded once, coalesced),
// and reach the FMAs through v_readlane, which has no latency to wait for:
// 28 lane reads and 15 FP64 operations per row.  (Scalar loads, four rows per wait on a
// 24 KB table that the 16 KB scalar cache does not hold, kept a wave waiting.)
// Lane reads cost issue slots instead: on fields that stay in cache, pentadiagonal
// lines of 64 to 200 points along y and z take 5 to 20% longer than with scalar
// loads (38 x 200 x 200, one derivative along z, 13.4 us then and 16.5 now), all
// else less.  Blocks of up to 16 waves leave a wave 128 registers: the solves
// along y and z keep within them, those of contiguous lines put 7 to 9
// (tridiagonal) or 26 to 32 registers of a lane into scratch memory, and pairs
// 161 to 185 or 240 to 243.
// Where the factored matrix is tridiagonal (p = e = 0: the schemes of order 6
// and below) a second instance drops p, e, A, D and one of the two exchanged
// values: 20 lane reads and 11 operations.
// Measured, before (scalar loads, contiguous lines read and written lane by
// lane, blocks in launch order) and now: one derivative along x / y / z of
// 201 x 256 x 187, in cache, 80 / 75 / 88 -> 45 / 49 / 43 us (154 MB; a copy
// takes 31), all three from HBM 256 -> 186 us; six fields of 192 x 256 x 192
// 400 / 413 / 404 -> 205 / 238 / 255 us (4.4-3.6 TB/s); 64^3 16 -> 12 us;
// 49 152 contiguous lines of 192 points, one lane per line before, 130 -> 30 us.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <vector>

namespace mf {

constexpr int SEG_LEN = 32;     // longest segment, on lines of up to 16 of them
constexpr int SEG_LONG = 33;    // longest on the lines just beyond (an instance of its own)
// Whether the lines along y or z of a field of nx columns go in groups of
// `lines` aligned in memory: rows of whole cache lines (16 points), and few
// lanes lost at the rows' ends.  Six fields of 192 x 256 x 192 along y / z 253 / 272
// -> 238 / 253 us, three of 256^3 212 / 227 -> 191 / 200 us; the same time either
// way on fields that stay in cache (64^3, 496 x 64 x 60).
inline bool seg_aligned(int nx, int lines) {
  return nx % 16 == 0 && 16 * ((nx + lines - 1) / lines * lines - nx) <= 2 * nx;
}

// Contiguous lines: the wave shuffles 32-bit line offsets, so 64 lines that lie
// `stride` points apart have to stay within 2^31 points.
inline bool seg_fits(long stride) { return stride <= 0x7fffffffL / 64; }

constexpr int SEG_KMAX = 16;    // segments per line (wavefronts per block)
constexpr int SEG_PACK = 512;   // coefficient doubles per segment
constexpr int SEG_CHAIN = 64;   // doubles per chain table (4 per segment)

// Segmentation of a line of n points: K segments of seg_len(n, K) rows, the last
// one the rest (of several at least 8 rows: it holds the 7-point
// closure's inputs and row n-4).  Even segments, since a block takes as long
// as its longest.  Lines of 513 to 528 points (2^9 intervals and a few more)
// take 16 segments of up to 33 rows: 513 x 64 x 65, one derivative along x / y / z
// 300 / 299 / 293 us one lane per line, 25 / 85 / 82 us in segments (512 points:
// 24 / 80 / 80 us).  Pentadiagonal lines of 17 to 32 points take two segments, since
// their rows' 28 lane reads make one long wave: 32^3 along x / y / z 12.0 / 13.0 /
// 13.4 -> 9.8 / 8.9 / 8.9 us, 49 152 lines of 32 points 14.8 -> 12.4 us (400 000 of
// them, where the rows read twice count, 46.6 -> 49.2 us).  Tridiagonal ones keep
// one segment, which is as fast there and 10% faster on 400 000 lines.
inline int seg_count(int n, bool tri) {
  if (!tri && n >= 17 && n <= SEG_LEN) return 2;
  const int K = (n + SEG_LEN - 1) / SEG_LEN;
  return K > SEG_KMAX && n <= SEG_KMAX * SEG_LONG ? SEG_KMAX : K;
}
inline int seg_len(int n, int K) { return (n + K - 1) / K; }

// LDS doubles per wave: the forward and backward exchange arrays, 2 x 64
// each; on contiguous lines the wave's 64 x 16 transpose tile, whose start
// doubles as the forward exchange (the tile is idle between the loads and the
// last barrier), and the backward exchange
constexpr int SEG_TP = 17;  // pitch of the transpose tile
__host__ __device__ constexpr int seg_wave_doubles(bool xt) { return xt ? 64 * SEG_TP + 128 : 256; }
// dynamic LDS doubles of a block running a scheme of K segments
inline int seg_lds_doubles(int K, bool xt) { return seg_wave_doubles(xt) * K; }
// doubles of a scheme's table: the segments' packs, then the two chain tables
inline size_t seg_table_doubles(int K) { return (size_t)SEG_PACK * K + 2 * SEG_CHAIN; }

// The right-hand side sum_m dr_m f_m of an interior row is formed on the
// differences of its window,
//   s f_2 + sum_j t_j (f_{j+1} - f_j),
//   s = sum_m dr_m,  t_j = sum_{m > j} dr_m (j >= 2),  -sum_{m <= j} dr_m (j < 2),
// the same sum (s is the rounding residue of a derivative's weights) without
// the cancellation of the f_m themselves, for one subtraction per row.  The
// 7-point rows at the ends, whose rounding the closure's small pivots
// amplify, keep their weights as they are.
//
// A segment's pack, row k of the segment at seg_cw(tri) k:
//   s, t(0..3) | dr(0..4), p, f, e, d, 1/c, A, B, C, D      (14 per row)
//   s, t(0..3) | dr(0..4), f, d, 1/c, B, C                  (10 per row, tridiagonal)
// and, from 496, what the line's ends need: dr(5..6) of rows 0 and 1, of
// rows n-2 and n-1, alpha, beta.
template <bool TRI>
struct SegSlot {
  static constexpr int P = 5, F = TRI ? 5 : 6, E = 7, D = TRI ? 6 : 8, RC = TRI ? 7 : 9,
                       HA = 10, HB = TRI ? 8 : 11, HC = TRI ? 9 : 12, HD = 13;
};
__host__ __device__ constexpr int seg_cw(bool tri) { return tri ? 10 : 14; }
constexpr int SEG_XHEAD = 496, SEG_XTAIL = 500, SEG_XALPHA = 504, SEG_XBETA = 505;
static_assert(SEG_LONG * 14 <= SEG_XHEAD, "a segment's rows fit the pack");
static_assert(4 * SEG_KMAX <= SEG_CHAIN, "the chain tables fit one register pair");
// Chain tables, 4 doubles per segment j: forward A, B of its last row but one
// and of its last row; backward C, D of its first and second row.

struct SegTab {
  const double *pack;  // K x SEG_PACK, then the chain tables
  int n, K, len;       // points, segments, segment length
};

struct SegLines {
  // line l of the launch starts at (a0 + l % na) * sa + (b0 + l / na) * sb;
  // stride s between its points
  long sa, sb, s;
  int a0, na, b0, nb;
  int nlines;
  // not 0: groups of a block's lines (64) at a = 64 g .. 64 g + 63, this many
  // for each b (lines outside a0 .. a0 + na - 1 are left out); 0: 64 in turn
  int groups;
};

// lane `lane` (uniform) of v, in scalar registers
__device__ __forceinline__ double seg_lane(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// the wave's own LDS tile: its writes before its reads (no other wave uses it)
__device__ __forceinline__ void seg_tile_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// What a block solves: the derivative of one field, 64 lines, one per lane ...
struct SegDer {
  static constexpr bool PAIR = false;
  const double *__restrict__ x;
  double *__restrict__ out;
  __device__ __forceinline__ const double *in(bool) const { return x; }
  __device__ __forceinline__ void edge(long o) const { out[o] = 0.0; }
};

// ... or one component's share of the convective term along one axis,
//   out = acc + (u d(q) + d(q u)) / 2
// on 32 lines: the lower half of the wave solves for d(q), the upper half for
// d(q u).  Each half loads one of the two factors and they exchange them
// (v_permlane32_swap); afterwards they exchange every other row, so that both
// halves form and store results.
template <bool ACC>
struct SegConv {
  static constexpr bool PAIR = true, HAS_ACC = ACC;
  const double *__restrict__ q, *__restrict__ u, *__restrict__ acc;
  double *__restrict__ out;
  __device__ __forceinline__ const double *in(bool up) const { return up ? u : q; }
  __device__ __forceinline__ void edge(long o) const { out[o] = 0.0; }
};
template <class Job>
__host__ __device__ constexpr int seg_lines() { return Job::PAIR ? 32 : 64; }

// a's upper half of the wave <-> b's lower half
__device__ __forceinline__ void seg_swap(double &a, double &b) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  a = __longlong_as_double(((long long)hi[0] << 32) | lo[0]);
  b = __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}

// One wavefront's segment [s0, s0 + len).  LEN rows are unrolled; DYN: the
// length is the runtime len <= LEN (rows beyond it are skipped), else len =
// LEN.  HEAD: segment 0 (7-point rows 0 and 1, the alpha term of row 0);
// TAIL: the last segment (7-point rows n-2 and n-1, the beta term of row n-1).
// base: the block's first line; rel: this lane's line from there; lo, hi:
// lines lo .. hi - 1 of the block are its own (the others repeat one and
// are not stored).  lds: the block's arrays; w, K: this segment
// and the count.
// XT: contiguous lines (s = 1).  A lane's line then lies in memory away from
// the next lane's, so the wave moves 16 rows x 64 lines at a time through
// its transpose tile: each load and store covers 128 contiguous bytes of four
// lines (stored lane by lane, 8 bytes per line and instruction, HBM wrote
// 1.56 x the field, and x took 85 us where y and z took 54-58 at
// 201 x 256 x 187).
template <int LEN, bool HEAD, bool TAIL, bool DYN, bool TRI, bool XT, class Job>
__device__ __forceinline__ void seg_wave(const Job &job, long base, long rel, int lo, int hi,
                                         long s, const SegTab &T, int w, int K, int s0, int len,
                                         double *lds) {
  constexpr bool PAIR = Job::PAIR;
  const int n = T.n;
  const int lane = threadIdx.x & 63;
  const bool up = PAIR && lane >= 32;       // this lane solves for d(q u)
  const int line = PAIR ? lane & 31 : lane;
  typedef SegSlot<TRI> Slot;
  constexpr int CW = seg_cw(TRI);
  constexpr int NC = (LEN * CW + 63) / 64;  // register pairs of the rows
  constexpr int WD = seg_wave_doubles(XT), WB = XT ? 64 * SEG_TP : 128;
  const double *xl = job.in(up) + base + rel;
  // a loaded value as the solve takes it: the halves' factors become q and q u
  auto factor = [&](double v) {
    if constexpr (PAIR) {
      double o = v;
      seg_swap(v, o);
      return up ? v * o : v;
    } else {
      return v;
    }
  };
  // exchange slots of wave j: forward Ef[j WD ..], backward Eb[j WD ..]
  double *Ef = lds + lane, *Eb = lds + WB + lane;
  double *tile = lds + (long)WD * w;
  // XT: this lane's place in a coalesced access, row tr of line 4 q + tl
  const int tr = lane & 15, tl = lane >> 4;
  auto on = [&](int k) { return !DYN || k < len; };
  // tail rows: k = len - 2 (row n-2) and k = len - 1 (row n-1)
  auto is_n2 = [&](int k) { return TAIL && (DYN ? k == len - 2 : k == LEN - 2); };
  auto is_n1 = [&](int k) { return TAIL && (DYN ? k == len - 1 : k == LEN - 1); };
  double cv[NC], cx = 0.0, cf = 0.0, cb = 0.0;
  auto load_rows = [&]() {
    const double *pk = T.pack + (long)SEG_PACK * w + lane;
#pragma unroll
    for (int j = 0; j < NC; ++j) cv[j] = pk[64 * j];
    if (HEAD || TAIL) cx = pk[SEG_PACK - 64];
  };
  if (!XT) load_rows();
  const double *ch = T.pack + (long)SEG_PACK * K + lane;  // loaded once V's registers free up
  auto C = [&](int k, int m) { return seg_lane(cv[(k * CW + m) / 64], (k * CW + m) % 64); };
  auto X = [&](int m) { return seg_lane(cx, m - (SEG_PACK - 64)); };
  // inputs V[k] = x[s0 - 2 + k]; the two before the line (segment 0) and the
  // two after it (last segment of exactly LEN rows) are never read; a
  // runtime-length segment clamps into the line
  double V[LEN + 4];
  constexpr int NR = LEN / 16;  // 16-row tiles (rows beyond them go lane by lane)
  if constexpr (XT) {
    double R[NR][16];
#pragma unroll
    for (int t = 0; t < NR; ++t)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        int r = s0 + 16 * t + tr;
        if (DYN) r = r > n - 1 ? n - 1 : r;
        R[t][q] = job.in(PAIR && q >= 8)[base + __shfl((int)rel, 4 * q + tl, 64) + r];
      }
    // the rows next to the segment (the rows of a DYN segment's tile that lie
    // beyond its len are its successor's: nothing more to fetch)
    V[0] = HEAD ? 0.0 : xl[s0 - 2];
    V[1] = HEAD ? 0.0 : xl[s0 - 1];
#pragma unroll
    for (int r = 16 * NR; r < LEN + 2; ++r)
      V[2 + r] = TAIL && r >= LEN ? 0.0 : xl[s0 + r > n - 1 ? n - 1 : s0 + r];
#pragma unroll
    for (int t = 0; t < NR; ++t) {
#pragma unroll
      for (int q = 0; q < 16; ++q) tile[(4 * q + tl) * SEG_TP + tr] = R[t][q];
      seg_tile_sync();
#pragma unroll
      for (int r = 0; r < 16; ++r) V[2 + 16 * t + r] = factor(tile[lane * SEG_TP + r]);
      seg_tile_sync();
      if (t == 0) load_rows();
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (PAIR) {
      V[0] = factor(V[0]);
      V[1] = factor(V[1]);
      V[LEN + 2] = factor(V[LEN + 2]);
      V[LEN + 3] = factor(V[LEN + 3]);
    }
  } else if constexpr (PAIR) {
    // the halves' pointers walk the rows (36 addresses would not fit the
    // registers)
    auto none = [](int k) { return (HEAD && k < 2) || (TAIL && !DYN && k >= LEN + 2); };
    const double *xp = xl + (long)(HEAD ? 0 : s0 - 2) * s;
#pragma unroll
    for (int k = 0; k < LEN + 4; ++k) {
      V[k] = none(k) ? 0.0 : *xp;
      if (!none(k) && (!DYN || s0 - 2 + k < n - 1)) xp += s;
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int k = 0; k < LEN + 4; ++k) {
      if (!none(k)) V[k] = factor(V[k]);
      if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int k = 0; k < LEN + 4; ++k) {
      if ((HEAD && k < 2) || (TAIL && !DYN && k >= LEN + 2)) {
        V[k] = 0.0;
        continue;
      }
      int q = s0 - 2 + k;
      if (DYN) q = q > n - 1 ? n - 1 : q;
      V[k] = xl[(long)q * s];
    }
  }
  // forward particular solution from zero incoming values (segment 0 starts
  // at the true start); df[j]: the differences of the row's window
  double Y[LEN];
  double ym1 = 0.0, ym2 = 0.0, ym3 = 0.0, yl0 = 0.0, yl1 = 0.0;
  double df[4] = {0.0, V[1] - V[0], V[2] - V[1], V[3] - V[2]};
  // a 7-point row on x[0..6] = V[v0..v0+6]; its last two weights at X(m)
  auto row7 = [&](int k, int v0, int m) {
    double r = C(k, 0) * V[v0];
#pragma unroll
    for (int j = 1; j < 7; ++j) r = fma(j < 5 ? C(k, j) : X(m + j - 5), V[v0 + j], r);
    return r;
  };
#pragma unroll
  for (int k = 0; k < LEN; ++k) {
#pragma unroll
    for (int j = 0; j < 3; ++j) df[j] = df[j + 1];
    df[3] = V[k + 4] - V[k + 3];
    if (on(k)) {
      double yi;
      // the row's window: V[k..k+4] inside, x[0..6] on the 7-point rows 0 and 1,
      // x[n-7..n-1] on rows n-2 (V[k-3..k+3]) and n-1 (V[k-4..k+2])
      if (HEAD && k < 2) {
        yi = row7(k, 2, SEG_XHEAD + 2 * k);
      } else if (k >= 4 && is_n2(k)) {
        yi = row7(k, k >= 4 ? k - 3 : 0, SEG_XTAIL);
      } else if (k >= 4 && is_n1(k)) {
        yi = row7(k, k >= 4 ? k - 4 : 0, SEG_XTAIL + 2);
      } else {
        yi = C(k, 0) * V[k + 2];
#pragma unroll
        for (int j = 0; j < 4; ++j) yi = fma(C(k, 1 + j), df[j], yi);
      }
      // what the sweep waits for comes last
      if (!TRI && is_n1(k)) yi = fma(-X(SEG_XBETA), ym3, yi);
      if (!TRI && !(HEAD && k < 2)) yi = fma(-C(k, Slot::P), ym2, yi);
      if (!(HEAD && k == 0)) yi = fma(-C(k, Slot::F), ym1, yi);
      Y[k] = yi;
      ym3 = ym2; ym2 = ym1; ym1 = yi;
      if (DYN ? k == len - 2 : k == LEN - 2) yl0 = yi;
      if (DYN ? k == len - 1 : k == LEN - 1) yl1 = yi;
    }
    if (k == LEN / 2 && !HEAD) cf = ch[0];
    if (k == LEN / 2 && !TAIL) cb = ch[SEG_CHAIN];
    // keep the lane reads near their rows (hoisting them exhausts the SGPRs)
    if (k % 2 == 1) __builtin_amdgcn_sched_barrier(0);
  }
  // publish the segment's last particular values
  if (!TRI) Ef[w * WD] = yl0;
  Ef[w * WD + 64] = yl1;
  __syncthreads();
  double v0 = 0.0, v1 = 0.0;
  if (!HEAD) {
    // incoming (y_{s0-2}, y_{s0-1}): segment 0 ends on its own values, later
    // segments map theirs through their homogeneous responses
    if (!TRI) v0 = Ef[0];
    v1 = Ef[64];
    for (int j = 1; j < w; ++j) {
      const double p1 = Ef[j * WD + 64];
      if (TRI) {
        v1 = fma(seg_lane(cf, 4 * j + 3), v1, p1);
      } else {
        const double p0 = Ef[j * WD];
        const double n0 = fma(seg_lane(cf, 4 * j + 1), v1, fma(seg_lane(cf, 4 * j + 0), v0, p0));
        v1 = fma(seg_lane(cf, 4 * j + 3), v1, fma(seg_lane(cf, 4 * j + 2), v0, p1));
        v0 = n0;
      }
    }
  }
  // backward particular solution from zero incoming values (the last segment
  // ends at the true end), in place in Y, on the corrected forward values
  double xp1 = 0.0, xp2 = 0.0, x3 = 0.0;
#pragma unroll
  for (int k = LEN - 1; k >= 0; --k) {
    if (on(k)) {
      double xi = Y[k];
      if (!HEAD) {
        if (!TRI) xi = fma(C(k, Slot::HA), v0, xi);
        xi = fma(C(k, Slot::HB), v1, xi);
      }
      if (!is_n1(k)) {
        if (HEAD && k == 0 && !TRI) xi = fma(-X(SEG_XALPHA), x3, xi);
        if (!TRI) xi = fma(-C(k, Slot::E), xp2, xi);
        xi = fma(-C(k, Slot::D), xp1, xi);
      }
      xi *= C(k, Slot::RC);
      Y[k] = xi;
      xp2 = xp1; xp1 = xi;
      if (HEAD && k == 3) x3 = xi;
    }
    if (k % 2 == 0) __builtin_amdgcn_sched_barrier(0);
  }
  Eb[w * WD] = Y[0];
  if (!TRI) Eb[w * WD + 64] = Y[1];
  // a field at byte offset v (of the lane) from row ro of the segment
  auto at = [&](auto *f, long ro, unsigned v) -> auto & {
    return *(decltype(f))((char *)(f + base + (long)s0 * s + ro) + v);
  };
  // a pair's u and acc, 4 groups of 4 values per lane (the rows k0 + 2 j + up,
  // or 4 lines of a 16-row tile), fetched two groups ahead of their use: the
  // first two while the other segments finish
  constexpr int GR = 4, NG = LEN / 8;
  static_assert(!PAIR || LEN % 16 == 0, "a pair's groups are whole tiles");
  double uv[2][GR], av[2][GR];
  // opaque to the compiler, so that the offsets of the stores are formed here
  // rather than shared with those of the loads and held through the segment
  long so = s;
  int relo = (int)rel;
  asm volatile("" : "+s"(so), "+v"(relo));
  auto goff = [&](int g, int j) -> unsigned {
    if constexpr (XT) {
      const int r = 16 * (g / 2) + tr;
      return 8u * (unsigned)(__shfl(relo, 16 * (g % 2) + 4 * j + tl, 64) + (DYN ? min(r, len - 1) : r));
    } else {
      const int k = 8 * g + 2 * j;
      return 8u * (unsigned)relo + (up && (!DYN || k + 1 < len) ? 8u * (unsigned)so : 0u);
    }
  };
  auto grow = [&](int g, int j) -> long {
    const int k = 8 * g + 2 * j;
    return XT ? 0 : (long)(DYN ? min(k, len - 1) : k) * so;
  };
  auto fetch = [&](int g) {
    if constexpr (PAIR) {
#pragma unroll
      for (int j = 0; j < GR; ++j) {
        uv[g % 2][j] = at(job.u, grow(g, j), goff(g, j));
        if (Job::HAS_ACC) av[g % 2][j] = at(job.acc, grow(g, j), goff(g, j));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto share = [&](int g, int j, double dq, double dp) {
    const double v = 0.5 * fma(uv[g % 2][j], dq, dp);
    if constexpr (PAIR) return Job::HAS_ACC ? av[g % 2][j] + v : v;
    return v;
  };
  fetch(0);
  fetch(1);
  __syncthreads();
  v0 = v1 = 0.0;
  if (!TAIL) {
    // incoming (x_{e0}, x_{e0+1}) from the segments after this one
    v0 = Eb[(K - 1) * WD];
    if (!TRI) v1 = Eb[(K - 1) * WD + 64];
    for (int j = K - 2; j > w; --j) {
      const double q0 = Eb[j * WD];
      if (TRI) {
        v0 = fma(seg_lane(cb, 4 * j + 0), v0, q0);
      } else {
        const double q1 = Eb[j * WD + 64];
        const double n0 = fma(seg_lane(cb, 4 * j + 1), v1, fma(seg_lane(cb, 4 * j + 0), v0, q0));
        v1 = fma(seg_lane(cb, 4 * j + 3), v1, fma(seg_lane(cb, 4 * j + 2), v0, q1));
        v0 = n0;
      }
    }
  }
  auto fixed = [&](int k) {
    double xi = Y[k];
    if (!TAIL) {
      xi = fma(C(k, Slot::HC), v0, xi);
      if (!TRI) xi = fma(C(k, Slot::HD), v1, xi);
    }
    return xi;
  };
  if constexpr (XT) {
#pragma unroll
    for (int t = 0; t < NR; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (on(16 * t + r)) tile[lane * SEG_TP + r] = fixed(16 * t + r);
        if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
      seg_tile_sync();
      const bool rok = 16 * t + tr < (DYN ? len : LEN);
      if constexpr (PAIR) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int g = 2 * t + h;
#pragma unroll
          for (int j = 0; j < GR; ++j) {
            const int l = 16 * h + 4 * j + tl;
            const double v = share(g, j, tile[l * SEG_TP + tr], tile[(l + 32) * SEG_TP + tr]);
            const unsigned o = goff(g, j);  // (all lanes take part)
            if (rok && l < hi) at(job.out, 0, o) = v;
          }
          if (g + 2 < NG) fetch(g + 2);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int l = 4 * q + tl;
          const int o = __shfl(relo, l, 64) + s0 + 16 * t + tr;
          const double v = tile[l * SEG_TP + tr];
          if (rok && l < hi) job.out[base + o] = v;
          if (q % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
      seg_tile_sync();
    }
    if constexpr (16 * NR < LEN) {
      const bool act = line >= lo && line < hi;
#pragma unroll
      for (int r = 16 * NR; r < LEN; ++r)
        if (on(r)) {
          const double xi = fixed(r);
          if (act) job.out[base + relo + s0 + r] = xi;
        }
    }
  } else if constexpr (PAIR) {
    const bool act = line >= lo && line < hi;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
#pragma unroll
      for (int j = 0; j < GR; ++j) {
        const int k = 8 * g + 2 * j;
        if (on(k)) {
          double a = fixed(k), b = on(k + 1) ? fixed(k + 1) : 0.0;
          seg_swap(a, b);  // this half's row: a = d(q), b = d(q u)
          const double v = share(g, j, a, b);
          if (act && (!DYN || k + up < len)) at(job.out, grow(g, j), goff(g, j)) = v;
        }
      }
      if (g + 2 < NG) fetch(g + 2);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    double *po = job.out + base + rel + (long)s0 * so;
    const bool act = line >= lo && line < hi;
#pragma unroll
    for (int k = 0; k < LEN; ++k) {
      if (on(k)) {
        const double xi = fixed(k);
        if (act) po[(long)k * so] = xi;
      }
      if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Solve the scheme on 64 lines per block (32 of a pair), wave w = segment w.
// LONG: segments of up to SEG_LONG rows.
// off: added to every line's start; lines per SegLines (one family of lines).
// lds: seg_lds_doubles(K, XT) (of the longest scheme of the launch).
// Every wave of the block passes the same two barriers.
template <bool TRI, bool XT, bool LONG, class Job>
__device__ __forceinline__ void seg_solve(const Job &job, long off, const SegTab &T,
                                          const SegLines &L, int lblock, double *lds) {
  constexpr int NL = seg_lines<Job>();
  const int n = T.n;
  const int K = T.K;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w >= K) {
    // waves beyond K (blocks sized for a longer scheme) only join the barriers
    __syncthreads();
    __syncthreads();
    return;
  }
  // the block's first line, and this lane's from there
  const int line = threadIdx.x & (NL - 1);
  int lo = 0, hi;
  long base, rel;
  if (!XT && L.groups) {
    const int ag = NL * (lblock % L.groups), b = lblock / L.groups;
    lo = max(0, L.a0 - ag);
    hi = min(NL, L.a0 + L.na - ag);
    base = (long)ag * L.sa + (long)(L.b0 + b) * L.sb;
    rel = min(max(line, lo), hi - 1) * L.sa;
  } else {
    const int l0 = lblock * NL;
    hi = min(NL, L.nlines - l0);
    const int l = l0 + min(line, hi - 1);
    const int a0 = l0 % L.na, b0 = l0 / L.na;
    base = (long)(L.a0 + a0) * L.sa + (long)(L.b0 + b0) * L.sb;
    rel = (long)(l % L.na - a0) * L.sa + (long)(l / L.na - b0) * L.sb;
  }
  base += off;
  const int s0 = T.len * w;
  const int len = (w == K - 1) ? n - s0 : T.len;
  auto go = [&](auto head, auto tail, auto dyn) {
    seg_wave<LONG ? SEG_LONG : SEG_LEN, decltype(head)::value, decltype(tail)::value,
             decltype(dyn)::value, TRI, XT>(job, base, rel, lo, hi, L.s, T, w, K, s0, len, lds);
  };
  typedef std::true_type yes;
  typedef std::false_type no;
  if constexpr (LONG) {
    if (w == 0) go(yes(), no(), yes());
    else if (w < K - 1) go(no(), no(), yes());
    else go(no(), yes(), yes());
  } else if (K == 1) {
    go(yes(), yes(), yes());
  } else if (len == SEG_LEN) {
    if (w == 0) go(yes(), no(), no());
    else if (w < K - 1) go(no(), no(), no());
    else go(no(), yes(), no());
  } else {
    if (w == 0) go(yes(), no(), yes());
    else if (w < K - 1) go(no(), no(), yes());
    else go(no(), yes(), yes());
  }
}

// Table of a scheme of n points (host side) from its dr (n,7) column-major
// and packed p, f, d, e, 1/c: the segments' packs and the chain tables, formed
// in extended precision and rounded once.  The homogeneous responses are zero
// on segment 0 (forward) and on the last one (backward).
inline void seg_tables(int n, const double *dr, const double *p, const double *f,
                       const double *d, const double *e, const double *rc, double alpha,
                       double beta, bool tri, double *out) {
  typedef long double real;
  const int K = seg_count(n, tri), len = seg_len(n, K), CW = seg_cw(tri);
  double *fch = out + (size_t)SEG_PACK * K, *bch = fch + SEG_CHAIN;
  std::fill(out, out + seg_table_doubles(K), 0.0);
  std::vector<real> R[4];  // A, B, C, D
  for (int u = 0; u < 4; ++u) R[u].assign(n, 0);
  for (int w = 0; w < K; ++w) {
    const int s0 = len * w, e0 = (w == K - 1) ? n : s0 + len;
    for (int u = 0; u < 2 && w > 0; ++u) {
      real m2 = u ? 0 : 1, m1 = u ? 1 : 0;  // y_{s0-2}, y_{s0-1}
      for (int i = s0; i < e0; ++i) {
        real yi = -(real)p[i] * m2 - (real)f[i] * m1;
        if (i == n - 1) yi -= beta * R[u][n - 4];
        R[u][i] = yi;
        m2 = m1;
        m1 = yi;
      }
    }
    for (int u = 2; u < 4 && w < K - 1; ++u) {
      real p1 = u == 2 ? 1 : 0, p2 = u == 2 ? 0 : 1;  // x_{e0}, x_{e0+1}
      for (int i = e0 - 1; i >= s0; --i) {
        real xi = -(real)e[i] * p2 - (real)d[i] * p1;
        if (i == 0) xi -= alpha * R[u][3];
        xi *= rc[i];
        R[u][i] = xi;
        p2 = p1;
        p1 = xi;
      }
    }
    double *pk = out + (size_t)SEG_PACK * w;
    for (int i = s0; i < e0; ++i) {
      double *r = pk + (size_t)CW * (i - s0);
      auto w = [&](int m) { return (real)dr[i + (size_t)n * m]; };
      if (i < 2 || i >= n - 2) {
        for (int m = 0; m < 5; ++m) r[m] = (double)w(m);
        const int x = i < 2 ? SEG_XHEAD + 2 * i : SEG_XTAIL + 2 * (i - (n - 2));
        pk[x] = (double)w(5);
        pk[x + 1] = (double)w(6);
      } else {
        r[0] = (double)(w(0) + w(1) + w(2) + w(3) + w(4));
        r[1] = (double)-w(0);
        r[2] = (double)(-w(0) - w(1));
        r[3] = (double)(w(3) + w(4));
        r[4] = (double)w(4);
      }
      auto put = [&](auto slot) {
        typedef decltype(slot) S;
        r[S::F] = f[i]; r[S::D] = d[i]; r[S::RC] = rc[i];
        r[S::HB] = (double)R[1][i]; r[S::HC] = (double)R[2][i];
        if (!tri) {
          r[S::P] = p[i]; r[S::E] = e[i];
          r[S::HA] = (double)R[0][i]; r[S::HD] = (double)R[3][i];
        }
      };
      if (tri) put(SegSlot<true>());
      else put(SegSlot<false>());
    }
    pk[SEG_XALPHA] = alpha;
    pk[SEG_XBETA] = beta;
    fch[4 * w + 0] = (double)R[0][e0 - 2];
    fch[4 * w + 1] = (double)R[1][e0 - 2];
    fch[4 * w + 2] = (double)R[0][e0 - 1];
    fch[4 * w + 3] = (double)R[1][e0 - 1];
    bch[4 * w + 0] = (double)R[2][s0];
    bch[4 * w + 1] = (double)R[3][s0];
    bch[4 * w + 2] = (double)R[2][s0 + 1];
    bch[4 * w + 3] = (double)R[3][s0 + 1];
  }
}

}  // namespace mf
