// Hot-path kernels of the multislice STEM engine (gfx950).
//
//  * k_pass_rows  -- per slice, along rows:  [inverse row FFT, 1/N^2] -> x t(window) -> forward row FFT
//  * k_pass_cols  -- per slice, along columns: forward column FFT -> x propagator ->
//                    [annular detectors] -> inverse column FFT   (exit slice: detectors only)
//  * k_reduce_det -- per finished probe: fixed-order compensated FP64 sum of detector partials
//  * k_form_table / k_phase / k_accumulate_mfma16 -- projected potential in reciprocal space,
//                    several slices per launch (structure-factor sums on the matrix cores, 16 x 16
//                    pixel tiles)
//  * k_fft_rows / k_fft_cols -- plain batched 2-D FFT passes (potential IFFT, tests)
//
// A full 2-D forward+inverse FFT per slice therefore costs two read+write
// passes over the probe wave in HBM: 32 f N^2 bytes per probe.slice, where f is the
// fraction of reciprocal-space columns in which the propagator has a nonzero entry
// (the wave is zero elsewhere after every propagator multiply, so neither pass
// reads or writes those columns; 2/3 with the 2/3 band limit).
#include "fft_block.h"
#include "host_common.h"
#include "kernels.h"
#include "launch.h"
#include "unit_map.h"
#include "unit_round.h"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>

// Tuning knobs (compile-time).
#ifndef TOTEM_ROWS_MINWAVES
#define TOTEM_ROWS_MINWAVES 1  // minimum waves per SIMD the rows pass is compiled for
#endif
#ifndef TOTEM_COLS_MINWAVES
#define TOTEM_COLS_MINWAVES 1
#endif
// Columns per columns-pass workgroup.  The workgroup exchanges C whole columns
// through LDS ((N + N/16) * C float2 with the bank padding), which must stay within
// 64 KiB: 16 columns of 512 points would need 68 KiB, and 4 columns of 2048 points
// fit only with the exchange split into two rounds of half the buffer.
#ifndef TOTEM_COLS_C512
#define TOTEM_COLS_C512 8
#endif
#ifndef TOTEM_COLS_C1024
#define TOTEM_COLS_C1024 4
#endif
#ifndef TOTEM_COLS_C1536
#define TOTEM_COLS_C1536 4
#endif
#ifndef TOTEM_COLS_C2048
#define TOTEM_COLS_C2048 4
#endif
#ifndef TOTEM_COLS_SPLIT2048
#define TOTEM_COLS_SPLIT2048 1  // 2048-point columns exchange through half buffers
#endif
#ifndef TOTEM_ROWS_SPLIT2048
#define TOTEM_ROWS_SPLIT2048 0  // 2048-point rows: half-buffer exchanges, 4 rows per workgroup
#endif
#ifndef TOTEM_ROWS_PP
#define TOTEM_ROWS_PP 0        // rows pass: ping-pong LDS (1) or one buffer (0)
#endif
#ifndef TOTEM_COLS_PP
#define TOTEM_COLS_PP 0
#endif

namespace totem {

// ------------------------------------------------------------------------- helpers

#ifndef TOTEM_ROWS_K
#define TOTEM_ROWS_K 1  // row groups per workgroup (loads of the next one overlap the FFTs of this one)
#endif
#ifndef TOTEM_ROWS_TPREFETCH
#define TOTEM_ROWS_TPREFETCH 1  // load the transmission window together with the wave
#endif
#ifndef TOTEM_ROWS_THREADS
#define TOTEM_ROWS_THREADS 256  // threads per rows-pass workgroup
#endif
#ifndef TOTEM_ROWS_THREADS_SMALL
#define TOTEM_ROWS_THREADS_SMALL 128  // ... at 768 and 1024 points
#endif
// Rows per rows-pass workgroup also sets the wave tile (TR = min(RW, 4) rows of
// 16 / TR columns).  At 1024 points two rows per workgroup (2 x 8 tiles) measured
// best over the two passes together (rows 110 -> 97 us, columns 90 -> 98 us per
// launch of 26 probes); at 768 points 128-thread workgroups (4 rows, tiles
// unchanged) take the rows pass from 100.5 to 96.5 us; 2048 points keep 2 x 8
// tiles from 128 lanes per row.
// Pass variants ("plans"): each grid side has one or more schedules for its two
// passes -- the radix plan of each pass, rows per rows workgroup (which also sets
// the wave tile shared by both passes), columns per columns workgroup and whether
// the column exchanges run through half buffers.  Variant 0 is the default; the
// others are chosen at run time per device (totem_stem_set_plan, or measured by
// totem_stem_autotune), for a whole run or served grid side at a time.
// Base schedules whose passes run in fused form: the grid sides at which it is no less
// exact than separate twiddle products, by the exit waves of 80 slices against
// complex128 (relative L2, separate -> fused; the images' error falls more, by up to a
// factor of ten, with the balanced factors): 128 2.7e-6 -> 2.5e-6, 512 2.8e-6 -> 2.7e-6,
// 1024 3.3e-6 -> 3.1e-6, 1536 3.8e-6 -> 3.6e-6.  At 2048 (120 slices) the rows alone
// 4.2e-6 -> 4.2e-6, both passes 4.5e-6, and the columns pass gains nothing; 64 2.1e-6 ->
// 3.0e-6, 256 1.5e-6 -> 2.6e-6, 320 4.1e-6 -> 4.9e-6 and 768 4.1e-6 -> 4.4e-6 stay separate.  Rows / columns pass, us per launch of
// the full batch: 512 50.6 / 53.4 -> 48.3 / 51.8, 1024 70.6 / 54.9 -> 63.4 / 51.9 (24
// probes on average), 2048 rows 88 -> 81.
constexpr bool fused_cols(int n) { return n == 128 || n == 512 || n == 1024 || n == 1536; }
constexpr bool fused_rows(int n) { return fused_cols(n) || n == 2048; }
template <int N> struct PassSpecBase {
  using RowPlan = std::conditional_t<fused_rows(N), Fused<Plan<N>>, Plan<N>>;
  using ColPlan = std::conditional_t<fused_cols(N), Fused<Plan<N>>, Plan<N>>;
  static constexpr int rows_threads = (N == 1024 || N == 768) ? TOTEM_ROWS_THREADS_SMALL
                                      : (N == 2048 && TOTEM_ROWS_SPLIT2048) ? 2 * TOTEM_ROWS_THREADS
                                                                             : TOTEM_ROWS_THREADS;
  static constexpr bool rows_split = N == 2048 && TOTEM_ROWS_SPLIT2048;
  static constexpr int cols_c = N < 512 ? 16
                                : N == 512 ? TOTEM_COLS_C512
                                : N == 1024 ? TOTEM_COLS_C1024
                                : N == 1536 ? TOTEM_COLS_C1536
                                : N == 2048 ? TOTEM_COLS_C2048 : 8;
  static constexpr bool cols_split = N == 2048 && TOTEM_COLS_SPLIT2048;
  static constexpr bool rows_tprefetch = TOTEM_ROWS_TPREFETCH;  // transmission loaded with the wave
  static constexpr int rows_k = TOTEM_ROWS_K;                   // row groups per rows workgroup, in turn
};
template <int N, int V> struct PassSpec : PassSpecBase<N> {};
// The plain 2-D FFT kernels (potential build, fft2d) use the base schedule of each
// side whatever the pass variants specialise.
constexpr int kBaseSpec = 15;
// Variant 1 of most sizes: the rows pass loads its transmission window after the
// inverse transform, not with the wave (fewer registers live across the
// transform: 1024 points 118 -> 88 VGPRs, the load latency then hidden by more waves).
template <int N> struct PassSpecLateT : PassSpecBase<N> {
  static constexpr bool rows_tprefetch = false;
};
template <> struct PassSpec<256, 1> : PassSpecLateT<256> {};
template <> struct PassSpec<512, 1> : PassSpecLateT<512> {};
template <> struct PassSpec<1024, 1> : PassSpecLateT<1024> {};
template <> struct PassSpec<1536, 1> : PassSpecLateT<1536> {};
template <> struct PassSpec<2048, 1> : PassSpecLateT<2048> {};
// 768: rows transformed by the 12-element plan 4.4.4.4.3 on 64 lanes (one row per
// wave, 2 x 8 tiles); variant 0 also the columns, 4 per columns workgroup, variant 1
// the columns by the 24-element plan, variant 2 both passes by the 24-element plan.
template <> struct PassSpec<768, 1> : PassSpecBase<768> {
  using RowPlan = PlanB<768>;
  static constexpr int rows_threads = 128;
};
template <> struct PassSpec<768, 0> : PassSpec<768, 1> {
  using ColPlan = PlanB<768>;
  static constexpr int cols_c = 4;
};
template <> struct PassSpec<768, 2> : PassSpecBase<768> {};
// 1024, variant 2: rows transformed by 8.8.8.2 on 128 lanes (8 elements per lane,
// fewer registers per wave, one more exchange), two rows per workgroup (2 x 8 tiles).
template <> struct PassSpec<1024, 2> : PassSpecBase<1024> {
  using RowPlan = PlanB<1024>;
  static constexpr int rows_threads = 256;
};
// ... and with the transmission loaded after the inverse transform (59 VGPRs, 8 waves/SIMD).
template <> struct PassSpec<1024, 3> : PassSpec<1024, 2> {
  static constexpr bool rows_tprefetch = false;
};
// (Each workgroup taking two row groups in turn, the second group's wave loads
// issued before the first group's transforms -- rows_k = 2 on this plan, 95 VGPRs
// -- measured 90.2 against 88.9 us per 26-probe launch and is not compiled.)
// 512, variant 2: rows transformed by 8.8.8 on 64 lanes (8 elements per lane), four
// rows per workgroup (4 x 4 tiles, as variant 0).
template <> struct PassSpec<512, 2> : PassSpecBase<512> {
  using RowPlan = PlanB<512>;
  static constexpr int rows_threads = 256;
};
// 1536, variant 2: rows by 4.4.4.4.2.3 on 128 lanes (12 elements per lane), two rows
// per rows workgroup (2 x 8 tiles); columns by the 24-element plan, 4 per workgroup.
// Per 26-probe launch: rows 102.6, columns 121.6 us against variant 0's 110.1 and
// 113.7 (the 2 x 8 tiles cost the columns pass what the rows pass gains; four rows
// per workgroup keep variant 0's tiles but take the rows pass to 136.8 us).
template <> struct PassSpec<1536, 2> : PassSpecBase<1536> {
  using RowPlan = PlanB<1536>;
  static constexpr int rows_threads = 256;
};
template <int N> constexpr int pass_variants() {
  return N == 1024 ? 4 : (N == 512 || N == 768 || N == 1536) ? 3 : (N >= 256 && N != 320) ? 2 : 1;
}

// Calls f(std::integral_constant<int, V>) for the compiled variant V == v of grid side S.
template <int S, int V = 0, class F> static auto on_variant(int v, F&& f) {
  if constexpr (V + 1 < pass_variants<S>()) {
    if (v != V) return on_variant<S, V + 1>(v, static_cast<F&&>(f));
  }
  return f(std::integral_constant<int, V>{});
}

template <int N, int V = 0> struct RowCfg {
  using Spec = PassSpec<N, V>;
  using PL = typename Spec::RowPlan;
  static constexpr bool TPREFETCH = Spec::rows_tprefetch;
  static constexpr int K = Spec::rows_k;
  static constexpr int T = PL::T;
  static constexpr int RW = (Spec::rows_threads / T) > 0 ? Spec::rows_threads / T : 1;  // rows per workgroup
  static constexpr int THREADS = RW * T;
  static constexpr bool SPLIT = Spec::rows_split;
  static constexpr int LL = SPLIT ? row_lds_len<N / 2>() : row_lds_len<N>();
  static constexpr bool PP = TOTEM_ROWS_PP != 0 && !SPLIT;
  static constexpr int NBUF = PP ? 2 : 1;
};
template <int N, int V = 0> struct ColCfg {
  using Spec = PassSpec<N, V>;
  using PL = typename Spec::ColPlan;
  static constexpr bool SPLIT = Spec::cols_split;
  static constexpr bool PP = TOTEM_COLS_PP != 0 && !SPLIT;
  static constexpr int NBUF = PP ? 2 : 1;
  static constexpr int T = PL::T;
  static constexpr int C = Spec::cols_c;  // columns per workgroup
  static constexpr int THREADS = T * C;
  static constexpr int LC = SPLIT ? col_lds_len<N / 2, C>() : col_lds_len<N, C>();  // one exchange buffer
};
template <int N> using FftRowCfg = RowCfg<N, kBaseSpec>;
template <int N> using FftColCfg = ColCfg<N, kBaseSpec>;
// Every pass kernel's static LDS (transform buffers plus the detector's wave sums)
// stays within 64 KiB per workgroup.
#ifndef TOTEM_LDS_LIMIT
#define TOTEM_LDS_LIMIT (64 * 1024)
#endif
constexpr int kLdsLimit = TOTEM_LDS_LIMIT;

#ifndef TOTEM_TILED
#define TOTEM_TILED 1  // in-flight waves in the tiled layout below (0: row-major)
#endif

// Layout of an in-flight wave [N][N] (the probe, the transmission, the propagator
// and the outputs stay row-major).  Tiled: TR x TC tiles of 16 elements (one
// 128-byte line), tiles row-major, elements row-major inside a tile.  A rows-pass
// workgroup (TR rows at a time) then streams whole lines, and a columns-pass
// wave (C >= TC columns x 64/C consecutive rows) touches whole lines instead of
// C x 8-byte segments of 64/C rows.  Element (r, c) sits at
//   ((r / TR) * (N / TC) + c / TC) * 16 + (r % TR) * TC + c % TC.
template <int N, int V = 0> struct WaveLay {
  static constexpr int RW = RowCfg<N, V>::RW, RT = RowCfg<N, V>::T, CT = ColCfg<N, V>::T;
  static constexpr int TR = TOTEM_TILED ? (RW < 4 ? RW : 4) : 1;
  static constexpr int TC = TOTEM_TILED ? 16 / TR : 1;
  static_assert(!TOTEM_TILED || (TR * TC == 16 && N % TC == 0 && RT % TC == 0 && RT % TR == 0 && RW % TR == 0 &&
                                 CT % TR == 0),
                "tile shape");
  __device__ static int at(int r, int c) {
    if constexpr (!TOTEM_TILED) return r * N + c;
    return ((r / TR) * (N / TC) + c / TC) * 16 + (r % TR) * TC + c % TC;
  }
  // element stride between (r, c + T*v) and (r, c + T*(v+1)) for T a multiple of TC
  static constexpr int row_step(int T) { return TOTEM_TILED ? 16 * (T / TC) : T; }
};

#ifndef TOTEM_ROWS_WAVESYNC
#define TOTEM_ROWS_WAVESYNC 1  // rows that fit in one wave exchange with wave-local barriers
#endif
#ifndef TOTEM_ROWS_LANE_TILED
#define TOTEM_ROWS_LANE_TILED 2  // 0: never, 1: always, 2: the sizes that keep workgroup barriers
#endif
// Rows-pass lane mapping, two forms:
//  * row-major lanes: T consecutive lanes per row, so a row with T <= 64 stays
//    inside one wave and its LDS exchanges need only wave-local barriers; the TR
//    rows of a tile are read by TR waves of the workgroup and share each line in
//    the caches;
//  * lane-tiled: the 64 lanes of a wave cover TR rows x 64/TR columns, whole
//    128-byte tiles per load and store instruction; a row then spans TR waves
//    (workgroup barriers), and the LDS rows are padded by 4 float2 so that the
//    TR rows of a wave fall on different banks.
// Measured with cache-fit batches (us per launch of the rows pass, workgroup
// barriers -> wave-local row-major -> lane-tiled): 256: 94 -> 88 -> 95,
// 512: 103.5 -> 100 -> 104, 768: 177 -> 100 -> 133, 1024: 110.5 -> 113 -> 107,
// 1536: 185 -> 116 -> 137, 2048 (T = 128, no wave-local form): 111 -> - -> 97.
template <int N, int V = 0> constexpr bool rows_lane_tiled() {
  return TOTEM_ROWS_LANE_TILED == 1 ||
         (TOTEM_ROWS_LANE_TILED == 2 && !(TOTEM_ROWS_WAVESYNC && RowCfg<N, V>::T <= 64 && N != 1024));
}
// LDS row pad of the lane-tiled form: the TR rows of a wave start 16 / TR float2
// apart modulo 16, so one instruction's accesses of the TR rows fall on disjoint banks.
#ifndef TOTEM_ROWS_PAD
#define TOTEM_ROWS_PAD 0  // 0: 16 / TR
#endif
template <int N, int V = 0> constexpr int rows_lds_pad();
template <int N, int V = 0> constexpr bool rows_wave_local() {
  return TOTEM_ROWS_WAVESYNC && !rows_lane_tiled<N, V>() && RowCfg<N, V>::T <= 64 && 64 % RowCfg<N, V>::T == 0;
}
template <int N, int V> constexpr int rows_lds_pad() {
  return !rows_lane_tiled<N, V>() ? 0 : TOTEM_ROWS_PAD ? TOTEM_ROWS_PAD : 16 / WaveLay<N, V>::TR;
}
// How the passes store the wave (kWriteThrough: fft_block.h).  Rows: through where one
// store instruction covers at least half of each line it touches (the other half comes
// from the next wave of the workgroup): the wave holds all TR rows of a tile (lane-tiled)
// or 64 / T of them.  Columns: through where the workgroup's C columns cover a tile's TC;
// with half lines the other half comes from another workgroup, later.  Both sides of the
// line, 20 slices, written back -> through (rows and columns as the rule says; us at 1/8 of
// the full batch, at the full batch): 64 622 -> 435, 3867 -> 3665; 128 680 -> 556, 5476 ->
// 5309; 256 683 -> 613, 5624 -> 5481; 320 948 -> 836, 7112 -> 7069; 512 744 -> 583, 5280 ->
// 5247; 768 819 -> 698, 6492 -> 6564; 1024 703 -> 641, 5490 -> 5461; 1536 (columns) 814 ->
// 818, 7324 -> 7153; 2048 (two probes) 1418 -> 1393, 6420 -> 6403.  Against the rule, full
// batches: columns through at 768 6647 -> 7096, 1024 5588 -> 6084, 2048 6522 -> 6778, rows
// through at 1536 7392 -> 7775.  Loads or stores past the caches (nt) cost 10 to 50%.
template <int N, int V> constexpr int rows_store_policy() {
  using L = WaveLay<N, V>;
  constexpr int rows = rows_lane_tiled<N, V>() ? L::TR : 64 / L::RT < 1 ? 1 : 64 / L::RT < L::TR ? 64 / L::RT : L::TR;
  return rows * L::TC * (int)sizeof(float2) >= 64 ? kWriteThrough : kWriteBack;
}
template <int N, int V> constexpr int cols_store_policy() {
  return ColCfg<N, V>::C >= WaveLay<N, V>::TC ? kWriteThrough : kWriteBack;
}
template <int N, int V> __device__ __forceinline__ void row_lane(int tid, int& lr, int& t) {
  constexpr int T = RowCfg<N, V>::T, TR = rows_lane_tiled<N, V>() ? WaveLay<N, V>::TR : 1;
  const int q = tid / (TR * T), rem = tid - q * (TR * T);
  lr = q * TR + rem % TR;
  t = rem / TR;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// ------------------------------------------------------------------------ pass R

#ifndef TOTEM_COLS_HPREFETCH
#define TOTEM_COLS_HPREFETCH 1  // load the propagator before the forward transform
#endif

// The wave source (the probe, row-major, at slice 0; the item's tiled wave after)
// and destination are buffer resources: lanes hold 32-bit byte offsets and the
// offsets between a lane's elements are uniform (scalar registers), so the wave
// accesses need no 64-bit address arithmetic per element.
struct RowUnit {
  bool active;
  int slice;
  __amdgpu_buffer_rsrc_t src, dst;
  int src_off, src_step;  // bytes: the lane's first element, stride between consecutive v
  int dst_off;
  __amdgpu_buffer_rsrc_t trs;  // the transmission slice
  int t_off;                   // bytes: the lane's row in it
  int c0, np;
  int lo, len;                 // the job's column band
};

// A lane offset beyond every buffer resource's range: buffer loads there return 0
// and stores are dropped, without a memory access.
constexpr int kNoAccess = (int)0x80000000u;
// off if column c0 + T*v lies in a job's band [lo, lo + len) (mod N) (base = c0 - lo),
// else kNoAccess
template <int N, int T> __device__ __forceinline__ int band_off(int base, int v, int len, int off) {
  int d = base + T * v;
  if constexpr ((N & (N - 1)) == 0) {
    d &= N - 1;
  } else {
    d = d < 0 ? d + N : d;
  }
  return d < len ? off : kNoAccess;
}

template <int N, int V, int K>
__device__ __forceinline__ RowUnit row_unit(const ItemDev* __restrict__ items, const JobDev* __restrict__ jobs,
                                            int step, int u, int lr, int t) {
  using Cfg = RowCfg<N, V>;
  using Lay = WaveLay<N, V>;
  constexpr int RW = Cfg::RW, G = N / RW;
  RowUnit r;
  int item, rg;
  unit_map<K>(blockIdx.x, u, G, item, rg);
  const ItemDev it = items[item];
  const JobDev& jb = jobs[it.job];
  r.slice = step - it.start_step;
  r.active = r.slice >= 0 && r.slice < jb.S;
  const int row = rg * RW + lr;
  constexpr unsigned kBytes = (unsigned)N * N * sizeof(float2);
  r.dst = buf_rsrc(it.wave, kBytes);
  r.dst_off = Lay::at(row, t) * (int)sizeof(float2);
  const bool probe = r.slice == 0;
  r.src = buf_rsrc(probe ? it.probe : it.wave, kBytes);
  r.src_off = probe ? (row * N + t) * (int)sizeof(float2) : r.dst_off;
  r.src_step = (probe ? Cfg::T : Lay::row_step(Cfg::T)) * (int)sizeof(float2);
  r.np = jb.np;
  int pr = it.r0 + row;
  if (pr >= r.np) pr -= r.np;  // only reachable with wrap (validated on the host)
  const size_t np2 = (size_t)r.np * r.np;
  r.trs = buf_rsrc(jb.t + (size_t)(r.active ? r.slice : 0) * np2, (unsigned)(np2 * sizeof(float2)));
  r.t_off = pr * r.np * (int)sizeof(float2);
  r.c0 = it.c0;
  r.lo = jb.band_lo;
  r.len = jb.band_len;
  return r;
}

template <int N, int V>
__global__ void __launch_bounds__((RowCfg<N, V>::THREADS), TOTEM_ROWS_MINWAVES)
k_pass_rows(const ItemDev* __restrict__ items, const JobDev* __restrict__ jobs, int step, const float2* __restrict__ tw) {
  using Cfg = RowCfg<N, V>;
  using PL = typename Cfg::PL;
  constexpr int T = Cfg::T, RW = Cfg::RW, E = N / T, K = Cfg::K;
  constexpr int LLP = Cfg::LL + rows_lds_pad<N, V>();
  static_assert(Cfg::NBUF * RW * LLP * sizeof(float2) <= kLdsLimit, "rows-pass LDS above 64 KiB");
  __shared__ float2 lds[Cfg::NBUF * RW * LLP];
  float2* const lds1 = lds + (Cfg::NBUF - 1) * RW * LLP;
  int lr, t;
  row_lane<N, V>(threadIdx.x, lr, t);
  const RowLayT<rows_wave_local<N, V>()> lay{lr * LLP};
  constexpr int DSTEP = WaveLay<N, V>::row_step(T) * (int)sizeof(float2);
  float2 xa[E], xb[E];
  RowUnit ua = row_unit<N, V, K>(items, jobs, step, 0, lr, t);
  // After slice 0 the wave is zero outside the job's band and only its band columns are read.
  if (ua.active) {
    if (ua.slice == 0) {
#pragma unroll
      for (int v = 0; v < E; ++v) xa[v] = bld(ua.src, ua.src_off, ua.src_step * v);
    } else {
#pragma unroll
      for (int v = 0; v < E; ++v)
        xa[v] = bld(ua.src, band_off<N, T>(t - ua.lo, v, ua.len, ua.src_off), ua.src_step * v);
    }
  }
#pragma unroll
  for (int u = 0; u < K; ++u) {
    RowUnit ub;
    if (u + 1 < K) {
      ub = row_unit<N, V, K>(items, jobs, step, u + 1, lr, t);
      if (ub.active) {
#pragma unroll
        for (int v = 0; v < E; ++v)
          xb[v] = bld(ub.src, ub.slice == 0 ? ub.src_off : band_off<N, T>(t - ub.lo, v, ub.len, ub.src_off),
                      ub.src_step * v);
      }
    }
    if (ua.active) {  // uniform over the workgroup
      float2 tv[Cfg::TPREFETCH ? E : 1];
      if constexpr (Cfg::TPREFETCH) {
#pragma unroll
        for (int v = 0; v < E; ++v) {
          int pc = ua.c0 + t + T * v;
          if (pc >= ua.np) pc -= ua.np;
          tv[v] = bld(ua.trs, ua.t_off + pc * (int)sizeof(float2), 0);
        }
      }
      if (ua.slice > 0) {
        block_fft<N, +1, Cfg::PP, 0, Cfg::SPLIT, PL>(xa, lds, lds1, lay, t, tw);
        const float s = 1.0f / (float)(N * N);
#pragma unroll
        for (int v = 0; v < E; ++v) xa[v] = cscale(xa[v], s);
      }
#pragma unroll
      for (int v = 0; v < E; ++v) {
        if constexpr (Cfg::TPREFETCH) {
          xa[v] = cmul(xa[v], tv[v]);
        } else {
          int pc = ua.c0 + t + T * v;
          if (pc >= ua.np) pc -= ua.np;
          xa[v] = cmul(xa[v], bld(ua.trs, ua.t_off + pc * (int)sizeof(float2), 0));
        }
      }
      block_fft<N, -1, Cfg::PP, next_start<N, Cfg::PP, PL>(0), Cfg::SPLIT, PL>(xa, lds, lds1, lay, t, tw);
#pragma unroll
      for (int v = 0; v < E; ++v)  // the columns pass reads band columns only
        bst<rows_store_policy<N, V>()>(ua.dst, band_off<N, T>(t - ua.lo, v, ua.len, ua.dst_off), DSTEP * v, xa[v]);
      if (u + 1 < K) __syncthreads();  // LDS reuse by the next unit
    }
    if (u + 1 < K) {
      ua = ub;
#pragma unroll
      for (int v = 0; v < E; ++v) xa[v] = xb[v];
    }
  }
}

// ------------------------------------------------------------------------ pass C

template <int N, int E, int T, int C>
__device__ __forceinline__ void detector_partial(const float2* x, const double* __restrict__ masks, bool centred,
                                                 int A, int t, int col, double* red, double* out, int G, int cg) {
  // sum_k |Psi(k)|^2 * mask(k) over this workgroup's columns, FP64
  double acc[kMaxAper];
#pragma unroll
  for (int a = 0; a < kMaxAper; ++a) acc[a] = 0.0;
  const int mcol = centred ? ((col + N / 2) % N) : col;
#pragma unroll
  for (int v = 0; v < E; ++v) {
    const int row = t + T * v;
    const int mrow = centred ? ((row + N / 2) % N) : row;
    const double inten = (double)x[v].x * (double)x[v].x + (double)x[v].y * (double)x[v].y;
    const double* m = masks + (size_t)mrow * N + mcol;
#pragma unroll
    for (int a = 0; a < kMaxAper; ++a)
      if (a < A) acc[a] += inten * gldd(m + (size_t)a * N * N);
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  constexpr int NW = (T * C + 63) / 64;
#pragma unroll
  for (int a = 0; a < kMaxAper; ++a) {
    if (a < A) {
      double s = wave_sum(acc[a]);
      if (lane == 0) red[wave * kMaxAper + a] = s;
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < A) {
    double s = 0.0;
    for (int q = 0; q < NW; ++q) s += red[q * kMaxAper + threadIdx.x];
    out[(size_t)threadIdx.x * G + cg] = s;
  }
  __syncthreads();
}

// One column group per workgroup, idle ones leaving at once and nothing carried between
// units (as a loop over one unit, with a flag around each part and copies for a next unit:
// us per launch at the full batch 51.0 -> 49.6 at 1024 points, 50.5 ->
// 47.4 at 256, 45.1 -> 44.4 at 768).
// One kernel for every slice; the detector work is a run-time branch (uniform
// per workgroup).  A variant compiled without the detector code was measured
// slower at every size (its register allocation gives fewer waves per SIMD:
// at 1024 points 160 vs 128 VGPRs, 101 vs 89 us per launch of 26 probes).
template <int N, int V>
__global__ void __launch_bounds__((ColCfg<N, V>::THREADS), TOTEM_COLS_MINWAVES)
k_pass_cols(const ItemDev* __restrict__ items, const JobDev* __restrict__ jobs, int step, int groups,
            const float2* __restrict__ tw) {
  using Cfg = ColCfg<N, V>;
  using PL = typename Cfg::PL;
  using Lay = WaveLay<N, V>;
  constexpr int T = Cfg::T, C = Cfg::C, E = N / T, G = N / C;
  constexpr int NW = (Cfg::THREADS + 63) / 64;
  constexpr int LC = Cfg::LC;
  static_assert(Cfg::NBUF * LC * sizeof(float2) + NW * kMaxAper * sizeof(double) <= kLdsLimit,
                "columns-pass LDS above 64 KiB");
  __shared__ float2 lds[Cfg::NBUF * LC];
  __shared__ double red[NW * kMaxAper];
  float2* const lds1 = lds + (Cfg::NBUF - 1) * LC;
  constexpr unsigned kBytes = (unsigned)N * N * sizeof(float2);
  constexpr int kStep = T * N * (int)sizeof(float2);
  // `groups` groups per item from the first group of the job's band on (all G groups with
  // the default band); a launch runs the largest band of its jobs, and groups beyond a
  // job's own band are idle, as is an item before its first slice or after its last
  int item, gi;
  unit_map(blockIdx.x, 0, groups, item, gi);
  const ItemDev it = items[item];
  const JobDev& jb = jobs[it.job];
  const int slice = step - it.start_step;
  if (slice < 0 || slice >= jb.S || gi >= jb.band_ng) return;  // uniform over the workgroup
  int cg = gi + jb.band_g0;
  if (cg >= G) cg -= G;
  const int c = threadIdx.x % C;
  const int t = threadIdx.x / C;
  const ColLay<C> lay{c};
  const int col = cg * C + c;
  // byte offsets of (row t, column): in the wave (WaveLay) and in row-major arrays (H, exit wave);
  // both advance by T*N elements per v
  const auto wr = buf_rsrc(it.wave, kBytes);
  const int voff = Lay::at(t, col) * (int)sizeof(float2);
  const int hoff = (t * N + col) * (int)sizeof(float2);
  float2 x[E], hv[TOTEM_COLS_HPREFETCH ? E : 1];
#pragma unroll
  for (int v = 0; v < E; ++v) x[v] = bld(wr, voff, v * kStep);
  const auto hr = buf_rsrc(jb.prop, kBytes);
  // the propagator in column-group order: a wave's 64 lanes read 512 contiguous bytes
  const bool grouped = jb.prop_cols == C;
  const int poff = grouped ? ((cg * N + t) * C + c) * (int)sizeof(float2) : hoff;
  const int pstep = grouped ? T * C * (int)sizeof(float2) : kStep;
  if constexpr (TOTEM_COLS_HPREFETCH) {
#pragma unroll
    for (int v = 0; v < E; ++v) hv[v] = bld(hr, poff, v * pstep);
  }
  block_fft<N, -1, Cfg::PP, 0, Cfg::SPLIT, PL>(x, lds, lds1, lay, t, tw);
#pragma unroll
  for (int v = 0; v < E; ++v) x[v] = cmul(x[v], TOTEM_COLS_HPREFETCH ? hv[v] : bld(hr, poff, v * pstep));
  const int mid = jb.mid_of_slice ? jb.mid_of_slice[slice] : -1;
  if (mid >= 0) {
    for (int a0 = 0; a0 < jb.A; a0 += kMaxAper)
      detector_partial<N, E, T, C>(x, jb.aper2 + (size_t)a0 * N * N, false, min(kMaxAper, jb.A - a0), t, col, red,
                                   it.part + ((size_t)mid * jb.A + a0) * G, G, cg);
  }
  if (slice == jb.S - 1) {  // the exit face needs no inverse transform
    for (int a0 = 0; a0 < jb.A; a0 += kMaxAper)
      detector_partial<N, E, T, C>(x, jb.aper + (size_t)a0 * N * N, true, min(kMaxAper, jb.A - a0), t, col, red,
                                   it.part + ((size_t)jb.L * jb.A + a0) * G, G, cg);
    if (jb.exit) {
      const auto er = buf_rsrc(jb.exit + (size_t)it.out * N * N, kBytes);
#pragma unroll
      for (int v = 0; v < E; ++v) bst(er, hoff, v * kStep, x[v]);
    }
  } else {
    block_fft<N, +1, Cfg::PP, next_start<N, Cfg::PP, PL>(0), Cfg::SPLIT, PL>(x, lds, lds1, lay, t, tw);
#pragma unroll
    for (int v = 0; v < E; ++v) bst<cols_store_policy<N, V>()>(wr, voff, v * kStep, x[v]);
  }
}

// Fixed-order Kahan sum of the detector partials of the listed items.  One thread a sum
// and few threads: bound by the latency of the partials' loads, so 16 are loaded before
// they are added in turn (one at a time, behind the band test: 28.4 us on average over
// finishing launches of 256 to 1024 points, so 9.5).
__global__ void k_reduce_det(const ItemDev* __restrict__ items, const int* __restrict__ list, int n,
                             const JobDev* __restrict__ jobs, int G, int lmax1, int amax) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * lmax1 * amax) return;
  const int a = idx % amax;
  const int layer = (idx / amax) % lmax1;
  const int e = idx / (amax * lmax1);
  const ItemDev it = items[list ? list[e] : e];
  const JobDev& jb = jobs[it.job];
  if (a >= jb.A || layer > jb.L) return;
  double s = 0.0;
  if (layer == jb.L || jb.layer_hit[layer]) {
    const double* p = it.part + ((size_t)layer * jb.A + a) * G;
    double comp = 0.0;
    auto add = [&](double v) {
      const double y = v - comp;
      const double tt = s + y;
      comp = (tt - s) - y;
      s = tt;
    };
    // only the job's band groups are written (the rest is zero): in order of g, those of
    // the band beyond the last group, then the others; a step's partials are loaded together
    auto sum = [&](int g, int end) {
      constexpr int U = 16;
      for (; g + U <= end; g += U) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = p[g + u];
#pragma unroll
        for (int u = 0; u < U; ++u) add(v[u]);
      }
      for (; g < end; ++g) add(p[g]);
    };
    const int past = jb.band_g0 + jb.band_ng;
    sum(0, min(max(past - G, 0), jb.band_g0));
    sum(jb.band_g0, min(past, G));
  }
  jb.det[((size_t)layer * jb.A + a) * jb.n_out + it.out] = s;
}

// --------------------------------------------------------------- plain 2-D FFT passes

template <int N, int SIGN>
__global__ void __launch_bounds__(FftRowCfg<N>::THREADS) k_fft_rows(float2* __restrict__ data, long rows, const float2* __restrict__ tw) {
  using Cfg = FftRowCfg<N>;
  constexpr int T = Cfg::T, RW = Cfg::RW, E = N / T;
  static_assert(RW * Cfg::LL * sizeof(float2) <= kLdsLimit, "row FFT LDS above 64 KiB");
  __shared__ float2 lds[RW * Cfg::LL];
  const int lr = threadIdx.x / T;
  const int t = threadIdx.x - lr * T;
  const long row = (long)blockIdx.x * RW + lr;
  float2* w = data + row * N;
  float2 x[E];
  const bool ok = row < rows;
#pragma unroll
  for (int v = 0; v < E; ++v) x[v] = ok ? w[t + T * v] : make_float2(0.f, 0.f);
  block_fft<N, SIGN, false, 0, Cfg::SPLIT>(x, lds, lds, RowLay{lr * Cfg::LL}, t, tw);
  if (ok) {
#pragma unroll
    for (int v = 0; v < E; ++v) w[t + T * v] = x[v];
  }
}

// epi: 0 store, 1 store exp(i*sigma*V) (transmission), 2 store scaled by 1/N^2
template <int N, int SIGN>
__global__ void __launch_bounds__(FftColCfg<N>::THREADS)
k_fft_cols(const float2* __restrict__ src, float2* __restrict__ dst, int epi, float sigma,
           const float2* __restrict__ tw) {
  using Cfg = FftColCfg<N>;
  constexpr int T = Cfg::T, C = Cfg::C, E = N / T, G = N / C;
  static_assert(Cfg::LC * sizeof(float2) <= kLdsLimit, "column FFT LDS above 64 KiB");
  __shared__ float2 lds[Cfg::LC];
  // neighbouring column groups, which share 128-byte lines, run on one XCD's L2 (dispatched
  // round-robin instead, four XCDs fetched and wrote every line: 5 x 1024^2 44.6 us, so 22.6)
  int mat, cg;
  unit_map(blockIdx.x, 0, G, mat, cg);
  const int c = threadIdx.x % C;
  const int t = threadIdx.x / C;
  const int col = cg * C + c;
  const float2* s = src + (size_t)mat * N * N + col;
  float2* d = dst + (size_t)mat * N * N + col;
  float2 x[E];
#pragma unroll
  for (int v = 0; v < E; ++v) x[v] = s[(size_t)(t + T * v) * N];
  block_fft<N, SIGN, false, 0, Cfg::SPLIT>(x, lds, lds, ColLay<C>{c}, t, tw);
#pragma unroll
  for (int v = 0; v < E; ++v) {
    float2 y = x[v];
    if (epi == 1) {
      // t = exp(i sigma V) = exp(-sigma Im V) (cos(sigma Re V) + i sin(sigma Re V))
      const float amp = expf(-sigma * y.y);
      float sn, cs;
      sincosf(sigma * y.x, &sn, &cs);
      y = make_float2(amp * cs, amp * sn);
    } else if (epi == 2) {
      y = cscale(y, 1.0f / (float)((long)N * N));
    }
    d[(size_t)(t + T * v) * N] = y;
  }
}

// ------------------------------------------------------------------- potential build

// ex[j][c] = w_j exp(-2 pi i kx1[c] x_j), ey[j][r] = exp(-2 pi i ky1[r] y_j); the
// product k.x is formed and reduced modulo 1 in FP64 before the (FP64) sincospi, and
// the term's weight is applied in FP64 before the rounding to FP32.  Only the first
// nc entries of each row are formed and stored (the accumulation reads no more);
// entries at or beyond np, in the last tile's overhang, are zero.  Terms of runs that
// k_repeated_runs marked are left out: nothing reads them.
__global__ void __launch_bounds__(256) k_phase(const double* __restrict__ tx, const double* __restrict__ ty,
                                               const double* __restrict__ wt,
                                               const unsigned char* __restrict__ dup,
                                               const double* __restrict__ kx1, const double* __restrict__ ky1, int np,
                                               int nc, float2* __restrict__ ex, float2* __restrict__ ey) {
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  const int j = blockIdx.x;
  if (c >= nc || (dup && dup[j])) return;
  const size_t at = (size_t)j * nc + c;
  if (c >= np) {
    ex[at] = ey[at] = make_float2(0.f, 0.f);
    return;
  }
  double fx = kx1[c] * tx[j];
  fx -= rint(fx);
  double fy = ky1[c] * ty[j];
  fy -= rint(fy);
  double sx, cx, sy, cy;
  sincospi(2.0 * fx, &sx, &cx);
  sincospi(2.0 * fy, &sy, &cy);
  const double w = wt[j];
  ex[at] = make_float2((float)(w * cx), (float)(-w * sx));
  ey[at] = make_float2((float)cy, (float)-sy);
}

// Terms with a zero coefficient are skipped: the one-term classes of erf-weighted
// slicing keep a single Gaussian (the branch is uniform: one class per wave).
__device__ __forceinline__ double peng5(const double* p, double s2) {
  double f = 0.0;
#pragma unroll
  for (int q = 0; q < 5; ++q)
    if (p[2 * q] != 0.0) f += p[2 * q] * exp(-p[2 * q + 1] * s2);
  return f;
}
__device__ __forceinline__ double lobato5(const double* p, double g2) {
  double f = 0.0;
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const double d = 1.0 + p[2 * q + 1] * g2;
    f += p[2 * q] * (2.0 + p[2 * q + 1] * g2) / (d * d);
  }
  return f;
}

// Form factor of a class at one reciprocal-space pixel (FP64, complex when absorptive).
__device__ __forceinline__ double2 form_factor(const PotClass& k, double s2, const double* __restrict__ corr,
                                               size_t pix, size_t np2) {
  double re = 0.0;
  switch (k.kind) {
    case kPeng: re = peng5(k.p1, s2); break;
    case kLobato: re = lobato5(k.p1, 4.0 * s2) * exp(-k.B * s2); break;
    case kPengIon: re = k.w1 * peng5(k.p1, s2) + k.w2 * peng5(k.p2, s2); break;
    case kLobatoIon: re = (k.w1 * lobato5(k.p1, 4.0 * s2) + k.w2 * lobato5(k.p2, 4.0 * s2)) * exp(-k.B * s2); break;
    case kCorr: re = corr[(size_t)k.i1 * np2 + pix] * exp(-k.B * s2); break;
    case kCorrIon:
      re = (k.w1 * corr[(size_t)k.i1 * np2 + pix] + k.w2 * corr[(size_t)k.i2 * np2 + pix]) * exp(-k.B * s2);
      break;
    default: break;
  }
  const double im = k.has_abs ? peng5(k.ab, s2) : 0.0;
  return make_double2(re, im);
}

// Runs of a slice whose terms repeat an earlier run's (same x, y and weight, in order): an
// atom's correction term stands beside its own term, at the same place and weight, in
// another class, and the structure-factor sum, which is most of a build, is the same for
// both.  Each such run is linked to the earlier one (`next`) and marked (`dup`), its terms
// in dup[].  One workgroup per slice; runs are compared by length and a hash of their
// terms' bits, and a match is checked term by term.  Slices of more than kMaxRuns runs are
// left as they are.
constexpr int kMaxRuns = 512;
__global__ void __launch_bounds__(256) k_repeated_runs(const PotSlice* __restrict__ slices, PotSeg* __restrict__ segs,
                                                       const double* __restrict__ tx, const double* __restrict__ ty,
                                                       const double* __restrict__ wt,
                                                       unsigned char* __restrict__ dup) {
  __shared__ unsigned long long hash[kMaxRuns];
  __shared__ int same[kMaxRuns], len[kMaxRuns], differ;
  const PotSlice ps = slices[blockIdx.x];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = ps.n_seg <= kMaxRuns ? ps.n_seg : 0;
  for (int i = 0; i < ps.n_seg; ++i) {
    const PotSeg sg = segs[ps.seg + i];
    for (int j = sg.begin + (int)threadIdx.x; j < sg.end; j += 256) dup[ps.term + j] = 0;
  }
  for (int i = wave; i < n; i += 4) {
    const PotSeg sg = segs[ps.seg + i];
    unsigned long long h = 0;
    for (int j = sg.begin + lane; j < sg.end; j += 64) {
      const size_t at = ps.term + j;
      const unsigned long long v = (unsigned long long)__double_as_longlong(tx[at]) * 0x9E3779B97F4A7C15ull ^
                                   (unsigned long long)__double_as_longlong(ty[at]) * 0xC2B2AE3D27D4EB4Full ^
                                   (unsigned long long)__double_as_longlong(wt[at]);
      h += (v ^ (v >> 29)) * (2ull * (unsigned)(j - sg.begin) + 1ull);
    }
    for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o, 64);
    if (lane == 0) {
      hash[i] = h;
      len[i] = sg.end - sg.begin;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 256) {
    int f = i;  // first run like run i
    for (int j = 0; j < i && f == i; ++j)
      if (hash[j] == hash[i] && len[j] == len[i]) f = j;
    same[i] = f;
  }
  __syncthreads();
  for (int i = 0; i < n; ++i) {  // uniform over the workgroup
    const int f = same[i];
    if (f == i) continue;
    if (threadIdx.x == 0) differ = 0;
    __syncthreads();
    const size_t a = ps.term + segs[ps.seg + f].begin, b = ps.term + segs[ps.seg + i].begin;
    for (int j = threadIdx.x; j < len[i]; j += 256)
      if (tx[a + j] != tx[b + j] || ty[a + j] != ty[b + j] || wt[a + j] != wt[b + j]) differ = 1;
    __syncthreads();
    if (!differ) {
      for (int j = threadIdx.x; j < len[i]; j += 256) dup[b + j] = 1;
      if (threadIdx.x == 0) {  // to the end of run f's chain
        int k = ps.seg + f;
        while (segs[k].next >= 0) k = segs[k].next;
        segs[k].next = ps.seg + i;
        segs[ps.seg + i].dup = 1;
      }
    }
    __syncthreads();
  }
}

// ff_re[cls][pix] (and ff_im where some class is absorptive): the form factors of
// every class at every pixel, formed once per build.  A slice's accumulation then reads
// 8 bytes per class and pixel instead of evaluating up to ten FP64 exponentials there,
// which every slice of the stack would repeat.
__global__ void __launch_bounds__(256) k_form_table(const PotClass* __restrict__ classes, const double* __restrict__ s2,
                                                    const double* __restrict__ corr, size_t np2,
                                                    double* __restrict__ ff_re, double* __restrict__ ff_im) {
  const size_t pix = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= np2) return;
  const double2 f = form_factor(classes[blockIdx.y], s2[pix], corr, pix, np2);
  ff_re[blockIdx.y * np2 + pix] = f.x;
  if (ff_im) ff_im[blockIdx.y * np2 + pix] = f.y;
}

// Slices of a chunk: V_k(r,c) = PARAMETER * AperTrue * sum_classes f_cls(k) * sum_{j in cls} w_j ex_j[c] ey_j[r],
// written at the ifftshifted position (the reference's quadrant swap) as complex64.
//
// Per class the sum over terms is a complex matrix product, A[r][j] = ey_j[r] times
// B[j][c] = ex_j[c] (the weight w_j already in ex), on the matrix cores in FP32
// (v_mfma_f32_16x16x4f32, four terms per product): lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16], and accumulator element i of lane l is C[4 (l / 16) + i][l % 16].  The
// four real products are kept apart,
//   P1 = Ar Br,  P2 = Ai Bi,  P3 = Ar Bi,  P4 = Ai Br  (summed over terms),
// because the weights are real and the grid's frequencies come in pairs
// (ky[N - r] = -ky[r], kx[N - c] = -kx[c]): then ey_j[N - r] = conj(ey_j[r]) and
// ex_j[N - c] = conj(ex_j[c]), and one tile's products give four pixels,
//   S(r, c)         = (P1 - P2) + i (P3 + P4)
//   S(r, N - c)     = (P1 + P2) + i (P4 - P3)
//   S(N - r, c)     = (P1 + P2) + i (P3 - P4)
//   S(N - r, N - c) = (P1 - P2) - i (P3 + P4).
// With `sym` set the tiles cover rows and columns [0, N/2] (r = 0 and N/2 have no pair)
// and rows / columns in [1, N/2 - 1] also write their pair N - r: every pixel is
// written once.  Without it (a grid whose frequencies are not paired) the tiles cover
// the grid.
// Eight waves share a 16 x 16 tile, each taking every eighth group of 16 terms of a class;
// the partial products of the waves that hold terms are summed in LDS and each thread
// weights two pixels by the class's FP64 form factors there, formed or fetched before the
// sum (formed after it, 64^2 and 128^2 slices of many classes take 6 to 20% longer).  The
// waves also keep FP32 chains short: a sum in chains of L terms is off by about
// 2.5e-8 sqrt(L / 2), here L = n / 8 of a run's n (V of one class of 1600 / 16000 terms at
// 256^2: 3.0e-7 / 7.4e-7; 3.9e-7 / 1.0e-6 with chains of n / 4).  Runs of up to 64 terms go
// in groups of 8 for the same reason (16 terms 1.68e-7 -> 1.63e-7), and a group of 8 or
// fewer skips its other half's products.
// Bound by the phases from L2 and the matrix cores where runs are long, by each run's
// reduction where they are short; 56 VGPRs and 32 KiB let four tiles share a CU.  Tiles of
// 32 x 32 by four waves (half the operands, but a quarter of the workgroups, eight times the
// pixels per thread and 242 VGPRs) are slower throughout, us per launch 32 / 16: one slice
// of 600 terms in 3 classes 68 / 15 at 256^2, 97 / 49 at 1024^2; 16 x 256^2 of 600 48 / 38;
// 8 x 1024^2 of 4000 980 / 850, and of 120 in 30 classes 542 / 458; whole builds 80 x 1024^2
// with corrections 3.68 / 3.54 ms, 30 x 512^2 erf-weighted 1.70 / 1.52.
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kAccWaves = 8;  // waves sharing a tile
// tiles along a side: of [0, np / 2] (paired frequencies) or of [0, np)
__host__ __device__ constexpr int acc_tiles(int np, bool sym) { return sym ? np / 32 + 1 : np / 16; }
enum FormMode : int { kFormEval, kFormRe, kFormComplex };
template <int FORM>
__global__ void __launch_bounds__(64 * kAccWaves)
k_accumulate_mfma16(const float2* __restrict__ ex, const float2* __restrict__ ey, const PotSlice* __restrict__ slices,
                    long term_base, const PotSeg* __restrict__ segs, const PotClass* __restrict__ classes,
                    const double* __restrict__ ff_re, const double* __restrict__ ff_im, const double* __restrict__ s2,
                    const double* __restrict__ aper_true, const double* __restrict__ corr, double parameter, int np,
                    int nc, int sym, float2* __restrict__ vshift) {
  constexpr int W = kAccWaves, NO = 1024 / (64 * W);  // waves; pixels per thread
  constexpr int U = 4, GT = 4 * U;                      // matrix steps, terms per group
  static_assert(W == 8, "two pixels per thread");
  __shared__ float red[W][4][256];  // [wave][product][64 * element + lane]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int half = np / 2;
  const int dt = acc_tiles(np, sym != 0), tiles = dt * dt;
  const int sl = blockIdx.x / tiles, tile = blockIdx.x - sl * tiles;
  const int tr = tile / dt, tc = tile - tr * dt;
  const int r0 = tr * 16, c0 = tc * 16;
  const int li = lane & 15, lk = lane >> 4;
  const PotSlice ps = slices[sl];
  const size_t np2 = (size_t)np * np;
  // this thread's tile position, where its sums stand in LDS, and its pixels
  const int pos = threadIdx.x & 255, pr = pos >> 4, pc = pos & 15;
  const int src = 64 * (pr & 3) + (pr >> 2) * 16 + pc;
  int pix[NO];  // -1: no such pixel
  bool cj_r[NO], cj_c[NO];
  double s2v[NO], vr[NO], vi[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    const int quad = (threadIdx.x >> 8) + 2 * o;  // bit 0: column pair, bit 1: row pair
    const int r = r0 + pr, c = c0 + pc;
    cj_c[o] = quad & 1;
    cj_r[o] = quad >> 1;
    const bool ok = sym ? (r <= half && c <= half && (!cj_r[o] || (r >= 1 && r < half)) &&
                           (!cj_c[o] || (c >= 1 && c < half)))
                        : quad == 0;
    pix[o] = ok ? (cj_r[o] ? np - r : r) * np + (cj_c[o] ? np - c : c) : -1;
    s2v[o] = FORM == kFormEval && ok ? s2[pix[o]] : 0.0;
    vr[o] = vi[o] = 0.0;
  }
  int oa[U], ob[U];  // byte offsets of this lane's phases in a group of terms
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int row = (4 * u + lk) * nc;
    oa[u] = (row + r0 + li) * (int)sizeof(float2);
    ob[u] = (row + c0 + li) * (int)sizeof(float2);
  }
  const int base = (int)(ps.term - term_base);  // within the chunk
  const int last = ps.seg + ps.n_seg - 1;
  PotSeg sg, coming;
  if (ps.n_seg > 0) coming = segs[ps.seg];
  for (int sgi = ps.seg; sgi <= last; ++sgi) {
    sg = coming;
    coming = segs[min(sgi + 1, last)];  // in flight during this run
    if (sg.dup) continue;
    floatx4 p[4] = {};
    const int gt = sg.end - sg.begin <= 8 * W ? 8 : GT;  // short runs: half groups, on more waves
    for (int j = sg.begin + gt * wave; j < sg.end; j += gt * W) {
      const int left = min(sg.end - j, gt);  // the phases of later terms read as zero
      const size_t at = (size_t)(base + j) * nc;
      const auto ra = buf_rsrc(ey + at, (unsigned)(left * nc * (int)sizeof(float2)));
      const auto rb = buf_rsrc(ex + at, (unsigned)(left * nc * (int)sizeof(float2)));
      float2 a[U], b[U];
      auto load = [&](int u0) {
#pragma unroll
        for (int u = u0; u < u0 + U / 2; ++u) {
          a[u] = bld(ra, oa[u], 0);
          b[u] = bld(rb, ob[u], 0);
        }
      };
      auto products = [&](int u0) {
#pragma unroll
        for (int u = u0; u < u0 + U / 2; ++u) {
          p[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].x, b[u].x, p[0], 0, 0, 0);
          p[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].y, b[u].y, p[1], 0, 0, 0);
          p[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].x, b[u].y, p[2], 0, 0, 0);
          p[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].y, b[u].x, p[3], 0, 0, 0);
        }
      };
      if (left > GT / 2) {
        load(0);
        load(U / 2);
        products(0);
        products(U / 2);
      } else {  // the other half holds zeros
        load(0);
        products(0);
      }
    }
    double fr[NO], fi[NO];
    auto factors = [&](int cls) {
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        if constexpr (FORM == kFormEval) {
          const double2 f = pix[o] < 0 ? make_double2(0.0, 0.0)
                                       : form_factor(classes[cls], s2v[o], corr, pix[o], np2);
          fr[o] = f.x;
          fi[o] = f.y;
        } else {
          const size_t at = cls * np2 + max(pix[o], 0);
          fr[o] = ff_re[at];
          if constexpr (FORM == kFormComplex) fi[o] = ff_im[at];
        }
      }
    };
    factors(sg.cls);  // tabulated ones in flight during the sums
    const int waves = min((sg.end - sg.begin + gt - 1) / gt, W);  // that hold terms of the run
    if (wave < waves) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][k][64 * i + lane] = p[k][i];
    }
    __syncthreads();
    float q[4] = {};
    if (waves == W) {
#pragma unroll
      for (int w = 0; w < W; ++w)
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] += red[w][k][src];
    } else {
      for (int w = 0; w < waves; ++w)
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] += red[w][k][src];
    }
    __syncthreads();  // read before the next run's sums are stored
    for (int next = sg.next;;) {  // the run's class and those of its repetitions
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        const double sre = cj_r[o] == cj_c[o] ? (double)(q[0] - q[1]) : (double)(q[0] + q[1]);
        const double sim = (double)(cj_c[o] ? -q[2] : q[2]) + (double)(cj_r[o] ? -q[3] : q[3]);
        if constexpr (FORM == kFormRe) {
          vr[o] += fr[o] * sre;
          vi[o] += fr[o] * sim;
        } else {
          vr[o] += fr[o] * sre - fi[o] * sim;
          vi[o] += fr[o] * sim + fi[o] * sre;
        }
      }
      if (next < 0) break;
      factors(segs[next].cls);
      next = segs[next].next;
    }
  }
  float2* const out = vshift + sl * np2;
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    if (pix[o] < 0) continue;
    const int R = pix[o] / np, C = pix[o] - R * np;
    const double scale = parameter * aper_true[pix[o]];
    const int rs = R < half ? R + half : R - half, cs = C < half ? C + half : C - half;
    out[(size_t)rs * np + cs] = make_float2((float)(vr[o] * scale), (float)(vi[o] * scale));
  }
}

// prop [N][N] row-major -> column groups of C columns, rows in order: element
// (r, g*C + c) at (g*N + r)*C + c.
__global__ void k_prop_cols(const float2* __restrict__ prop, float2* __restrict__ out, int n, int C) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)n * n) return;
  const int r = (int)(i / n), col = (int)(i - (long)r * n);
  const int g = col / C, c = col - g * C;
  out[((long)g * n + r) * C + c] = prop[i];
}

// flags[c] = 0 for every column, then one thread per (column, chunk of n / kFlagChunks
// rows) sets it to 1 on a nonzero entry (every writer stores the same value);
// consecutive threads read consecutive entries of a row.
constexpr int kFlagChunks = 32;
__global__ void k_zero_i32(int* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}
__global__ void k_column_flags(const float2* __restrict__ prop, int* __restrict__ flags, int n) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const int rows = (n + kFlagChunks - 1) / kFlagChunks;
  const int r0 = blockIdx.y * rows, r1 = min(n, r0 + rows);
  for (int r = r0; r < r1; ++r) {
    const float2 h = prop[(size_t)r * n + c];
    if (h.x != 0.f || h.y != 0.f) {
      flags[c] = 1;
      return;
    }
  }
}

// x moved to the next float towards +2 (dir > 0) or -2 (dir < 0), |x| < 2
__device__ __forceinline__ float neighbour(float x, int dir) {
  if (dir == 0) return x;
  if (x == 0.f) return __uint_as_float(dir > 0 ? 0x00000001u : 0x80000001u);
  return __int_as_float(__float_as_int(x) + ((x > 0.f) == (dir > 0) ? 1 : -1));
}
// out[i] = complex64 of (re[i], im[i]); with `unit`, values of unit modulus are rounded
// as unit_float2 rounds them on the host (the same operations in the same order, no
// contraction: the same floats).  Bound by its 24 bytes per value; on one host thread the
// nine candidates took about 40 ns a value, 3 of the 5.4 ms of a call with 256^2 windows.
__global__ void __launch_bounds__(256) k_complex64(const double* __restrict__ re, const double* __restrict__ im,
                                                   float2* __restrict__ out, long n, int unit) {
#pragma clang fp contract(off)
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double c = re[i], s = im[i];
  float bc = (float)c, bs = (float)s;
  if (unit && fabs(c * c + s * s - 1.0) < 1e-12) {
    const float c0 = bc, s0 = bs;
    double best = 1e300;
    for (int a = -1; a <= 1; ++a)
      for (int b = -1; b <= 1; ++b) {
        const float cc = neighbour(c0, a), ss = neighbour(s0, b);
        const double dn = fabs((double)cc * cc + (double)ss * ss - 1.0);
        const double dv = fabs(cc - c) + fabs(ss - s);
        const double score = dn * 1e6 + dv;
        if (score < best) {
          best = score;
          bc = cc;
          bs = ss;
        }
      }
  }
  out[i] = make_float2(bc, bs);
}

__global__ void k_fill_c64(float2* __restrict__ p, long n, float re, float im) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = make_float2(re, im);
}
__global__ void k_fill_f64(double* __restrict__ p, long n, double v) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// --------------------------------------------------------------------- launchers

#define TOTEM_FOR_SIZES(X) X(64) X(128) X(256) X(320) X(512) X(768) X(1024) X(1536) X(2048)

// Twiddle tables of every plan in one static device array (no allocation on any
// path that launches the passes); each table starts at an even entry so that its
// float4 reads stay 16-byte aligned.
constexpr int tw_even(int n) { return (n + 1) & ~1; }
template <class Q, class... PLS> struct TwOffset {
  static constexpr int value = -(1 << 28);  // not registered
};
template <class Q, class P0, class... PLS> struct TwOffset<Q, P0, PLS...> {
  static constexpr int value =
      std::is_same<Q, P0>::value ? 0 : tw_even(plan_twiddle_len<P0>()) + TwOffset<Q, PLS...>::value;
};
template <class... PLS> struct PlanSet {
  static constexpr int total = (0 + ... + tw_even(plan_twiddle_len<PLS>()));
  template <class Q> static constexpr int offset() {
    constexpr int o = TwOffset<Q, PLS...>::value;
    static_assert(o >= 0, "plan without a twiddle table");
    return o;
  }
};
using AllPlans = PlanSet<Plan<64>, Plan<128>, Plan<256>, Plan<320>, Plan<512>, Plan<768>, Plan<1024>, Plan<1536>,
                         Plan<2048>, Fused<Plan<128>>, Fused<Plan<512>>, Fused<Plan<1024>>, Fused<Plan<1536>>,
                         Fused<Plan<2048>>, PlanB<768>, PlanB<1024>, PlanB<512>, PlanB<1536>>;
__device__ __align__(16) float2 g_twiddles[AllPlans::total];

// Stage (P, R) of a plan, P > 1: the factor exp(-2 pi i q k / (P R)) of input q of a
// butterfly with k = b mod P.  Laid out q-major so that one load instruction, whose
// lanes hold neighbouring k, reads neighbouring entries: for even R the pair
// (q, q + 1) = (2j, 2j + 1) of block k sits at [(j P + k) 2 + {0, 1}] (one 16-byte
// load per pair), for odd R entry q of block k at [q P + k].
template <class PL> void twiddle_host_plan(std::vector<float2>& out) {
  out.clear();
  int p = 1;
  for (int i = 0; i < PL::NRAD; ++i) {
    const int r = PL::radix(i);
    if (p > 1 && PL::FUSED && fused_radix(r)) {
      const int f = r / 2;
      const size_t base = out.size();
      out.resize(base + (size_t)stage_table_len(p * f), make_float2(0.f, 0.f));
      std::vector<double> sum(f, 0.0);
      for (int k = 0; k < p; ++k)
        for (int q = 0; q < f; ++q) {
          // w^a W_r^b with w = exp(-2 pi i k / (p r)): angle a k / (p r) + b / r turns
          const double a = -2.0 * M_PI * ((double)fused_power(r, q, false) * k / (double)(p * r) +
                                          (double)fused_power(r, q, true) / (double)r);
          const size_t at = f % 2 == 0 ? ((size_t)(q / 2) * p + k) * 2 + q % 2 : (size_t)q * p + k;
          out[base + at] = balanced_float2(std::cos(a), std::sin(a), sum[q]);
        }
    } else if (p > 1) {
      const size_t base = out.size();
      out.resize(base + (size_t)stage_table_len(p * r), make_float2(0.f, 0.f));
      for (int k = 0; k < p; ++k)
        for (int q = 0; q < r; ++q) {
          const double a = -2.0 * M_PI * (double)q * (double)k / (double)(p * r);
          const size_t at = r % 2 == 0 ? ((size_t)(q / 2) * p + k) * 2 + q % 2 : (size_t)q * p + k;
          out[base + at] = unit_float2(std::cos(a), std::sin(a));
        }
    }
    p *= r;
  }
}
template <class PL> static void put_table(std::vector<float2>& all) {
  std::vector<float2> h;
  twiddle_host_plan<PL>(h);
  std::copy(h.begin(), h.end(), all.begin() + AllPlans::offset<PL>());
}
template <class... PLS> static void put_tables(std::vector<float2>& all, PlanSet<PLS...>*) {
  (put_table<PLS>(all), ...);
}

// Device address of g_twiddles on the current device, filled on first use.
static float2* twiddle_base() {
  int dev = 0;
  HIP_OK(hipGetDevice(&dev));
  static std::mutex mu;
  static std::map<int, float2*> base;
  std::lock_guard<std::mutex> lk(mu);
  auto it = base.find(dev);
  if (it == base.end()) {
    float2* p = nullptr;
    HIP_OK(hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(g_twiddles)));
    std::vector<float2> all(AllPlans::total, make_float2(0.f, 0.f));
    put_tables(all, static_cast<AllPlans*>(nullptr));
    HIP_OK(hipMemcpy(p, all.data(), all.size() * sizeof(float2), hipMemcpyHostToDevice));
    it = base.emplace(dev, p).first;
  }
  return it->second;
}
template <class PL> static const float2* tw_for() { return twiddle_base() + AllPlans::offset<PL>(); }

void twiddle_host(int n, std::vector<float2>& out) {
  out.clear();
#define X(S) if (n == S) { twiddle_host_plan<Plan<S>>(out); return; }
  TOTEM_FOR_SIZES(X)
#undef X
}

const float2* tw_table(int n) {
#define X(S) if (n == S) return tw_for<Plan<S>>();
  TOTEM_FOR_SIZES(X)
#undef X
  require(false, "no FFT plan for n=" + std::to_string(n), TOTEM_ERR_UNSUPPORTED);
  return nullptr;
}

template <int N, int V> void launch_pass_rows(hipStream_t st, const ItemDev* items, int n_items, const JobDev* jobs,
                                              int step) {
  using Cfg = RowCfg<N, V>;
  constexpr int K = Cfg::K;
  static_assert((N / Cfg::RW) % K == 0, "row groups per probe must be a multiple of K");
  const dim3 grid((unsigned)(n_items * (N / Cfg::RW) / K));
  hipLaunchKernelGGL((k_pass_rows<N, V>), grid, dim3(Cfg::THREADS), 0, st, items, jobs, step,
                     tw_for<typename Cfg::PL>());
}
template <int N, int V> void launch_pass_cols(hipStream_t st, const ItemDev* items, int n_items, const JobDev* jobs,
                                              int step, int groups) {
  using Cfg = ColCfg<N, V>;
  if (groups <= 0 || groups > N / Cfg::C) throw std::runtime_error("columns pass: bad group count");
  const dim3 grid((unsigned)(n_items * groups));
  hipLaunchKernelGGL((k_pass_cols<N, V>), grid, dim3(Cfg::THREADS), 0, st, items, jobs, step, groups,
                     tw_for<typename Cfg::PL>());
}
template <int N> void launch_fft2d(hipStream_t st, float2* data, float2* dst, int batch, int sign, int epi,
                                   float sigma) {
  using R = FftRowCfg<N>;
  using Cc = FftColCfg<N>;
  const long rows = (long)batch * N;
  const dim3 rgrid((unsigned)((rows + R::RW - 1) / R::RW));
  const float2* tw = tw_for<Plan<N>>();
  if (sign < 0) hipLaunchKernelGGL((k_fft_rows<N, -1>), rgrid, dim3(R::THREADS), 0, st, data, rows, tw);
  else hipLaunchKernelGGL((k_fft_rows<N, +1>), rgrid, dim3(R::THREADS), 0, st, data, rows, tw);
  const dim3 cgrid((unsigned)(batch * (N / Cc::C)));
  if (sign < 0) hipLaunchKernelGGL((k_fft_cols<N, -1>), cgrid, dim3(Cc::THREADS), 0, st, data, dst, epi, sigma, tw);
  else hipLaunchKernelGGL((k_fft_cols<N, +1>), cgrid, dim3(Cc::THREADS), 0, st, data, dst, epi, sigma, tw);
}

template <class PL> static std::string plan_radices() {
  std::string r;
  for (int i = 0; i < PL::NRAD; ++i) r += (i ? "." : "") + std::to_string(PL::radix(i));
  return r;
}
template <int N, int V> static std::string variant_desc() {
  using R = RowCfg<N, V>;
  using C = ColCfg<N, V>;
  return "rows " + plan_radices<typename R::PL>() + " on " + std::to_string(R::T) + " lanes x " +
         std::to_string(R::RW) + " rows" + (R::SPLIT ? " (half-buffer exchanges)" : "") +
         (R::TPREFETCH ? "" : " (transmission loaded after the inverse transform)") + "; columns " +
         plan_radices<typename C::PL>() + " on " + std::to_string(C::T) + " lanes x " + std::to_string(C::C) +
         " columns" + (C::SPLIT ? " (half-buffer exchanges)" : "") + "; tiles " +
         std::to_string(WaveLay<N, V>::TR) + " x " + std::to_string(WaveLay<N, V>::TC);
}

bool size_supported(int n) {
#define X(S) if (n == S) return true;
  TOTEM_FOR_SIZES(X)
#undef X
  return false;
}

int pass_variant_count(int n) {
#define X(S) if (n == S) return pass_variants<S>();
  TOTEM_FOR_SIZES(X)
#undef X
  return 0;
}

std::string pass_variant_desc(int n, int v) {
#define X(S) \
  if (n == S) return on_variant<S>(v, [](auto vc) { return variant_desc<S, decltype(vc)::value>(); });
  TOTEM_FOR_SIZES(X)
#undef X
  return "";
}

int detector_groups(int n, int v) {
#define X(S) \
  if (n == S) return on_variant<S>(v, [](auto vc) { return S / ColCfg<S, decltype(vc)::value>::C; });
  TOTEM_FOR_SIZES(X)
#undef X
  return 0;
}

int detector_groups_max(int n) {
  int g = 0;
  for (int v = 0; v < pass_variant_count(n); ++v) g = std::max(g, detector_groups(n, v));
  return g;
}

void pass_rows(int n, int v, hipStream_t st, const ItemDev* items, int n_items, const JobDev* jobs, int step) {
#define X(S)                                                                                          \
  if (n == S) {                                                                                       \
    on_variant<S>(v, [&](auto vc) { launch_pass_rows<S, decltype(vc)::value>(st, items, n_items, jobs, step); }); \
    return;                                                                                           \
  }
  TOTEM_FOR_SIZES(X)
#undef X
}

void pass_cols(int n, int v, hipStream_t st, const ItemDev* items, int n_items, const JobDev* jobs, int step,
               int groups) {
#define X(S)                                                                                          \
  if (n == S) {                                                                                       \
    on_variant<S>(v, [&](auto vc) {                                                                   \
      launch_pass_cols<S, decltype(vc)::value>(st, items, n_items, jobs, step, groups);              \
    });                                                                                               \
    return;                                                                                           \
  }
  TOTEM_FOR_SIZES(X)
#undef X
}

void reduce_det(hipStream_t st, const ItemDev* items, const int* list, int n, const JobDev* jobs, int groups,
                int lmax1, int amax) {
  const int total = n * lmax1 * amax;
  if (total <= 0) return;
  hipLaunchKernelGGL(k_reduce_det, dim3((total + 255) / 256), dim3(256), 0, st, items, list, n, jobs, groups, lmax1,
                     amax);
}

int pass_cols_width(int n, int v) {
#define X(S) \
  if (n == S) return on_variant<S>(v, [](auto vc) { return ColCfg<S, decltype(vc)::value>::C; });
  TOTEM_FOR_SIZES(X)
#undef X
  return 0;
}

void prop_column_groups(hipStream_t st, const float2* prop, float2* out, int n, int C) {
  const long total = (long)n * n;
  hipLaunchKernelGGL(k_prop_cols, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, prop, out, n, C);
}

void column_flags(hipStream_t st, const float2* prop, int* flags, int n) {
  const unsigned nb = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(k_zero_i32, dim3(nb), dim3(256), 0, st, flags, n);
  hipLaunchKernelGGL(k_column_flags, dim3(nb, kFlagChunks), dim3(256), 0, st, prop, flags, n);
}

void complex64(hipStream_t st, const double* re, const double* im, float2* out, long n, bool unit) {
  if (n > 0)
    hipLaunchKernelGGL(k_complex64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, re, im, out, n,
                       unit ? 1 : 0);
}

void fill(hipStream_t st, float2* p, long n, float re, float im) {
  if (n > 0) hipLaunchKernelGGL(k_fill_c64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n, re, im);
}
void fill(hipStream_t st, double* p, long n, double v) {
  if (n > 0) hipLaunchKernelGGL(k_fill_f64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n, v);
}

void fft2d(int n, hipStream_t st, float2* data, float2* dst, int batch, int sign, int epi, float sigma) {
#define X(S) if (n == S) { launch_fft2d<S>(st, data, dst, batch, sign, epi, sigma); return; }
  TOTEM_FOR_SIZES(X)
#undef X
}

bool hermitian_pairs(const double* kx1, const double* ky1, int np) {
  if (np % 2 != 0) return false;
  for (int r = 1; r < np / 2; ++r)
    if (ky1[np - r] != -ky1[r] || kx1[np - r] != -kx1[r]) return false;
  return true;
}

// whole 16-entry tiles of [0, np/2] (paired frequencies) or of [0, np)
int phase_columns(int np, bool sym) { return 16 * acc_tiles(np, sym); }

void repeated_runs(hipStream_t st, const PotSlice* slices, int n_slices, PotSeg* segs, const double* tx,
                   const double* ty, const double* wt, unsigned char* dup) {
  if (n_slices > 0)
    hipLaunchKernelGGL(k_repeated_runs, dim3(n_slices), dim3(256), 0, st, slices, segs, tx, ty, wt, dup);
}

void phase_tables(hipStream_t st, const double* tx, const double* ty, const double* wt, const unsigned char* dup,
                  int n_terms, const double* kx1, const double* ky1, int np, bool sym, float2* ex, float2* ey) {
  if (n_terms <= 0) return;
  const int nc = phase_columns(np, sym);
  hipLaunchKernelGGL(k_phase, dim3(n_terms, (nc + 255) / 256), dim3(256), 0, st, tx, ty, wt, dup, kx1, ky1, np, nc,
                     ex, ey);
}

void form_table(hipStream_t st, const PotClass* classes, int n_classes, const double* s2, const double* corr, int np,
                double* ff_re, double* ff_im) {
  const size_t np2 = (size_t)np * np;
  if (n_classes > 0)
    hipLaunchKernelGGL(k_form_table, dim3((unsigned)((np2 + 255) / 256), n_classes), dim3(256), 0, st, classes, s2,
                       corr, np2, ff_re, ff_im);
}

void accumulate(hipStream_t st, const float2* ex, const float2* ey, const PotSlice* slices, int n_slices,
                long term_base, const PotSeg* segs, const PotClass* classes, const double* ff_re, const double* ff_im,
                const double* s2, const double* aper_true, const double* corr, double parameter, int np, bool sym,
                float2* vshift) {
#define X(S) static_assert(S % 16 == 0 && S <= 32768, "potential tiles: whole tiles without pairs, 32-bit pixels");
  TOTEM_FOR_SIZES(X)
#undef X
  const int nc = phase_columns(np, sym), dt = acc_tiles(np, sym);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(n_slices * dt * dt)), dim3(64 * kAccWaves), 0, st, ex, ey, slices,
                       term_base, segs, classes, ff_re, ff_im, s2, aper_true, corr, parameter, np, nc, sym ? 1 : 0,
                       vshift);
  };
  if (ff_im) launch(k_accumulate_mfma16<kFormComplex>);
  else if (ff_re) launch(k_accumulate_mfma16<kFormRe>);
  else launch(k_accumulate_mfma16<kFormEval>);
}

}  // namespace totem
