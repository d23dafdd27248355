// Wide request groups of the flow: many drafts share every weight stream.
//
// A batch of drafts is run in groups of up to 16 requests (128 activation rows for the second
// chunk expert at draft_length 8) whose rows all multiply each packed weight fragment as it
// streams past, so a group costs about one draft's weight traffic instead of one per two drafts.
// The narrow streaming kernel (cfh_stream.h) stages its whole K chunk once and holds at most 16
// rows; here the activation rows are staged in K chunks of WCH columns through three LDS buffers,
// refilled while the weights stream:
//
//   chunk c:  multiply the chunk's WCH/32 k-steps of fragments, each against every 16-row group of the
//             rows in LDS; the rows of a k-step are read while the one before multiplies, those of
//             the chunk's last k-step's successor from chunk c + 1's buffer, complete since the last
//             barrier, so that neither the barrier nor the LDS latency stands before a multiply
//             place chunk c + 2's rows (loaded during chunk c - 2) in the buffer chunk c - 1 left
//             issue the loads of chunk c + 4's rows into the registers just freed
//             one LDS barrier
//
// What bounds it (13 requests at d = 2560, the 157 MB up-projection, 35 us): copies of the kernel with
// one part each taken out run at 24 us with the matrix instructions alone (no rows, no weights: about
// 14 ns each a SIMD), 25 us with the rows' LDS reads too, 33 us with the rows' staging, 35 us
// with the weights; of these 2 us are the launch, 1 us its start, 2-5 us the epilogue's stores.
//
// A wave owns WT adjacent 16-column tiles of one (expert, k-split) unit and keeps one accumulator
// per (tile, 16-row group).  Self attention, which the narrow kernel computes while staging, runs as its own
// small kernel per (request, head), and the context rows' LayerNorm of every block is computed
// once per draft into rows the cross K/V stream reads.
#pragma once
#include <algorithm>
#include <type_traits>

#include "cfh_stream.h"

namespace {

constexpr int WCH = 128;          // K columns staged per chunk (4 k-steps)
constexpr int WMAXR = 128;        // max activation rows of one expert in a wide group

struct WEx {
  const h16x8* w;      // packed weights: fragment (tile t, k-step s) at ((t * K/32) + s) * 64
  const h16* a;        // activation rows [S][lda]; the unit's K range [kc K/ks, (kc+1) K/ks) is read
  int lda;
  const h16* bias;     // E_BIAS16 / E_GELU16 / E_GELUF16 bias [N]
  void* out;           // E_PART: float [ks][S][N]; E_PART16: h16 (as SEx); otherwise h16 (below)
  int S;               // activation rows (1 .. WMAXR)
  int pack, hrows;     // E_PART16: as SEx
  int nsplit;          // E_BIAS16: column n goes to block n / nsplit, stored [blocks][S][nsplit] (0: [S][N])
  const int* ids;      // row i of the operand is a[max(ids[i * ids_stride], 0)] (a gather), or row i (null)
  int ids_stride;
};

struct WArgs {
  WEx ex[4];
  int nex, N, K, ks, wg_per_kc;
  int gelu_r16;        // E_GELU16: as SArgs (E_GELUF16: gelu16_erff of the rounded sum)
  int pair;            // entries e and e + nex/2 stream the same weights (two request groups of one
                       // expert): their workgroups for a unit run side by side on one XCD
  int map;             // workgroup order (set by launch_wide): MAP_PLAIN, MAP_PAIR or MAP_XCD
};

// Workgroup -> (entry, k-split, tile group) orders.  Workgroups go to the 8 XCDs round robin,
// each XCD with its own L2, starting from an XCD that depends on the dispatches before the launch:
// workgroups b and b' share an XCD when b = b' mod 8 (below, "XCD x" is the XCD of the workgroups
// b = x mod 8, whichever it is).
//   MAP_PLAIN: entry-major.
//   MAP_PAIR:  workgroups b and b + 8 take the same unit of entries e and e + nex/2.
//   MAP_XCD:   (split-K) XCD x takes every unit of the (entry, k-split) combinations x, x + 8, ...:
//              each XCD reads the operand rows of its own K ranges only, instead of every XCD
//              reading all of them (W2's 128 rows x 24576 columns are 6.3 MB an entry), and with
//              nex/2 * ks a multiple of 8 the two groups' combinations of one weight range share
//              an XCD.
enum { MAP_PLAIN = 0, MAP_PAIR = 1, MAP_XCD = 2 };

// CH: K columns staged per chunk.  WCH everywhere but in the folded cross attention's factor launches
// (E_PART16, K split by head), whose k-splits are one head wide: the widest of 128, 64 and 32 that
// divides the head width (320 at d = 2560: five chunks of 64).  A wave keeps RC 128-column chunks of
// fragments in flight at every CH.
template <int I, int N, typename F>
__device__ __forceinline__ void unrolled(F&& f) {   // f(0), f(1), .. f(N - 1), each a compile-time constant
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unrolled<I + 1, N>(f);
  }
}

// LDS rows of one staged chunk: the NG row groups, rounded up to whole passes of the workgroup's threads.
constexpr int wide_rows(int ng, int wv, int ch) {
  const int rpv = wv * 64 / (ch / 8);
  return (ng * 16 + rpv - 1) / rpv * rpv;
}

template <int EPI, int NG, int WV, int CH, int WT, int RS, int RC, bool GA>
__device__ __forceinline__ void wide_unit(const WArgs& a, const WEx& ex, int kc, int tg) {
  constexpr int WKS = CH / 32;      // k-steps per chunk
  constexpr int WRC = RC * WCH / CH;     // chunks of fragments in flight per wave
  constexpr int WSPF = WRC * WKS * WT;   // fragment loads in flight per wave
  // AP: a k-step's rows are read while the one before multiplies.  Eight-wave workgroups have no
  // registers for it, and two waves a SIMD that cover the reads for each other.
  constexpr bool AP = WKS % 2 == 0 && WV <= 4;
  constexpr int WLDA = CH + 8;      // LDS row stride (halves): rows of a chunk start on different banks
  extern __shared__ __align__(16) h16 lds[];
  // (the wave index read as a scalar keeps the weight pointers out of the vector registers)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int S = ex.S;
  const int ksteps = a.K / 32;
  const int KCW = a.K / a.ks, nsteps = KCW / 32, nchunk = KCW / CH;
  // wave w: columns' share w % WC (WT adjacent 16-column tiles), rows' share w / WC (NGW of the NG groups)
  constexpr int WC = WV / RS, NGW = NG / RS;
  const int t0 = (tg * WC + wave % WC) * WT, g0 = wave / WC * NGW;
  const int k0 = kc * KCW;
  // staging of one chunk: thread t's vector u is row t / NVR + u NT / NVR, columns (t % NVR) * 8 .. +7;
  // rows past S repeat the last one (every load unconditional, see Stage; the LDS rows they fill
  // only reach output rows that are never stored)
  constexpr int NT = WV * 64;
  constexpr int NVR = CH / 8;                         // 16-byte vectors per row of a chunk
  constexpr int RPV = NT / NVR;                       // rows between a thread's vectors
  constexpr int NSV = (NG * 16 + RPV - 1) / RPV;      // vectors per thread
  static_assert(NSV * RPV == wide_rows(NG, WV, CH), "LDS rows of a chunk");
  const int trow = (int)threadIdx.x / NVR, tcol = (int)threadIdx.x % NVR;
  // each vector's byte offset in the operand, the same at every chunk (a gathered row's
  // index is read once)
  typename std::conditional<GA, size_t, unsigned>::type soff[NSV];
#pragma unroll
  for (int u = 0; u < NSV; ++u) {
    const int i = min(trow + u * RPV, S - 1);
    if constexpr (GA) soff[u] = (size_t)max(ex.ids[(size_t)i * ex.ids_stride], 0) * ex.lda * 2 + tcol * 16;
    else soff[u] = (unsigned)(i * ex.lda * 2 + tcol * 16);
  }
  h16x8 st0[NSV], st1[NSV];                           // rows of two chunks on their way to LDS
  auto load_chunk = [&](int c, h16x8 (&st)[NSV]) {
    const char* base = (const char*)(ex.a + k0 + c * CH);
#pragma unroll
    for (int u = 0; u < NSV; ++u) st[u] = *(const h16x8*)(base + soff[u]);
  };
  h16* const wbuf = lds + trow * WLDA + tcol * 8;
  constexpr int BUF = NSV * RPV * WLDA;               // halves of one chunk buffer, of three
  auto place_chunk = [&](int off, const h16x8 (&st)[NSV]) {
#pragma unroll
    for (int u = 0; u < NSV; ++u) *(h16x8*)(wbuf + off + u * (RPV * WLDA)) = st[u];
  };
  // the wave's fragments, k-step by k-step, the WT tiles of a k-step together; past the last
  // k-step the pointers stay there, so the ring's surplus refills re-read lines just fetched
  const char* lw = (const char*)(ex.w + ((size_t)t0 * ksteps + (size_t)kc * nsteps) * 64);
  const size_t tstride = (size_t)ksteps * 1024;       // bytes to the next tile, same k-step
  const unsigned loff = lane * 16;
  int lleft = nsteps;
  auto issue = [&](int u) -> h16x8 {
    const h16x8 v = __builtin_nontemporal_load((const h16x8*)(lw + u * tstride + loff));
    if (u == WT - 1) {
      const bool adv = lleft > 1;
      lw += adv ? 1024 : 0;
      lleft -= adv;
    }
    return v;
  };
  // the products are taken as weights x rows: lane l's accumulator q is row l % 16 of the group, column
  // cbase + q of the tile, so that a lane stores four adjacent columns at once
  const int row = lane & 15, kg = lane >> 4, cbase = 4 * kg;
  h16x4 bias[WT];
  if constexpr (EPI == E_BIAS16 || EPI == E_GELU16 || EPI == E_GELUF16) {
#pragma unroll
    for (int u = 0; u < WT; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) bias[u][q] = ex.bias[(t0 + u) * 16 + cbase + q];   // (any alignment)
  }
  // operand chunks 0 and 1 first, then the weight prefetch (independent of them), then chunks 2 and 3
  h16x8 ring[WSPF];
  {
    h16x8 p0[NSV], p1[NSV];
    load_chunk(0, p0);
    load_chunk(min(1, nchunk - 1), p1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < WSPF; ++p) {
      ring[p] = issue(p % WT);
      // issued in slot order: each multiply then waits for its own slot alone (with the order left
      // free, slot 0 went out seventh and the first multiply waited for the whole ring)
      __builtin_amdgcn_sched_barrier(0);
    }
    load_chunk(min(2, nchunk - 1), st0);
    load_chunk(min(3, nchunk - 1), st1);
    __builtin_amdgcn_sched_barrier(0);
    place_chunk(0, p0);
    place_chunk(BUF, p1);
  }
  lds_barrier();
  f32x4 acc[WT][NGW];
#pragma unroll
  for (int u = 0; u < WT; ++u)
#pragma unroll
    for (int g = 0; g < NGW; ++g) acc[u][g] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // (every row group is multiplied, which keeps the loop free of branches)
  const h16* const rbuf = lds + (g0 * 16 + row) * WLDA + kg * 8;
  int off0 = 0, off1 = BUF, off2 = 2 * BUF;           // buffers of chunks c, c + 1, c + 2
  h16x8 av[AP ? 2 : 1][NGW];
  auto read = [&](int off, int q, int set) __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < NGW; ++g) av[set][g] = *(const h16x8*)(rbuf + off + g * (16 * WLDA) + q * 32);
  };
  if constexpr (AP) read(0, 0, 0);
  constexpr int CYC = WRC % 2 ? 2 * WRC : WRC;        // chunks per ring cycle, an even count
  auto chunk = [&](int c, auto hc) __attribute__((always_inline)) {
    constexpr int h = decltype(hc)::value;            // c % CYC
    constexpr int hs = h % WRC * WKS;
#pragma unroll
    for (int q = 0; q < WKS; ++q) {
      if constexpr (AP) {
        if (q + 1 < WKS) read(off0, q + 1, (q + 1) & 1);
        else read(off1, 0, 0);                        // (past the last chunk: never used)
        __builtin_amdgcn_sched_barrier(0);
      } else {
        read(off0, q, 0);
      }
#pragma unroll
      for (int g = 0; g < NGW; ++g) {
#pragma unroll
        for (int u = 0; u < WT; ++u) acc[u][g] = mfma_f16(ring[(hs + q) * WT + u], av[AP ? q & 1 : 0][g], acc[u][g]);
      }
#pragma unroll
      for (int u = 0; u < WT; ++u) ring[(hs + q) * WT + u] = issue(u);
      if (q == (WKS > 1 ? 1 : 0)) {
        place_chunk(off2, h & 1 ? st1 : st0);
        load_chunk(min(c + 4, nchunk - 1), h & 1 ? st1 : st0);
      }
      // left free, the scheduler hoists every read of the chunk ahead of the multiplies and runs
      // out of registers
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
    const int o = off0;
    off0 = off1; off1 = off2; off2 = o;
  };
  int c0 = 0;
  for (; c0 + CYC <= nchunk; c0 += CYC) unrolled<0, CYC>([&](auto h) __attribute__((always_inline)) { chunk(c0 + h, h); });
  unrolled<0, CYC - 1>([&](auto h) __attribute__((always_inline)) { if (c0 + h < nchunk) chunk(c0 + h, h); });
  // epilogue: row g * 16 + row, columns n .. n + 3
#pragma unroll
  for (int g = 0; g < NGW; ++g) {
    const int r = (g0 + g) * 16 + row;
    if (r >= S) break;
#pragma unroll
    for (int u = 0; u < WT; ++u) {
      const int n = (t0 + u) * 16 + cbase;
      const f32x4 v = acc[u][g];
      if constexpr (EPI == E_PART) {
        *(f32x4*)((float*)ex.out + ((size_t)kc * S + r) * a.N + n) = v;
      } else if constexpr (EPI == E_PART16) {
        const int hr = ex.hrows > 0 ? ex.hrows : S, hb = r / hr, rr = r - hb * hr;
        h16* o = (h16*)ex.out + ((size_t)kc * (S / hr) + hb) * hr * a.N;
        *(h16x4*)(o + (ex.pack ? frag_index(rr, n, hr) : (size_t)rr * a.N + n)) =
            (h16x4){(h16)v[0], (h16)v[1], (h16)v[2], (h16)v[3]};
      } else {
        h16x4 w;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float y = v[q] + (float)bias[u][q];
          if constexpr (EPI == E_GELUF16) w[q] = gelu16_erff(r16(y));
          else w[q] = EPI == E_BIAS16 ? (h16)y : (h16)gelu_erf(a.gelu_r16 ? r16(y) : y);
        }
        h16* o = (h16*)ex.out + (size_t)r * a.N + n;
        if (EPI == E_BIAS16 && ex.nsplit > 0) {
          const int part = n / ex.nsplit;
          o = (h16*)ex.out + ((size_t)part * S + r) * ex.nsplit + (n - part * ex.nsplit);
        }
        *(h16x4*)o = w;
      }
    }
  }
}

template <int EPI, int NG, int WV, int CH, int WT, int RS, int RC, bool GA, bool HALF>
__global__ void __launch_bounds__(WV * 64) k_wide(WArgs a) {
  int b = blockIdx.x;
  const int per_ex = a.ks * a.wg_per_kc;
  int e, kc, tg;
  if (a.map == MAP_XCD) {
    const int x = b & 7, j = b >> 3;
    const int cl = j / a.wg_per_kc;
    const int combo = x + 8 * cl;
    tg = j - cl * a.wg_per_kc;
    e = combo / a.ks;
    kc = combo - e * a.ks;
  } else {
    if (a.map == MAP_PAIR) {
      // workgroups b and b + 8 (dispatched together, on the same XCD) take the same unit of the
      // two groups, so the second reads the weight fragments the first has just brought into the
      // XCD's L2 instead of from HBM
      const int lo = b & 7, hi = b >> 3;
      b = (((hi >> 1) << 3) | lo) + (hi & 1) * (a.nex / 2) * per_ex;
    }
    e = b / per_ex;
    b -= e * per_ex;
    kc = b / a.wg_per_kc;
    tg = b - kc * a.wg_per_kc;
  }
  const WEx& ex = a.ex[e];
  // an entry with at most half the rows (the first chunk expert) multiplies half the row groups
  if (HALF && ex.S <= NG * 8) wide_unit<EPI, NG / 2, WV, CH, WT, RS, RC, GA>(a, ex, kc, tg);
  else wide_unit<EPI, NG, WV, CH, WT, RS, RC, GA>(a, ex, kc, tg);
}

template <int EPI, int NG, int WV, int CH, int WT, int RS, int RC, bool GA, bool HALF>
int launch_wide_k(const WArgs& a, hipStream_t st) {
  constexpr size_t lds = (size_t)3 * wide_rows(NG, WV, CH) * (CH + 8) * 2;
  static_assert(lds <= 150 * 1024, "three chunk buffers fit the LDS");
  static unsigned long long attr_set = 0;
  int dev = 0;
  CFH_HIP(hipGetDevice(&dev));
  if (dev < 64 && !(attr_set & (1ull << dev))) {
    CFH_HIP(hipFuncSetAttribute((const void*)k_wide<EPI, NG, WV, CH, WT, RS, RC, GA, HALF>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                150 * 1024));
    attr_set |= 1ull << dev;
  }
  const long long wgs = (long long)a.nex * a.ks * a.wg_per_kc;
  hipLaunchKernelGGL((k_wide<EPI, NG, WV, CH, WT, RS, RC, GA, HALF>), dim3((unsigned)wgs), dim3(WV * 64), lds, st, a);
  CFH_LAUNCH_CHECK();
  return CFH_OK;
}

// Shape of a wide launch's workgroups: wv waves, wv / rs of them side by side on wt adjacent 16-column
// tiles each, every rs-th part of the rows.
struct WShape {
  int wv, wt, rs;
  int tiles() const { return wv / rs * wt; }
};
constexpr WShape WSHAPES[] = {{4, 1, 2}, {4, 1, 1}, {4, 2, 1}, {4, 3, 1}, {8, 2, 1}, {8, 3, 1}};

// 128-column chunks of fragments a wave keeps in flight.  The loads in flight are not what bounds these
// launches: four chunks at {4, 2, 1} were 7% slower than one over a 13-request d = 2560 flow (each
// workgroup's start and end carry the surplus), two at {8, 3, 1} do not fit the registers.
constexpr int wide_rc(int wv, int wt) { return wv * wt == 8 || wv * wt == 24 ? 1 : 2; }

// Shape checks of a wide launch (also used by the plan): CFH_OK when every workgroup covers whole
// units, every k-split a whole number of chunks, and the rows fit.
int wide_check(const WArgs& a, WShape s, int S_max, int ch = WCH) {
  if (a.nex < 1 || a.nex > 4 || a.N <= 0 || a.N % 16 || a.ks <= 0 || a.K % a.ks || (a.K / a.ks) % ch)
    return CFH_E_UNSUPPORTED;
  bool known = false;
  for (const WShape& w : WSHAPES) known = known || (w.wv == s.wv && w.wt == s.wt && w.rs == s.rs);
  if (!known || (a.N / 16) % s.tiles() || S_max < 1 || S_max > WMAXR)
    return CFH_E_UNSUPPORTED;
  if (a.pair && a.nex % 2) return CFH_E_UNSUPPORTED;
  return CFH_OK;
}

// Shape of a full-K launch of `units` units of `tiles` column tiles: the one with the least rounds of
// 256 workgroups x (tiles a workgroup + 4), the 4 for what a workgroup costs whatever its tiles (its
// start, the staging of the rows); the last listed on ties.  Without the 4, flow passes (4 layers, 2
// steps) take 2.89 ms where this takes 2.67 (16 requests, d = 4096), 3.33 where 3.25 (8, d = 5120), 1.32
// where 1.23 (16, d = 2048); at d = 1024 up to 16 requests and in the latent drafter the two agree.
WShape wide_shape_for(int tiles, int units) {
  constexpr int CUS = 256;
  WShape best = {};
  long long best_load = 0;
  for (const WShape& s : WSHAPES) {
    if (tiles % s.tiles()) continue;
    const long long wgs = (long long)units * tiles / s.tiles();
    const long long load = (wgs + CUS - 1) / CUS * (s.tiles() + 4);
    if (!best.wv || load <= best_load) {
      best = s;
      best_load = load;
    }
  }
  return best;
}

// k-splits of a split-K launch: the most workgroups up to one a CU (the operand buffers of more than 64
// rows leave room for one).  The first split to give 256, whose last round is then nearly empty, takes
// 4.35 ms where this takes 3.97 (flow pass of 4 layers and 2 steps, 16 requests, d = 5120: 160 workgroups
// for 320), 1.27 where 1.17 (8 requests, d = 2560) and 1.76 where 1.66 (16 requests of the latent
// drafter); at d = 1024, 2048 and 4096 the two agree.
int wide_ks(int N, int K, int units, WShape s) {
  constexpr int CUS = 256;
  int best = 0;
  for (int ks = 1; ks <= K / WCH; ++ks) {
    if (K % ks || (K / ks) % WCH) continue;
    if (best && (long long)units * (N / 16 / s.tiles()) * ks > CUS) break;
    best = ks;
  }
  return best;
}

// GA: the operand rows are gathered by WEx::ids.  HALVES: entries of at most half the largest one's
// row groups multiply half as many (the flow's chunk experts).
template <int EPI, bool HALVES = false, int CH = WCH, bool GA = false>
int launch_wide(const WArgs& a0, WShape s, hipStream_t st) {
  WArgs a = a0;
  int S_max = 0;
  for (int e = 0; e < a.nex; ++e) S_max = std::max(S_max, a.ex[e].S);
  if (wide_check(a, s, S_max, CH)) return CFH_E_UNSUPPORTED;
  for (int e = 0; e < a.nex; ++e)
    if (a.ex[e].S < 1 || a.ex[e].lda < a.K || !a.ex[e].w || !a.ex[e].a || !a.ex[e].out || !a.ex[e].ids == GA) return CFH_E_INVALID;
  a.wg_per_kc = (a.N / 16) / s.tiles();
  // the side-by-side order needs a whole number of 8-workgroup runs per half (narrow widths such as
  // d = 640 have 5 a k-split: their paired launches keep the plain order, still one launch for both)
  const bool pair_runs = a.pair && ((long long)(a.nex / 2) * a.ks * a.wg_per_kc) % 8 == 0;
  if (a.ks > 1 && (a.nex * a.ks) % 8 == 0 && (!a.pair || ((a.nex / 2) * a.ks) % 8 == 0))
    a.map = MAP_XCD;
  else
    a.map = pair_runs ? MAP_PAIR : MAP_PLAIN;
  const int ng = (S_max + 15) / 16;
  [[maybe_unused]] bool half = false;
  for (int e = 0; e < a.nex; ++e) half = half || a.ex[e].S <= (ng <= 2 ? 0 : ng <= 4 ? 32 : 64);
#define CFH_WIDE_S(G, W, T, R)                                                                                       \
  if (ng <= G && s.wv == W && s.wt == T && s.rs == R) {                                                                        \
    if constexpr (G > 2 && HALVES)                                                                                \
      if (half) return launch_wide_k<EPI, G, W, CH, T, R, wide_rc(W, T), GA, true>(a, st);                           \
    return launch_wide_k<EPI, G, W, CH, T, R, wide_rc(W, T), GA, false>(a, st);                                      \
  }
#define CFH_WIDE(W, T, R) CFH_WIDE_S(2, W, T, R) CFH_WIDE_S(4, W, T, R) CFH_WIDE_S(8, W, T, R)
  CFH_WIDE(4, 2, 1)
  // (the factor launches come in one shape only, the gathered ones in two)
  if constexpr (EPI != E_PART16) { CFH_WIDE(8, 2, 1) }
  if constexpr (EPI != E_PART16 && !GA) {
    CFH_WIDE(4, 1, 2) CFH_WIDE(4, 1, 1) CFH_WIDE(4, 3, 1) CFH_WIDE(8, 3, 1)
  }
#undef CFH_WIDE
#undef CFH_WIDE_S
  return CFH_E_UNSUPPORTED;
}

// Self attention of a wide group (causal, or with no mask), one workgroup per (entry, request,
// head): the request's Sr rows of q, k, v (columns of head h of the [S][3d] rows) staged in LDS,
// then `attend` (the narrow kernel's attention, same arithmetic), written as fp16 rows [S][d] of
// the attention output.
struct SelfArgs {
  const h16* qkv[4];   // [S][3d]
  h16* out[4];         // [S][d]
  int S[4], Sr[4];     // rows, rows per request
  int nex, R, H, d, hd;
  int bidir;           // 0: causal (the flow's draft rows); 1: no mask (the VAE's sequences)
};

constexpr int SAT = 256;          // threads of a self-attention workgroup

__global__ void __launch_bounds__(SAT) k_self_attn(SelfArgs a) {
  extern __shared__ __align__(16) h16 sm[];
  int b = blockIdx.x;
  const int h = b % a.H;
  b /= a.H;
  const int j = b % a.R, e = b / a.R;
  const int Sr = a.Sr[e], hd = a.hd, d = a.d;
  if ((j + 1) * Sr > a.S[e]) return;                  // (a request the group does not hold)
  const h16* src = a.qkv[e] + (size_t)j * Sr * 3 * d + h * hd;
  h16* sq = sm;
  h16* sk = sq + Sr * hd;
  h16* sv = sk + Sr * hd;
  float* P = (float*)(sv + Sr * hd);                  // [Sr][Sr]
  const int nv = hd / 8;
  for (int idx = threadIdx.x; idx < 3 * Sr * nv; idx += blockDim.x) {
    const int part = idx / (Sr * nv), rem = idx - part * Sr * nv;
    const int i = rem / nv, c = (rem - i * nv) * 8;
    *(h16x8*)(sq + (size_t)(part * Sr + i) * hd + c) = *(const h16x8*)(src + (size_t)i * 3 * d + part * d + c);
  }
  lds_barrier();
  attend(Sr, Sr, Sr, Sr, hd, hd, !a.bidir, sq, sk, sv, P, a.out[e] + (size_t)j * Sr * d + h * hd, d);
}

int launch_self_attn(const SelfArgs& a, hipStream_t st) {
  if (a.hd % 8 || a.hd <= 0 || a.nex < 1 || a.nex > 4) return CFH_E_UNSUPPORTED;
  int Srm = 0;
  for (int e = 0; e < a.nex; ++e) {
    if (a.Sr[e] < 1 || a.Sr[e] > 16 || a.S[e] > a.R * a.Sr[e]) return CFH_E_UNSUPPORTED;
    Srm = std::max(Srm, a.Sr[e]);
  }
  const size_t lds = (size_t)3 * Srm * a.hd * 2 + (size_t)Srm * Srm * 4;
  if (lds > 64 * 1024) return CFH_E_UNSUPPORTED;
  hipLaunchKernelGGL(k_self_attn, dim3((unsigned)(a.nex * a.R * a.H)), dim3(SAT), lds, st, a);
  CFH_LAUNCH_CHECK();
  return CFH_OK;
}

// Cross attention of a wide group whose heads do not fold (head widths such as 80: two heads an
// MFMA k-chunk), one workgroup per (expert, request, head): the request's Sr rows of q (columns of
// head h of the [S][d] rows, bias included), its C context rows of K and V (block l's [2][Ct][d]
// image, the request's rows [j C, j C + C)), staged in LDS, then `attend` without a mask, written
// as fp16 rows [S][d] of the attention output.
struct CrossArgs {
  const h16* q[4];     // [S][d]
  const h16* kv[4];    // [2][Ct][d]: K rows then V rows
  h16* out[4];         // [S][d]
  int S[4], Sr[4], Ct[4];
  int nex, R, H, d, hd, C;
};

__global__ void __launch_bounds__(SAT) k_cross_attn(CrossArgs a) {
  extern __shared__ __align__(16) h16 sm[];
  int b = blockIdx.x;
  const int h = b % a.H;
  b /= a.H;
  const int j = b % a.R, e = b / a.R;
  const int Sr = a.Sr[e], C = a.C, hd = a.hd, d = a.d;
  if ((j + 1) * Sr > a.S[e] || (j + 1) * C > a.Ct[e]) return;   // (a request the group does not hold)
  const h16* qs = a.q[e] + (size_t)j * Sr * d + h * hd;
  const h16* ks = a.kv[e] + (size_t)j * C * d + h * hd;
  const h16* vs = ks + (size_t)a.Ct[e] * d;
  h16* sq = sm;
  h16* sk = sq + Sr * hd;
  h16* sv = sk + C * hd;
  float* P = (float*)(sv + C * hd);                   // [Sr][C]
  const int nv = hd / 8;
  for (int idx = threadIdx.x; idx < (Sr + 2 * C) * nv; idx += blockDim.x) {
    const int i = idx / nv, c = (idx - i * nv) * 8;
    const h16* src = i < Sr ? qs + (size_t)i * d : i < Sr + C ? ks + (size_t)(i - Sr) * d : vs + (size_t)(i - Sr - C) * d;
    *(h16x8*)(sq + (size_t)i * hd + c) = *(const h16x8*)(src + c);
  }
  lds_barrier();
  attend(Sr, C, Sr, C, hd, hd, false, sq, sk, sv, P, a.out[e] + (size_t)j * Sr * d + h * hd, d);
}

size_t cross_attn_lds(int Sr, int C, int hd) { return (size_t)(Sr + 2 * C) * hd * 2 + (size_t)Sr * C * 4; }

int launch_cross_attn(const CrossArgs& a, hipStream_t st) {
  if (a.hd % 8 || a.hd <= 0 || a.nex < 1 || a.nex > 4 || a.C < 1 || a.C > 16) return CFH_E_UNSUPPORTED;
  int Srm = 0;
  for (int e = 0; e < a.nex; ++e) {
    if (a.Sr[e] < 1 || a.Sr[e] > 16 || a.S[e] > a.R * a.Sr[e] || a.Ct[e] > a.R * a.C) return CFH_E_UNSUPPORTED;
    Srm = std::max(Srm, a.Sr[e]);
  }
  const size_t lds = cross_attn_lds(Srm, a.C, a.hd);
  if (lds > 64 * 1024) return CFH_E_UNSUPPORTED;
  hipLaunchKernelGGL(k_cross_attn, dim3((unsigned)(a.nex * a.R * a.H)), dim3(SAT), lds, st, a);
  CFH_LAUNCH_CHECK();
  return CFH_OK;
}

// The context rows' LayerNorm of every block, once per draft: rows[e][l][c] =
// fp16((ctx[c] - mean_c) rstd_c g_l + b_l) with the row moments the ROWS kernel left in mom (the
// narrow cross K/V stream applies the same formula while staging).
struct CtxLnArgs {
  const h16* ctx;      // [Ct][d]
  const float* mom;    // [Ct][2]
  const h16* g0[4];    // block 0's context_norm weight of each expert; block l at + l * vstride bytes
  const h16* b0[4];
  h16* out[4];         // [L][Ct][d]
  long long vstride;
  int nex, nl, Ct, d;
};

__global__ void __launch_bounds__(256) k_ctx_ln(CtxLnArgs a) {
  const int nv = a.d / 8;
  const size_t per_l = (size_t)a.Ct * nv, per_e = per_l * a.nl, total = per_e * a.nex;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    const int e = (int)(i / per_e);
    size_t r = i - (size_t)e * per_e;
    const int l = (int)(r / per_l);
    r -= (size_t)l * per_l;
    const int c = (int)(r / nv), k = (int)(r - (size_t)c * nv) * 8;
    const h16* gw = (const h16*)((const char*)a.g0[e] + (size_t)l * a.vstride);
    const h16* gb = (const h16*)((const char*)a.b0[e] + (size_t)l * a.vstride);
    const h16x8 xv = *(const h16x8*)(a.ctx + (size_t)c * a.d + k);
    const h16x8 gv = *(const h16x8*)(gw + k);
    const h16x8 bv = *(const h16x8*)(gb + k);
    const float mu = a.mom[2 * c], rs = a.mom[2 * c + 1];
    h16x8 o;
#pragma unroll
    for (int t = 0; t < 8; ++t) o[t] = (h16)(((float)xv[t] - mu) * rs * (float)gv[t] + (float)bv[t]);
    *(h16x8*)(a.out[e] + ((size_t)l * a.Ct + c) * a.d + k) = o;
  }
}

}  // namespace
