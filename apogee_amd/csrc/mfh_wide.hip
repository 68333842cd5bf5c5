// Flat filter for n = 8192 ... 65536 with 32 points per thread: one workgroup
// per pair (n = 8192, 16384) or per half of a pair's lags (32768, 65536), with
// the whole transform in registers.
//
// Transform.  n = 4096 RF, passes of radix RF, 16, 16, 16 (Stockham autosort),
// the arithmetic and tables of inverse_fft<n> (mfh_flat.h) at n <= 16384, so
// the two kernels agree bit for bit.  At n = 32768 and 65536 a pair is two
// workgroups: the lags k = 2 kl + h come from the half of the first pass's
// outputs with r' = h mod 2, and from there on the two halves never meet, so
// nothing but the product is computed twice.
//
// Exchanges go through LDS one component at a time: the real parts of all
// points, then the imaginary parts through the same space (4.25 n bytes per
// local point count instead of 8.5).  That is what lets two workgroups of 512
// threads share a CU at n = 16384 and 32768 (68 KiB each), so that one computes
// while the other waits at a barrier or for its rows; with 16 points per
// thread and both components at once one workgroup of 1024 threads filled the
// CU and every phase was exposed (n = 16384, 16 x 256: 157 us, now 104).
//
// Rows are read with 16-byte loads.  The vector cache serves a wave's load
// instruction in 16 clocks whether its lanes ask for 8 or for 16 bytes: with
// 8-byte loads the same kernel took 127 us at n = 16384 and 138 us at 65536
// (4 x 128), with 16-byte loads 118 and, with the spills of the wider
// prefetch gone, 103.
//
// Bound.  VALU issue: about 62 instructions per point at n = 16384 (70 at
// 65536, whose product is formed twice), i.e. 16 k clocks per pair and CU at
// n = 16384 against 15.6 k waiting at nothing; measured 16.8 k (104 us for
// 4096 pairs).  At n = 65536 one workgroup of 1024 threads fills the CU
// (136 KiB of LDS), and loads, exchanges and arithmetic overlap only within
// it: 36 k of 59 k clocks issue.  Measured against the kernels before (us,
// threshold 5.5, one filter's buffers warm): n = 8192 16 x 256: 89 to 50;
// 16384 16 x 256: 157 to 104; 32768 4 x 256: 118 to 74; 65536 4 x 128: 120 to
// 99 -- and 180 to 99 when several filters take turns, since the two-kernel
// path's scratch is then written through to memory.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mfh_flat.h"
#include "mfh_internal.h"

namespace mfh {

namespace {

// From how many pairs a call takes this path at 8192, 16384 and 32768.  Below, more
// threads per pair win: at 8192 and 16384 one workgroup per CU of the 16-point
// kernel (256 pairs: 8.2 against 9.4 us and 12.1 against 12.4; 384 pairs: 11.5
// against 10.8 and 22.1 against 17.6), at 32768 the two-kernel path (24 pairs:
// 16.8 against 15.8 us, but 25.7 against 26.3 with three filters in turn; 32:
// 20.6 and 17.3, 28.5 and 27.2).
constexpr long long kWideMinPairs[3] = {257, 257, 32};

// n = 65536: one workgroup of 1024 threads fills a CU, so pairs run in rounds of
// 128, each 25 us (36 with every sample a candidate), while the two-kernel
// path takes 0.17 (0.22) us a pair and 8 more per 256, one chunk of its
// scratch.  A round that the call does not fill must therefore hold enough
// pairs.  us a call, this path / two kernels, in brackets with three filters in
// turn, whose scratch leaves the caches; threshold 5.5, 64 bins: 64 pairs 26.9 /
// 30.8 (39.4 / 37.0), 72 26.2 / 32.2 (39.3 / 39.6); 132 51.1 / 41.6 (61.6 / 56.9),
// 160 50.2 / 45.8 (62.0 / 70.2), 192 51.0 / 49.3 (62.1 / 79.0); 260 74.8 / 71.7,
// 268 74.4 / 72.6 (86.0 / 112.2); 388 98.1 / 97.3; 512 101 / 119 (113 / 182).
// Without a threshold: 64 pairs 37.2 / 34.5 (50.9 / 40.2), 104 40.2 / 42.4 (51.3 /
// 51.7); 256 76.2 / 75.6 (87.6 / 112); 352 110.5 / 107.2 (122 / 155); 512 148 /
// 142 (160 / 207); from eight rounds on, where the spectra leave the caches,
// 1000 pairs 288 / 329.
bool wide_rounds_pay(long long pairs, bool dense) {
  constexpr long long kRound = 128;
  const long long rounds = (pairs + kRound - 1) / kRound, last = pairs - (rounds - 1) * kRound;
  if (dense) return rounds >= 8 || (rounds == 1 && last >= 104);
  constexpr int kFill[3] = {72, 64, 12};
  return rounds > 3 || (rounds > 0 && last >= kFill[rounds - 1]);
}

struct WideArgs {
  FlatArgs f;              // rows, window, bins, outputs, list
  long long p0;            // first pair (tiled) or list position of this launch
  long long np;            // pairs of this launch, at most
  uint64_t *pkey;          // S > 1: per-part bin tables [pair of the launch][part][nb]
  cf *pval;
  int *done;               // tiled, S > 1: part_is_last's counter per pair of the launch
};

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Ends a scheduling region: the scheduler would otherwise run independent
// butterflies side by side and spill, and other waves already fill their
// latency.
__device__ __forceinline__ void wide_fence() { __builtin_amdgcn_sched_barrier(0); }

// n = 4096 RF, S = RF / FL parts per pair.  Part h holds the lags k = S kl + h,
// kl < NL = 4096 FL, and is one workgroup of T = 128 FL threads with 32 points
// each.
template <int RF_, int FL_>
struct WideShape {
  static constexpr int RF = RF_, FL = FL_;
  static constexpr int S = RF / FL;
  static constexpr int N = 4096 * RF, NL = 4096 * FL;
  static constexpr int T = 128 * FL;
  static constexpr int XCH = NL + NL / 16;  // floats of the exchange space, padded
};

// The outputs k = 2 m + H, m < RF / 2, of an RF-point inverse DFT from
// c[i] = x[i] + x[i + RF/2] (H = 0) or x[i] - x[i + RF/2] (H = 1): the rest of
// dftR's arithmetic for that half of its outputs, so a pair's two parts
// repeat no operation of it.
template <int RF, int H>
__device__ __forceinline__ void wide_half_dft(cf *c) {
  if constexpr (RF == 4) {
    const cf u = H ? cmul_i(c[1]) : c[1];
    c[1] = csub(c[0], u);
    c[0] = cadd(c[0], u);
  } else if constexpr (RF == 8) {
    if constexpr (H) {
      c[1] = rot_w8_1(c[1]);
      c[2] = cmul_i(c[2]);
      c[3] = rot_w8_3(c[3]);
    }
    dft4(c[0], c[1], c[2], c[3]);
  } else {
    static_assert(RF == 16, "radix");
    cf y0[4], y1[4];  // k1 = H and k1 = H + 2
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const cf u = H ? cmul_i(c[i + 4]) : c[i + 4];
      y0[i] = cadd(c[i], u);
      y1[i] = csub(c[i], u);
    }
    if constexpr (H) {
      dft4_w16<+1>(y0[0], y0[1], y0[2], y0[3]);
      dft4_w16<-1>(y1[0], y1[1], y1[2], y1[3]);
    } else {
      dft4(y0[0], y0[1], y0[2], y0[3]);
      dft4_k2(y1[0], y1[1], y1[2], y1[3]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      c[2 * i] = y0[i];
      c[2 * i + 1] = y1[i];
    }
  }
}

// First pass (radix RF, no twiddles): butterflies j = 2 (t + q T) + e, e = 0 and
// 1, q < 16 / FL, read the products at j + 4096 r and keep the outputs
// r' = S m + H of their RF, which are the part's local elements FL j + m:
// v[(2 q + e) FL + m].  Two neighbouring points per 16-byte load (dword
// alignment is enough for it, so any complex64 row qualifies): 8-byte loads
// fill half of the vector cache's 64 bytes per clock.
template <class W, int H>
__device__ __forceinline__ void wide_first(cf *v, __amdgpu_buffer_rsrc_t rd, __amdgpu_buffer_rsrc_t rt, int t) {
  constexpr int RF = W::RF, FL = W::FL, S = W::S;
  static_assert(S <= 2, "one or two parts");
  auto load = [&](__amdgpu_buffer_rsrc_t row, int step, int half) {
    const int q = step / FL, r = step % FL + half * FL;
    return __builtin_bit_cast(
        f32x4, __builtin_amdgcn_raw_buffer_load_b128(row, t * 16, (2 * q * W::T + 4096 * r) * (int)sizeof(cf), 0));
  };
  // Steps of one r (S = 1) or of r and r + RF / 2, issued AHEAD steps before
  // they are used: eight loads in flight per wave (four cost 1-4%, sixteen gave
  // nothing).  The fences keep the scheduler from issuing more and spilling.
  constexpr int STEPS = 16, AHEAD = 4 / S;
  f32x4 x[AHEAD][S], y[AHEAD][S];
  auto issue = [&](int step) {
#pragma unroll
    for (int i = 0; i < S; i++) {
      x[step % AHEAD][i] = load(rd, step, i);
      y[step % AHEAD][i] = load(rt, step, i);
    }
  };
  wide_fence();
#pragma unroll
  for (int s = 0; s < AHEAD; s++) issue(s);
  cf b[2][FL];  // FL = RF / S
#pragma unroll
  for (int step = 0; step < STEPS; step++) {
    const int q = step / FL, r = step % FL;
    cf p[2][S];
#pragma unroll
    for (int i = 0; i < S; i++) {
      const f32x4 a = x[step % AHEAD][i], c = y[step % AHEAD][i];
      p[0][i] = cmul_conj(cf{a.x, a.y}, cf{c.x, c.y});
      p[1][i] = cmul_conj(cf{a.z, a.w}, cf{c.z, c.w});
    }
#pragma unroll
    for (int e = 0; e < 2; e++) {
      if constexpr (S == 1) b[e][r] = p[e][0];
      else b[e][r] = H ? csub(p[e][0], p[e][1]) : cadd(p[e][0], p[e][1]);
    }
    wide_fence();
    if (step + AHEAD < STEPS) issue(step + AHEAD);
    wide_fence();
    if (r == FL - 1) {
#pragma unroll
      for (int e = 0; e < 2; e++) {
        if constexpr (S == 1) dftR<RF>(b[e]);
        else wide_half_dft<RF, H>(b[e]);
#pragma unroll
        for (int m = 0; m < FL; m++) v[(2 * q + e) * FL + m] = b[e][m];
        wide_fence();
      }
    }
  }
}

// One component of an exchange: the pass outputs to LDS.
template <class W, int STAGE, int C>
__device__ __forceinline__ void wide_put(const cf *v, int t, float *x) {
  constexpr int FL = W::FL, T = W::T;
  auto comp = [&](int i) { return C ? v[i].y : v[i].x; };
  if constexpr (STAGE == 1) {
    // 2 FL consecutive elements per q, in 16-byte chunks; their order within
    // eight chunks (32 banks) is permuted so that eight neighbouring lanes'
    // stores of one i fall in distinct banks, as 64 lanes' reads still do
    constexpr int CH = FL / 2;
    const int sw = (CH * t >> 3) & (CH - 1);
    f32x4 *p = reinterpret_cast<f32x4 *>(x) + CH * t;
#pragma unroll
    for (int i = 0; i < CH; i++) {
      f32x4 *pi = p + (i ^ sw);
#pragma unroll
      for (int q = 0; q < 16 / FL; q++) {
        const int e = q * 2 * FL + 4 * i;
        pi[q * CH * T] = f32x4{comp(e), comp(e + 1), comp(e + 2), comp(e + 3)};
      }
    }
  } else if constexpr (STAGE == 2) {
    float *p = x + (t / FL) * (17 * FL) + t % FL;
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int r = 0; r < 16; r++) p[q * (T / FL) * (17 * FL) + FL * r] = comp(q + 2 * r);
  } else {
    float *p = x + (t / (16 * FL)) * (272 * FL) + t % (16 * FL);
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int r = 0; r < 16; r++) p[q * (T / (16 * FL)) * (272 * FL) + 16 * FL * r] = comp(q + 2 * r);
  }
}

// The same component back: element t + u T.
template <class W, int STAGE, int C>
__device__ __forceinline__ void wide_get(cf *v, int t, const float *x) {
  constexpr int FL = W::FL, T = W::T;
  const float *p;
  if constexpr (STAGE == 1) p = x + (t ^ (((t >> 5) & (FL / 2 - 1)) << 2));
  else if constexpr (STAGE == 2) p = x + t + FL * (t / (16 * FL));
  else p = x + t;
#pragma unroll
  for (int u = 0; u < 32; u++) {
    int o;
    if constexpr (STAGE == 1) o = u * T;
    else if constexpr (STAGE == 2) o = u * 136 * FL;
    else o = u * T + 16 * FL * (u >> 1);
    if constexpr (C) v[u].y = p[o];
    else v[u].x = p[o];
  }
}

// Exchange between passes, one component at a time through one buffer of half
// the size: the second component waits in its registers meanwhile.
template <class W, int STAGE>
__device__ __forceinline__ void wide_exchange(cf *v, int t, float *x) {
  if constexpr (STAGE > 1) __syncthreads();  // the previous exchange's last reads
  wide_put<W, STAGE, 0>(v, t, x);
  __syncthreads();
  wide_get<W, STAGE, 0>(v, t, x);
  __syncthreads();
  wide_put<W, STAGE, 1>(v, t, x);
  __syncthreads();
  wide_get<W, STAGE, 1>(v, t, x);
}

// Twiddles of butterflies Q0 .. Q0 + NQ - 1: register q + 2 r times w^r, with
// the powers from the table rows w^1, w^4 (and w^2, w^8) by power_twiddles' products,
// each used as soon as it is known (w^1 ... w^8 are all that stays live).
template <int Q0, int NQ>
__device__ __forceinline__ void wide_twiddle(cf *v, cf w1, cf w2, cf w4, cf w8) {
  auto use = [&](int r, cf w) {
#pragma unroll
    for (int q = Q0; q < Q0 + NQ; q++) v[q + 2 * r] = cmul(v[q + 2 * r], w);
  };
  cf w[8];
  w[1] = w1;
  w[2] = w2;
  w[3] = cmul(w1, w[2]);
  w[4] = w4;
  w[5] = cmul(w1, w4);
  w[6] = cmul(w[2], w4);
  w[7] = cmul(w[3], w4);
  use(8, w8);
#pragma unroll
  for (int r = 1; r < 8; r++) {
    use(r, w[r]);
    use(r + 8, cmul(w[r], w8));
  }
}

template <int Q0, int NQ>
__device__ __forceinline__ void wide_twiddle(cf *v, cf w1, cf w4) {
  wide_twiddle<Q0, NQ>(v, w1, cmul(w1, w1), w4, cmul(w4, w4));
}

// One radix-16 butterfly in place, registers q + 2 r.
__device__ __forceinline__ void wide_dft16(cf *v, int q) {
  cf b[16];
#pragma unroll
  for (int r = 0; r < 16; r++) b[r] = v[q + 2 * r];
  dft16(b);
#pragma unroll
  for (int r = 0; r < 16; r++) v[q + 2 * r] = b[r];
}

// Inverse transform of the part: v[u] ends as z[S (t + u T) + h].
template <class W>
__device__ __forceinline__ void wide_transform(cf *v, int t, int h, float *x, const cf *tw) {
  using L = TwiddleLayout<W::N>;
  constexpr int FL = W::FL, RF = W::RF, S = W::S, T = W::T;
  // tables of the passes NS = RF, 16 RF, 256 RF (RF = 16: the second, third and
  // fourth radix-16 pass)
  constexpr int p0 = L::NS0 == 1 ? 1 : 0;
  const cf *tw2 = tw + L::offset(p0), *tw3 = tw + L::offset(p0 + 1), *tw4 = tw + L::offset(p0 + 2);
  wide_exchange<W, 1>(v, t, x);
  wide_fence();
  {
    const cf *p = tw2 + S * (t % FL) + h;
    wide_twiddle<0, 2>(v, p[0], p[RF]);
  }
  wide_fence();
  wide_dft16(v, 0);
  wide_fence();
  wide_dft16(v, 1);
  wide_fence();
  wide_exchange<W, 2>(v, t, x);
  wide_fence();
  {
    const int k = S * (t % (16 * FL)) + h;
    const cf *p = tw3 + k;
    if constexpr (L::EXTRA_NS > 0) {
      const cf *e = tw + L::extra() + k;
      wide_twiddle<0, 2>(v, p[0], e[0], p[16 * RF], e[16 * RF]);
    } else {
      wide_twiddle<0, 2>(v, p[0], p[16 * RF]);
    }
  }
  wide_fence();
  wide_dft16(v, 0);
  wide_fence();
  wide_dft16(v, 1);
  wide_fence();
  wide_exchange<W, 3>(v, t, x);
  wide_fence();
  const cf *p = tw4 + S * t + h;
  wide_twiddle<0, 1>(v, p[0], p[256 * RF]);
  wide_fence();
  wide_dft16(v, 0);
  wide_fence();
  wide_twiddle<1, 1>(v, p[S * T], p[S * T + 256 * RF]);
  wide_fence();
  wide_dft16(v, 1);
  wide_fence();
}

typedef float f32x32 __attribute__((ext_vector_type(32)));

// A thread's samples for loops over u that stay loops (the index is uniform:
// register indexing).  Unrolled 32 times the selection is tens of KiB of code
// that a wave with a peak, rare under a threshold, fetches cold.
struct WideSamples {
  f32x32 x, y;
  __device__ __forceinline__ explicit WideSamples(const cf *v) {
#pragma unroll
    for (int u = 0; u < 32; u++) {
      x[u] = v[u].x;
      y[u] = v[u].y;
    }
  }
  __device__ __forceinline__ cf operator[](int u) const { return cf{x[u], y[u]}; }
};

// The u at which some lane of the wave has |z|^2 above the seed inside the
// window, as bits: one or two under a threshold, all 32 without.
template <class W>
__device__ __forceinline__ uint32_t wide_hot(const FlatArgs &a, const cf *v, int t, int h) {
  uint32_t hot = 0u;
#pragma unroll
  for (int u = 0; u < 32; u++) {
    const uint32_t k = (uint32_t)(W::S * (t + u * W::T) + h);
    const float m2 = __builtin_fmaf(v[u].x, v[u].x, v[u].y * v[u].y);
    if (__ballot(m2 > a.seed && k - a.ws < a.we - a.ws)) hot |= 1u << u;
  }
  return hot;
}

// The largest |z|^2 above the seed seen so far and its lag, lowest lag first
// among equals (samples come in rising lag order; a NaN is never taken).
struct WideBest {
  float m2;
  uint32_t lag;  // 0xffffffff: none
  __device__ __forceinline__ void start(float seed) {
    m2 = seed;
    lag = 0xffffffffu;
  }
  __device__ __forceinline__ void see(cf z, uint32_t k, bool in) {
    const float m = __builtin_fmaf(z.x, z.x, z.y * z.y);
    const bool take = in && m > m2;
    m2 = take ? m : m2;
    lag = take ? k : lag;
  }
  // raise `bin` to the wave's key (every lane of the wave calls this): only
  // the lanes that hold the wave's largest value go to the atomic
  __device__ __forceinline__ void flush(uint64_t *bin) const {
    const uint32_t m = lag != 0xffffffffu ? __float_as_uint(m2) : 0u;
    const uint32_t mw = wave_umax(m);
    if (mw && m == mw) atomicMax((unsigned long long *)bin, ((unsigned long long)m << 32) | (unsigned long long)(~lag));
  }
};

// Raises the bin keys of samples seen in rising lag order.  A wave's 64 lags at
// one u, kf ... kl, mostly share a bin: scalar compares against the current
// bin's end tell, and only the lanes of a wave that straddles an edge (or the
// window's) compute a bin of their own.
template <class W, bool ONE>
struct WideSelect {
  static constexpr int S = W::S, T = W::T;
  const FlatArgs &a;
  uint64_t *bins;
  int t, h;
  uint32_t kw;
  WideBest best;
  int cur = -1;
  uint32_t edge = 0u;  // first lag past bin `cur`
  __device__ __forceinline__ WideSelect(const FlatArgs &a_, uint64_t *bins_, int t_, int h_)
      : a(a_), bins(bins_), t(t_), h(h_), kw((uint32_t)(S * __builtin_amdgcn_readfirstlane(t_) + h_)) {
    best.start(a.seed);
  }
  __device__ __forceinline__ void see(cf z, int u) {
    const uint32_t k = (uint32_t)(S * (t + u * T) + h);
    if constexpr (ONE) {
      best.see(z, k, k - a.ws < a.we - a.ws);
    } else {
      const uint32_t kf = kw + (uint32_t)(S * T * u), kl = kf + 63u * S;
      bool same = kf >= a.ws && kl < a.we;
      if (same && kf >= edge) {
        if (cur >= 0) best.flush(bins + cur);
        best.start(a.seed);
        cur = __builtin_amdgcn_readfirstlane((int)bin_of(kf, a));
        edge = a.ws + (uint32_t)(cur + 1) * a.binsize;
      }
      same = same && kl < edge;
      if (same) {
        best.see(z, k, true);
      } else if (k - a.ws < a.we - a.ws) {
        const uint64_t key = make_key(z, k, a.seed);
        if (key) atomicMax((unsigned long long *)&bins[bin_of(k, a)], (unsigned long long)key);
      }
    }
  }
  __device__ __forceinline__ void end() {
    if constexpr (ONE) best.flush(bins);
    else if (cur >= 0) best.flush(bins + cur);
  }
};

// The samples at the `hot` u.  DENSE (no threshold: every u is hot): unrolled,
// since register indexing and the loop around it cost more than the rest of
// the selection.  In one kernel the two forms would keep the samples in two
// register layouts and spill, so the host picks.
template <class W, bool ONE, bool DENSE>
__device__ __forceinline__ void wide_select(const FlatArgs &a, const cf *v, uint32_t hot, int t, int h,
                                            uint64_t *bins) {
  WideSelect<W, ONE> sel(a, bins, t, h);
  if constexpr (DENSE) {
#pragma unroll
    for (int u = 0; u < 32; u++) {
      sel.see(v[u], u);
      wide_fence();
    }
  } else {
    const WideSamples s(v);
#pragma unroll 1
    for (; hot; hot &= hot - 1u) {
      const int u = __builtin_ctz(hot);
      sel.see(s[u], u);
    }
  }
  sel.end();
}

// Write the peaks of the bins whose winning lag this wave holds, at o + bin of
// the outputs (S = 1) or only their values, to pval (the keys go apart).  Up to
// kWideLook bins, each lane looks at one bin's key and the wave then visits its
// own winners one by one; past that the `hot` samples, 32 at most, look up
// theirs.  The line: without a threshold a wave of n = 8192 wins a quarter of the
// bins (2048 bins, 2052 pairs: 2.5 times the 16-point kernel's time by visits,
// 0.74 by lookups; 256 bins 1.05 and 1.05; 128 bins 0.88 and 0.94).
constexpr int kWideLook = 256;
template <class W, bool ONE>
__device__ __forceinline__ void wide_write(const FlatArgs &a, const WideSamples &v, uint32_t hot, int t, int h,
                                           int lane, int nb, const uint64_t *bins, long long o, cf *pval) {
  constexpr int S = W::S, T = W::T;
  auto put = [&](int b, uint32_t k, cf z) {
    if constexpr (S == 1) a.out.put(o + b, (long long)k, z);
    else part_put((uint64_t *)pval + o + b, __builtin_bit_cast(uint64_t, z));
  };
  if (ONE || nb <= kWideLook) {
    const int w0 = __builtin_amdgcn_readfirstlane(t);
#pragma unroll 1
    for (int b0 = 0; b0 < nb; b0 += 64) {
      const uint64_t key = b0 + lane < nb ? bins[b0 + lane] : 0ull;
      const uint32_t kwin = ~(uint32_t)key;
      unsigned long long mine = __ballot(key != 0ull && (int)((kwin / S) % T) - w0 >= 0 && (int)((kwin / S) % T) - w0 < 64);
#pragma unroll 1
      for (; mine; mine &= mine - 1ull) {
        const int j = __builtin_ctzll(mine);
        const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)kwin, j);
        const cf z = v[(int)(k / S / T)];
        if ((int)((k / S) % T) == t) put(b0 + j, k, z);
      }
    }
  } else {
#pragma unroll 1
    for (; hot; hot &= hot - 1u) {
      const int u = __builtin_ctz(hot);
      const cf z = v[u];
      const uint32_t k = (uint32_t)(S * (t + u * T) + h);
      if (k - a.ws < a.we - a.ws) {
        const uint32_t b = bin_of(k, a);
        if (k == ~(uint32_t)bins[b]) put((int)b, k, z);  // an empty bin's key is 0: past every lag
      }
    }
  }
}

// One (pair, bin) cell: the largest key over the parts (keys are distinct per
// lag) and that part's value.
template <int S>
__device__ __forceinline__ void wide_cell(const WideArgs &wa, long long pl, int b, long long o) {
  const int nb = (int)wa.f.nb;
  uint64_t best = 0ull;
  int bw = 0;
#pragma unroll
  for (int h = 0; h < S; h++) {
    const uint64_t key = part_get(wa.pkey + (pl * S + h) * nb + b);
    bw = key > best ? h : bw;
    best = key > best ? key : best;
  }
  if (best)
    wa.f.out.put(o, (long long)(~(uint32_t)best),
                 __builtin_bit_cast(cf, part_get((const uint64_t *)wa.pval + (pl * S + bw) * nb + b)));
  else
    wa.f.out.none(o);
}

template <class W, bool ONE, bool DENSE, bool LIST>
__global__ void __launch_bounds__(W::T) __attribute__((amdgpu_waves_per_eu(4))) wide_kernel(WideArgs wa) {
  constexpr int S = W::S, T = W::T, N = W::N;
  FlatArgs &a = wa.f;
  extern __shared__ __align__(16) unsigned char smem[];
  float *x = reinterpret_cast<float *>(smem);
  uint64_t *bins = reinterpret_cast<uint64_t *>(smem);  // after the last exchange, in the same space
  const int lane = threadIdx.x & 63;
  const int nb = (int)a.nb;
  if (a.zero && blockIdx.x == 0 && threadIdx.x == 0) *a.zero = 0;
  long long pairs = wa.np;
  if constexpr (LIST) {
    const int have = *a.list_count;
    if (a.hint && blockIdx.x == 0 && threadIdx.x == 0) *a.hint = have;
    pairs = min(pairs, (long long)have - wa.p0);
  }
  const long long units = pairs * S;
  // tiled: one workgroup per unit; list: drained grid-stride
  long long w = blockIdx.x;
  if (w >= units) return;
  do {
    // workgroups are dealt to the XCDs in turn (8 of them): give each XCD a
    // run of neighbouring units, which share spectra in its L2
    const long long c = w & 7, i = w >> 3, per = units >> 3, rem = units & 7;
    const long long unit = c * per + min(c, rem) + i;
    const long long pl = unit / S;
    const int h = (int)(unit % S);
    int d, tt;
    if constexpr (LIST) {
      const int2 pr = a.list[wa.p0 + pl];
      d = pr.x;
      tt = pr.y;
    } else {
      tt = (int)((wa.p0 + pl) / a.nd);
      d = (int)((wa.p0 + pl) % a.nd);
    }
    if constexpr (!LIST) {
      if (a.win) {
        a.ws = a.win[d].x;
        a.we = a.win[d].y;
      }
    }
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<cf *>(uniform_ptr(a.data + (long long)d * a.data_stride)), (short)0, N * (int)sizeof(cf),
        0x00020000);
    const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<cf *>(uniform_ptr(a.tmpl + (long long)tt * a.tmpl_stride)), (short)0, N * (int)sizeof(cf),
        0x00020000);
    cf v[32];
    if (S == 1 || h == 0) wide_first<W, 0>(v, rd, rt, t);
    else wide_first<W, S - 1>(v, rd, rt, t);
    wide_transform<W>(v, t, h, x, a.twiddle);
    // the thread's largest |z|^2: a wave with none above the seed raises no
    // key (nonnegative floats order like their bits; a NaN's bits, above all
    // of them, only send the wave on to wide_hot, which never takes one)
    uint32_t mloc = 0;
#pragma unroll
    for (int u = 0; u < 32; u++) mloc = max(mloc, __float_as_uint(__builtin_fmaf(v[u].x, v[u].x, v[u].y * v[u].y)));
    wide_fence();
    asm volatile("" : "+v"(t));
    uint32_t hot = 0u;
    if (wave_umax(mloc) > __float_as_uint(a.seed)) hot = DENSE ? 0xffffffffu : wide_hot<W>(a, v, t, h);
    __syncthreads();  // the last exchange is read
    for (int b = threadIdx.x; b < nb; b += T) bins[b] = 0ull;
    __syncthreads();
    if (hot) wide_select<W, ONE, DENSE>(a, v, hot, t, h, bins);
    __syncthreads();
    long long o;
    if constexpr (S > 1) o = unit * nb;
    else o = (LIST && a.list_ooff) ? a.list_ooff[wa.p0 + pl] : ((long long)d * a.nt + tt) * a.ostride;
    if (hot) wide_write<W, ONE>(a, WideSamples(v), hot, t, h, lane, nb, bins, o, wa.pval);
    for (int b = threadIdx.x; b < nb; b += T) {
      if constexpr (S > 1) part_put(wa.pkey + o + b, bins[b]);
      else if (bins[b] == 0ull) a.out.none(o + b);
    }
    if constexpr (S > 1 && !LIST) {
      if (part_is_last(wa.done + pl, S, *reinterpret_cast<int *>(smem))) {
        const long long ro = ((long long)d * a.nt + tt) * a.ostride;
        for (int b = threadIdx.x; b < nb; b += T) wide_cell<S>(wa, pl, b, ro + b);
      }
    }
    if constexpr (LIST) __syncthreads();  // the space is free for the next unit's exchange
    w += gridDim.x;
  } while (LIST && w < units);
}

// The cells of a list launch.  Its workgroups go on to further pairs, one at a time
// per CU, and would wait for their tables to arrive each time: 65536-point
// requests of a mixed queue take 340 us with this launch and 347 without.
template <int S>
__global__ void __launch_bounds__(256) wide_finish_kernel(WideArgs wa) {
  const FlatArgs &a = wa.f;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long pl = i / (int)a.nb;
  const int b = (int)(i % (int)a.nb);
  if (pl >= min(wa.np, (long long)*a.list_count - wa.p0)) return;
  const int2 pr = a.list[wa.p0 + pl];
  const long long o = a.list_ooff ? a.list_ooff[wa.p0 + pl] : ((long long)pr.x * a.nt + pr.y) * a.ostride;
  wide_cell<S>(wa, pl, b, o + b);
}

template <class W>
constexpr size_t wide_lds() {
  return (size_t)W::XCH * sizeof(float);
}

using WideKernel = void (*)(WideArgs);

// The kernel for a launch of nb bins and this seed, its LDS limit raised.  List
// launches take the rolled selection without a threshold too: beside the list's own
// state the unrolled one spills (a mixed queue without thresholds: 812 us a run
// against 692; 757 before this path).
template <class W, bool LIST>
WideKernel wide_pick(Ctx *c, size_t nb, bool dense) {
  const WideKernel k =
      nb == 1 ? (dense ? wide_kernel<W, true, !LIST, LIST> : wide_kernel<W, true, false, LIST>)
              : (dense ? wide_kernel<W, false, !LIST, LIST> : wide_kernel<W, false, false, LIST>);
  return lds_limit((const void *)k, c->dev, wide_lds<W>()) ? k : nullptr;
}

// The per-part tables of `total` pairs of nb bins, at most 64 MiB: `chunk` is
// the pairs that they hold.  A list launch has no part counters: they would have
// to be of the largest chunk, which is that of the fewest bins.
template <class W, bool LIST>
int wide_tables(Ctx *c, WideArgs &wa, long long total, size_t nb, long long &chunk) {
  chunk = std::max<long long>(1, std::min<long long>(total, (64ll << 20) / ((long long)W::S * (long long)nb * 16)));
  if (c->no_alloc || c->capturing) {  // the tables that are there, in more launches if need be
    const auto have = c->bufs.find("wide_key");
    const long long fit = have == c->bufs.end() ? 0 : (long long)(have->second.bytes / (W::S * nb * sizeof(uint64_t)));
    if (fit > 0) chunk = std::min(chunk, fit);
  }
  const size_t cells = (size_t)chunk * W::S * nb;
  wa.pkey = (uint64_t *)c->scratch("wide_key", cells * sizeof(uint64_t));
  wa.pval = (cf *)c->scratch("wide_val", cells * sizeof(cf));
  wa.done = LIST ? nullptr : c->part_counters((size_t)chunk);
  return wa.pkey && wa.pval && (LIST || wa.done) ? 0 : -1;
}

template <class W, bool LIST>
int wide_piece(Ctx *c, WideArgs &wa, long long total, size_t nb) {
  const WideKernel kern = wide_pick<W, LIST>(c, nb, wa.f.seed == 0.f);
  if (!kern) return -1;
  long long chunk = total;
  if (W::S > 1 && wide_tables<W, LIST>(c, wa, total, nb, chunk) < 0) return -1;
  chunk = std::min(chunk, 1ll << 20);  // a launch holds fewer than 2^32 threads
  for (long long p0 = 0; p0 < total; p0 += chunk) {
    wa.p0 = p0;
    wa.np = std::min(chunk, total - p0);
    long long grid = wa.np * W::S;
    // a list is drained grid-stride: its length is known on the device only
    if (LIST) grid = std::min<long long>(grid, 1024);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(W::T), wide_lds<W>(), c->stream, wa);
    if (!hip_ok(hipGetLastError(), "wide_kernel")) return -1;
    wa.f.zero = nullptr;
    wa.f.hint = nullptr;
    if (W::S > 1 && LIST) {
      const long long cells = wa.np * (long long)nb;
      hipLaunchKernelGGL(wide_finish_kernel<W::S>, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, c->stream, wa);
      if (!hip_ok(hipGetLastError(), "wide_finish_kernel")) return -1;
    }
  }
  return 0;
}

template <class W>
constexpr size_t wide_max_bins() {
  return wide_lds<W>() / sizeof(uint64_t);
}

template <class W>
int wide_run(Ctx *c, const FlatRun &r) {
  WideArgs wa{};
  const size_t nb_total = (r.we - r.ws + r.binsize - 1) / r.binsize;
  const size_t maxb = wide_max_bins<W>();
  const long long total = r.list ? (long long)r.list_cap : (long long)r.nd * r.nt;
  Ctx::ProfScope ps(c, r.list ? r.list_prof_name : r.prof_name);
  // bins past one LDS table split the window into pieces of whole bins, each
  // with its own transform; bins are independent
  for (size_t b0 = 0; b0 < nb_total; b0 += maxb) {
    const size_t cnt = std::min(maxb, nb_total - b0);
    const size_t ws = r.ws + b0 * r.binsize;
    const size_t we = std::min(r.we, ws + cnt * r.binsize);
    if (flat_base_args(c, W::N, r, ws, we, nb_total, b0, cnt, wa.f) < 0) return -1;
    if ((r.list ? wide_piece<W, true>(c, wa, total, cnt) : wide_piece<W, false>(c, wa, total, cnt)) < 0) return -1;
  }
  return 0;
}

// What a captured or allocation-free list launch of this shape needs.
template <class W>
int wide_ready(Ctx *c, const FlatRun &r) {
  WideArgs wa{};
  const size_t nb = (r.we - r.ws + r.binsize - 1) / r.binsize, most = std::min(nb, wide_max_bins<W>());
  const bool dense = !(r.threshold > 0.f);
  long long chunk;
  if (!wide_pick<W, true>(c, most, dense) || !wide_pick<W, true>(c, 1, dense)) return -1;
  return W::S == 1 || wide_tables<W, true>(c, wa, (long long)r.list_cap, most, chunk) == 0 ? 0 : -1;
}

}  // namespace

size_t wide_table_bins(size_t n) {
  switch (n) {
    case 8192: return wide_max_bins<WideShape<2, 2>>();
    case 16384: return wide_max_bins<WideShape<4, 4>>();
    case 32768: return wide_max_bins<WideShape<8, 4>>();
    case 65536: return wide_max_bins<WideShape<16, 8>>();
    default: return 0;
  }
}

bool wide_takes(const Ctx *c, size_t n, const FlatRun &r) {
  if (n < 8192 || n > 65536 || c->wide == 2) return false;
  if (c->wide == 1) return true;
  long long pairs = r.list ? (long long)r.list_cap : (long long)r.nd * r.nt;
  // without a threshold and with several bins every sample is a candidate, which
  // costs a thread with 32 of them more
  const bool multi = r.we - r.ws > r.binsize, dense = multi && !(r.threshold > 0.f);
  // a list's length as of the previous call (results never depend on it); a
  // captured or allocation-free call must find the buffers of the route that
  // it takes, so it goes by the list's capacity
  if (r.list && r.hint && !c->capturing && !c->no_alloc) {
    pairs = std::min<long long>(pairs, std::max(0, (int)*(volatile int *)r.hint));
    // the two-kernel path launches every chunk that the list could fill: 65536, 640
    // pairs of which 0 / 24 / 136 are left, one bin: 37 / 43 / 63 us a
    // hierarchical call, here 21 / 38 / 62
    if (n >= 32768 && !dense && (long long)r.list_cap * (long long)n * (long long)sizeof(cf) > c->big_chunk_bytes)
      return true;
  }
  // n = 8192, several bins: the 16-point kernel selects bins on the 64-lag grid in
  // runs, and holds its own to two workgroups per CU (us, here / there: without a
  // threshold, 1024-lag bins, 512 pairs 16.8 / 14.4, 600 19.4 / 22.2; threshold 3,
  // 1% of the samples, 400 pairs 1.16 of its time, 520 1.01).  Bins that several
  // lanes of a wave share but a wave straddles: 24 lags, 1030 pairs 1.19.
  if (n == 8192 && multi && !r.list) {
    const bool runs = r.binsize % 64 == 0 && r.ws % 64 == 0 && r.we % 64 == 0;
    if (dense && r.binsize > 8 && r.binsize < 64) return false;
    return pairs >= (dense && !runs && r.binsize >= 200 ? kWideMinPairs[0] : 513);
  }
  if (n <= 16384 || !multi) return n == 65536 ? wide_rounds_pay(pairs, false) : pairs >= kWideMinPairs[ilog2((int)n) - 13];
  // n = 32768 and 65536, several bins.  Tables that fill most of the LDS leave the
  // rows of two kernels few workgroups per CU: 65536, without a threshold, 16
  // lags to a bin, 64 pairs 0.83 of their time, 132 0.91; 8 lags, 24 pairs 0.93;
  // 32768, 8 lags, 40 pairs 0.99.
  const size_t nb = (r.we - r.ws + r.binsize - 1) / r.binsize;
  if (n == 65536 && nb > 3000) return pairs >= (nb >= 8192 ? 24 : 64);
  if (n == 32768 && nb >= 4096) return pairs >= (dense ? 48 : 40);
  // A wave's lags at one step span 128: without a threshold, bins down to a few
  // lanes wide straddle it (64 lags: 32768, 130 pairs 1.37 of the other path's
  // time, 600 1.17, 1030 0.91; 65536, 128 pairs 1.16, 1000 1.11, 2000 1.22; 300
  // lags: 32768, 260 pairs 1.10; 65536, 104 1.06, 1000 0.85; 512: 0.80 ... 1.0).
  if (n == 32768) return pairs >= (!dense ? 56 : r.binsize > 16 && r.binsize <= 400 ? 1024 : 104);
  if (dense && r.binsize <= (pairs >= 1024 ? 200 : 400)) return false;
  // with a threshold that 1% of the samples beat, a round costs up to 1.2 times
  // what the lines are for; search thresholds leave 1e-4 and fewer
  return wide_rounds_pay(pairs, dense);
}

int launch_wide(Ctx *c, size_t n, const FlatRun &r) {
  switch (n) {
    case 8192: return wide_run<WideShape<2, 2>>(c, r);
    case 16384: return wide_run<WideShape<4, 4>>(c, r);
    case 32768: return wide_run<WideShape<8, 4>>(c, r);
    case 65536: return wide_run<WideShape<16, 8>>(c, r);
    default: return fail("transform length %zu does not take this path", n);
  }
}

int wide_reserve(Ctx *c, size_t n, const FlatRun &r) {
  switch (n) {
    case 8192: return wide_ready<WideShape<2, 2>>(c, r);
    case 16384: return wide_ready<WideShape<4, 4>>(c, r);
    case 32768: return wide_ready<WideShape<8, 4>>(c, r);
    case 65536: return wide_ready<WideShape<16, 8>>(c, r);
    default: return 0;
  }
}

}  // namespace mfh
