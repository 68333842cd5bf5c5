// Flat filter for n >= 32768 across two kernels, columns and rows.
//
// n >= 131072: a four-step split.  A length-n transform does not fit one
// workgroup, so n = N1 x 256 with f = f1 + N1 f2 and k = k2 + 256 k1:
//   Y[f1][k2] = w_n^(f1 k2) sum_f2 P[f1 + N1 f2] w_256^(f2 k2)     kernel A
//   z[k2 + 256 k1] = sum_f1 Y[f1][k2] w_N1^(f1 k1)                 kernel B
// n = 32768 and 65536 (RF = n / 4096), for calls of few pairs: the four passes
// of the one-workgroup transform (mfh_wide.hip), the first two in kernel A
// (256 columns of 16 RF points), the last two in kernel B (16 RF rows of 256
// points), with the same arithmetic and so the same bits.  Spread over many
// workgroups, one pair takes 14 us instead of 33 at n = 65536; from some 30 (70 at
// 65536) pairs on the scratch round trip costs more than it gives (wide_takes).
// Kernel A forms the product D*conj(T) on load, runs the column transforms (256
// points, 16 RF at 32768 and 65536) over 16 columns per workgroup and writes Y
// k2-major to scratch (each 16-lane group writes 128 contiguous bytes).
// Kernel B gives each pair a few workgroups that walk k2 in groups, run the row
// transforms, and keep a per-bin (key, value) table in LDS: keys rise by
// ds_max_u64, and after each group the lane holding the bin's key writes its
// value, so the table always pairs the largest |z|^2 (lowest lag among equals)
// with its own z.  Only the final per-bin result leaves the chip.
//
// Reference behaviour: the same selection rule as the flat kernel
// (src/balanced-inl.h:876-969 in the reference checkout); the reference's GPU
// carried these lengths in one workgroup with R = 32/64 points per thread
// (src/gpu/tierb.slang:13-22), which wave64 register budgets do not allow.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "mfh_flat.h"
#include "mfh_internal.h"

namespace mfh {

namespace {

// ROWS rows of ROW points; columns of ROWS points, CT threads each.  RF > 0:
// the passes of the one-workgroup transform of n = 4096 RF.
template <int N1, int RF_ = 0>
struct BigShape {
  static constexpr int RF = RF_;
  static constexpr int ROWS = RF ? 16 * RF : 256;
  static constexpr int ROW = RF ? 256 : N1;
  static constexpr int N = ROWS * ROW;
  static constexpr int CT = ROWS / 16;
  static constexpr int COL_STRIDE = FlatShape<ROWS>::XCH + 1;  // see kColStride; 137 for 128 points
};

struct BigArgs {
  const cf *data, *tmpl;
  long long data_stride, tmpl_stride;
  int nd, nt;           // tiled mode: pair p = p0 + blockIdx -> (d, t) = (p % nd, p / nd)
  long long p0;         // first pair (tiled) or list position (list) of this chunk
  const int2 *list;     // list mode
  const int *list_count;
  int *hint;            // if set, the first workgroup stores the list length there (host-mapped)
  const long long *list_ooff;  // list mode: output element offset per pair
  cf *scratch;          // [chunk pair][ROWS][ROW]
  const cf *twCol, *twRow;  // Stockham tables of the column and the row passes
  const cf *rootH, *rootL; // w_N1^h (h < N1) and w_n^l (l < 256)
  int nsplit;               // rows workgroups per pair (gridDim.y of the rows kernel)
  uint64_t *pkey;           // nsplit > 1: per-part bin tables [pair][part][nb]
  cf *pval;
  int *done;                // RF > 0, if set: the pair's last part merges them (part_is_last)
  PeakOut out;
  uint32_t ws, we, binsize, nb, ostride;
  int bshift;
  float inv_bs, seed;
};

__device__ __forceinline__ bool big_pair(const BigArgs &a, long long p, int &d, int &t) {
  if (a.list) {
    if (p >= *a.list_count) return false;
    const int2 pr = a.list[p];
    d = pr.x;
    t = pr.y;
    return true;
  }
  if (p >= (long long)a.nd * a.nt) return false;
  // template-major: the nd pairs of one template are neighbours, so its
  // spectrum is re-read from L2 rather than HBM (2.5% at n = 65536, 4 x 128)
  t = (int)(p / a.nd);
  d = (int)(p % a.nd);
  return true;
}

// w_n^m for 0 <= m < n from the two root tables (global, a few KiB, cached).
__device__ __forceinline__ cf big_root(const BigArgs &a, int m) { return cmul(a.rootH[m >> 8], a.rootL[m & 255]); }

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Where a pair's outputs start.
__device__ __forceinline__ long long pair_out(const BigArgs &a, long long pl, int d, int t) {
  return a.list_ooff ? a.list_ooff[a.p0 + pl] : ((long long)d * a.nt + t) * a.ostride;
}

// One (pair, bin) cell of a chunk after its rows launch: the largest key over
// the parts (keys are distinct per lag, so exactly one part holds it) and that
// part's value.  The keys are read first, all independent loads, then the one value.
__device__ __forceinline__ void finish_cell(const BigArgs &a, long long np, long long i) {
  const int nb = (int)a.nb;
  if (i >= np * nb) return;
  const long long pl = i / nb;
  const int b = (int)(i % nb);
  int d = 0, tt = 0;
  if (!big_pair(a, a.p0 + pl, d, tt)) return;
  const uint64_t *keys = a.pkey + pl * a.nsplit * (long long)nb + b;
  uint64_t best = 0ull;
  int bw = 0;
#pragma unroll 8
  for (int w = 0; w < a.nsplit; w++) {
    const uint64_t key = keys[(long long)w * nb];
    bw = key > best ? w : bw;
    best = key > best ? key : best;
  }
  const long long o = pair_out(a, pl, d, tt) + b;
  if (best) a.out.put(o, (long long)(~(uint32_t)best), a.pval[(pl * a.nsplit + bw) * (long long)nb + b]);
  else a.out.none(o);
}

// Columns: 16 columns f1 of one pair per workgroup; lane = 16 * t + s, so the
// 16 lanes of a row group touch 16 consecutive columns (128-byte accesses).
// The pair's rows and its Y block are wave-uniform, so loads and stores go
// through buffer descriptors: one vector offset per thread and the per-u
// stride as a scalar offset, with no vector address arithmetic per point.
// A workgroup keeps its columns and walks pairs, so the closing twiddles are
// found once and the next pair's template columns, which come from HBM, are
// read into registers while this pair is transformed and stored.  One tile
// per workgroup, all in step, first read, then wrote: n = 262144, 2 x 31 pairs,
// cold templates: 63.2 us, of which reading alone takes 35 and writing alone
// 23; with the walk 53.0 (195 MB, 3.7 TB/s; the same at three or four
// workgroups per CU and with the data columns read ahead too).  At 4 waves per SIMD
// the registers spill (59.9 us).  WALK false: one tile per workgroup (kColTiles).
template <class B, bool WALK>
__global__ void __launch_bounds__(16 * B::CT) __attribute__((amdgpu_waves_per_eu(WALK ? 3 : 4)))
big_cols_kernel(BigArgs a, int np) {
  constexpr int N = B::N, ROW = B::ROW, CT = B::CT;
  extern __shared__ __align__(16) unsigned char smem[];
  const int s = threadIdx.x & 15;
  const int t = threadIdx.x >> 4;
  cf *xch = reinterpret_cast<cf *>(smem) + s * B::COL_STRIDE;
  // The four-step closing twiddle of output k2 = t + 16 u of column f1 splits as
  // w_n^(f1 k2) = w_n^(f1 t) * w_n^(16 f1 u): the first factor is one per
  // thread, the second one per (column, u), 256 per workgroup, kept in LDS
  // as bt[17 s + u] (rows of 17: the 16 columns a wave reads in one step
  // fall in distinct banks, its 4 row groups read the same words).
  cf *bt = reinterpret_cast<cf *>(smem) + 16 * B::COL_STRIDE;
  if (a.hint && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *a.hint = *a.list_count;
  int pl = (int)blockIdx.y;  // pair within the chunk
  int d = 0, tt = 0;
  if (!big_pair(a, a.p0 + pl, d, tt)) return;  // uniform; no barrier has run yet
  const int f1 = blockIdx.x * 16 + s;
  cf wt{1.f, 0.f};
  auto closing_roots = [&]() {
    if constexpr (!B::RF) {
      bt[17 * s + t] = big_root(a, 16 * f1 * t);  // u = t; 16 f1 t < n
      wt = big_root(a, f1 * t);
    }
  };
  cf w1{1.f, 0.f}, w4{1.f, 0.f};  // the column passes' twiddles depend on t only
  if constexpr (WALK) {
    w1 = a.twCol[TwiddleLayout<256>::offset(1) + t];
    w4 = a.twCol[TwiddleLayout<256>::offset(1) + 16 + t];
  }
  const int voff = (f1 + ROW * t) * (int)sizeof(cf);  // element f1 + ROW (t + CT u) at voff + u * CT ROW * 8
  auto row_rsrc = [](const cf *row) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<cf *>(uniform_ptr(row)), (short)0, N * (int)sizeof(cf),
                                             0x00020000);
  };
  auto load = [&](cf *x, __amdgpu_buffer_rsrc_t r) {
#pragma unroll
    for (int u = 0; u < 16; u++)
      x[u] = __builtin_bit_cast(cf, __builtin_amdgcn_raw_buffer_load_b64(r, voff, u * CT * ROW * (int)sizeof(cf), 0));
  };
  // inverse transform of the columns and Y[k2][f1], k2 = t + CT u; its barriers
  // order the bt stores before the reads
  auto finish = [&](cf *v, int pl) {
    if constexpr (WALK) {
      dft16(v);
      stockham_store<256, 16, 1>(v, t, xch);
      __syncthreads();
      stockham_load<256>(v, t, xch);
      cf w[15];
      power_twiddles(w, w1, w4);
#pragma unroll
      for (int r = 1; r < 16; r++) v[r] = cmul(v[r], w[r - 1]);
      dft16(v);
      __builtin_amdgcn_sched_barrier(0);
    } else {
      inverse_fft<B::ROWS>(v, t, xch, a.twCol);
    }
    const __amdgpu_buffer_rsrc_t ry = row_rsrc(a.scratch + (long long)pl * N);
    const int yoff = (t * ROW + f1) * (int)sizeof(cf);
#pragma unroll
    for (int u = 0; u < 16; u++) {
      if constexpr (!B::RF) v[u] = cmul(v[u], cmul(wt, bt[17 * s + u]));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v[u]), ry, yoff, u * CT * ROW * (int)sizeof(cf),
                                            0);
    }
  };
  if constexpr (!WALK) {
    closing_roots();
    const __amdgpu_buffer_rsrc_t rd = row_rsrc(a.data + (long long)d * a.data_stride);
    const __amdgpu_buffer_rsrc_t rt = row_rsrc(a.tmpl + (long long)tt * a.tmpl_stride);
    cf v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int so = u * CT * ROW * (int)sizeof(cf);
      const cf x = __builtin_bit_cast(cf, __builtin_amdgcn_raw_buffer_load_b64(rd, voff, so, 0));
      const cf y = __builtin_bit_cast(cf, __builtin_amdgcn_raw_buffer_load_b64(rt, voff, so, 0));
      v[u] = cmul_conj(x, y);
    }
    finish(v, pl);
  } else {
    cf y[16];
    load(y, row_rsrc(a.tmpl + (long long)tt * a.tmpl_stride));
    closing_roots();
    for (;;) {
      cf v[16];
      load(v, row_rsrc(a.data + (long long)d * a.data_stride));
      const int next = pl + (int)gridDim.y;
      const bool more = next < np && big_pair(a, a.p0 + next, d, tt);
#pragma unroll
      for (int u = 0; u < 16; u++) v[u] = cmul_conj(v[u], y[u]);
      // the next pair's template is read while this one is transformed and stored
      if (more) load(y, row_rsrc(a.tmpl + (long long)tt * a.tmpl_stride));
      __builtin_amdgcn_sched_barrier(0);
      finish(v, pl);
      if (!more) break;
      pl = next;
      __syncthreads();  // the exchange is read
    }
  }
}

// The table rows of the last two passes of the one-workgroup transform over row
// k of its 16 RF rows: the third pass's depend on the row only, the fourth's on
// k + 16 RF t.  Read ahead of the row itself (65536, 160 pairs: rows 19.3 -> 18.7 us).
template <int RF>
struct ClosingTwiddles {
  cf w3[4], w4[2];  // w^1, w^2, w^4, w^8 and w^1, w^4
  __device__ __forceinline__ ClosingTwiddles(int t, int k, const cf *tw) {
    using L = TwiddleLayout<4096 * RF>;
    constexpr int p0 = L::NS0 == 1 ? 1 : 0;  // the table of NS = RF
    const cf *tw3 = tw + L::offset(p0 + 1) + k, *tw4 = tw + L::offset(p0 + 2) + k + 16 * RF * t;
    const cf *e = tw + L::extra() + k;
    w3[0] = tw3[0];
    w3[1] = e[0];
    w3[2] = tw3[16 * RF];
    w3[3] = e[16 * RF];
    w4[0] = tw4[0];
    w4[1] = tw4[256 * RF];
  }
};

// Those passes: 256 points, thread t holding t + 16 u.
template <int RF>
__device__ __forceinline__ void closing_passes(cf *v, int t, cf *xch, const ClosingTwiddles<RF> &c) {
  cf w[15];
  power_twiddles(w, c.w3[0], c.w3[1], c.w3[2], c.w3[3]);
#pragma unroll
  for (int r = 1; r < 16; r++) v[r] = cmul(v[r], w[r - 1]);
  dft16(v);
  stockham_store<256, 16, 1>(v, t, xch);
  __syncthreads();
  stockham_load<256>(v, t, xch);
  power_twiddles(w, c.w4[0], c.w4[1]);
#pragma unroll
  for (int r = 1; r < 16; r++) v[r] = cmul(v[r], w[r - 1]);
  dft16(v);
}

// Rows: nsplit workgroups per pair (workgroup = pair * nsplit + part), each
// walking its share of the rows k2, SLOTS rows at a time.  With one part
// the table is the result; with several, each part leaves its (key, value)
// table and the largest key per bin is kept: by the pair's last part (RF > 0
// and small tables), else by finish_cell in the next chunk's rows launch or in
// big_rows_finish_kernel after the last chunk.
template <class B>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
big_rows_kernel(BigArgs a, BigArgs fin, long long fin_np, int fin_blocks) {
  // the last fin_blocks workgroups finish the previous chunk (its tables
  // were completed by the previous launch): one thread per (pair, bin)
  const int row_blocks = (int)gridDim.x - fin_blocks;
  if ((int)blockIdx.x >= row_blocks) {
    finish_cell(fin, fin_np, (long long)(blockIdx.x - row_blocks) * 256 + threadIdx.x);
    return;
  }
  constexpr int ROW = B::ROW, ROWS = B::ROWS;
  using S = FlatShape<ROW>;
  constexpr int TPT = S::TPT;
  constexpr int SLOTS = S::SLOTS;
  extern __shared__ __align__(16) unsigned char smem[];
  cf *xch_all = reinterpret_cast<cf *>(smem);
  uint64_t *bkey = reinterpret_cast<uint64_t *>(xch_all + SLOTS * S::XSTRIDE);
  cf *bval = reinterpret_cast<cf *>(bkey + a.nb);
  const int slot = threadIdx.x / TPT;
  const int t = threadIdx.x % TPT;
  cf *xch = xch_all + slot * S::XSTRIDE;
  const long long pl = blockIdx.x / a.nsplit;  // pair within the chunk
  const int part = (int)(blockIdx.x % a.nsplit);
  int d = 0, tt = 0;
  if (!big_pair(a, a.p0 + pl, d, tt)) return;  // uniform; before any barrier
  const int nb = (int)a.nb;
  for (int b = threadIdx.x; b < nb; b += 256) bkey[b] = 0ull;
  __syncthreads();
  const cf *Y = a.scratch + pl * (long long)B::N;
  constexpr int G = ROWS / SLOTS;  // row groups of the pair
  const int gbeg = part * G / a.nsplit, gend = (part + 1) * G / a.nsplit;
  const bool whole = a.ws == 0 && a.we == (uint32_t)B::N;
  const bool full8 = whole && a.bshift == ilog2(B::N / 8);
  FlatArgs fa;  // for bin_of / make_key
  fa.ws = a.ws;
  fa.we = a.we;
  fa.binsize = a.binsize;
  fa.bshift = a.bshift;
  fa.inv_bs = a.inv_bs;
  // the first twiddled pass's twiddles depend on t only: derived once for
  // all the part's row groups where the registers allow (rows of up to 512 points)
  constexpr bool HOIST = !B::RF && ROW <= 512;
  cf wf[HOIST ? 15 : 1];
  if constexpr (HOIST) first_twiddles<ROW>(wf, t, a.twRow);
  for (int g = gbeg; g < gend; g++) {
    const int k2 = g * SLOTS + slot;
    cf v[16];
    auto load = [&]() {
#pragma unroll
      for (int u = 0; u < 16; u++) v[u] = Y[(long long)k2 * ROW + t + TPT * u];
    };
    if constexpr (B::RF > 0) {
      const ClosingTwiddles<B::RF> w(t, k2, a.twRow);
      load();
      closing_passes<B::RF>(v, t, xch, w);
    } else {
      load();
      inverse_fft<ROW, HOIST>(v, t, xch, a.twRow, wf);
    }
    // thread t holds z[k2 + ROWS (t + TPT u)]; lags rise with u.  A wave none
    // of whose window lags has |z|^2 above the seed raises no key and records
    // no value, so it skips both steps below (wave-uniform; nonnegative
    // floats order like their bits, and a NaN's bits, above all of them,
    // send the wave through the steps, which never select it)
    uint32_t mloc = 0;
    if (whole) {
#pragma unroll
      for (int u = 0; u < 16; u++) mloc = max(mloc, __float_as_uint(__builtin_fmaf(v[u].x, v[u].x, v[u].y * v[u].y)));
    } else {
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const uint32_t k = (uint32_t)(k2 + ROWS * (t + TPT * u));
        const uint32_t m = __float_as_uint(__builtin_fmaf(v[u].x, v[u].x, v[u].y * v[u].y));
        mloc = (k >= a.ws && k < a.we) ? max(mloc, m) : mloc;
      }
    }
    const bool hot = wave_umax(mloc) > __float_as_uint(a.seed);
    if (!hot) {
    } else if (full8) {
      // n/8 bins over the whole transform: every wave's 64 lanes put u and
      // u + 1 = 2 rho, 2 rho + 1 in bin rho (their lags span < ROWS TPT)
      const int lane = threadIdx.x & 63;
      const int k2w = __builtin_amdgcn_readfirstlane(k2);
      runs8_max_to_bins<ROWS * TPT>(v, (uint32_t)(k2 + ROWS * t), (uint32_t)k2w, lane, a.seed, a.bshift, bkey);
    } else {
    uint64_t acc = 0ull;
    int acc_bin = -1;
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const uint32_t k = (uint32_t)(k2 + ROWS * (t + TPT * u));
      if (k >= a.ws && k < a.we) {
        const uint64_t key = make_key(v[u], k, a.seed);
        const int b = (int)bin_of(k, fa);
        if (b != acc_bin) {
          if (acc) atomicMax((unsigned long long *)&bkey[acc_bin], (unsigned long long)acc);
          acc = 0ull;
          acc_bin = b;
        }
        acc = key > acc ? key : acc;
      }
    }
    if (acc) atomicMax((unsigned long long *)&bkey[acc_bin], (unsigned long long)acc);
    }
    __syncthreads();
    // the holder of each bin's key records its value
    if (hot) {
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const uint32_t k = (uint32_t)(k2 + ROWS * (t + TPT * u));
        if (k >= a.ws && k < a.we) {
          const uint64_t key = make_key(v[u], k, a.seed);
          if (key) {
            const uint32_t b = bin_of(k, fa);
            if (bkey[b] == key) bval[b] = v[u];
          }
        }
      }
    }
    __syncthreads();  // values settled before the next group raises keys; xch reusable
  }
  const long long o = pair_out(a, pl, d, tt);
  if (a.nsplit > 1) {
    const long long po = (pl * a.nsplit + part) * (long long)nb;
    if (!B::RF || !a.done) {
      for (int b = threadIdx.x; b < nb; b += 256) {
        const uint64_t key = bkey[b];
        a.pkey[po + b] = key;
        a.pval[po + b] = key ? bval[b] : cf{0.f, 0.f};
      }
      return;
    }
    for (int b = threadIdx.x; b < nb; b += 256) {
      const uint64_t key = bkey[b];
      part_put(a.pkey + po + b, key);
      part_put((uint64_t *)a.pval + po + b, key ? __builtin_bit_cast(uint64_t, bval[b]) : 0ull);
    }
    if (!part_is_last(a.done + pl, a.nsplit, *reinterpret_cast<int *>(smem))) return;
    // the others' keys into this part's own table, all loads at once; then a
    // bin's value from the part that holds its winning lag's row
    const uint64_t *keys = a.pkey + pl * a.nsplit * (long long)nb;
#pragma unroll 4
    for (int i = threadIdx.x; i < a.nsplit * nb; i += 256) {
      const uint64_t key = part_get(keys + i);
      if (key) atomicMax((unsigned long long *)&bkey[i % nb], (unsigned long long)key);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += 256) {
      const uint64_t key = bkey[b];
      if (!key) {
        a.out.none(o + b);
        continue;
      }
      const uint32_t k = ~(uint32_t)key;
      const int w = (int)(k % ROWS) / SLOTS * a.nsplit / G;  // both powers of two
      const uint64_t *vals = (const uint64_t *)a.pval + (pl * a.nsplit + w) * (long long)nb;
      a.out.put(o + b, (long long)k, __builtin_bit_cast(cf, part_get(vals + b)));
    }
    return;
  }
  for (int b = threadIdx.x; b < nb; b += 256) {
    const uint64_t key = bkey[b];
    if (key) a.out.put(o + b, (long long)(~(uint32_t)key), bval[b]);
    else a.out.none(o + b);
  }
}

// The last chunk's finish (every other chunk's runs inside the next rows
// launch): one thread per (pair, bin) cell.
__global__ void __launch_bounds__(256) big_rows_finish_kernel(BigArgs a, long long np) {
  finish_cell(a, np, (long long)blockIdx.x * 256 + threadIdx.x);
}

__global__ void roots_kernel(cf *out, int L, int period) {
  // out[k] = exp(+2 pi i k / period), k < L
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < L) {
    double sn, cs;
    sincospi(2.0 * (double)k / (double)period, &sn, &cs);
    out[k] = cf{(float)cs, (float)sn};
  }
}

constexpr size_t kLds = 160 * 1024;
// n = 32768 and 65536: a pair's last part merges the parts' tables where a launch has
// no more than so many rows workgroups and a pair so many table entries; else a
// finish launch does.  Each workgroup that counts itself in waits for its
// entries first, and the next one on its CU for it: with 1024 of them the rows
// launch takes 14.9 us in place of 9.1, more than the finish launch's 4.6; one
// workgroup takes 3 us for 4096 entries.  us a call with its wait, merged /
// finish launch: 65536, 64 bins, threshold 5.5: 4 pairs (64 workgroups) 23.3 /
// 24.3, 8 24.9 / 24.9, 16 29.1 / 27.6; without a threshold 64 pairs 45.6 / 43.5;
// 4 pairs of 256 bins 31.6 / 28.5; 32768, one bin: 8 pairs 21.8 / 22.5, 16 23.8
// / 23.6, 64 33.0 / 32.1; several calls on their way gain another 0.7.  Longer
// rows keep the finish launch, most of which run inside the next chunk's rows
// launch: merging there took 2 x 31 pairs at 262144 from 104.8 to 102.7, but
// 1 x 20 from 53.7 to 57.8 and 4 x 64 from 321 to 330.
constexpr long long kMergeBlocks = 128;
constexpr size_t kMergeCells = 1024;
// Walking pairs pays from a good third more tiles than a launch has resident (us a
// call, walk / one tile each; tiles): 1280 49.5 / 48.2 and 53.9 / 53.7, 1440 57.6 /
// 60.2, 1536 66.7 / 67.5, 1792 67.7 / 69.0, 3968 104.8 / 111.
constexpr int kColTiles = 1400;
constexpr int kColGrid = 1024;  // columns workgroups per launch: four per CU, of which three are resident at a time

template <class B>
constexpr size_t big_cols_lds() {
  return (16 * B::COL_STRIDE + 16 * 17) * sizeof(cf);
}

template <class B>
size_t rows_max_bins() {
  using S = FlatShape<B::ROW>;
  return (kLds - (size_t)S::SLOTS * S::XSTRIDE * sizeof(cf)) / (sizeof(uint64_t) + sizeof(cf));
}

// What launches of up to `total` pairs with nb_total bins run in: pairs per chunk,
// rows workgroups per pair, and the buffers, which `a` and `b` then point to.
struct BigBuffers {
  long long chunk;
  size_t part_cells;
  uint64_t *pkey2 = nullptr;
  cf *pval2 = nullptr;
};

template <class B>
int big_buffers(Ctx *c, long long total, size_t nb_total, BigArgs &a, BigBuffers &b) {
  constexpr int N = B::N;
  using S = FlatShape<B::ROW>;
  a.twCol = c->twiddles(B::ROWS);
  a.twRow = c->twiddles(B::RF ? N : B::ROW);
  if (!a.twCol || !a.twRow) return -1;
  a.rootH = a.rootL = nullptr;
  if (!B::RF) {
    const cf *roots = big_roots(c, B::ROW);
    if (!roots) return -1;
    a.rootH = roots;
    a.rootL = roots + B::ROW;
  }
  // scratch in chunks of pairs: at most c->big_chunk_bytes of intermediate data
  b.chunk = std::max<long long>(1, std::min<long long>(total, c->big_chunk_bytes / ((long long)N * 8)));
  a.scratch = (cf *)c->scratch("big_scratch", (size_t)b.chunk * N * sizeof(cf));
  if (!a.scratch) return -1;
  if (!lds_limit((const void *)big_cols_kernel<B, false>, c->dev, big_cols_lds<B>()) ||
      !lds_limit((const void *)big_cols_kernel<B, !B::RF>, c->dev, big_cols_lds<B>()) ||
      !lds_limit((const void *)big_rows_kernel<B>, c->dev, kLds))
    return -1;
  // rows workgroups per pair: enough for about 1024 workgroups per launch (at
  // least 8, at most one per row group), as long as the per-part tables stay
  // within 64 MiB
  constexpr int G = B::ROWS / S::SLOTS;
  const size_t nb_piece = std::min(rows_max_bins<B>(), nb_total);
  int nsplit = (int)std::min<long long>(G, std::max<long long>(8, (1024 + b.chunk - 1) / b.chunk));
  nsplit = 1 << ilog2(nsplit);  // a power of two: parts split the row groups evenly
  while (nsplit > 1 && (size_t)b.chunk * nsplit * nb_piece * 16 > (64ull << 20)) nsplit /= 2;
  a.nsplit = nsplit;
  a.pkey = nullptr;
  a.pval = nullptr;
  // part tables in two halves, by chunk parity: a rows launch writes one
  // while its finishing blocks read the previous chunk's
  b.part_cells = (size_t)b.chunk * nsplit * nb_piece;
  if (nsplit > 1) {
    b.pkey2 = (uint64_t *)c->scratch("big_part_key", 2 * b.part_cells * sizeof(uint64_t));
    b.pval2 = (cf *)c->scratch("big_part_val", 2 * b.part_cells * sizeof(cf));
    if (!b.pkey2 || !b.pval2) return -1;
  }
  // where the pairs' last parts do not merge the tables, the finish of a chunk
  // runs in the next rows launch when the window is one piece (one rows launch
  // per chunk), and after each rows launch when not
  a.done = nullptr;
  if (B::RF && nsplit > 1) {
    a.done = c->part_counters((size_t)b.chunk);  // in any case: a later, captured call may have fewer bins
    if (!a.done) return -1;
    if (b.chunk * nsplit > kMergeBlocks || nb_piece * nsplit > kMergeCells) a.done = nullptr;
  }
  return 0;
}

template <class B>
int launch_big_shape(Ctx *c, const FlatRun &r) {
  using S = FlatShape<B::ROW>;
  BigArgs a;
  a.data = r.data;
  a.tmpl = r.tmpl;
  a.data_stride = r.data_stride;
  a.tmpl_stride = r.tmpl_stride;
  a.nd = r.nd;
  a.nt = r.nt;
  a.list = r.list;
  a.list_count = r.list_count;
  a.hint = r.list ? r.hint : nullptr;
  a.list_ooff = r.list_ooff;
  const float thr = r.threshold;
  a.seed = thr > 0.f ? (float)((double)thr * (double)thr) : 0.f;
  a.binsize = (uint32_t)r.binsize;
  const bool pow2 = (r.binsize & (r.binsize - 1)) == 0;
  a.bshift = pow2 ? ilog2((int)r.binsize) : -1;
  a.inv_bs = 1.0f / (float)r.binsize;
  const long long total = r.list ? (long long)r.list_cap : (long long)r.nd * r.nt;
  const size_t nb_total = (r.we - r.ws + r.binsize - 1) / r.binsize;
  const size_t maxb = rows_max_bins<B>();
  BigBuffers b;
  if (big_buffers<B>(c, total, nb_total, a, b) < 0) return -1;
  const long long chunk = b.chunk;
  const int nsplit = a.nsplit;
  const bool fold = nsplit > 1 && nb_total <= maxb;
  BigArgs fin = a;
  long long fin_np = 0;
  int fin_blocks = 0;
  long long ci = 0;  // chunk index
  Ctx::ProfScope ps(c, r.list ? r.list_prof_name : r.prof_name);
  for (long long p0 = 0; p0 < total; p0 += chunk, ci++) {
    const long long np = std::min(chunk, total - p0);
    a.p0 = p0;
    if (nsplit > 1) {
      a.pkey = b.pkey2 + (ci & 1) * b.part_cells;
      a.pval = b.pval2 + (ci & 1) * b.part_cells;
    }
    // the first with one tile per workgroup
    const long long tiles = np * (B::ROW / 16);
    if (!B::RF && tiles > kColTiles) {
      hipLaunchKernelGGL((big_cols_kernel<B, !B::RF>), dim3(B::ROW / 16, kColGrid / (B::ROW / 16)), dim3(16 * B::CT),
                         big_cols_lds<B>(), c->stream, a, (int)np);
    } else {
      hipLaunchKernelGGL((big_cols_kernel<B, false>), dim3(B::ROW / 16, (unsigned)np), dim3(16 * B::CT),
                         big_cols_lds<B>(), c->stream, a, (int)np);
    }
    if (!hip_ok(hipGetLastError(), "big_cols_kernel")) return -1;
    a.hint = nullptr;
    for (size_t b0 = 0; b0 < nb_total; b0 += maxb) {
      const size_t cnt = std::min(maxb, nb_total - b0);
      a.ws = (uint32_t)(r.ws + b0 * r.binsize);
      a.we = (uint32_t)std::min(r.we, r.ws + (b0 + cnt) * r.binsize);
      a.nb = (uint32_t)cnt;
      a.ostride = (uint32_t)nb_total;
      a.out = r.out.at(b0);
      const size_t lds = (size_t)S::SLOTS * S::XSTRIDE * sizeof(cf) + cnt * (sizeof(uint64_t) + sizeof(cf));
      const long long row_blocks = np * nsplit;
      hipLaunchKernelGGL(big_rows_kernel<B>, dim3((unsigned)(row_blocks + fin_blocks)), dim3(256), lds, c->stream, a,
                         fin, fin_np, fin_blocks);
      if (!hip_ok(hipGetLastError(), "big_rows_kernel")) return -1;
      fin_blocks = 0;
      if (nsplit > 1 && !a.done) {
        const long long cells = np * (long long)cnt;
        if (fold) {  // finished by the next rows launch, or after the loop
          fin = a;
          fin_np = np;
          fin_blocks = (int)((cells + 255) / 256);
        } else {
          hipLaunchKernelGGL(big_rows_finish_kernel, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, c->stream,
                             a, np);
          if (!hip_ok(hipGetLastError(), "big_rows_finish_kernel")) return -1;
        }
      }
    }
  }
  if (fin_blocks) {
    hipLaunchKernelGGL(big_rows_finish_kernel, dim3((unsigned)fin_blocks), dim3(256), 0, c->stream, fin, fin_np);
    if (!hip_ok(hipGetLastError(), "big_rows_finish_kernel")) return -1;
  }
  return 0;
}

}  // namespace

const cf *big_roots(Ctx *c, int n1) {
  const int n = n1 * 256;
  char rname[32];
  snprintf(rname, sizeof rname, "bigroots%d", n);
  cf *roots = (cf *)c->scratch(rname, (n1 + 256) * sizeof(cf));
  if (!roots) return nullptr;
  if (!c->big_roots_ready[ilog2(n1)]) {
    hipLaunchKernelGGL(roots_kernel, dim3((n1 + 255) / 256), dim3(256), 0, c->stream, roots, n1, n1);
    hipLaunchKernelGGL(roots_kernel, dim3(1), dim3(256), 0, c->stream, roots + n1, 256, n);
    if (!hip_ok(hipGetLastError(), "roots_kernel")) return nullptr;
    c->big_roots_ready[ilog2(n1)] = true;
  }
  return roots;
}

template <class B>
static int reserve_shape(Ctx *c, long long pairs, size_t nb) {
  BigArgs a;
  BigBuffers b;
  return big_buffers<B>(c, pairs, nb, a, b);
}

int big_reserve(Ctx *c, size_t n, const FlatRun &r) {
  const size_t nb = (r.we - r.ws + r.binsize - 1) / r.binsize;
  switch (n) {
    case 32768: return reserve_shape<BigShape<0, 8>>(c, r.list_cap, nb);
    case 65536: return reserve_shape<BigShape<0, 16>>(c, r.list_cap, nb);
    default: return 0;
  }
}

int launch_big(Ctx *c, size_t n, const FlatRun &r) {
  switch (n) {
    case 32768: return launch_big_shape<BigShape<0, 8>>(c, r);
    case 65536: return launch_big_shape<BigShape<0, 16>>(c, r);
    case 131072: return launch_big_shape<BigShape<512>>(c, r);
    case 262144: return launch_big_shape<BigShape<1024>>(c, r);
    case 524288: return launch_big_shape<BigShape<2048>>(c, r);
    case 1048576: return launch_big_shape<BigShape<4096>>(c, r);
    default: return fail("transform length %zu is not a two-kernel length", n);
  }
}

}  // namespace mfh
