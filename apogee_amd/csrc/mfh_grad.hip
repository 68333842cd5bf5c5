// Gradients of reported peak values with respect to the data and template
// spectra, from the stored peak indices alone (no correlation series).
//
// A reported peak of pair (d, t) at lag k has the value
//     z = sum_f D_d[f] conj(T_t[f]) w^(f k),   w = exp(+2 pi i / n),
// so, with g = dL/dRe z + i dL/dIm z the incoming gradient of a real loss
// (PyTorch's convention for complex tensors),
//     dL/dD_d[f] = sum_{t, bins} g       T_t[f] w^(-f k)
//     dL/dT_t[f] = sum_{d, bins} conj(g) D_d[f] w^(+f k)
// Bins that reported nothing (index -1) hold the constant 0 and contribute
// nothing.  Each output element is an ordered sum (no atomics), so the result
// is deterministic.  w^m, m = (f k) mod n in exact integer
// arithmetic, is the product of two FP64-generated roots, w^(256 (m >> 8)) and
// w^(m & 255), read from a 4 KiB copy of both tables in LDS: the indices are
// scattered across lanes, which the vector cache serves poorly.
//
// The same table gives the peak value itself at a stored lag (a direct sum
// over f per peak, one wave each), which is how a caller recomputes z at the
// argmax without keeping the series.
//
// Reference behaviour: the forward value is the flat filter's
// (src/balanced-inl.h:876-969); the reference has no derivative.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mfh_dft.h"
#include "mfh_internal.h"
#include "mfhip.h"

namespace mfh {

namespace {

// Two-level root table of length n: hi[h] = w^(256 h) for h < max(1, n/256),
// then lo[l] = w^l for l < 256.
__global__ void circle_tables_kernel(cf *out, int n) {
  const int nh = n >= 256 ? n / 256 : 1;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nh + 256) {
    const long long e = i < nh ? 256ll * i : (long long)(i - nh);
    double sn, cs;
    sincospi(2.0 * (double)(e % n) / (double)n, &sn, &cs);
    out[i] = cf{(float)cs, (float)sn};
  }
}

// The block's LDS copy of the two tables; returns (hi, lo) in *lds.
__device__ __forceinline__ void stage_circle(const cf *tables, int n, cf *lds) {
  const int nh = n >= 256 ? n / 256 : 1;
  for (int i = threadIdx.x; i < nh + 256; i += blockDim.x) lds[i] = tables[i];
  __syncthreads();
}

__device__ __forceinline__ cf circle(const cf *lds, int n, uint32_t m) {
  const int nh = n >= 256 ? n / 256 : 1;
  return cmul(lds[m >> 8], lds[nh + (m & 255u)]);
}

// dL/dT (TEMPL = true) or dL/dD, n < 1024: one workgroup per (row, 64 F
// consecutive f); the row is blockIdx.y, the other side's rows are summed over.  The row's
// (lag, gradient) list is staged through LDS in chunks, so the inner loop
// reads LDS instead of waiting on one global load per term.  The eight
// waves take the other side's rows in turn (row j to wave j mod 8), so each
// reads its row's F spectrum values once for all of that row's bins; a
// fixed-order sum of the eight partial sums keeps the result deterministic.
// Each lane covers F consecutive f: w^(f k) for the first comes from the
// tables (one scattered lookup), the rest by F - 1 products with w^k (one
// lookup at a uniform address per term), so scattered LDS reads -- whose
// bank conflicts bound this kernel -- drop F-fold.
template <bool TEMPL, int F>
__global__ void __launch_bounds__(512) peak_grad_kernel(const cf *__restrict__ other, long long other_stride,
                                                        int nother, const int64_t *__restrict__ idx,
                                                        const cf *__restrict__ gval, int nd, int nt, int nb,
                                                        const cf *__restrict__ tables, int n, cf *__restrict__ out,
                                                        long long out_stride) {
  constexpr int CH = 1024;  // (lag, gradient) entries per LDS chunk
  constexpr int W = 8;      // waves
  __shared__ cf roots[512];
  __shared__ uint32_t sk[CH];
  __shared__ cf sg[CH];
  __shared__ cf part[W][64 * F];
  stage_circle(tables, n, roots);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int fb = blockIdx.x * 64 * F;  // n is a multiple of 64 F
  const int f0 = fb + lane * F;
  const int row = blockIdx.y;
  const uint32_t mask = (uint32_t)n - 1u;
  float ax[F], ay[F];
#pragma unroll
  for (int q = 0; q < F; q++) ax[q] = ay[q] = 0.f;
  const long long total = (long long)nother * nb;
  for (long long e0 = 0; e0 < total; e0 += CH) {
    const int cnt = (int)(total - e0 < CH ? total - e0 : CH);
    __syncthreads();  // the previous chunk is consumed
    for (int i = threadIdx.x; i < cnt; i += blockDim.x) {
      const long long e = e0 + i;
      const int j = (int)(e / nb), b = (int)(e % nb);
      const long long pair = TEMPL ? (long long)j * nt + row : (long long)row * nt + j;
      const long long k = idx[pair * nb + b];
      sk[i] = k < 0 ? 0xffffffffu : (uint32_t)k;
      sg[i] = gval[pair * nb + b];
    }
    __syncthreads();
    // this wave's rows of the chunk: j = w (mod W)
    const long long j0 = e0 / nb, j1 = (e0 + cnt - 1) / nb;
    for (long long j = j0 + ((w - j0 % W) + W) % W; j <= j1; j += W) {
      const int ib = (int)(j * nb - e0 > 0 ? j * nb - e0 : 0);
      const int ie = (int)((j + 1) * nb - e0 < cnt ? (j + 1) * nb - e0 : cnt);
      cf x[F];
      const cf *xr = other + j * other_stride + f0;
#pragma unroll
      for (int q = 0; q < F; q++) x[q] = xr[q];
      for (int i = ib; i < ie; i++) {
        const uint32_t k = sk[i];
        if (k == 0xffffffffu) continue;  // uniform: one term for the whole wave
        const cf g = sg[i];
        cf wk = circle(roots, n, ((uint32_t)f0 * k) & mask);
        const cf step = circle(roots, n, k & mask);
#pragma unroll
        for (int q = 0; q < F; q++) {
          if (q > 0) wk = cmul(wk, step);
          // templates: conj(g) x w ; data: g x conj(w)
          cf xw;
          if (TEMPL) {
            xw = cmul(x[q], wk);
            ax[q] += g.x * xw.x + g.y * xw.y;
            ay[q] += g.x * xw.y - g.y * xw.x;
          } else {
            xw = cmul_conj(x[q], wk);
            ax[q] += g.x * xw.x - g.y * xw.y;
            ay[q] += g.x * xw.y + g.y * xw.x;
          }
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < F; q++) part[w][lane * F + q] = cf{ax[q], ay[q]};
  __syncthreads();
  for (int c = threadIdx.x; c < 64 * F; c += blockDim.x) {
    float sx = 0.f, sy = 0.f;
#pragma unroll
    for (int v = 0; v < W; v++) {
      sx += part[v][c].x;
      sy += part[v][c].y;
    }
    out[(long long)row * out_stride + fb + c] = cf{sx, sy};
  }
}

// The same sums on the matrix cores, n >= 1024.  With f = 64 f1 + f2,
//   G_j[f] = sum_b g_b w^(f k_b) = sum_b (g_b w^(64 f1 k_b)) (w^(f2 k_b))
// is a product of a (f1 x bins) and a (bins x f2) complex matrix, one per row j
// of the other side, and the output is sum_j x_j[f] G_j[f].  A root is looked up
// per row and per column of a tile instead of per element, and the elements'
// products run on v_mfma_f32_32x32x2_f32 (FP32 in and out).
//
// Tile: 16 f1 x 32 f2, i.e. 512 f per workgroup.  The 32 rows of a matrix tile
// are the real and imaginary parts of 16 f1 in turn, so that a lane's
// accumulators are (re, im) pairs; the two inner indexes are the column
// factor's parts.  One instruction adds one (row j, bin) term to the tile.
// A lane's operands are real parts: its row's Re or Im of conj(g) w^m is
// Re(conj(g) w^(m + s n/4)) with an s of the lane's own, so that an operand
// costs a product sum and no selection.  Sums run over at most 64 bins before
// x_j multiplies them, and lanes hold those 64 (lag, gradient) entries, so a
// wave walks the reported ones with scalar code.
// Eight waves take the other side's rows in turn, as above, and a split of
// those rows gets a workgroup of its own (grid.z): partial sums are added in
// a fixed order, so the result is deterministic.
//
// Bound: instruction issue.  A term costs a wave 64 clocks of the matrix core
// and 14 VALU instructions (56 clocks), which on this card add up in FP32; a
// row another 50 for x_j.  n = 4096, 64 x 32 rows, eight bins: 14.0 us (data)
// and 16.8 us (templates), against 32.6 and 33.2 us with peak_grad_kernel's
// root recurrence; one or two terms in all: 5.2 us against 5.4.
// The error against FP64 is smaller too (1.7e-7 of the largest element against
// 2.4e-7): no recurrence, and sums of 64 bins at most.
typedef float f32x16 __attribute__((ext_vector_type(16)));

// One term's operands on the way: the entry's gradient, its lane's roots.
struct GradTerm {
  float gx, gy;
  cf wa, hi, lo;
};

template <bool TEMPL>
__global__ void __launch_bounds__(512) peak_grad_mfma_kernel(const cf *__restrict__ other, long long other_stride,
                                                             int nother, int per, const int64_t *__restrict__ idx,
                                                             const cf *__restrict__ gval, int nt, int nb,
                                                             const cf *__restrict__ tables, int n,
                                                             cf *__restrict__ out, long long out_stride) {
  constexpr int CH = 1024;  // (lag, gradient) entries per LDS chunk
  constexpr int W = 8;      // waves
  __shared__ cf roots[512];     // w^(256 h) from element 256 on, w^l before
  __shared__ cf roots64[1024];  // w^(64 h), h < n / 64
  __shared__ uint32_t sk[CH];
  __shared__ cf sg[CH];
  __shared__ cf part[W][512];
  const int nh = n / 256;
  if ((int)threadIdx.x < nh + 256) roots[threadIdx.x] = tables[threadIdx.x < 256 ? nh + threadIdx.x : threadIdx.x - 256];
  __syncthreads();
  for (int h = threadIdx.x; h < n / 64; h += 512) roots64[h] = cmul(roots[256 + (h >> 2)], roots[64 * (h & 3)]);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5;  // half: the inner index of this lane's operands
  const int g1 = blockIdx.x >> 1;
  const uint32_t f2 = 32u * (blockIdx.x & 1) + (uint32_t)col;
  const uint32_t f1 = 16u * (uint32_t)g1 + (uint32_t)(col >> 1);  // of this lane's A row
  const bool imag = (col & 1) != 0;                               // of this lane's A row
  // Quarter turns.  Templates: conj(g) w = ar + i ai; the row Re is (ar, -ai),
  // the row Im (ai, ar) against the column's (re, im); ai = Re(conj(g) w^(m - n/4)).
  // Data: g conj(w), ai = Re(conj(g) w^(m + n/4)), the column's conjugate.
  const uint32_t qa = imag == (half != 0) ? 0u : imag == TEMPL ? 3u : 1u;
  const uint32_t qb = half == 0 ? 0u : TEMPL ? 3u : 1u;
  const uint32_t oa = qa * (uint32_t)(n / 256) * 8u, ob = qb * (uint32_t)(n / 4) * 8u;  // in bytes of a table
  const uint32_t mask_a = (uint32_t)(n / 64 - 1) * 8u, mask_h = (uint32_t)(nh - 1) * 8u;
  const int row = blockIdx.y;
  const int jfirst = blockIdx.z * per, jlast = min(nother, jfirst + per);
  // element p of a lane: f = 64 (16 g1 + m) + f2, m = 4 (p >> 1) + 2 half + (p & 1)
  const int fbase = 64 * (16 * g1 + 2 * half) + (int)f2;
  cf acc[8];
#pragma unroll
  for (int p = 0; p < 8; p++) acc[p] = cf{0.f, 0.f};
  // Chunks of whole rows, or of one row's bins
  const int chunk_bins = min(nb, CH), chunk_rows = CH / chunk_bins;
  for (int j0 = jfirst; j0 < jlast; j0 += chunk_rows) {
    for (int b0 = 0; b0 < nb; b0 += chunk_bins) {
      const int rows = min(chunk_rows, jlast - j0), bins = min(chunk_bins, nb - b0);
      __syncthreads();  // the tables are staged; the previous chunk is consumed
      for (int i = threadIdx.x; i < rows * bins; i += 512) {
        const int r = (uint32_t)i / (uint32_t)bins, j = j0 + r, b = b0 + i - r * bins;
        const long long pair = TEMPL ? (long long)j * nt + row : (long long)row * nt + j;
        const long long k = idx[pair * nb + b];
        sk[i] = k < 0 ? 0xffffffffu : (uint32_t)k & ((uint32_t)n - 1u);
        sg[i] = gval[pair * nb + b];
      }
      __syncthreads();
      // (row, up to 64 bins) by (row, up to 64 bins), waves in turn
      const int segs = (bins + 63) / 64;
      for (int it = w; it < rows * segs; it += W) {
        const int r = segs == 1 ? it : (int)((uint32_t)it / (uint32_t)segs);
        const int i0 = r * bins + 64 * (it - r * segs), ie = (r + 1) * bins;
        uint32_t k8 = 0xffffffffu;
        cf g = cf{0.f, 0.f};
        if (i0 + lane < ie) {
          k8 = sk[i0 + lane];
          g = sg[i0 + lane];
        }
        unsigned long long left = __ballot(k8 != 0xffffffffu);
        if (!left) continue;  // a row with nothing reported adds nothing, whatever it holds
        const int terms = __popcll(left);
        k8 *= 8u;
        const cf *xr = other + (long long)(j0 + r) * other_stride;
        cf x[8];
#pragma unroll
        for (int p = 0; p < 8; p++) x[p] = xr[(uint32_t)(fbase + 64 * (4 * (p >> 1) + (p & 1)))];
        // past the last entry: any lane's, masked into the tables, and not used
        auto fetch = [&]() {
          const int l = __builtin_ctzll(left | 1ull << 63);
          left &= left - 1;
          const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)k8, l);
          GradTerm t;
          t.gx = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(g.x), l));
          t.gy = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(g.y), l));
          const uint32_t ma = __umul24(f1, k) + oa, mb = __umul24(f2, k) + ob;
          t.wa = *(const cf *)((const char *)roots64 + (ma & mask_a));
          t.lo = *(const cf *)((const char *)roots + (mb & 255u * 8u));
          t.hi = *(const cf *)((const char *)(roots + 256) + (mb >> 8 & mask_h));
          return t;
        };
        f32x16 c = {};
        auto add = [&](const GradTerm &t) {
          c = __builtin_amdgcn_mfma_f32_32x32x2f32(t.gx * t.wa.x + t.gy * t.wa.y,
                                                   t.hi.x * t.lo.x - t.hi.y * t.lo.y, c, 0, 0, 0);
        };
        // two by two: the second's roots are read while the first's products run
        for (int i = terms; i > 3; i -= 4) {
          const GradTerm t = fetch(), u = fetch(), v = fetch(), x4 = fetch();
          add(t);
          add(u);
          add(v);
          add(x4);
        }
        if (terms & 2) {
          const GradTerm t = fetch(), u = fetch();
          add(t);
          add(u);
        }
        if (terms & 1) add(fetch());
#pragma unroll
        for (int p = 0; p < 8; p++) {
          acc[p].x = acc[p].x + x[p].x * c[2 * p] - x[p].y * c[2 * p + 1];
          acc[p].y = acc[p].y + x[p].x * c[2 * p + 1] + x[p].y * c[2 * p];
        }
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 8; p++) part[w][32 * (4 * (p >> 1) + 2 * half + (p & 1)) + col] = acc[p];
  __syncthreads();
  {
    const int e = threadIdx.x;  // 32 m + column
    float sx = 0.f, sy = 0.f;
#pragma unroll
    for (int v = 0; v < W; v++) {
      sx += part[v][e].x;
      sy += part[v][e].y;
    }
    const long long f = 64 * (16 * g1 + (e >> 5)) + 32 * (blockIdx.x & 1) + (e & 31);
    out[((long long)blockIdx.z * gridDim.y + row) * out_stride + f] = cf{sx, sy};
  }
}

// The splits' partial sums, [split][elements], in order.
__global__ void __launch_bounds__(256) grad_sum_kernel(const cf *__restrict__ part, long long elems, int splits,
                                                       cf *__restrict__ out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= elems) return;
  float sx = 0.f, sy = 0.f;
  for (int s = 0; s < splits; s++) {
    const cf p = part[s * elems + i];
    sx += p.x;
    sy += p.y;
  }
  out[i] = cf{sx, sy};
}

// z at stored lags: one wave per (pair, bin), FP32 throughout (FP64 on the
// device is kept to table generation and band-fraction sums): each lane sums
// its n/64 terms, then a fixed-order butterfly adds the lanes.
__global__ void __launch_bounds__(256) peak_value_kernel(const cf *__restrict__ D, long long dstride,
                                                         const cf *__restrict__ T, long long tstride, int nt,
                                                         int nb, long long npeaks, const int64_t *__restrict__ idx,
                                                         const cf *__restrict__ tables, int n, cf *__restrict__ out) {
  __shared__ cf roots[512];
  stage_circle(tables, n, roots);
  const long long p = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (p >= npeaks) return;  // uniform per wave, after the only barrier
  const long long k = idx[p];
  const long long pair = p / nb;
  const int d = (int)(pair / nt), t = (int)(pair % nt);
  float sx = 0.f, sy = 0.f;
  if (k >= 0) {
    const uint32_t mask = (uint32_t)n - 1u;
    const cf *dp = D + (long long)d * dstride;
    const cf *tp = T + (long long)t * tstride;
    for (int f = lane; f < n; f += 64) {
      const cf pr = cmul(cmul_conj(dp[f], tp[f]), circle(roots, n, ((uint32_t)f * (uint32_t)k) & mask));
      sx += pr.x;
      sy += pr.y;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sx += __shfl_xor(sx, off, 64);
    sy += __shfl_xor(sy, off, 64);
  }
  if (lane == 0) out[p] = k >= 0 ? cf{sx, sy} : cf{0.f, 0.f};
}

}  // namespace

// Elements of partial sums behind the root tables (n >= 1024): splits x rows x n
// is at most 256 workgroups' tiles of 512 whatever the call, so that one call
// of a context leaves all that any later, captured one needs.
constexpr size_t kGradPart = 256 * 512;

static const cf *unit_circle(Ctx *c) {
  char name[32];
  snprintf(name, sizeof name, "circle%zu", c->n);
  auto it = c->bufs.find(name);
  if (it != c->bufs.end() && it->second.p) return (const cf *)it->second.p;
  const int nh = c->n >= 256 ? (int)(c->n / 256) : 1;
  cf *r = (cf *)c->scratch(name, ((size_t)(nh + 256) + (c->n >= 1024 ? kGradPart : 0)) * sizeof(cf));
  if (!r) return nullptr;
  hipLaunchKernelGGL(circle_tables_kernel, dim3((unsigned)((nh + 256 + 255) / 256)), dim3(256), 0, c->stream, r,
                     (int)c->n);
  if (!hip_ok(hipGetLastError(), "circle_tables_kernel")) return nullptr;
  return r;
}

// Gradient of `rows` output rows (templates if TEMPL, else data rows) against the
// `nother` rows of the other side.  Where fewer than 256 workgroups would run,
// the other side's rows are split over up to 16 per tile, whose partial sums
// a second launch adds.  That launch costs 3 us, and a term alone on its SIMD
// 0.15 us: a split gets eight rows and 64 terms (eight per wave) at least.
// n = 2048, one data row x 64 templates x eight bins: 8.6 us split and
// 14.0 unsplit; 4096, 32 rows (256 workgroups): 15.6 us unsplit and 18.2 split.
template <bool TEMPL>
static int launch_grad_mfma(Ctx *c, const cf *other, long long other_stride, int nother, const int64_t *idx,
                            const cf *gval, int rows, int nt, int nb, const cf *roots, cf *out) {
  const int n = (int)c->n, tiles = n / 512;
  const long long wgs = (long long)tiles * rows;
  int splits = (int)std::min<long long>(16, std::max<long long>(1, 256 / wgs));
  splits = std::max(1, std::min(splits, nother / 8));
  splits = (int)std::max<long long>(1, std::min<long long>(splits, (long long)nother * nb / 64));
  const int per = (nother + splits - 1) / splits;
  splits = (nother + per - 1) / per;
  cf *dst = splits > 1 ? const_cast<cf *>(roots) + n / 256 + 256 : out;  // kGradPart
  hipLaunchKernelGGL(peak_grad_mfma_kernel<TEMPL>, dim3(tiles, rows, splits), dim3(512), 0, c->stream, other,
                     other_stride, nother, per, idx, gval, nt, nb, roots, n, dst, (long long)n);
  if (!hip_ok(hipGetLastError(), "peak_grad_mfma_kernel")) return -1;
  if (splits > 1) {
    const long long elems = (long long)rows * n;
    hipLaunchKernelGGL(grad_sum_kernel, dim3((unsigned)((elems + 255) / 256)), dim3(256), 0, c->stream, dst, elems,
                       splits, out);
    if (!hip_ok(hipGetLastError(), "grad_sum_kernel")) return -1;
  }
  return 0;
}

}  // namespace mfh

using mfh::cf;
using mfh::Ctx;
using mfh::fail;
using mfh::hip_ok;

extern "C" int mfh_peak_grad_async(mfh_ctx *ctx, const void *dev_data_c64, long long data_stride, int nd,
                                   const void *dev_tmpl_c64, long long tmpl_stride, int nt, size_t nb,
                                   const int64_t *dev_idx, const void *dev_gval_c64, void *dev_grad_data_c64,
                                   void *dev_grad_tmpl_c64) {
  if (!ctx) return fail("null context");
  Ctx *c = reinterpret_cast<Ctx *>(ctx);
  if (nd < 1 || nt < 1 || nb < 1) return fail("empty peak array (%d x %d x %zu)", nd, nt, nb);
  if (!dev_data_c64 || !dev_tmpl_c64 || !dev_idx || !dev_gval_c64) return fail("null input pointer");
  if (data_stride < (long long)c->n || tmpl_stride < (long long)c->n) return fail("row stride below n");
  if (nd > 65535 || nt > 65535) return fail("at most 65535 data and template rows per call");
  if (c->n > 65536 || c->n < 64) return fail("peak gradients are built for 64 <= n <= 65536");
  hipSetDevice(c->dev);
  const cf *roots = mfh::unit_circle(c);
  if (!roots) return -1;
  const int n = (int)c->n;
  if (n >= 1024) {
    if (dev_grad_tmpl_c64 &&
        mfh::launch_grad_mfma<true>(c, (const cf *)dev_data_c64, data_stride, nd, dev_idx, (const cf *)dev_gval_c64,
                                    nt, nt, (int)nb, roots, (cf *)dev_grad_tmpl_c64) < 0)
      return -1;
    if (dev_grad_data_c64 &&
        mfh::launch_grad_mfma<false>(c, (const cf *)dev_tmpl_c64, tmpl_stride, nt, dev_idx, (const cf *)dev_gval_c64,
                                     nd, nt, (int)nb, roots, (cf *)dev_grad_data_c64) < 0)
      return -1;
    return 0;
  }
  const dim3 block(512);
  // four frequencies per lane where n allows (n >= 256), else one
  const bool f4 = n >= 256;
  const int fcols = n / (f4 ? 256 : 64);
  auto *ktmpl = f4 ? &mfh::peak_grad_kernel<true, 4> : &mfh::peak_grad_kernel<true, 1>;
  auto *kdata = f4 ? &mfh::peak_grad_kernel<false, 4> : &mfh::peak_grad_kernel<false, 1>;
  if (dev_grad_tmpl_c64) {
    hipLaunchKernelGGL(ktmpl, dim3(fcols, nt), block,
                       0, c->stream, (const cf *)dev_data_c64, data_stride, nd, dev_idx, (const cf *)dev_gval_c64, nd,
                       nt, (int)nb, roots, n, (cf *)dev_grad_tmpl_c64, (long long)n);
    if (!hip_ok(hipGetLastError(), "peak_grad_kernel")) return -1;
  }
  if (dev_grad_data_c64) {
    hipLaunchKernelGGL(kdata, dim3(fcols, nd), block,
                       0, c->stream, (const cf *)dev_tmpl_c64, tmpl_stride, nt, dev_idx, (const cf *)dev_gval_c64, nd,
                       nt, (int)nb, roots, n, (cf *)dev_grad_data_c64, (long long)n);
    if (!hip_ok(hipGetLastError(), "peak_grad_kernel")) return -1;
  }
  return 0;
}

extern "C" int mfh_peak_values_async(mfh_ctx *ctx, const void *dev_data_c64, long long data_stride, int nd,
                                     const void *dev_tmpl_c64, long long tmpl_stride, int nt, size_t nb,
                                     const int64_t *dev_idx, void *dev_out_c64) {
  if (!ctx) return fail("null context");
  Ctx *c = reinterpret_cast<Ctx *>(ctx);
  if (nd < 1 || nt < 1 || nb < 1) return fail("empty peak array (%d x %d x %zu)", nd, nt, nb);
  if (!dev_data_c64 || !dev_tmpl_c64 || !dev_idx || !dev_out_c64) return fail("null pointer");
  if (data_stride < (long long)c->n || tmpl_stride < (long long)c->n) return fail("row stride below n");
  if (c->n > 65536) return fail("peak values are built for n <= 65536");
  hipSetDevice(c->dev);
  const cf *roots = mfh::unit_circle(c);
  if (!roots) return -1;
  const long long npeaks = (long long)nd * nt * (long long)nb;
  hipLaunchKernelGGL(mfh::peak_value_kernel, dim3((unsigned)((npeaks + 3) / 4)), dim3(256), 0, c->stream,
                     (const cf *)dev_data_c64, data_stride, (const cf *)dev_tmpl_c64, tmpl_stride, nt, (int)nb, npeaks,
                     dev_idx, roots, (int)c->n, (cf *)dev_out_c64);
  return hip_ok(hipGetLastError(), "peak_value_kernel") ? 0 : -1;
}
