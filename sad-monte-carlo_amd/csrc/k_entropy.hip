// Mean entropy S(E) of a walker set, reduced on the device.
//
// Per walker (plotting/parse-binning.py:150-171): inside [too_lo, too_hi]
// S = ln w; below too_lo S = ln w(i_lo) + (E - too_lo)/min_T + ln(H/<H>),
// above too_hi S = ln w(i_hi) + ln(H/<H>), <H> the mean histogram over
// [i_lo, i_hi] and i_lo, i_hi the bins whose centres are nearest too_lo and
// too_hi.  Bins outside the range with H = 0 carry no estimate and are
// skipped (the reference's script sets them to 0 for its one walker).  Each
// walker's free constant is removed by subtracting its mean S over a common
// energy window [ga, gb) of global bins (a walker without an estimate in
// every window bin is left out), then S is averaged over the walkers
// covering each bin.
//
// k_entropy_walker: one wavefront per walker computes i_lo, i_hi, <H> and the
// window mean.  k_entropy_bins: two global bins per lane, looping over the
// walkers; consecutive lanes read consecutive bins of the same walker, so
// every load of the 16-byte hot records is coalesced.
// Both are bound by HBM: 16384 LJ31 walkers of 7900 bins are 2.07 GB a pass,
// 377 us for the first (5.5 TB/s; it read the window a second time before)
// and about 430 us for the second.
#include "sadmc_kernels.h"

namespace sadmc {

struct EntropyWalker {
  double too_lo, too_hi, min_T, lnw_lo, lnw_hi, mean_hist, c, bmin;
  int64_t off, base, len;
  int32_t ok, pad;
};

__global__ __launch_bounds__(64) void k_entropy_walker(const sadmc_walker_state *ws, const HotBin *hot, int64_t cap,
                                                       double width, double gmin, int64_t ga, int64_t gb,
                                                       EntropyWalker *out) {
  const int w = blockIdx.x;
  const sadmc_walker_state &s = ws[w];
  const int64_t len = s.len, base = s.base;
  const double bmin = s.bins_min;
  const HotBin *H = hot + (int64_t)w * cap + base;
  const int64_t off = (int64_t)llround((bmin - gmin) / width);
  if (len <= 0 || s.status != 0 || s.method != SADMC_SAD) {
    if (threadIdx.x == 0) {
      EntropyWalker e = {};
      e.ok = 0;
      out[w] = e;
    }
    return;
  }
  // bin nearest a given energy: first index of the smallest |E_i - e|
  auto nearest = [&](double e) {
    int64_t i = (int64_t)floor((e - bmin) / width);
    i = i < 0 ? 0 : (i > len - 1 ? len - 1 : i);
    int64_t best = i;
    double bd = fabs(bmin + ((double)i + 0.5) * width - e);
    for (int64_t j = i - 1; j <= i + 1; j++) {
      if (j < 0 || j >= len) continue;
      double d = fabs(bmin + ((double)j + 0.5) * width - e);
      if (d < bd || (d == bd && j < best)) {
        bd = d;
        best = j;
      }
    }
    return best;
  };
  const int64_t ilo = nearest(s.too_lo), ihi = nearest(s.too_hi);
  // Where the window lies inside the walker's range (the default one does),
  // its values are plain ln w and one sweep serves both sums: lane l takes the
  // bins g = ga + l (mod 64), as the window's sum below does, and the counts
  // add up exactly in any order.  Otherwise the window's sweep follows once <H>
  // is known.  Eight loads in flight per lane.
  const int64_t a0 = ga - off, b0 = gb - off;
  const bool inside = a0 >= 0 && b0 <= len && bmin + ((double)a0 + 0.5) * width >= s.too_lo &&
                      bmin + ((double)(b0 - 1) + 0.5) * width <= s.too_hi;
  double hsum = 0.0, csum = 0.0;
  int64_t ccount = 0;
  const int64_t ifrom = inside && a0 < ilo ? a0 : ilo, ito = inside && b0 - 1 > ihi ? b0 - 1 : ihi;
  for (int64_t i0 = ifrom + ((a0 + (int64_t)threadIdx.x - ifrom) & 63); i0 <= ito; i0 += 512) {
    HotBin h[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      h[u].lnw = 0.0;
      h[u].hist = 0;
      if (i0 + 64 * u <= ito) h[u] = H[i0 + 64 * u];
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int64_t i = i0 + 64 * u;
      if (i >= ilo && i <= ihi) hsum += (double)h[u].hist;
      if (inside && i >= a0 && i < b0) {
        csum += h[u].lnw;
        ccount += 1;
      }
    }
  }
  for (int d = 32; d >= 1; d >>= 1) hsum += __shfl_xor(hsum, d, 64);
  const double mean_hist = hsum / (double)(ihi - ilo + 1);
  const double lnw_lo = H[ilo].lnw, lnw_hi = H[ihi].lnw;
  // the window mean of the extended S; every window bin must carry an estimate
  for (int64_t g = ga + threadIdx.x; g < gb && !inside; g += 64) {
    const int64_t i = g - off;
    if (i < 0 || i >= len) continue;
    const HotBin b = H[i];
    const double E = bmin + ((double)i + 0.5) * width;
    if (E < s.too_lo) {
      if (b.hist == 0) continue;
      csum += lnw_lo + (E - s.too_lo) / s.min_T + log((double)b.hist / mean_hist);
    } else if (E > s.too_hi) {
      if (b.hist == 0) continue;
      csum += lnw_hi + log((double)b.hist / mean_hist);
    } else {
      csum += b.lnw;
    }
    ccount += 1;
  }
  for (int d = 32; d >= 1; d >>= 1) {
    csum += __shfl_xor(csum, d, 64);
    ccount += __shfl_xor(ccount, d, 64);
  }
  if (threadIdx.x == 0) {
    EntropyWalker e;
    e.too_lo = s.too_lo;
    e.too_hi = s.too_hi;
    e.min_T = s.min_T;
    e.lnw_lo = lnw_lo;
    e.lnw_hi = lnw_hi;
    e.mean_hist = mean_hist;
    e.c = ccount > 0 ? csum / (double)ccount : 0.0;
    e.bmin = bmin;
    e.off = off;
    e.base = base;
    e.len = len;
    e.ok = (s.status == 0 && s.method == SADMC_SAD && ccount == gb - ga && len > 0) ? 1 : 0;
    e.pad = 0;
    out[w] = e;
  }
}

// Each lane takes kBinsPerLane grid bins, 256 apart, and each block row a
// chunk of walkers: partial sums over the chunk's walkers in their order.  The
// shape is measured (16384 LJ31 walkers, whole call): bins per lane x walkers
// in flight 1 x 4 1098 us, 1 x 8 1085, 2 x 4 912, 2 x 8 1090, 3 x 4 969, 4 x 2
// 1003, 4 x 4 982.
constexpr int kBinsPerLane = 2, kWalkersInFlight = 4;
__global__ __launch_bounds__(256) void k_entropy_bins(const EntropyWalker *ew, int W, const HotBin *hot, int64_t cap,
                                                      double width, int64_t ng, int chunks, double *psum,
                                                      int64_t *pcnt) {
  const int64_t g0 = (int64_t)blockIdx.x * (256 * kBinsPerLane) + threadIdx.x;
  const int c = blockIdx.y;
  const int w0 = (int)((int64_t)W * c / chunks), w1 = (int)((int64_t)W * (c + 1) / chunks);
  double sum[kBinsPerLane];
  int32_t n[kBinsPerLane];
#pragma unroll
  for (int b = 0; b < kBinsPerLane; b++) {
    sum[b] = 0.0;
    n[b] = 0;
  }
  for (int wq = w0; wq < w1; wq += kWalkersInFlight) {
    // the records of a few walkers in flight, used in walker order
    HotBin bq[kWalkersInFlight][kBinsPerLane];
#pragma unroll
    for (int u = 0; u < kWalkersInFlight; u++) {
      const int w = wq + u < w1 ? wq + u : w1 - 1;
      const int64_t off = ew[w].off, len = ew[w].ok ? ew[w].len : 0;
      const HotBin *H = hot + (int64_t)w * cap + ew[w].base;
#pragma unroll
      for (int b = 0; b < kBinsPerLane; b++) {
        const int64_t i = g0 + 256 * b - off;
        bq[u][b].lnw = 0.0;
        bq[u][b].hist = 0;
        if (i >= 0 && i < len) bq[u][b] = H[i];
      }
    }
#pragma unroll
    for (int u = 0; u < kWalkersInFlight; u++) {
      const int w = wq + u;
      if (w >= w1) continue;
      const EntropyWalker e = ew[w];
      const int64_t len = e.ok ? e.len : 0;
#pragma unroll
      for (int b = 0; b < kBinsPerLane; b++) {
        const int64_t i = g0 + 256 * b - e.off;
        const double E = e.bmin + ((double)i + 0.5) * width;
        double v = bq[u][b].lnw;
        bool have = i >= 0 && i < len;
        if (have && (E < e.too_lo || E > e.too_hi)) {
          have = bq[u][b].hist != 0;
          if (have) {
            const double l = log((double)bq[u][b].hist / e.mean_hist);
            v = E < e.too_lo ? e.lnw_lo + (E - e.too_lo) / e.min_T + l : e.lnw_hi + l;
          }
        }
        if (have) {
          sum[b] += v - e.c;
          n[b] += 1;
        }
      }
    }
  }
#pragma unroll
  for (int b = 0; b < kBinsPerLane; b++) {
    const int64_t g = g0 + 256 * b;
    if (g < ng) {
      psum[(int64_t)c * ng + g] = sum[b];
      pcnt[(int64_t)c * ng + g] = n[b];
    }
  }
}

// The chunks' partial sums, combined in chunk order.
__global__ __launch_bounds__(256) void k_entropy_combine(int64_t ng, int chunks, const double *psum,
                                                         const int64_t *pcnt, double *S, int64_t *count) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (g >= ng) return;
  double sum = 0.0;
  int64_t n = 0;
  for (int c = 0; c < chunks; c++) {
    sum += psum[(int64_t)c * ng + g];
    n += pcnt[(int64_t)c * ng + g];
  }
  S[g] = n ? sum / (double)n : 0.0;
  count[g] = n;
}

// The set's common grid from the walker states, on the device: gmin = the
// smallest bins_min, lo / hi = the largest too_lo / smallest too_hi over the
// walkers still running with bins, then ng = the largest
// round((bins_min - gmin) / width) + len.  kEntropyRangeBlocks blocks reduce
// slices of the walkers into partial records, one block combines them
// (twice: ng needs gmin).  Minima and maxima do not depend on the order.
template <typename T, typename F>
__device__ __forceinline__ T block_reduce(T v, T *sh, F op) {
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int d = blockDim.x / 2; d > 0; d >>= 1) {
    if (t < d) sh[t] = op(sh[t], sh[t + d]);
    __syncthreads();
  }
  const T r = sh[0];
  __syncthreads();
  return r;
}
struct DMin {
  __device__ double operator()(double a, double b) const { return b < a ? b : a; }
};
struct DMax {
  __device__ double operator()(double a, double b) const { return b > a ? b : a; }
};
struct IMax {
  __device__ int64_t operator()(int64_t a, int64_t b) const { return b > a ? b : a; }
};

__global__ __launch_bounds__(256) void k_entropy_range_part(const sadmc_walker_state *ws, int W, EntropyRange *part) {
  __shared__ double sd[256];
  __shared__ int64_t si[256];
  double g = __builtin_inf(), lo = -__builtin_inf(), hi = __builtin_inf();
  int64_t any = 0;
  for (int w = blockIdx.x * 256 + threadIdx.x; w < W; w += gridDim.x * 256) {
    const sadmc_walker_state &x = ws[w];
    if (x.status || x.len <= 0) continue;
    g = x.bins_min < g ? x.bins_min : g;
    lo = x.too_lo > lo ? x.too_lo : lo;
    hi = x.too_hi < hi ? x.too_hi : hi;
    any = 1;
  }
  g = block_reduce(g, sd, DMin());
  lo = block_reduce(lo, sd, DMax());
  hi = block_reduce(hi, sd, DMin());
  any = block_reduce(any, si, IMax());
  if (threadIdx.x == 0) {
    EntropyRange r;
    r.gmin = g;
    r.lo = lo;
    r.hi = hi;
    r.ng = 0;
    r.any = (int32_t)any;
    r.pad = 0;
    part[blockIdx.x] = r;
  }
}

__global__ __launch_bounds__(256) void k_entropy_range_ng(const sadmc_walker_state *ws, int W, double width,
                                                          const EntropyRange *out, EntropyRange *part) {
  __shared__ int64_t si[256];
  const double gmin = out->gmin;
  int64_t ng = 0;
  for (int w = blockIdx.x * 256 + threadIdx.x; w < W; w += gridDim.x * 256) {
    const sadmc_walker_state &x = ws[w];
    if (x.status || x.len <= 0) continue;
    const int64_t e = (int64_t)llround((x.bins_min - gmin) / width) + x.len;
    ng = e > ng ? e : ng;
  }
  ng = block_reduce(ng, si, IMax());
  if (threadIdx.x == 0) part[blockIdx.x].ng = ng;
}

// One block of kEntropyRangeBlocks lanes combines the partial records; with
// `ng_only` only their ng.
__global__ __launch_bounds__(kEntropyRangeBlocks) void k_entropy_range_join(const EntropyRange *part,
                                                                            EntropyRange *out, int ng_only) {
  __shared__ double sd[kEntropyRangeBlocks];
  __shared__ int64_t si[kEntropyRangeBlocks];
  const EntropyRange p = part[threadIdx.x];
  if (ng_only) {
    const int64_t ng = block_reduce(p.ng, si, IMax());
    if (threadIdx.x == 0) out->ng = ng;
    return;
  }
  const double g = block_reduce(p.gmin, sd, DMin());
  const double lo = block_reduce(p.lo, sd, DMax());
  const double hi = block_reduce(p.hi, sd, DMin());
  const int64_t any = block_reduce((int64_t)p.any, si, IMax());
  if (threadIdx.x == 0) {
    EntropyRange r;
    r.gmin = g;
    r.lo = lo;
    r.hi = hi;
    r.ng = 0;
    r.any = (int32_t)any;
    r.pad = 0;
    *out = r;
  }
}

hipError_t launch_entropy_range(const sadmc_walker_state *ws, int W, double width, EntropyRange *out,
                                EntropyRange *part, hipStream_t s) {
  const dim3 nb(kEntropyRangeBlocks), nt(256);
  hipLaunchKernelGGL(k_entropy_range_part, nb, nt, 0, s, ws, W, part);
  hipLaunchKernelGGL(k_entropy_range_join, dim3(1), nb, 0, s, (const EntropyRange *)part, out, 0);
  hipLaunchKernelGGL(k_entropy_range_ng, nb, nt, 0, s, ws, W, width, (const EntropyRange *)out, part);
  hipLaunchKernelGGL(k_entropy_range_join, dim3(1), nb, 0, s, (const EntropyRange *)part, out, 1);
  return hipGetLastError();
}

// Chunks of walkers: 2048 pieces of 256 bins of a chunk, which k_entropy_bins
// takes 256 * kBinsPerLane at a time (two: 1024 blocks, 4 per CU).  The count
// is part of the result: the sums are added chunk by chunk.
int entropy_chunks(int W, int64_t ng) {
  const int64_t blocks = (ng + 255) / 256;
  int64_t c = (2048 + blocks - 1) / blocks;
  if (c > 64) c = 64;
  if (c > W) c = W;
  return c < 1 ? 1 : (int)c;
}

hipError_t launch_entropy(const sadmc_walker_state *ws, const HotBin *hot, int W, int64_t cap, double width,
                          double gmin, int64_t ga, int64_t gb, int64_t ng, void *ew, int chunks, double *psum,
                          int64_t *pcnt, double *S, int64_t *count, hipStream_t s) {
  hipLaunchKernelGGL(k_entropy_walker, dim3(W), dim3(64), 0, s, ws, hot, cap, width, gmin, ga, gb,
                     (EntropyWalker *)ew);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const unsigned bx = (unsigned)((ng + 255) / 256);
  const unsigned bins_x = (unsigned)((ng + 256 * kBinsPerLane - 1) / (256 * kBinsPerLane));
  hipLaunchKernelGGL(k_entropy_bins, dim3(bins_x, (unsigned)chunks), dim3(256), 0, s, (const EntropyWalker *)ew, W, hot,
                     cap, width, ng, chunks, psum, pcnt);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_entropy_combine, dim3(bx), dim3(256), 0, s, ng, chunks, (const double *)psum,
                     (const int64_t *)pcnt, S, count);
  return hipGetLastError();
}

size_t entropy_walker_bytes() { return sizeof(EntropyWalker); }

}  // namespace sadmc
