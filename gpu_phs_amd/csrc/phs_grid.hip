// Randoms on the device, drawn from each channel's adaptive grid, and the grid's update from
// the accepted events (the reference's rng.cpp:18-93 on the host: std::default_random_engine
// through a std::piecewise_constant_distribution per (channel, dimension), 10 equal bins whose
// weights are the accepted events' histogram).
//
// The uniform numbers come from Philox4x32-10 (J. K. Salmon, M. A. Moraes, R. O. Dror,
// D. E. Shaw, "Parallel random numbers: as easy as 1, 2, 3", SC 2011), a counter-based
// generator: the numbers of event e of segment s are a function of (seed, s, e, block), so
// every lane draws its own without state and a launch is reproducible whatever its shape.
// Two 32-bit outputs give one double u = (a 2^32 + b) >> 11 times 2^-53 in [0, 1).  u is
// mapped through the inverse distribution function of the piecewise-constant density of the
// bins: x = b_k + (u - F_k) / rho_k for the first bin k whose F_{k+1} > u.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "phs_device.h"
#include "phs_kernels.h"

namespace gphs {

namespace {

__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
  constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
  for (int r = 0; r < 10; r++) {
    // one 32 x 32 -> 64-bit product gives both halves
    const uint64_t p0 = (uint64_t)M0 * c[0], p1 = (uint64_t)M1 * c[2];
    const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
    const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    const uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
    c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
    k0 += W0; k1 += W1;
  }
}

// ((a 2^32 + b) >> 11) 2^-53: both terms and their sum are exact.
__device__ __forceinline__ double u53(uint32_t a, uint32_t b) {
  return __builtin_fma((double)a, 0x1.0p-32, (double)(b >> 11) * 0x1.0p-53);
}

// What a bin contributes: x = edge + (u - F) / rho, with the quotient's reciprocal at hand.  40
// bytes: lanes that read different bins of one dimension meet different LDS banks.
struct BinRec {
  double F, next, rho, inv, edge;   // F_b, F_{b+1}, density (F_{b+1} - F_b) / width, 1 / rho, b / kGridBins
};

// (u - F) / rho, correctly rounded as the division is: the product with the rounded reciprocal,
// then one step with the exact remainder (P. Markstein, IBM J. Res. Dev. 34 (1990) 111).  A bin
// that holds some u > 0 has rho > 2^-107; for the others (inv = 0) only u = F = 0 occurs.
__device__ __forceinline__ double in_bin(const BinRec& r, double u) {
  const double n = u - r.F;
  const double q = n * r.inv;
  return __builtin_fma(__builtin_fma(-r.rho, q, n), r.inv, q);
}

// cdf: [channel][dim][kGridBins + 1] cumulative bin probabilities of the plan's channels.
//
// Bound by integer and FP64 issue (10 rounds of two 32 x 32-bit products per two randoms), not by
// its writes, so the work per random is kept down: the top bits of u give the first bin it can lie
// in, and the bounds are compared from there (the bin is the number of interior bounds at or below
// u, and the bounds rise); the division by the bin's density is a product with its reciprocal,
// corrected; and the rows leave without a division per word.  A workgroup takes a contiguous range
// of the tile table (as the histogram below), builds the tables of a channel once per run of tiles
// in LDS, and its waves then take 64 events each: every lane puts its event's randoms into its column of the
// wave's table x[k][lane], and the wave stores the 64 rows as one contiguous run (16-byte words
// where the row length is even and the rows are 16-byte aligned).  4e6 events of 8 randoms: 68 us
// (56 VALU instructions per random, the vector units 73% busy; 79 us with both tables at strides
// whose lanes met the same banks), against 103 us with nine bounds read per random, two
// divisions and a division per word stored.  A run of at most kGenCellEvents events does not repay the first-bin
// table and compares with the nine bounds (20,000 events of 32 randoms in 12 channels 36 and 46 us, but 2e6
// of 8 60 and 58 us at twice as many events).
constexpr int kGenWaves = 4;   // at most (launch_grid_generate)
constexpr int kGenGroups = 4096;
constexpr int kGenRow = 68;   // the lanes that read one another's columns meet different LDS banks
constexpr int kGenCellBits = 6, kGenCells = 1 << kGenCellBits, kGenCellEvents = 256;

// per_group, extra: workgroup b takes per_group tiles, and one more for b < extra.
__global__ __launch_bounds__(64 * kGenWaves) void grid_generate_kernel(const TileDesc* __restrict__ tiles, int per_group,
                                                                    int extra,
                                                                    const SegDesc* __restrict__ segs,
                                                                    const ChannelDesc* __restrict__ chans,
                                                                    const double* __restrict__ cdf, int n_dim,
                                                                    uint64_t seed) {
  // n_dim * kGridBins records, per wave n_dim rows of kGenRow doubles, n_dim * kGenCells first bins
  extern __shared__ BinRec rec[];
  constexpr int NB1 = kGridBins + 1;
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  double* xs0 = (double*)(rec + n_dim * kGridBins);
  double* xs = xs0 + wave * n_dim * kGenRow;
  const int threads = (int)blockDim.x;
  uint8_t* first = (uint8_t*)(xs0 + (threads >> 6) * n_dim * kGenRow);
  const int b0 = (int)blockIdx.x;
  int t = b0 * per_group + (b0 < extra ? b0 : extra);
  const int t1 = t + per_group + (b0 < extra ? 1 : 0);
  while (t < t1) {
    const TileDesc td = tiles[t];
    const SegDesc sd = segs[td.seg];
    const int n_x = chans[sd.channel].n_x;
    const uint32_t div_nx = chans[sd.channel].div_nx;
    const double* F0 = cdf + (size_t)sd.channel * n_dim * NB1;
    // the run: this tile and the following ones of its segment, up to the range's end (a 64-bit division
    // only where the segment ends within it)
    int run = t1 - t;
    if (sd.n_events - td.e0 < (int64_t)run * td.count) run = (int)((sd.n_events - td.e0 + td.count - 1) / td.count);
    const int64_t e_run = td.e0 + (int64_t)run * td.count;
    const int64_t e_end = e_run < sd.n_events ? e_run : sd.n_events;
    t += run;
    __syncthreads();   // the previous run's records have been read
    for (int i = (int)threadIdx.x; i < n_x * kGridBins; i += threads) {
      const int k = i / kGridBins, b = i - k * kGridBins;
      const double f0 = F0[k * NB1 + b], f1 = F0[k * NB1 + b + 1];
      const double rho = (f1 - f0) * kGridBins;
      // (no u is above the last bin's bound)
      rec[i] = BinRec{f0, b < kGridBins - 1 ? f1 : 2.0, rho, rho > 0x1.0p-1000 ? 1.0 / rho : 0.0, (double)b / kGridBins};
    }
    // the first-bin table pays for itself from some hundred events on
    const bool cells = e_end - td.e0 > kGenCellEvents;
    for (int i = (int)threadIdx.x; cells && i < n_x * kGenCells; i += threads) {
      const double* F = F0 + i / kGenCells * NB1;
      const double u = (double)(i % kGenCells) / kGenCells;
      int b = 0;
      for (int q = 1; q < kGridBins; q++) b += F[q] <= u ? 1 : 0;
      first[i] = (uint8_t)b;
    }
    __syncthreads();
    const bool vec = (sd.align16 & 1) && (n_x % 2 == 0);
    // word w of a wave's rows holds doubles w * step ..: event (w * step) / n_x, random the rest;
    // 64 words on, both advance by constants
    const int step = vec ? 2 : 1;
    const int ev0 = (int)__umulhi((uint32_t)(lane * step), div_nx), k0 = lane * step - ev0 * n_x;
    const int dev = (int)__umulhi((uint32_t)(64 * step), div_nx), dk = 64 * step - dev * n_x;
    // (tiles start at multiples of 64 events, so an event's low index word is the unit's with the lane)
    for (int64_t e = td.e0 + 64 * wave; e < e_end; e += threads) {
      const int cnt = e_end - e < 64 ? (int)(e_end - e) : 64;
      const uint32_t e_lo = (uint32_t)e + (uint32_t)lane, e_hi = (uint32_t)((uint64_t)e >> 32);
      auto draw = [&](auto by_cells) {
        for (int j = 0; 2 * j < n_x; j++) {
          uint32_t c[4] = {e_lo, e_hi, (uint32_t)td.seg, (uint32_t)j};
          philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const int k = 2 * j + h;
            if (k >= n_x) break;
            const double u = u53(c[2 * h], c[2 * h + 1]);
            const BinRec* at = rec + k * kGridBins;
            BinRec r;
            if constexpr (decltype(by_cells)::value) {
              at += first[k * kGenCells + (int)(c[2 * h] >> (32 - kGenCellBits))];
              r = *at;
              while (r.next <= u) r = *++at;
            } else {
              int b = 0;
#pragma unroll
              for (int q = 1; q < kGridBins; q++) b += at[q].F <= u ? 1 : 0;
              r = at[b];
            }
            xs[k * kGenRow + lane] = r.edge + in_bin(r, u);
          }
        }
      };
      if (cells) draw(std::true_type{});
      else draw(std::false_type{});
      // the wave's lanes read one another's columns: no other wave is concerned
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // rows [e, e + cnt) of x are cnt * n_x consecutive doubles
      const int n = cnt * n_x;
      double* dst = const_cast<double*>(sd.x) + e * (int64_t)n_x;
      int ev = ev0, k = k0;
      if (vec) {
        gdouble2* d2 = (gdouble2*)dst;
        for (int w = lane; 2 * w < n; w += 64) {
          dvec2 v;   // k is even, so k + 1 < n_x
          v.x = xs[k * kGenRow + ev];
          v.y = xs[(k + 1) * kGenRow + ev];
          d2[w] = v;
          ev += dev;
          k += dk;
          if (k >= n_x) { k -= n_x; ev++; }
        }
      } else {
        gdouble* d1 = as_global(dst);
        for (int w = lane; w < n; w += 64) {
          d1[w] = xs[k * kGenRow + ev];
          ev += dev;
          k += dk;
          if (k >= n_x) { k -= n_x; ev++; }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();   // the table is read before the next events overwrite it
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
}

// Histogram of the accepted events' randoms per (channel, dim, bin) and the accepted count per
// channel.  Bound by reading the randoms once (8 n_x + 1 bytes per event).  A workgroup takes a
// contiguous range of the tile table, which it reads as runs of consecutive events of one segment
// (a segment's tiles follow one another in the table, in event order, all but the last of one
// size), and each thread keeps one dimension for a whole run: element t of a pass over
// kHistThreads / n_x events is event t / n_x, dimension t % n_x, so the loads are contiguous and
// a thread counts its bins in ten 6-bit fields of one register pair, without atomics.  The
// fields go to the workgroup's LDS histogram before they can overflow, and that to the global
// counts once per workgroup and channel: device atomics on the few hundred shared counters
// serialise (1.27 million of them, one set per 256-event tile, made the kernel 251 us for 4e6
// events of 8 randoms in 3 channels).  Four workgroups per CU fill it with loads in flight: eight
// randoms and flags per thread, which the whole batches load without a test (guarded, each load waits in a
// branch of its own: 63 us for the same events after a forward pass, 66 with the one element per thread tested
// for in the loop, 46 as it is, 5.6 TB/s of the randoms).  The flags come a batch ahead, and the randoms of
// rejected events are not read: deep trees reject most of theirs (2e6 events of 2 -> 8 trees 29 us, 54 with all
// rows read).  The workgroups were chosen on the first version: 49 us at 1024, 55 at 512, 87 at 256, 62 at
// 2048, where the atomics show again; fewer for few events (launch_grid_histogram).
constexpr int kHistThreads = 512;
constexpr int kHistGroups = 1024;
constexpr int kHistUnroll = 8;                                     // loads in flight per thread
constexpr int kHistField = 6;                                      // bits of a bin's private count
constexpr int kHistPasses = ((1 << kHistField) - 1) / kHistUnroll; // batches before a field is full
static_assert(kHistField * kGridBins <= 64, "a thread's counts fill one register pair");

// per_group, extra: workgroup b takes per_group tiles, and one more for b < extra.
__global__ __launch_bounds__(kHistThreads) void grid_histogram_kernel(const TileDesc* __restrict__ tiles,
                                                                      int per_group, int extra,
                                                                      const SegDesc* __restrict__ segs,
                                                                      const ChannelDesc* __restrict__ chans, int n_dim,
                                                                      unsigned long long* __restrict__ counts,
                                                                      unsigned long long* __restrict__ n_ok) {
  extern __shared__ unsigned int hist[];   // n_dim * kGridBins bins, then the accepted count
  const int nb = n_dim * kGridBins;
  const int tid = (int)threadIdx.x;
  const int b0 = (int)blockIdx.x;
  int t = b0 * per_group + (b0 < extra ? b0 : extra);
  const int t1 = t + per_group + (b0 < extra ? 1 : 0);
  for (int i = tid; i <= nb; i += kHistThreads) hist[i] = 0;
  __syncthreads();
  while (t < t1) {
    const TileDesc td = tiles[t];
    const SegDesc sd = segs[td.seg];
    const int n_x = chans[sd.channel].n_x;
    const uint32_t div_nx = chans[sd.channel].div_nx;
    // the run: this tile and the following ones of its segment, up to the range's end (the 64-bit division
    // only where the segment ends within it)
    int run = t1 - t;
    if (sd.n_events - td.e0 < (int64_t)run * td.count) run = (int)((sd.n_events - td.e0 + td.count - 1) / td.count);
    const int64_t e_run = td.e0 + (int64_t)run * td.count;
    const int64_t e_end = e_run < sd.n_events ? e_run : sd.n_events;
    const int per = (int)__umulhi((uint32_t)kHistThreads, div_nx);   // events per pass
    const int r = (int)__umulhi((uint32_t)tid, div_nx), k = tid - r * n_x;
    if (r < per) {
      const gdouble* xk = as_global(sd.x) + k;
      const guint8* ok = as_global(sd.ok);
      unsigned long long fields = 0;
      unsigned int accepted = 0;
      auto flush = [&]() {
#pragma unroll
        for (int b = 0; b < kGridBins; b++) {
          const unsigned int v = (unsigned int)(fields >> (kHistField * b)) & ((1u << kHistField) - 1);
          if (v) atomicAdd(&hist[k * kGridBins + b], v);
        }
        fields = 0;
      };
      // element u of a batch from its first one: its bin and whether it counts
      auto count = [&](double xe, bool accept) {
        int b = (int)(xe * kGridBins);   // rng.cpp:52
        b = b < 0 ? 0 : b > kGridBins - 1 ? kGridBins - 1 : b;
        const unsigned int one = accept ? 1u : 0u;
        fields += (unsigned long long)one << (kHistField * b);
        accepted += one;
      };
      int passes = 0;
      const int step = per * n_x;   // from one element of the thread to the next
      int64_t e = td.e0;            // first event of the pass
      const gdouble* px = xk + (e + r) * n_x;
      const guint8* po = ok + (e + r);
      const gdouble* x0 = as_global(sd.x);   // read in the place of the randoms of rejected events
      unsigned int in[kHistUnroll];
      auto load_flags = [&]() {
#pragma unroll
        for (int u = 0; u < kHistUnroll; u++) in[u] = po[u * per];
        po += kHistUnroll * per;
      };
      // whole batches: every load is inside, without a test; the flags of the next one with the randoms of this
      const int batch = per * kHistUnroll;
      if (e + batch <= e_end) load_flags();
      for (; e + batch <= e_end; e += batch) {
        bool accept[kHistUnroll], any = false;
#pragma unroll
        for (int u = 0; u < kHistUnroll; u++) {
          accept[u] = in[u] != 0;
          any = any || accept[u];
        }
        if (e + 2 * batch <= e_end) load_flags();
        if (__any(any)) {
          double xv[kHistUnroll];
#pragma unroll
          for (int u = 0; u < kHistUnroll; u++) xv[u] = *(accept[u] ? px + u * step : x0);
#pragma unroll
          for (int u = 0; u < kHistUnroll; u++) count(xv[u], accept[u]);
        }
        px += kHistUnroll * step;
        if (++passes == kHistPasses) { flush(); passes = 0; }
      }
      const int left = (int)(e_end - e);   // events after them
      if (left > per) {
        // elements past the end read the thread's first flag, which is inside, and do not count
        double xv[kHistUnroll];
#pragma unroll
        for (int u = 0; u < kHistUnroll; u++) {
          const bool inside = u * per + r < left;
          in[u] = po[inside ? u * per : 0];
          if (!inside) in[u] = 0;
        }
#pragma unroll
        for (int u = 0; u < kHistUnroll; u++) xv[u] = *(in[u] ? px + u * step : x0);
#pragma unroll
        for (int u = 0; u < kHistUnroll; u++) count(xv[u], in[u]);
      } else if (r < left) {   // one element per thread: counted at once
        const double xe = *px;
        if (*po) {
          const int b = (int)(xe * kGridBins);
          atomicAdd(&hist[k * kGridBins + (b < 0 ? 0 : b > kGridBins - 1 ? kGridBins - 1 : b)], 1u);
          accepted++;
        }
      }
      if (fields) flush();
      if (k == 0 && accepted) atomicAdd(&hist[nb], accepted);
    }
    t += run;
    // the range goes on in another channel, or ends: hand the counts over
    if (t < t1 && segs[tiles[t].seg].channel == sd.channel) continue;
    __syncthreads();
    for (int i = tid; i <= nb; i += kHistThreads) {
      const unsigned int v = hist[i];
      hist[i] = 0;
      if (v == 0) continue;
      if (i < nb) atomicAdd(&counts[(size_t)sd.channel * nb + i], (unsigned long long)v);
      else atomicAdd(&n_ok[sd.channel], (unsigned long long)v);
    }
    __syncthreads();
  }
}

// The same a tile per workgroup and a thread per event: nothing to set up, one pass.  For few events (18,067 of 2
// randoms 3.3 us, 4.6 with the kernel above; 1,003 of 8 3.2 and 5.0), and few tiles of any one channel, whose
// counts meet at the same addresses (whole updates of 1 x 10^5 and 2 x 10^5 events in 3 channels, 130 and 260
// tiles each: 33.3 and 39.0 us, 34.2 and 34.7 above; 2000 tiles of 70 events in 42 channels 40 and 44): at most
// kHistFew.  A row per thread is read less well than a row's words by neighbouring threads, which shows in large
// updates: 4.5 x 10^5 events 39.7 and 39.5 us (5 particles), 41.2 and 38.9 (6), 36.7 and 41.7 (8), 2 x 10^6
// 82 and 51 (5): at most kHistFewEvents.
constexpr int kHistFew = 192;
constexpr int64_t kHistFewEvents = 1 << 19;
__global__ __launch_bounds__(256) void grid_histogram_few_kernel(const TileDesc* __restrict__ tiles,
                                                                 const SegDesc* __restrict__ segs,
                                                                 const ChannelDesc* __restrict__ chans, int n_dim,
                                                                 unsigned long long* __restrict__ counts,
                                                                 unsigned long long* __restrict__ n_ok) {
  extern __shared__ unsigned int hist[];   // n_dim * kGridBins bins, then the accepted count
  const int nb = n_dim * kGridBins;
  const TileDesc td = tiles[blockIdx.x];
  const SegDesc sd = segs[td.seg];
  const int n_x = chans[sd.channel].n_x;
  for (int i = (int)threadIdx.x; i <= nb; i += (int)blockDim.x) hist[i] = 0;
  __syncthreads();
  for (int local = (int)threadIdx.x; local < td.count; local += (int)blockDim.x) {
    const int64_t e = td.e0 + local;
    if (!as_global(sd.ok)[e]) continue;
    const gdouble* xr = as_global((const double*)sd.x) + e * n_x;
    for (int k = 0; k < n_x; k++) {
      int b = (int)(xr[k] * kGridBins);   // rng.cpp:52
      b = b < 0 ? 0 : b > kGridBins - 1 ? kGridBins - 1 : b;
      atomicAdd(&hist[k * kGridBins + b], 1u);
    }
    atomicAdd(&hist[nb], 1u);
  }
  __syncthreads();
  for (int i = (int)threadIdx.x; i <= nb; i += (int)blockDim.x) {
    const unsigned int v = hist[i];
    if (v == 0) continue;
    if (i < nb) atomicAdd(&counts[(size_t)sd.channel * nb + i], (unsigned long long)v);
    else atomicAdd(&n_ok[sd.channel], (unsigned long long)v);
  }
}

__global__ void fill_u64_kernel(unsigned long long* p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0;
}

}  // namespace

hipError_t launch_grid_generate(const DevicePlan& dp, int64_t n_events, const double* cdf, int n_dim, uint64_t seed,
                                hipStream_t stream) {
  if (dp.n_tiles <= 0) return hipSuccess;
  const int groups = std::min(dp.n_tiles, kGenGroups);
  // waves of a workgroup: no more than have events to draw, and, where the launch fills the device, as many as let
  // a CU hold the most waves (2000 tiles of 70 events of 32 randoms: 118 us with four, 69 with two)
  const size_t limit = forward_lds_limit();
  auto lds = [&](int waves) {
    return (size_t)n_dim * (kGridBins * sizeof(BinRec) + waves * kGenRow * sizeof(double) + kGenCells);
  };
  int waves = kGenWaves;
  while (waves > 1 && n_events <= (int64_t)32 * waves * groups) waves /= 2;
  for (int w = waves / 2; w > 0 && (size_t)groups > 256 * (limit / lds(waves)); w /= 2)
    if (limit / lds(w) * w > limit / lds(waves) * waves) waves = w;
  const size_t shmem = lds(waves);
  if (shmem > limit) return hipErrorInvalidValue;
  hipLaunchKernelGGL(grid_generate_kernel, dim3(groups), dim3(64 * waves), shmem, stream, dp.tiles,
                     dp.n_tiles / groups, dp.n_tiles % groups, dp.segs, dp.chans, cdf, n_dim, seed);
  return hipGetLastError();
}

hipError_t launch_grid_histogram(const DevicePlan& dp, int64_t n_events, int busiest, int n_chans, int n_dim,
                                 unsigned long long* counts, hipStream_t stream) {
  unsigned long long* n_ok = counts + (size_t)n_chans * n_dim * kGridBins;
  const size_t n = (size_t)n_chans * n_dim * kGridBins + n_chans;
  hipLaunchKernelGGL(fill_u64_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 1024)), dim3(256), 0, stream,
                     counts, n);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || dp.n_tiles <= 0) return e;
  const size_t shmem = ((size_t)n_dim * kGridBins + 1) * sizeof(unsigned int);
  const int64_t batches = n_events * n_dim / (kHistThreads * kHistUnroll);
  if (busiest <= kHistFew && n_events <= kHistFewEvents) {
    hipLaunchKernelGGL(grid_histogram_few_kernel, dim3(dp.n_tiles), dim3(256), shmem, stream, dp.tiles, dp.segs, dp.chans,
                       n_dim, counts, n_ok);
    return hipGetLastError();
  }
  // at most a workgroup for each batch of loads beyond the first kHistFew of a channel: every workgroup's counts go
  // to the channel's few addresses one after the other, some 18 ns each (2 x 10^5 events of 2 randoms: 18 us at
  // one workgroup per tile, 782; 7.8 at 98)
  const int64_t channels = dp.n_tiles / std::max(1, busiest);
  const int groups = (int)std::min<int64_t>({dp.n_tiles, kHistGroups, std::max<int64_t>(kHistFew * channels, batches)});
  hipLaunchKernelGGL(grid_histogram_kernel, dim3(groups), dim3(kHistThreads), shmem, stream, dp.tiles,
                     dp.n_tiles / groups, dp.n_tiles % groups, dp.segs, dp.chans, n_dim, counts, n_ok);
  return hipGetLastError();
}

}  // namespace gphs
