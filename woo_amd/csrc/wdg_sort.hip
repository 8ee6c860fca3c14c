// Stable LSD radix sort of (key, value) pairs and exclusive prefix scan, for gfx950.
//
// Radix sort: 8-bit digits, one pass = histogram kernel (LDS bins per tile),
// exclusive scan of the digit-major histogram, stable scatter. The scatter
// ranks equal digits inside a 64-lane wavefront with eight ballots (lanes whose
// digit matches in every bit), then across the four wavefronts of the block
// through LDS counters, so the output keeps input order among equal keys.
#include "wdg_internal.hpp"

namespace wdg {

#if defined(__HIP_DEVICE_COMPILE__) && defined(__AMDGCN_WAVEFRONT_SIZE) && __AMDGCN_WAVEFRONT_SIZE != 64
#error "the ballot-based ranking assumes 64-lane wavefronts"
#endif

constexpr int SCAN_BS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_BS * SCAN_ITEMS;

// ------------------------------------------------------------------ scan
// One launch for any length: each workgroup takes the next tile (a ticket, so that every tile it
// waits for belongs to a workgroup that already runs), publishes its sum, and its first wavefront
// adds up the 64 tiles before it at a time until it meets one whose inclusive prefix is known.
// A tile's word holds the value, its state (1 sum, 2 inclusive prefix) and the number of the
// scan, so nothing is cleared between scans. Bound by the launch and the look-back's round trips
// across the XCDs; before, three to five launches (block sums, their scan, the add) took 12 us
// of GPU time and their gaps at 150,000 elements, now 5 us.
__device__ __forceinline__ uint64_t scan_word(uint32_t epoch, uint32_t state, uint32_t v) {
  return ((uint64_t)((epoch << 2) | state) << 32) | v;
}
__global__ __launch_bounds__(SCAN_BS) void k_scan(const uint32_t* in, uint32_t* out, int64_t n, uint64_t* words,
                                                   uint32_t epoch, uint32_t* ticket, uint32_t ticket0,
                                                   uint32_t first, int wide, uint32_t* dTotal) {
  __shared__ uint32_t sTile, sPrefix, wsum[SCAN_BS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid == 0) sTile = atomicAdd(ticket, 1u) - ticket0;
  __syncthreads();
  const uint32_t tile = sTile;
  const int64_t base = (int64_t)tile * SCAN_TILE + (int64_t)tid * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS], sum = 0;
  // wide: both arrays start on 16 bytes, so a thread's eight elements are two vector accesses
  const bool vec = wide && base + SCAN_ITEMS <= n;
  if (vec) {
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i += 4) {
      const uint4 x = *reinterpret_cast<const uint4*>(in + base + i);
      v[i] = x.x; v[i + 1] = x.y; v[i + 2] = x.z; v[i + 3] = x.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++) v[i] = base + i < n ? in[base + i] : 0u;
  }
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; i++) {
    const uint32_t x = v[i];
    v[i] = sum;
    sum += x;
  }
  uint32_t inc = sum;
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t t = __shfl_up(inc, off);
    if (lane >= off) inc += t;
  }
  if (lane == 63) wsum[wv] = inc;
  __syncthreads();
  uint32_t wpre = 0, tot = 0;
  for (int w = 0; w < SCAN_BS / 64; w++) {
    const uint32_t x = wsum[w];
    if (w < wv) wpre += x;
    tot += x;
  }
  if (wv == 0) {
    uint32_t prefix = 0;
    if (tile == 0) {
      prefix = first;
      if (lane == 0)
        __hip_atomic_store(&words[0], scan_word(epoch, 2u, first + tot), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      if (lane == 0)
        __hip_atomic_store(&words[tile], scan_word(epoch, 1u, tot), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // lane l reads the l-th tile before `at` (the first tile's prefix is always known, so the
      // walk ends there)
      for (int64_t at = (int64_t)tile - 1;; at -= 64) {
        const int64_t t = at - lane;
        uint32_t state = 2u, val = 0u;
        if (t >= 0) {
          uint64_t w;
          do {
            w = __hip_atomic_load(&words[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          } while ((uint32_t)(w >> 34) != (epoch & 0x3FFFFFFFu));
          state = (uint32_t)(w >> 32) & 3u;
          val = (uint32_t)w;
        }
        // the nearest tile with an inclusive prefix ends the walk
        const unsigned long long known = __ballot(state == 2u);
        const int stop = known ? __ffsll((long long)known) - 1 : 63;
        uint32_t x = lane <= stop ? val : 0u;
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
        prefix += x;
        if (known) break;
      }
      if (lane == 0)
        __hip_atomic_store(&words[tile], scan_word(epoch, 2u, prefix + tot), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    if (lane == 0) {
      sPrefix = prefix;
      if (((int64_t)tile + 1) * SCAN_TILE >= n) *dTotal = prefix + tot;
    }
  }
  __syncthreads();
  const uint32_t excl = sPrefix + wpre + (inc - sum);
  if (vec) {
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i += 4)
      *reinterpret_cast<uint4*>(out + base + i) =
          make_uint4(v[i] + excl, v[i + 1] + excl, v[i + 2] + excl, v[i + 3] + excl);
  } else {
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++)
      if (base + i < n) out[base + i] = v[i] + excl;
  }
}

// single-workgroup scan for short arrays (one launch); in may equal out
constexpr int S1_BS = 1024;
constexpr int S1_ITEMS = 8;
constexpr int64_t S1_MAX = 8192;
__global__ __launch_bounds__(S1_BS) void k_scan_one(const uint32_t* in, uint32_t* out, int64_t n, uint32_t first,
                                                     uint32_t* dTotal) {
  __shared__ uint32_t wsum[S1_BS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  uint32_t carry = first;
  for (int64_t base = 0; base < n; base += S1_BS * S1_ITEMS) {
    uint32_t v[S1_ITEMS], sum = 0;
    for (int i = 0; i < S1_ITEMS; i++) {
      const int64_t idx = base + (int64_t)tid * S1_ITEMS + i;
      const uint32_t x = idx < n ? in[idx] : 0u;
      v[i] = sum;
      sum += x;
    }
    uint32_t inc = sum;
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t t = __shfl_up(inc, off);
      if (lane >= off) inc += t;
    }
    if (lane == 63) wsum[wv] = inc;
    __syncthreads();
    uint32_t wpre = 0, tot = 0;
    for (int w = 0; w < S1_BS / 64; w++) {
      const uint32_t s = wsum[w];
      if (w < wv) wpre += s;
      tot += s;
    }
    const uint32_t excl = carry + wpre + (inc - sum);
    for (int i = 0; i < S1_ITEMS; i++) {
      const int64_t idx = base + (int64_t)tid * S1_ITEMS + i;
      if (idx < n) out[idx] = v[i] + excl;
    }
    carry += tot;
    __syncthreads();
  }
  if (tid == 0) *dTotal = carry;
}

void scan_exclusive(Ctx& c, const uint32_t* in, uint32_t* out, int64_t n, uint32_t* dTotal, uint32_t first) {
  if (n <= 0) {
    hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(S1_BS), 0, c.stream, in, out, (int64_t)0, first, dTotal);
    WDG_LAUNCH_CHECK();
    return;
  }
  if (n <= S1_MAX) {
    hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(S1_BS), 0, c.stream, in, out, n, first, dTotal);
    WDG_LAUNCH_CHECK();
    return;
  }
  const int64_t tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
  // the words of a new buffer, and of every buffer when the 30-bit scan number starts again, hold
  // no scan's number (0 is never used)
  const size_t before = c.scanWords.cap;
  c.scanWords.ensure((size_t)tiles);
  if (c.scanWords.cap != before || c.scanEpoch == 0x3FFFFFFFu) {
    WDG_HIP(hipMemsetAsync(c.scanWords.p, 0, c.scanWords.cap * sizeof(uint64_t), c.stream));
    c.scanEpoch = 0;
  }
  if (!c.scanTicket.p) {
    c.scanTicket.ensure(1);
    WDG_HIP(hipMemsetAsync(c.scanTicket.p, 0, sizeof(uint32_t), c.stream));
  }
  c.scanEpoch++;
  const int wide = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0u;
  hipLaunchKernelGGL(k_scan, dim3((unsigned)tiles), dim3(SCAN_BS), 0, c.stream, in, out, n, c.scanWords.p, c.scanEpoch,
                     c.scanTicket.p, c.scanTickets, first, wide, dTotal);
  WDG_LAUNCH_CHECK();
  c.scanTickets += (uint32_t)tiles;
}

uint32_t read_u32(Ctx& c, const uint32_t* d) {
  WDG_HIP(hipMemcpyAsync(c.hflags + 8, d, sizeof(uint32_t), hipMemcpyDeviceToHost, c.stream));
  WDG_HIP(hipStreamSynchronize(c.stream));
  return c.hflags[8];
}

// ------------------------------------------------------------------ radix sort
constexpr int RS_BS = 256;
constexpr int RS_ITEMS = 16;
constexpr int RS_TILE = RS_BS * RS_ITEMS;
constexpr int RS_WAVES = RS_BS / 64;

template <class K>
__global__ __launch_bounds__(RS_BS) void k_rs_hist(const K* __restrict__ keys, int64_t n, int shift,
                                                    uint32_t* hist, int nblk) {
  __shared__ uint32_t h[256];
  const int tid = threadIdx.x;
  h[tid] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * RS_TILE;
  for (int i = 0; i < RS_ITEMS; i++) {
    int64_t idx = base + (int64_t)i * RS_BS + tid;
    if (idx < n) atomicAdd(&h[(uint32_t)(keys[idx] >> shift) & 255u], 1u);
  }
  __syncthreads();
  hist[(int64_t)tid * nblk + blockIdx.x] = h[tid];
}

template <class K>
__global__ __launch_bounds__(RS_BS) void k_rs_scatter(const K* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                       K* __restrict__ kout, uint32_t* __restrict__ vout, int64_t n,
                                                       int shift, const uint32_t* __restrict__ histScan, int nblk) {
  __shared__ uint32_t base[256], running[256], wcount[RS_WAVES][256];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  base[tid] = histScan[(int64_t)tid * nblk + blockIdx.x];
  running[tid] = 0;
  for (int w = 0; w < RS_WAVES; w++) wcount[w][tid] = 0;
  __syncthreads();
  const int64_t tbase = (int64_t)blockIdx.x * RS_TILE;
  const uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
  for (int r = 0; r < RS_ITEMS; r++) {
    int64_t idx = tbase + (int64_t)r * RS_BS + tid;
    bool valid = idx < n;
    K key = valid ? kin[idx] : K(0);
    uint32_t val = valid ? vin[idx] : 0u;
    uint32_t d = (uint32_t)(key >> shift) & 255u;
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      bool bit = (d >> b) & 1u;
      uint64_t bb = __ballot(valid && bit);
      peers &= bit ? bb : ~bb;
    }
    uint32_t rank = 0;
    if (valid) {
      rank = (uint32_t)__popcll(peers & lt);
      int leader = 63 - __clzll((long long)peers);
      if (lane == leader) wcount[wave][d] = (uint32_t)__popcll(peers);
    }
    __syncthreads();
    if (valid) {
      uint32_t off = running[d] + rank;
      for (int w = 0; w < wave; w++) off += wcount[w][d];
      uint32_t dst = base[d] + off;
      kout[dst] = key;
      vout[dst] = val;
    }
    __syncthreads();
    uint32_t add = 0;
    for (int w = 0; w < RS_WAVES; w++) {
      add += wcount[w][tid];
      wcount[w][tid] = 0;
    }
    running[tid] += add;
    __syncthreads();
  }
}

template <class K>
void radix_sort_pairs(Ctx& c, K* keys, uint32_t* vals, K* keysTmp, uint32_t* valsTmp, int64_t n, int bits) {
  if (n <= 1) return;
  int passes = (bits + 7) / 8;
  int nblk = (int)((n + RS_TILE - 1) / RS_TILE);
  c.sortHist.ensure((size_t)256 * nblk + 64);
  K* ka = keys;
  K* kb = keysTmp;
  uint32_t* va = vals;
  uint32_t* vb = valsTmp;
  for (int p = 0; p < passes; p++) {
    int shift = 8 * p;
    hipLaunchKernelGGL(k_rs_hist<K>, dim3(nblk), dim3(RS_BS), 0, c.stream, (const K*)ka, n, shift, c.sortHist.p, nblk);
    WDG_LAUNCH_CHECK();
    scan_exclusive(c, c.sortHist.p, c.sortHist.p, (int64_t)256 * nblk, c.dflags.p + 3);
    hipLaunchKernelGGL(k_rs_scatter<K>, dim3(nblk), dim3(RS_BS), 0, c.stream, (const K*)ka, (const uint32_t*)va, kb, vb,
                       n, shift, (const uint32_t*)c.sortHist.p, nblk);
    WDG_LAUNCH_CHECK();
    std::swap(ka, kb);
    std::swap(va, vb);
  }
  if (ka != keys) {
    WDG_HIP(hipMemcpyAsync(keys, ka, n * sizeof(K), hipMemcpyDeviceToDevice, c.stream));
    WDG_HIP(hipMemcpyAsync(vals, va, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, c.stream));
  }
}

template void radix_sort_pairs<uint32_t>(Ctx&, uint32_t*, uint32_t*, uint32_t*, uint32_t*, int64_t, int);
template void radix_sort_pairs<uint64_t>(Ctx&, uint64_t*, uint32_t*, uint64_t*, uint32_t*, int64_t, int);

}  // namespace wdg
