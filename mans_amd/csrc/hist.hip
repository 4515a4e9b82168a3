// hist.hip -- per-byte-plane histograms with the probability normalisation
// fused into the last workgroup to finish.
//
// Reference: include/ans/GpuANSStatistics.h:23-151 (histogram),
// :186-406 (normalisation), :409-468 (launches).  The reference runs
// histogram -> quantizeWeights as two launches on one byte stream; here one
// launch counts every plane of the input (byte k of each element -> plane k),
// and the last workgroup (device-scope done counter) normalises each plane,
// writes the tables and the container's plane headers, and resets the
// accumulators so the next call needs no memset.
#include <algorithm>

#include "codec_device.hpp"
#include "hist_device.hpp"

namespace mans {
namespace {

// 512 threads: the launch's workgroups each add to the same counters (bins,
// chunks, workgroups done), and those atomics run one after another at 11 ns,
// so few large workgroups.
constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;

// One source, counted by the launch: a workgroup's first chunk of
// a.chunk_tiles tiles is its own, the others come from a device-wide counter
// (workgroups on different CUs stream at different rates, so a fixed share
// leaves the launch waiting for its slowest one), the next grab taken while
// the current chunk is counted; a chunk's tiles go round the wavefronts.  What is not a whole tile (the unaligned
// head, the bytes after the last whole tile) is counted byte by byte by
// workgroup 0.
template <int S>
__device__ __forceinline__ void count_source(const HistArgs& a, const HistSource& src, bool edges, uint32_t* grab,
                                             uint32_t* s_grab, uint32_t* lds) {
  const uint8_t* p = src.ptr;
  const uint64_t n = src.nbytes;
  const uint32_t mis = (uint32_t)((uintptr_t)p & 15u);
  const uint64_t head = mis ? ((16u - mis) < n ? (16u - mis) : n) : 0;
  const uint32_t ntiles = (uint32_t)((n - head) / (16u * kTileU4));
  const uint4* body = (const uint4*)(p + head);
  const uint32_t t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // planes are numbered from the source's start: with an unaligned head the
  // body starts at byte `head` of an element (a multiple of S: the source is
  // element aligned and S divides 16)
  int32_t sum[S][4];
#pragma unroll
  for (int k = 0; k < S; ++k)
#pragma unroll
    for (int v = 0; v < 4; ++v) sum[k][v] = 0;
  uint32_t* const ghist = a.hist + src.plane0 * kNumSymbols;
  const bool more = (uint64_t)gridDim.x * a.chunk_tiles < ntiles;
  if (t == 0) s_grab[0] = blockIdx.x;
  __syncthreads();
  uint32_t done = 0;
  for (uint32_t k = 0;; ++k) {
    const uint64_t t0 = (uint64_t)s_grab[k & 1u] * a.chunk_tiles;
    if (t0 >= ntiles) break;
    if (t == 0) s_grab[(k + 1) & 1u] = more ? gridDim.x + atomicAdd(grab, 1u) : ~0u;
    const uint32_t t1 = t0 + a.chunk_tiles < ntiles ? (uint32_t)t0 + a.chunk_tiles : ntiles;
    count_tiles<S>(body, (uint32_t)t0 + wave, t1, kWaves, sum);
    done += div_up(a.chunk_tiles, kWaves);
    if (done >= kTileFlush) {
      flush_counts<S, kThreads>(sum, lds, ghist);
      done = 0;
    }
    __syncthreads();
  }
  if (edges) {
    for (uint64_t i = t; i < head; i += kThreads) count_byte(lds, (uint32_t)i % S, p[i]);
    for (uint64_t i = head + 16ull * kTileU4 * ntiles + t; i < n; i += kThreads) count_byte(lds, (uint32_t)(i % S), p[i]);
    __syncthreads();
  }
  // (workgroups without a chunk have nothing to add)
  if (done || edges) flush_counts<S, kThreads>(sum, lds, ghist);
}

__global__ __launch_bounds__(kThreads, 4) void hist_kernel(HistArgs a) {
  __shared__ __align__(16) uint32_t s_cnt[kFlushWords];  // (the finisher's keys and ranks too)
  __shared__ int s_last_flag;
  int* s_last = &s_last_flag;
  __shared__ uint32_t s_grab[2];
  const int t = threadIdx.x;
  const int P = a.num_planes;

  // Clear the encode launch's look-back words (the previous user of this
  // workspace has finished: kernels on one stream run in order).
  for (uint64_t i = (uint64_t)blockIdx.x * kThreads + t; i < a.status_count;
       i += (uint64_t)gridDim.x * kThreads)
    a.status[i] = 0;

  for (int i = t; i < (int)kFlushWords; i += kThreads) s_cnt[i] = 0;
  __syncthreads();
  for (int s = 0; s < a.nsrc; ++s) {
    const HistSource& src = a.src[s];
    const bool edges = blockIdx.x == 0;
    if (src.stride == 1) count_source<1>(a, src, edges, a.grab + s, s_grab, s_cnt);
    else if (src.stride == 2) count_source<2>(a, src, edges, a.grab + s, s_grab, s_cnt);
    else count_source<4>(a, src, edges, a.grab + s, s_grab, s_cnt);
    __syncthreads();
  }
  // the adds are performed where every XCD sees them: once they have
  // completed, the finisher's device-scope loads read their sums
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (t == 0) *s_last = atomicAdd(a.done, 1u) == gridDim.x - 1;
  __syncthreads();
  if (!*s_last) return;

  // ---- finisher: normalise each plane (wavefront k plane k, the ranks by
  // all wavefronts), write tables and headers.  (A plane after another with
  // 256 threads: 3.5 us each.)
  const uint32_t wave = __builtin_amdgcn_readfirstlane((uint32_t)t >> 6), lane = (uint32_t)t & 63u;
  const bool owner = wave < (uint32_t)P;
  uint32_t* const s_keys = s_cnt;          // [P][256]
  uint32_t* const s_rank = s_cnt + 1024u;  // [P][256], zero
  uint32_t q[4] = {0, 0, 0, 0}, c[4], key[4], qsum = 0;
  const uint32_t total = owner ? (uint32_t)a.plane_nsym[wave] : 0u;
  if (owner) {
    uint32_t* const h = a.hist + wave * kNumSymbols + 4u * lane;
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = __hip_atomic_load(h + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *(uint4*)h = make_uint4(0, 0, 0, 0);
    if (a.hist_out) *(uint4*)(a.hist_out + wave * kNumSymbols + 4u * lane) = make_uint4(c[0], c[1], c[2], c[3]);
    if (total > 0) {
      qsum = quantize_syms(c, total, a.prob_bits, q, key);
      *(uint4*)(s_keys + wave * kNumSymbols + 4u * lane) = make_uint4(key[0], key[1], key[2], key[3]);
    }
  }
  __syncthreads();
  {
    // plane k's keys in kWaves / P parts (P is 1, 2 or 4)
    const uint32_t k = wave % (uint32_t)P, part = wave / (uint32_t)P, len = kNumSymbols * (uint32_t)P / kWaves;
    const uint4 kk = *(const uint4*)(s_keys + k * kNumSymbols + 4u * lane);
    const uint32_t mine[4] = {kk.x, kk.y, kk.z, kk.w};
    uint32_t r[4];
    rank_syms(mine, s_keys + k * kNumSymbols, part * len, (part + 1u) * len, r);
#pragma unroll
    for (int j = 0; j < 4; ++j) atomicAdd(s_rank + k * kNumSymbols + 4u * lane + (uint32_t)j, r[j]);
  }
  __syncthreads();
  bool bad = false;
  if (owner) {
    const uint4 rr = *(const uint4*)(s_rank + wave * kNumSymbols + 4u * lane);
    const uint32_t rank[4] = {rr.x, rr.y, rr.z, rr.w};
    uint4 e[4] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
    if (total > 0) settle_syms(q, qsum, rank, a.prob_bits, e, bad);  // (an empty plane's table is zero)
#pragma unroll
    for (int j = 0; j < 4; ++j) a.table[wave * kNumSymbols + 4u * lane + (uint32_t)j] = e[j];
    if (a.write_headers) {
      uint8_t* h = a.out + a.plane_section[wave];
      ((uint2*)(h + kAnsHeaderBytes))[lane] = make_uint2(e[0].x | (e[1].x << 16), e[2].x | (e[3].x << 16));
      if (lane < 8) {
        uint32_t f = 0;
        if (lane == 0) f = (kAnsMagic << 16) | a.version;
        if (lane == 1) f = (uint32_t)a.plane_nb[wave];
        if (lane == 2) f = (uint32_t)a.plane_nsym[wave];
        if (lane == 4) f = (uint32_t)a.prob_bits;
        ((uint32_t*)h)[lane] = f;  // totalCompressedWords (lane == 3) accumulates in encode
      }
      const uint64_t nb = a.plane_nb[wave];
      if ((nb & 1) && lane < 2) {
        uint32_t lanes = a.version == 2 ? 64u : 32u;
        ((uint32_t*)(h + kSectionFixed + 4ull * lanes * nb + 8ull * nb))[lane] = 0;
      }
    }
  }
  if (t == 0) {
    *a.done = 0;
    a.grab[0] = 0;
    a.grab[1] = 0;
    if (a.ticket) *a.ticket = 0;
  }
  if (a.write_headers && a.has_frame && t < 32) ((uint32_t*)a.out)[t] = a.frame_hdr[t];
  if (a.total_units == 0 && t == 0) {
    if (a.d_out_size32) *a.d_out_size32 = (uint32_t)a.empty_size;
    if (a.d_out_size64) *a.d_out_size64 = a.empty_size;
  }
  (void)bad;
}

__global__ void fill_u64_kernel(uint64_t* p, uint64_t n, uint64_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}
__global__ void fill_u32_kernel(uint32_t* p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}
// Zeroes n words at p and na / nb at a / b: one launch before a call.
__global__ void zero_kernel(uint64_t* p, uint64_t n, uint32_t* a, uint32_t na, uint32_t* b, uint32_t nb) {
  const uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i0 < na) a[i0] = 0;
  if (i0 < nb) b[i0] = 0;
  for (uint64_t i = i0; i < n; i += (uint64_t)gridDim.x * blockDim.x) p[i] = 0;
}
// na words of a, then nb of b, to pinned host memory.  (An asynchronous copy
// each is a kernel of the runtime's too, of 4-5 us, and 10 us of host time.)
__global__ void to_host_kernel(uint32_t* dst, const uint32_t* a, uint32_t na, const uint32_t* b, uint32_t nb) {
  const uint32_t i = threadIdx.x;
  if (i < na) dst[i] = a[i];
  else if (i < na + nb) dst[i] = b[i - na];
}

}  // namespace

hipError_t launch_hist(const HistArgs& args, int cu, hipStream_t s) {
  HistArgs a = args;
  uint64_t ntiles = 0;
  for (int i = 0; i < a.nsrc; ++i) ntiles = std::max<uint64_t>(ntiles, a.src[i].nbytes / (16u * kTileU4));
  int per_cu = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, hist_kernel, kThreads, 0);
  if (e != hipSuccess) return e;
  if (per_cu < 1) per_cu = 1;
  if (per_cu > 2) per_cu = 2;
  const uint64_t cap = (uint64_t)cu * (uint64_t)per_cu;
  // chunks: about four per workgroup, one tile a wavefront at least (small
  // inputs spread over the chip) and 4 at most (1 GiB: 0.230 ms with 4 tiles
  // a wavefront, 0.238 with 16; 128 MiB: 52 us with 2, 72 with 1)
  const uint64_t want = div_up(ntiles, cap * 4u * kWaves);
  a.chunk_tiles = (uint32_t)(kWaves * std::min<uint64_t>(std::max<uint64_t>(want, 1), 4));
  const uint64_t chunks = div_up(ntiles, a.chunk_tiles);
  const uint32_t grid = (uint32_t)std::max<uint64_t>(1, std::min(chunks, cap));
  hipLaunchKernelGGL(hist_kernel, dim3(grid), dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_fill_u64(uint64_t* p, uint64_t n, uint64_t v, hipStream_t s) {
  if (n == 0) return hipSuccess;
  uint32_t grid = (uint32_t)(div_up(n, 256) < 1024 ? div_up(n, 256) : 1024);
  hipLaunchKernelGGL(fill_u64_kernel, dim3(grid), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s) {
  if (n == 0) return hipSuccess;
  uint32_t grid = (uint32_t)(div_up(n, 256) < 1024 ? div_up(n, 256) : 1024);
  hipLaunchKernelGGL(fill_u32_kernel, dim3(grid), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}
hipError_t launch_zero(uint64_t* p, uint64_t n, uint32_t* a, uint32_t na, uint32_t* b, uint32_t nb, hipStream_t s) {
  const uint64_t most = std::max<uint64_t>(std::max<uint64_t>(n, 1), std::max(na, nb));
  const uint32_t grid = (uint32_t)std::min<uint64_t>(div_up(most, 256), 1024);
  if (std::max(na, nb) > grid * 256u) return hipErrorInvalidValue;
  hipLaunchKernelGGL(zero_kernel, dim3(grid), dim3(256), 0, s, p, n, a, na, b, nb);
  return hipGetLastError();
}
hipError_t launch_to_host(void* dst, const void* a, uint32_t na, const void* b, uint32_t nb, hipStream_t s) {
  if (na + nb > 256) return hipErrorInvalidValue;
  hipLaunchKernelGGL(to_host_kernel, dim3(1), dim3(64 * (uint32_t)div_up(na + nb, 64)), 0, s, (uint32_t*)dst,
                     (const uint32_t*)a, na, (const uint32_t*)b, nb);
  return hipGetLastError();
}

}  // namespace mans
