// adm.hip -- ADM byte mapping of uint16 data (code plane + bit-signal plane).
//
// Reference: mapping/cpu/mappingcpuV1.cpp:33-276 (semantics) and
// mapping/nv/mappingV15_fused_uint16.cu:24-121, 124-398, 400-730 (GPU
// kernels).  Group g = elements [512g, 512g + 512) = 32 lanes x 16 elements.
// center = floor(sum / count); per element d = |x - c|, len = 1 if x == c else
// ceil(d / 126), code = 1 if x == c else 2(d - 126(len - 1)) (+1 if x < c);
// each lane sets bit `bo` (MSB first) then advances bo by len; the group's
// lanes are padded to M_g = ceil(max L / 8) bytes (the byte holding bit L gets
// 0xFF >> (L % 8)), lanes without elements stay zero (mappingcpuV1.cpp:146);
// lane l's bytes go to 32 O_g + l M_g with O = exclusive prefix of M.
//
// Structure: a workgroup takes 4 x 32 groups per ticket, a wavefront 32 of
// them, two at a time (one per half-wave).  Each pair's codes and centers are
// written, its bits built in registers and put into the wavefront's LDS area,
// back to back; the workgroup publishes the ticket's byte total, and once its
// next ticket is mapped the look-back gives the offset and the area is copied
// out.  O_g is resolved by decoupled look-back over tickets (any number of
// groups; the reference's fused path is limited to 1024 groups,
// mappingV15_fused_uint16.cu:851), the whole wave reading 512 predecessors
// per round trip.  Unmap parses each lane's bytes with clz over 32-bit words.
#include "adm_device.hpp"
#include "codec_device.hpp"

namespace mans {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

// Sum and maximum over a half-wave (every lane gets it): within rows of 16
// lanes by DPP, then across the half's two rows.
template <typename F>
__device__ __forceinline__ uint32_t half_reduce(uint32_t v, F f) {
  v = f(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
  v = f(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
  v = f(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true));  // row_half_mirror
  v = f(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true));  // row_mirror
  return f(v, (uint32_t)__shfl_xor(v, 16, 64));
}
__device__ __forceinline__ uint32_t half_sum(uint32_t v) {
  return half_reduce(v, [](uint32_t x, uint32_t y) { return x + y; });
}
__device__ __forceinline__ uint32_t half_max(uint32_t v) {
  return half_reduce(v, [](uint32_t x, uint32_t y) { return x > y ? x : y; });
}

// Group pairs per wavefront and ticket.  One workgroup ticket (65536 elements)
// is one add on the ticket counter (11 ns each, all on one address) and one
// look-back entry: a ticket per wavefront cost 185 us in adds alone on
// 512 MiB.
constexpr uint32_t kPairs = kAdmTicketGroups / 2;
constexpr uint32_t kTicketGroups = kWaves * kAdmTicketGroups;
static_assert(kPairs % 2 == 0, "pairs are mapped two at a time");
// Bytes of a wavefront's area for its 32 groups' bits: 4 for each of the 1024
// lanes.  The pairs from the first on that does not fit are mapped a second
// time when their offset is known and the area has been copied out, in the area
// itself (lane buffers of kLaneWords words, padded to 9 so the lanes' words of
// one index fall in distinct LDS banks).  (All pairs mapped again: 4 M elements
// of 0.43 bytes of bits 66 us; a second pass over everything 59; so 48.)
constexpr uint32_t kAreaBytes = 4096;
constexpr uint32_t kLaneWords = kAdmLaneBytes / 4 + 1;
static_assert(64 * kLaneWords * 4 <= kAreaBytes, "the lane buffers fit the area");

// The 16 elements of one lane (half-wave = one group): raw_lane loads them
// (two 16-byte loads for a whole lane, element loads for the last, partial
// lane of the input); unpack_center spreads them and returns the group's
// center (all lanes of the half-wave).  Split so a pair's loads can be in
// flight while the previous pair is mapped.
struct LaneRaw {
  uint4 q0, q1;
  uint32_t cnt;
  uint64_t base;
};
// FULL: every lane of the ticket is whole (tickets before the input's end):
// no bounds, no branch around the loads.
template <bool FULL>
__device__ __forceinline__ LaneRaw raw_lane(const AdmMapArgs& a, uint64_t g, uint32_t lin) {
  LaneRaw r;
  r.base = g * kAdmGroup + (uint64_t)lin * kAdmChunk;
  if constexpr (FULL) {
    r.cnt = kAdmChunk;
    const uint4* p = (const uint4*)(a.in + r.base);
    r.q0 = p[0];
    r.q1 = p[1];
    return r;
  }
  const bool gactive = g < a.gsize;
  r.cnt = gactive && r.base < a.n ? (uint32_t)((a.n - r.base) < kAdmChunk ? (a.n - r.base) : kAdmChunk) : 0u;
  // (a partial lane, only at the end of the input, is loaded element by
  // element in unpack_center: no element loads here, so nothing makes the
  // wave wait for these loads before their pair is mapped)
  if (r.cnt == kAdmChunk) {
    const uint4* p = (const uint4*)(a.in + r.base);
    r.q0 = p[0];
    r.q1 = p[1];
  } else {
    r.q0 = make_uint4(0, 0, 0, 0);
    r.q1 = make_uint4(0, 0, 0, 0);
  }
  return r;
}
template <bool FULL>
__device__ __forceinline__ uint32_t unpack_center(const AdmMapArgs& a, const LaneRaw& r, uint32_t (&v)[kAdmChunk]) {
  uint32_t w[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
  if (!FULL && r.cnt > 0 && r.cnt < kAdmChunk) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t lo = (uint32_t)(2 * i) < r.cnt ? (uint32_t)a.in[r.base + 2 * i] : 0u;
      const uint32_t hi = (uint32_t)(2 * i + 1) < r.cnt ? (uint32_t)a.in[r.base + 2 * i + 1] : 0u;
      w[i] = lo | (hi << 16);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v[2 * i] = w[i] & 0xffffu;
    v[2 * i + 1] = w[i] >> 16;
  }
  uint32_t lsum = 0;
#pragma unroll
  for (int i = 0; i < (int)kAdmChunk; ++i) lsum += FULL || (uint32_t)i < r.cnt ? v[i] : 0u;
  if constexpr (FULL) return half_sum(lsum) / kAdmGroup;
  const uint32_t gsum = half_sum(lsum), gcnt = half_sum(r.cnt);
  return gcnt ? gsum / gcnt : 0u;  // mappingcpuV1.cpp:60-66
}

// Per element (mappingcpuV1.cpp:68-146): d = |x - c|, len = 1 if x == c else
// ceil(d / 126), code = 1 if x == c else 2 (d - 126 (len - 1)) (+1 if x < c);
// a one at bit `bo` (MSB first), then bo += len.  With `bits`, sets those
// bits in the lane's LDS buffer; returns bo (the lane's bit length).
template <bool PACK>
__device__ __forceinline__ uint32_t map_lane(const uint32_t (&v)[kAdmChunk], uint32_t cnt, uint32_t c,
                                             uint32_t (&codes)[4], uint32_t* bits) {
  uint32_t bo = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) codes[i] = 0;
  // (branch-free over the elements: an element past cnt adds no code byte
  // and no length)
#pragma unroll
  for (int i = 0; i < (int)kAdmChunk; ++i) {
    const bool ok = (uint32_t)i < cnt;
    const uint32_t x = v[i];
    const uint32_t d = x > c ? x - c : c - x;
    const uint32_t len = x == c ? 1u : (d + kAdmMod - 1) / kAdmMod;
    const uint32_t code = x == c ? 1u : ((d - kAdmMod * (len - 1)) * 2u + (x > c ? 0u : 1u));
    codes[i >> 2] |= (ok ? code & 0xffu : 0u) << (8 * (i & 3));
    if (PACK && ok && bo < 8 * kAdmLaneBytes)
      atomicOr(bits + (bo >> 5), 1u << (((bo >> 3) & 3u) * 8u + 7u - (bo & 7u)));
    bo += ok ? len : 0u;
  }
  return bo;
}

// map_lane for a whole lane whose bits fit 64: the same codes, and the bits
// in `word` (first bit on top).  With q = len - 1 = (max(d, 1) - 1) / 126 (the
// high word of a 24-bit product: exact for 16 bits) an element's string is a one and q zeros,
// and its code 2 (d - 126 q) + 1, less one if x > c.  Each half of the
// elements collects its bits in a 32-bit word; false if one does not fit.
__device__ __forceinline__ bool map_lane_word(const uint32_t (&v)[kAdmChunk], uint32_t c, uint32_t (&codes)[4],
                                              uint64_t& word, uint32_t& bo) {
  uint32_t acc[2] = {0, 0}, len[2] = {8, 8};
#pragma unroll
  for (int i = 0; i < 4; ++i) codes[i] = 0;
#pragma unroll
  for (int i = 0; i < (int)kAdmChunk; ++i) {
    const int32_t e = (int32_t)c - (int32_t)v[i];
    const uint32_t d = (uint32_t)(e < 0 ? -e : e);
    const uint32_t y = ((d > 1u ? d : 1u) << 8) - 256u;
    const uint32_t q = (uint32_t)(((uint64_t)(y & 0xffffffu) * 133153u) >> 32);
    const uint32_t code = 2u * (d - __umul24(kAdmMod, q)) + (uint32_t)(e >> 31);
    codes[i >> 2] |= code << (8 * (i & 3));
    acc[i >> 3] = ((acc[i >> 3] << 1) | 1u) << (q & 31u);
    len[i >> 3] += q;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) codes[i] += 0x01010101u;
  bo = len[0] + len[1];
  if (len[0] > 32u || len[1] > 32u) return false;
  word = ((uint64_t)acc[0] << (64u - len[0])) | ((uint64_t)acc[1] << (64u - bo));
  return true;
}

// A ticket's offset is resolved only after the workgroup's next ticket is
// mapped (two areas, used in turn): by then the predecessors have had a whole
// ticket's time to publish their totals, so the look-back sums published
// entries instead of waiting for the slowest.  A workgroup waits only on lower
// tickets, each of which publishes its total right after its mapping, so the
// launch drains.
// Bound by vector instructions (about 15 per element) and, from there, memory
// traffic (input, codes and bits once): 512 MiB 285 us; with a second
// pass over the input that built the bits by one LDS atomic per element, and
// a ticket per wavefront, 460.
__global__ __launch_bounds__(kThreads) void adm_map_kernel(AdmMapArgs a) {
  __shared__ uint4 s_area[2][kWaves][kAreaBytes / 16];
  __shared__ uint32_t s_sum[2][kWaves], s_next[2];
  const int t = threadIdx.x, lane = t & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane((uint32_t)t >> 6);
  const uint32_t half = (uint32_t)lane >> 5, lin = (uint32_t)lane & 31u;

  // the ticket mapped but not resolved (workgroup-uniform): its first group,
  // byte total (in units of 32 bytes, as all offsets here); of this
  // wavefront's groups the offset in the ticket, the total, and in lane g < 32
  // group g's offset
  bool pend = false;
  uint32_t p_tk = 0, p_agg = 0, p_off = 0, p_sum = 0, p_exlo = 0;

  // Pairs pr0 on, which did not fit the area: mapped again from the input,
  // pair by pair, with the lanes' bits in the area's lane buffers.
  auto direct = [&](uint32_t* area, uint64_t excl, uint64_t g0, uint32_t pr0) {
    uint32_t* const mybits = area + lane * kLaneWords;
    const uint8_t* const wavebytes = (const uint8_t*)area;
    for (uint32_t pr = pr0; pr < kPairs; ++pr) {
      const uint64_t g = g0 + 2 * pr + half;
      const LaneRaw cur = raw_lane<false>(a, g, lin);
      uint32_t v[kAdmChunk], codes[4];
      const uint32_t cnt = cur.cnt;
      const uint32_t c = unpack_center<false>(a, cur, v);
#pragma unroll
      for (int i = 0; i < (int)kLaneWords; ++i) mybits[i] = 0;
      __threadfence_block();
      const uint32_t bo = map_lane<true>(v, cnt, c, codes, mybits);
      const uint32_t ex0 = __shfl(p_exlo, (int)(2 * pr), 64), ex1 = __shfl(p_exlo, (int)(2 * pr + 1), 64);
      const uint32_t ex2 = pr + 1 < kPairs ? __shfl(p_exlo, (int)((2 * pr + 2) & 63u), 64) : p_sum;
      const uint32_t m = half ? ex2 - ex1 : ex1 - ex0;
      if (cnt && bo < 8u * m) {
        const uint32_t pad = (bo & 7u) == 0 ? 0xffu : (0xffu >> (bo & 7u));
        atomicOr(mybits + (bo >> 5), pad << (((bo >> 3) & 3u) * 8u));
      }
      __threadfence_block();
      if (g < a.gsize && m > 0) {
        const uint64_t dst0 = 32ull * (excl + (half ? ex1 : ex0));
        const uint32_t total = 32u * m;
        const uint32_t inv = (65536u + m - 1u) / m;
        const uint64_t valid_lanes = a.n > g * kAdmGroup ? div_up(a.n - g * kAdmGroup, kAdmChunk) : 0;
        if (dst0 + total <= a.bits_capacity) {
          for (uint32_t q = lin; q < total; q += 32u) {
            const uint32_t l = (q * inv) >> 16, j = q - l * m;
            const uint8_t byte = l < valid_lanes ? wavebytes[(half * 32u + l) * (4u * kLaneWords) + j] : (uint8_t)0;
            a.bits[dst0 + q] = byte;
          }
        } else if (lin == 0) {
          atomicOr(a.err, kErrCapacity);
        }
      }
      __threadfence_block();
    }
  };

  // the pending ticket's offsets and bits
  auto finish_pending = [&](uint32_t slot) {
    // (every wavefront resolves; all write the same prefix)
    uint64_t excl = resolve_prefix(a.status, p_tk / kTicketGroups, p_agg, lane);
    excl = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(excl >> 32)) << 32) |
           (uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)excl);
    if ((uint64_t)p_tk + kTicketGroups >= a.gsize && t == 0) a.offsets[a.gsize] = (int32_t)(excl + p_agg);
    excl += p_off;
    const uint64_t g0 = (uint64_t)p_tk + wave * kAdmTicketGroups;
    if ((uint32_t)lane < kAdmTicketGroups && g0 + lane < a.gsize) a.offsets[g0 + lane] = (int32_t)(excl + p_exlo);
    // the pairs in the area (each ends where the next begins) and their bytes
    uint32_t pairs = kPairs, held = p_sum;
    if (32u * p_sum > kAreaBytes) {
      pairs = (uint32_t)__popcll(__ballot((lane & 1) == 0 && lane >= 2 && (uint32_t)lane < kAdmTicketGroups &&
                                          32u * p_exlo <= kAreaBytes));
      held = __builtin_amdgcn_readlane(p_exlo, 2u * pairs);
    }
    uint32_t pr0 = 0;
    if (32ull * (excl + held) <= a.bits_capacity) {
      uint8_t* const dst = a.bits + 32ull * excl;
      if (((uintptr_t)a.bits & 15u) == 0) {
        const uint4* const src = s_area[slot][wave];
        for (uint32_t q = (uint32_t)lane; q < 2u * held; q += 64u) ((uint4*)dst)[q] = src[q];
      } else {
        const uint8_t* const src = (const uint8_t*)s_area[slot][wave];
        for (uint32_t q = (uint32_t)lane; q < 32u * held; q += 64u) dst[q] = src[q];
      }
      __threadfence_block();  // (the area is written again)
      pr0 = pairs;
    }
    if (pr0 < kPairs && p_sum > 0) direct((uint32_t*)s_area[slot][wave], excl, g0, pr0);
  };

  if (t == 0) s_next[0] = atomicAdd(a.ticket, kTicketGroups);
  __syncthreads();
  for (uint32_t k = 0;; ++k) {
    const uint32_t slot = k & 1u;
    const uint32_t tk = __builtin_amdgcn_readfirstlane(s_next[slot]);
    const bool more = (uint64_t)tk < a.gsize;
    uint32_t ex = 0, exlo = 0;
    if (more) {
      const uint64_t g0 = (uint64_t)tk + wave * kAdmTicketGroups;
      uint8_t* const area = (uint8_t*)s_area[slot][wave];
      bool over = false;
      auto pair = [&](uint32_t pr, const LaneRaw& cur, auto full) {
        constexpr bool FULL = decltype(full)::value;
        const uint64_t g = g0 + 2 * pr + half;
        uint32_t v[kAdmChunk], codes[4];
        const uint32_t cnt = cur.cnt;
        const uint32_t c = unpack_center<FULL>(a, cur, v);
        uint64_t word = 0;
        uint32_t bo;
        bool narrow = false;
        if constexpr (FULL) narrow = __ballot(!map_lane_word(v, c, codes, word, bo)) == 0;
        else bo = map_lane<false>(v, cnt, c, codes, nullptr);
        if (bo > 8 * kAdmLaneBytes) over = true;
        uint32_t m = half_max(cnt ? (bo + 7u) / 8u : 0u);
        if (m > kAdmLaneBytes) m = kAdmLaneBytes;
        if (cnt == kAdmChunk) {
          *(uint4*)(a.codes + cur.base) = make_uint4(codes[0], codes[1], codes[2], codes[3]);
        } else {
          for (uint32_t i = 0; i < cnt; ++i) a.codes[cur.base + i] = (uint8_t)(codes[i >> 2] >> (8 * (i & 3)));
        }
        if (g < a.gsize && lin == 0) a.centers[g] = (uint16_t)c;
        const uint32_t m0 = __builtin_amdgcn_readlane(m, 0), m1 = __builtin_amdgcn_readlane(m, 32);
        const uint32_t at = 32u * (ex + (half ? m0 : 0u)) + lin * m;  // this lane's bytes in the area
        // (the pairs that fit are the first ones: the sum only grows)
        const bool fits = 32u * (ex + m0 + m1) <= kAreaBytes;
        if (fits && narrow) {
          // the byte that holds bit bo, if the lane has one: ones from there
          if (bo < 8u * m) word |= ((1ull << (8u - (bo & 7u))) - 1u) << (63u - (bo | 7u));
          word = __builtin_bswap64(word);
          const uint32_t mm = m0 > m1 ? m0 : m1;
          for (uint32_t j = 0; j < mm; ++j) {
            if (j < m) area[at + j] = (uint8_t)word;
            word >>= 8;
          }
        } else if (fits) {
          for (uint32_t i = (uint32_t)lane; i < 8u * (m0 + m1); i += 64u) ((uint32_t*)area)[8u * ex + i] = 0;
          __threadfence_block();
          uint32_t p = 0;  // bit of the lane, `at` bytes into the area
          auto set = [&](uint32_t bit, uint32_t byte_bits) {
            const uint32_t y = at + (bit >> 3);
            atomicOr((uint32_t*)area + (y >> 2), byte_bits << (8u * (y & 3u)));
          };
#pragma unroll
          for (int i = 0; i < (int)kAdmChunk; ++i) {
            const bool ok = (uint32_t)i < cnt;
            const uint32_t d = v[i] > c ? v[i] - c : c - v[i];
            if (ok && p < 8u * m) set(p, 128u >> (p & 7u));
            p += ok ? (d == 0 ? 1u : (d + kAdmMod - 1) / kAdmMod) : 0u;
          }
          if (cnt && p < 8u * m) set(p, 0xffu >> (p & 7u));
        }
        exlo = (uint32_t)lane == 2 * pr ? ex : exlo;
        exlo = (uint32_t)lane == 2 * pr + 1 ? ex + m0 : exlo;
        ex += m0 + m1;
      };
      // two buffers used in turn (no register copy between them, so the next
      // pair's loads stay in flight while a pair is mapped)
      auto pass = [&](auto full) {
        constexpr bool FULL = decltype(full)::value;
        LaneRaw ra = raw_lane<FULL>(a, g0 + half, lin), rb;
        for (uint32_t pr = 0; pr < kPairs; pr += 2) {
          rb = raw_lane<FULL>(a, g0 + 2 * (pr + 1) + half, lin);
          pair(pr, ra, full);
          if (pr + 2 < kPairs) ra = raw_lane<FULL>(a, g0 + 2 * (pr + 2) + half, lin);
          pair(pr + 1, rb, full);
        }
      };
      // (before the input's end: whole lanes only)
      if ((g0 + kAdmTicketGroups) * kAdmGroup <= a.n) pass(std::true_type{});
      else pass(std::false_type{});
      if (__ballot(over) && lane == 0) atomicOr(a.err, kErrAdmDomain);
      if (lane == 0) s_sum[slot][wave] = ex;
      // (not earlier: a ticket held long before it is mapped keeps those
      // after it waiting)
      if (t == 0) s_next[slot ^ 1u] = atomicAdd(a.ticket, kTicketGroups);
    }
    __threadfence_block();
    __syncthreads();
    uint32_t agg = 0, off = 0;
    if (more) {
#pragma unroll
      for (uint32_t w = 0; w < (uint32_t)kWaves; ++w) {
        const uint32_t v = __builtin_amdgcn_readfirstlane(s_sum[slot][w]);
        off += w < wave ? v : 0u;
        agg += v;
      }
      if (wave == 0) publish_aggregate(a.status, tk / kTicketGroups, agg, lane);
    }
    if (pend) finish_pending(slot ^ 1u);
    if (!more) break;
    pend = true;
    p_tk = tk;
    p_agg = agg;
    p_off = off;
    p_sum = ex;
    p_exlo = exlo;
  }
}

__global__ __launch_bounds__(kThreads) void adm_unmap_kernel(AdmUnmapArgs a) {
  __shared__ uint8_t s_sig[kThreads][kAdmChunk];
  const int t = threadIdx.x;
  const uint64_t nlanes = (uint64_t)gridDim.x * kThreads;
  for (uint64_t li = (uint64_t)blockIdx.x * kThreads + t; li < a.gsize * kAdmLanes; li += nlanes) {
    const uint64_t base = li * kAdmChunk;
    if (base >= a.n) continue;
    const uint32_t cnt = (uint32_t)((a.n - base) < kAdmChunk ? (a.n - base) : kAdmChunk);
    const uint8_t* cp = a.codes + base;
    uint32_t cw[4];
    if (cnt == kAdmChunk) {
      const uint4 q = *(const uint4*)cp;
      cw[0] = q.x; cw[1] = q.y; cw[2] = q.z; cw[3] = q.w;
    } else {
      for (int i = 0; i < 4; ++i) cw[i] = 0;
      for (uint32_t i = 0; i < cnt; ++i) cw[i >> 2] |= (uint32_t)cp[i] << (8 * (i & 3));
    }
    adm_restore_lane(a, li, cnt, cw, s_sig[t]);
  }
}

}  // namespace

hipError_t launch_adm_map(const AdmMapArgs& a, int cu, hipStream_t s) {
  if (a.gsize == 0) return hipSuccess;
  int per_cu = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, adm_map_kernel, kThreads, 0);
  if (e != hipSuccess) return e;
  if (per_cu < 1) per_cu = 1;
  uint64_t grid = div_up(a.gsize, kTicketGroups);
  const uint64_t cap = (uint64_t)cu * per_cu;
  if (grid > cap) grid = cap;
  hipLaunchKernelGGL(adm_map_kernel, dim3((uint32_t)grid), dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_adm_unmap(const AdmUnmapArgs& a, hipStream_t s) {
  if (a.gsize == 0) return hipSuccess;
  uint64_t grid = div_up(a.gsize * kAdmLanes, kThreads);
  if (grid > 8192) grid = 8192;
  hipLaunchKernelGGL(adm_unmap_kernel, dim3((uint32_t)grid), dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

}  // namespace mans
