// adm_device.hpp -- the ADM restore of one 16-element lane (the unmap
// kernel's per-thread work), split so that the bit bytes, center and codes
// may come from global memory or LDS.  mappingcpuV1.cpp:195-276;
// mappingV15_fused_uint16.cu:24-121.
#pragma once
#include "mans_internal.hpp"

namespace mans {

__device__ __forceinline__ uint32_t adm_clz(uint32_t w) { return (uint32_t)__builtin_clz(w); }
__device__ __forceinline__ uint32_t adm_clz(uint64_t w) { return (uint32_t)__builtin_clzll(w); }
// The element of code byte `code` with signal `sig` around center c.
__device__ __forceinline__ uint32_t adm_element(uint32_t code, uint32_t sig, uint32_t c) {
  const uint32_t d = (code >> 1) + kAdmMod * sig;
  const uint32_t below = 0u - (code & 1u);
  return ((d ^ below) + (c - below)) & 0xffffu;  // c - d or c + d
}
// A lane's elements (two per word of o) from its bits in w, the first on top,
// with a one right after the last.  mappingcpuV1.cpp:233-243: the zeros after
// the i-th one are signal[i]; the one past the end closes the last signal,
// and what has no one before it stays 0.
template <typename W>
__device__ __forceinline__ void adm_restore_word(W w, uint32_t c, const uint32_t (&cw)[4], uint32_t (&o)[8]) {
  w = (w << adm_clz(w)) << 1;  // (w has a one)
#pragma unroll
  for (int i = 0; i < (int)kAdmChunk; ++i) {
    const uint32_t sig = w ? adm_clz(w) : 0u;
    w = (w << sig) << 1;
    const uint32_t x = adm_element((cw[i >> 2] >> (8 * (i & 3))) & 0xffu, sig & 0xffu, c);
    if (i & 1) o[i >> 1] |= x << 16; else o[i >> 1] = x;
  }
}

// Restores the cnt elements at out from the lane's m bytes of the bit plane
// at src (global memory or LDS): parses them into per-element signals and
// sets x = c + d or c - d with d = code / 2 + 126 signal (code & 1: below
// the center).  cw holds the 16 code bytes, little endian; sig is 16 bytes
// of this lane's own LDS scratch.  Lanes of at most 7 bytes, nearly all (16
// elements without signals take 2), are parsed in a register; by words in LDS
// as the longer ones, 512 MiB took 215 us instead of 188.
__device__ inline void adm_restore_core(uint32_t m, const uint8_t* src, uint32_t c, uint32_t cnt,
                                        const uint32_t (&cw)[4], uint8_t* sig, uint16_t* out) {
  uint32_t o[8];
  auto store = [&]() {
    if (cnt == kAdmChunk) {
      uint4* op = (uint4*)out;
      op[0] = make_uint4(o[0], o[1], o[2], o[3]);
      op[1] = make_uint4(o[4], o[5], o[6], o[7]);
    } else {
      for (uint32_t i = 0; i < cnt; ++i) out[i] = (uint16_t)(o[i >> 1] >> (16 * (i & 1)));
    }
  };
  if (m <= 3) {
    uint32_t v = 0x80000000u >> (8u * m);
    if (m > 0) v |= (uint32_t)src[0] << 24;
    if (m > 1) v |= (uint32_t)src[1] << 16;
    if (m > 2) v |= (uint32_t)src[2] << 8;
    adm_restore_word(v, c, cw, o);
    store();
    return;
  }
  if (m <= 7) {
    uint64_t v = (1ull << 63) >> (8u * m);
#pragma unroll
    for (uint32_t i = 0; i < 7; ++i) v |= (uint64_t)(i < m ? src[i] : 0u) << (56u - 8u * i);
    adm_restore_word(v, c, cw, o);
    store();
    return;
  }
  uint32_t w[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    uint32_t v = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint32_t i = 4u * r + b;
      v = (v << 8) | (i < m ? (uint32_t)src[i] : 0u);
    }
    w[r] = v;  // bit position 32r + j is bit (31 - j) of w[r]
  }
#pragma unroll
  for (int i = 0; i < (int)kAdmChunk; ++i) sig[i] = 0;
  // mappingcpuV1.cpp:233-243: a one advances the element index (stop at
  // 16), zeros after the i-th one count into signal[i] (uint8)
  int idx = -1;
  uint32_t prev = 0;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    uint32_t v = w[r];
    while (v != 0 && idx < (int)kAdmChunk) {
      const uint32_t z = (uint32_t)__clz((int)v);
      const uint32_t pos = 32u * r + z;
      if (idx >= 0) sig[idx] = (uint8_t)(pos - prev - 1u);
      ++idx;
      prev = pos;
      v &= ~(0x80000000u >> z);
    }
  }
  if (idx >= 0 && idx < (int)kAdmChunk) sig[idx] = (uint8_t)(8u * m - prev - 1u);
#pragma unroll
  for (int i = 0; i < (int)kAdmChunk; ++i) {
    const uint32_t x = adm_element((cw[i >> 2] >> (8 * (i & 3))) & 0xffu, sig[i], c);
    if (i & 1) o[i >> 1] |= x << 16; else o[i >> 1] = x;
  }
  store();
}

// Offsets o0 = O_g, o1 = O_{g+1} of a group are usable when the lane bytes
// they give fit the lane buffer and the bit plane.
__device__ __forceinline__ bool adm_offsets_ok(int32_t o0, int32_t o1, uint64_t bits_len) {
  return o0 >= 0 && o1 >= o0 && o1 - o0 <= (int32_t)kAdmLaneBytes && 32ull * (uint64_t)o1 <= bits_len;
}

// Lane li of the frame (elements [16 li, 16 li + cnt), group li / 32), all
// inputs from global memory.  Inconsistent offsets raise kErrBlockWords and
// store nothing.
__device__ inline void adm_restore_lane(const AdmUnmapArgs& a, uint64_t li, uint32_t cnt, const uint32_t (&cw)[4],
                                        uint8_t* sig) {
  const uint64_t g = li / kAdmLanes;
  const uint32_t lin = (uint32_t)(li % kAdmLanes);
  const int32_t o0 = a.offsets[g], o1 = a.offsets[g + 1];
  if (!adm_offsets_ok(o0, o1, a.bits_len)) {
    atomicOr(a.err, kErrBlockWords);
    return;
  }
  const uint32_t m = (uint32_t)(o1 - o0);
  adm_restore_core(m, a.bits + 32ull * (uint64_t)o0 + (uint64_t)lin * m, a.centers[g], cnt, cw, sig,
                   a.out + li * kAdmChunk);
}

}  // namespace mans
