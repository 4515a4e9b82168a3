// codec_device.hpp -- device-side pieces shared by the single-buffer and
// batched rANS kernels: the per-symbol encode and decode steps, the
// decoupled look-back, and the staging bound.
#pragma once
#include "mans_internal.hpp"

namespace mans {

template <int S> struct ElemOf;
template <> struct ElemOf<1> { using T = uint8_t; };
template <> struct ElemOf<2> { using T = uint16_t; };
template <> struct ElemOf<4> { using T = uint32_t; };

constexpr uint64_t kFlagAgg = 1ull << 62;
constexpr uint64_t kFlagPrefix = 2ull << 62;
constexpr uint64_t kValueMask = (1ull << 62) - 1;

// Words per chain per wavefront of one unit at most: 64 lanes x 128 symbols
// (one native unit, or two 32-lane reference units, one per half), rounded
// to 16 words so every area is 32-byte aligned.
template <int PB>
constexpr uint32_t chain_stage_words() {
  return (uint32_t)round_up(64ull * lane_max_words(128u, PB), 16u);
}

// One symbol of one chain with its table entry e already in registers.  The
// emit is branch-free: every lane stores, lanes that emit nothing store into
// their own dummy slot, so the steps of several chains can be interleaved by
// the scheduler (the table reads of the next step are issued before these
// stores; no wait on the LDS counter sits between them).  Slots are u16
// indices from the wave's staging base wbase: an emitted word goes to soff
// (the chain's region) + ((cnt + rank) & MASK), where cnt is the unit's words
// so far (wave-uniform in the 64-lane format) and rank the number of
// emitting lanes of its unit below it; a lane that emits nothing writes its
// dummy slot doff.
template <int L, uint32_t MASK>
__device__ __forceinline__ void enc_step(uint32_t& x, uint32_t& cnt, uint16_t* wbase, uint32_t soff, uint32_t doff,
                                         const uint4& e, bool v, uint32_t half) {
  const bool w = v && (x >= e.x);
  const uint64_t m = __ballot(w);
  const uint32_t mlo = (uint32_t)m, mhi = (uint32_t)(m >> 32);
  uint32_t add, below;
  if (L == 64) {
    add = (uint32_t)__popcll(m);
    below = 0;
  } else {
    add = half ? (uint32_t)__popc(mhi) : (uint32_t)__popc(mlo);
    below = half ? (uint32_t)__popc(mlo) : 0u;
  }
  const uint32_t rank = __builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, 0u)) - below;
  // the slot goes through an opaque register so the compiler keeps one
  // unconditional store instead of splitting the select into two branches
  uint32_t slot = w ? soff + ((cnt + rank) & MASK) : doff;
  __asm__ volatile("" : "+v"(slot));
  wbase[slot] = (uint16_t)x;
  x = w ? x >> 16 : x;
  cnt += add;
  const uint32_t q = (__umulhi(x, e.y) + x) >> (e.z & 31u);
  const uint32_t xn = __umul24(q, e.w) + x + (e.z >> 8);
  x = v ? xn : x;
}

typedef __attribute__((address_space(3))) uint16_t lds_u16;

// LDS byte address of a generic pointer into shared memory.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// Encoder table entry of the multi-chain coders for probability precision p,
// 8 bytes, from a normalised symbol {pdf, cdf, magic, shift}:
//   x = (2^p - pdf) << 16 | cdf << 5 | s,   s = ceil(log2 pdf)
//   y = m = ceil(2^(31 + s) / pdf)
// (2^p - pdf and cdf are below 2^11 and s <= 11; a shift by x takes its low
// five bits, s.)  floor(floor(2 x m / 2^32) / 2^s) = floor(x / pdf) for every
// x < 2^31: with e = m pdf - 2^(31 + s) < pdf <= 2^s, x m / 2^(31 + s) =
// x / pdf + x e / (pdf 2^(31 + s)), and the second term is below 1 / pdf.
// The reference's magic (GpuANSCodec.h:36-61) is floor(2^32 (2^s - pdf) / pdf)
// + 1, so m = 2^31 + ceil(magic / 2) (for a power of two one more than the
// ceiling: then e = 2^s, still below since x < 2^31).
// (16-byte entries took 12 LDS cycles a wave read on random symbols, these 7.)
__device__ __forceinline__ uint2 enc_entry(const uint4& t, int p) {
  return make_uint2((((1u << p) - t.x) << 16) | (t.y << 5) | t.w, 0x80000000u + (t.z >> 1) + (t.z & 1u));
}

// floor(x / pdf) for the entry e.  (The doubling as v_add_u32: the compiler
// would pick a shift.)
__device__ __forceinline__ uint32_t enc_quot(uint32_t x, const uint2& e) {
  uint32_t x2;
  __asm__("v_add_u32 %0, %1, %1" : "=v"(x2) : "v"(x));
  return __umulhi(x2, e.y) >> (e.x & 31u);
}
// The next state q 2^p + (x - q pdf) + cdf of a renormalised state x with
// quotient q = x / pdf (below 2^22).
__device__ __forceinline__ uint32_t enc_next(uint32_t x, uint32_t q, const uint2& e) {
  uint32_t qf;
  __asm__("v_mul_u32_u24_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1"
          : "=v"(qf)
          : "v"(q), "v"(e.x));
  return qf + x + ((e.x >> 5) & 0x7ffu);
}

// sbase += 2 * popcount(m) in two scalar instructions
__device__ __forceinline__ void advance2(uint32_t& sbase, uint64_t m) {
  uint32_t c;
  // (the compiler cannot always see that the base is wave-uniform)
  sbase = __builtin_amdgcn_readfirstlane(sbase);
  __asm__("s_bcnt1_i32_b64 %0, %1" : "=s"(c) : "s"(m) : "scc");
  __asm__("s_lshl1_add_u32 %0, %1, %0" : "+s"(sbase) : "s"(c) : "scc");
}

// Emits and renormalises CH chains: chain c's lanes in m[c] store the low half
// of x[c] at LDS byte address addr[c] and shift x[c] and its quotient q[c]
// right by 16 (floor((x >> 16) / pdf) = floor(x / pdf) >> 16).  exec is
// narrowed per chain and set back to all lanes (every caller runs whole
// wavefronts, with no lane masked off); s_mov does not write SCC.
template <int CH>
__device__ __forceinline__ void emit_renorm(const uint64_t (&m)[CH], const uint32_t (&addr)[CH], uint32_t (&x)[CH],
                                            uint32_t (&q)[CH]) {
  static_assert(CH == 1 || CH == 2 || CH == 4, "chains per lane");
  if constexpr (CH == 1) {
    __asm__ volatile(
        "s_mov_b64 exec, %2\n\tds_write_b16 %3, %0\n\tv_lshrrev_b32 %0, 16, %0\n\tv_lshrrev_b32 %1, 16, %1\n\t"
        "s_mov_b64 exec, -1"
        : "+v"(x[0]), "+v"(q[0])
        : "s"(m[0]), "v"(addr[0])
        : "memory");
  } else {
#pragma unroll
    for (int c = 0; c < CH; c += 2)
      __asm__ volatile(
          "s_mov_b64 exec, %4\n\tds_write_b16 %5, %0\n\tv_lshrrev_b32 %0, 16, %0\n\tv_lshrrev_b32 %1, 16, %1\n\t"
          "s_mov_b64 exec, %6\n\tds_write_b16 %7, %2\n\tv_lshrrev_b32 %2, 16, %2\n\tv_lshrrev_b32 %3, 16, %3\n\t"
          "s_mov_b64 exec, -1"
          : "+v"(x[c]), "+v"(q[c]), "+v"(x[c + 1]), "+v"(q[c + 1])
          : "s"(m[c]), "v"(addr[c]), "s"(m[c + 1]), "v"(addr[c + 1])
          : "memory");
  }
}

// One symbol of each of CH chains in the 64-lane format with linear stages,
// table entries e (enc_entry).  A lane emits when its state is at or above
// pdf << (31 - p), that is when its quotient has reached 2^(31 - p).  Chain
// c's emitted words go to LDS byte address sb[c] + 2 * rank, sb[c] (wave
// uniform) where the chain's next word goes and rank the number of emitting
// lanes below this one; sb[c] advances by two bytes per emitted word.  The
// phases (quotients and emitting lanes; ranks; stores and renormalisation;
// next states) each run over all chains, so the dependent operations of one
// chain have the others' between them.  13 vector operations a symbol bound
// the step (about 4.2 cycles each per SIMD).  FULL: every lane codes a
// symbol; else lanes with v[c] false keep their state and emit nothing.
template <int PB, int CH, bool FULL = true>
__device__ __forceinline__ void enc_steps64(uint32_t (&x)[CH], uint32_t (&sb)[CH], const uint2 (&e)[CH],
                                            const bool (&v)[CH]) {
  uint64_t m[CH];
  uint32_t q[CH], addr[CH], x0[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    q[c] = enc_quot(x[c], e[c]);
    m[c] = __ballot((FULL || v[c]) && q[c] >= (1u << (31 - PB)));
    x0[c] = x[c];
  }
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const uint32_t rank =
        __builtin_amdgcn_mbcnt_hi((uint32_t)(m[c] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m[c], 0u));
    addr[c] = sb[c] + 2u * rank;
  }
  emit_renorm<CH>(m, addr, x, q);
#pragma unroll
  for (int c = 0; c < CH; ++c) advance2(sb[c], m[c]);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const uint32_t xn = enc_next(x[c], q[c], e[c]);
    x[c] = FULL || v[c] ? xn : x0[c];
  }
}

// The 32-lane format on a 64-lane wavefront: lanes 0-31 code one unit of a
// chain and lanes 32-63 another (halfv = 0 / 1 per lane), each unit with its
// own stage.  An emitted word of the lower half goes to sbA + 2 * rank, one
// of the upper half to sbB + 2 * (rank - emitters of the lower half); the two
// bases are scalars, the per-lane choice one 24-bit multiply-add:
// emit = (sbA + 2 rank) + halfv * (sbB - sbA - 2 lo).
__device__ __forceinline__ uint32_t emit32(uint64_t m, uint32_t& sbA, uint32_t& sbB, uint32_t halfv) {
  const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  const uint32_t lo = (uint32_t)__popc((uint32_t)m), hi = (uint32_t)__popc((uint32_t)(m >> 32));
  const uint32_t a2 = __builtin_amdgcn_readfirstlane(sbA + 2u * lo);
  const int32_t delta = (int32_t)(sbB - a2);
  const uint32_t emit = (uint32_t)((int32_t)(sbA + 2u * rank) + __mul24((int32_t)halfv, delta));
  sbA = a2;
  sbB = __builtin_amdgcn_readfirstlane(sbB + 2u * hi);
  return emit;
}

// enc_steps64 for the 32-lane format: chain c's lower half advances sb[c],
// its upper half sb[CH + c].
template <int PB, int CH, bool FULL = true>
__device__ __forceinline__ void enc_steps32(uint32_t (&x)[CH], uint32_t (&sb)[2 * CH], uint32_t halfv,
                                            const uint2 (&e)[CH], const bool (&v)[CH]) {
  uint64_t m[CH];
  uint32_t q[CH], addr[CH], x0[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    q[c] = enc_quot(x[c], e[c]);
    m[c] = __ballot((FULL || v[c]) && q[c] >= (1u << (31 - PB)));
    x0[c] = x[c];
  }
#pragma unroll
  for (int c = 0; c < CH; ++c) addr[c] = emit32(m[c], sb[c], sb[CH + c], halfv);
  emit_renorm<CH>(m, addr, x, q);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const uint32_t xn = enc_next(x[c], q[c], e[c]);
    x[c] = FULL || v[c] ? xn : x0[c];
  }
}

// 8 * byte B of w: a byte offset into a table of 8-byte entries.
template <int B>
__device__ __forceinline__ uint32_t byte_x8(uint32_t w) {
  uint32_t r;
  if constexpr (B == 0)
    __asm__("v_lshlrev_b32_sdwa %0, 3, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_0"
            : "=v"(r) : "v"(w));
  else if constexpr (B == 1)
    __asm__("v_lshlrev_b32_sdwa %0, 3, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_1"
            : "=v"(r) : "v"(w));
  else if constexpr (B == 2)
    __asm__("v_lshlrev_b32_sdwa %0, 3, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2"
            : "=v"(r) : "v"(w));
  else
    __asm__("v_lshlrev_b32_sdwa %0, 3, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_3"
            : "=v"(r) : "v"(w));
  return r;
}

__device__ __forceinline__ uint64_t wave_sum(uint64_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Sum of the aggregates of status entries j, j - 1, ... back to and including
// the nearest inclusive prefix (entries below `first` read as a zero prefix).
// Lane l reads entries j - l - 64 k, k < K: 64 K entries per round trip.
// Groups of 64 are taken in order; a group with an unpublished entry before
// its nearest prefix ends the round (the groups before it are kept) and the
// wave sleeps briefly before reading again; with TRY it returns ~0 instead
// (an entry still unpublished: the caller resolves later).  dec(raw, flag,
// value) splits a status word (flag 0: not yet published, 1: aggregate,
// 2: inclusive prefix).
template <int K, bool TRY = false, typename Dec>
__device__ __forceinline__ uint64_t look_back_window(const uint64_t* status, int64_t j, int64_t first,
                                                     uint64_t zero_prefix, int lane, Dec dec) {
  uint64_t excl = 0;
  for (;;) {
    uint64_t raw[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t i = j - lane - 64 * k;
      raw[k] = i >= first ? __hip_atomic_load(status + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : zero_prefix;
    }
    uint64_t part = 0;
    int groups = 0;
    bool found = false;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      uint32_t f;
      uint64_t val;
      dec(raw[k], f, val);
      const uint64_t pm = __ballot(f == 2), nm = __ballot(f == 0);
      // lanes up to and including the nearest prefix (all 64 if none)
      const uint64_t upto = pm ? (pm & (0 - pm)) * 2u - 1u : ~0ull;
      if (nm & upto) {
        if constexpr (TRY) return ~0ull;
        break;
      }
      part += ((upto >> lane) & 1u) ? val : 0u;
      ++groups;
      if (pm) {
        found = true;
        break;
      }
    }
    excl += wave_sum(part);
    if (found) return excl;
    j -= 64 * groups;
    if (groups < K) __builtin_amdgcn_s_sleep(1);
  }
}

// First half of a look-back: publish entry `chain`'s own count (the first
// entry's is already its inclusive prefix).
__device__ __forceinline__ void publish_aggregate(uint64_t* status, uint64_t chain, uint64_t agg, int lane) {
  if (lane == 0)
    __hip_atomic_store(status + chain, (chain == 0 ? kFlagPrefix : kFlagAgg) | agg, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
// Second half: sum the predecessors back to the nearest published prefix,
// publish this entry's inclusive prefix and return the exclusive one.  Any
// time may pass between the two halves; the predecessors only need to have
// published their aggregates.  K groups of 64 entries per round trip.
template <int K = 8>
__device__ __forceinline__ uint64_t resolve_prefix(uint64_t* status, uint64_t chain, uint64_t agg, int lane) {
  if (chain == 0) return 0;
  const uint64_t excl = look_back_window<K>(status, (int64_t)chain - 1, 0, kFlagPrefix, lane,
                                            [](uint64_t v, uint32_t& f, uint64_t& val) {
                                              f = (uint32_t)(v >> 62);
                                              val = v & kValueMask;
                                            });
  if (lane == 0)
    __hip_atomic_store(status + chain, kFlagPrefix | (excl + agg), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return excl;
}
// Decoupled look-back for ticket group `chain` with aggregate agg (all
// lanes): publishes the aggregate, sums predecessors back to the nearest
// inclusive prefix (512 per round trip), publishes this group's inclusive
// prefix and returns the exclusive one.  Each status word holds its flag and
// value together and carries nothing else, so relaxed device-scope atomics
// suffice (release / acquire at agent scope would write back / invalidate
// the XCD's whole L2 on every publish and poll).
__device__ __forceinline__ uint64_t look_back(uint64_t* status, uint64_t chain, uint64_t agg, int lane) {
  publish_aggregate(status, chain, agg, lane);
  return resolve_prefix(status, chain, agg, lane);
}

// One symbol of each of the CH chains; returns the CH decoded bytes packed
// into an element.  Every lane reads a word (no branch, so the chains'
// steps interleave): lanes that take none read some in-range slot and keep
// their state.  ptr (words of the unit not yet taken) never drops below a
// step's count on a valid stream; on a corrupt one it is clamped at 0 so
// every read stays inside the stage, and `taken` (the words taken so far)
// then ends above the unit's word count.  Word i of a unit sits at
// stage[i & MASK] (MASK = R - 1 for a ring, all ones for a whole-unit
// stage); a step reads stage[(base & MASK) + rank] with rank <= 64, which the
// ring's mirror covers.  The three phases (LUT reads; state update and word
// reads; selects) each run over all chains, so one chain's LDS latency
// overlaps the others' work.
// Decoder LUT entries.  uint2 {pdf | sym << 24, slot - cdf}: the 24-bit
// multiply ignores the symbol byte, so the update is one shift and one
// multiply-add.  uint32_t (slot - cdf) << 20 | pdf << 8 | sym: half the LDS,
// two more operations per symbol.
template <int PB>
__device__ __forceinline__ uint32_t lut_next(uint2 e, uint32_t x) { return __umul24(e.x, x >> PB) + e.y; }
template <int PB>
__device__ __forceinline__ uint32_t lut_next(uint32_t e, uint32_t x) {
  return __umul24((e >> 8) & 0xfffu, x >> PB) + (e >> 20);
}
__device__ __forceinline__ uint32_t lut_sym(uint2 e) { return e.x >> 24; }
__device__ __forceinline__ uint32_t lut_sym(uint32_t e) { return e & 0xffu; }
// The CH decoded symbols packed into an element (chain c's byte at bits
// 8c..8c+7) with byte permutes: a uint2 entry's symbol is byte 3 of e.x, a
// uint32_t entry's byte 0.  v_perm selector bytes 0-3 pick the second
// operand's bytes, 4-7 the first's, 0x0c gives zero.
__device__ __forceinline__ uint32_t sym_word(uint2 e) { return e.x; }
__device__ __forceinline__ uint32_t sym_word(uint32_t e) { return e; }
template <typename LE>
constexpr uint32_t sym_byte() { return sizeof(LE) == 8 ? 3u : 0u; }
template <int CH, typename LE>
__device__ __forceinline__ uint32_t pack_syms(const LE (&e)[CH]) {
  constexpr uint32_t b = sym_byte<LE>();
  if constexpr (CH == 1) {
    return lut_sym(e[0]);
  } else if constexpr (CH == 2) {
    return __builtin_amdgcn_perm(sym_word(e[1]), sym_word(e[0]), 0x0c0c0000u | ((4u + b) << 8) | b);
  } else if constexpr (CH == 4) {
    const uint32_t lo = __builtin_amdgcn_perm(sym_word(e[1]), sym_word(e[0]), 0x0c0c0000u | ((4u + b) << 8) | b);
    const uint32_t hi = __builtin_amdgcn_perm(sym_word(e[3]), sym_word(e[2]), ((4u + b) << 24) | (b << 16) | 0x0c0cu);
    return lo | hi;
  } else {
    uint32_t el = 0;
#pragma unroll
    for (int c = 0; c < CH; ++c) el |= lut_sym(e[c]) << (8 * c);
    return el;
  }
}

// CLAMP: ptr stops at 0 (whole-unit stages, where a read past the unit's
// words must stay inside the stage); without it (rings, every read masked
// into the ring) ptr goes below 0 on a corrupt stream and stays there, and
// `taken` is not kept.
template <int L, int PB, int CH, uint32_t MASK, typename LE = uint2, bool CLAMP = true>
__device__ __forceinline__ uint32_t dec_steps(uint32_t (&x)[CH], uint32_t (&ptr)[CH], uint32_t (&taken)[CH],
                                              const LE* const (&lut)[CH], const uint16_t* const (&stage)[CH],
                                              const bool (&v)[CH], uint32_t half) {
  constexpr uint32_t W = 1u << PB;
  LE e[CH];
  uint32_t word[CH];
  bool r[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) e[c] = lut[c][x[c] & (W - 1u)];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const uint32_t xn = lut_next<PB>(e[c], x[c]);
    x[c] = v[c] ? xn : x[c];
    r[c] = v[c] && (x[c] < kMinState);
    const uint64_t m = __ballot(r[c]);
    const uint32_t mlo = (uint32_t)m, mhi = (uint32_t)(m >> 32);
    uint32_t cnt, below;
    if (L == 64) {
      cnt = (uint32_t)__popcll(m);
      below = 0;
    } else {
      cnt = half ? (uint32_t)__popc(mhi) : (uint32_t)__popc(mlo);
      below = half ? (uint32_t)__popc(mlo) : 0u;
    }
    uint32_t base;
    if constexpr (CLAMP) {
      taken[c] += cnt;
      // ptr < 2^16 and cnt <= 64: a signed max keeps this scalar (s_max_i32)
      const int32_t bd = (int32_t)ptr[c] - (int32_t)cnt;
      base = (uint32_t)(bd > 0 ? bd : 0);
    } else {
      base = ptr[c] - cnt;
    }
    // slot of this lane's word: (base & MASK) + rank, the base taken in as
    // mbcnt's accumulator (no scalar shift / add for the address)
    const uint32_t slot = __builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, base & MASK)) - below;
    word[c] = stage[c][slot];
    ptr[c] = base;
  }
  // keep the reads unconditional: without this the compiler moves each under
  // its `r` and puts a branch between the chains
#pragma unroll
  for (int c = 0; c < CH; ++c) __asm__ volatile("" : "+v"(word[c]));
#pragma unroll
  for (int c = 0; c < CH; ++c) x[c] = r[c] ? (x[c] << 16) | word[c] : x[c];
  return pack_syms<CH>(e);
}

// Sum of a 32-bit value over the 64 lanes (every lane gets it).
__device__ __forceinline__ uint32_t wave_sum32(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Normalisation of one plane, by a wavefront whose lane l owns symbols 4l ..
// 4l + 3 (element j is symbol 4l + j).  Restates GpuANSStatistics.h:186-385
// exactly, in three parts:
//  * quantize_syms: q = (u32)(float(2^p) * (float(count) / float(total))),
//    IEEE round to nearest on both operations, truncating conversion; present
//    symbols get at least 1.  Returns their sum;
//  * rank_syms: rank = position of (q << 16 | s) in descending order, the
//    number of the keys [k0, k1) (multiples of 4) above this lane's;
//  * settle_syms: with the sum below 2^p, q[s] += diff / 256 + (s < diff %
//    256) (the reference's repeated "+1 to symbol ids < min(diff, 256)"
//    loop); above, repeatedly G = #{q > 1}, it = min(diff, G), one subtracted
//    at the ranks [G - it, G) of the original order.  Then cdf = exclusive
//    scan in symbol order, shift = 32 - clz(pdf - 1), magic = 2^32 (2^shift -
//    pdf) / pdf + 1 (0 for pdf == 0), giving {pdf, cdf, magic, shift}.
__device__ __forceinline__ uint32_t quantize_syms(const uint32_t (&count)[4], uint32_t total, int p, uint32_t (&q)[4],
                                                  uint32_t (&key)[4]) {
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t qs = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float ratio = __fdiv_rn((float)count[j], (float)total);
    const float prod = __fmul_rn((float)(1u << p), ratio);
    q[j] = (uint32_t)prod;
    if (count[j] > 0 && q[j] == 0) q[j] = 1;
    qs += q[j];
    key[j] = (q[j] << 16) | (4u * lane + (uint32_t)j);
  }
  return wave_sum32(qs);
}
__device__ __forceinline__ void rank_syms(const uint32_t (&key)[4], const uint32_t* s_keys, uint32_t k0, uint32_t k1,
                                          uint32_t (&rank)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) rank[j] = 0;
#pragma unroll 4
  for (uint32_t i = k0; i < k1; i += 4) {
    const uint4 k = *(const uint4*)(s_keys + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) rank[j] += (k.x > key[j]) + (k.y > key[j]) + (k.z > key[j]) + (k.w > key[j]);
  }
}
__device__ __forceinline__ void settle_syms(uint32_t (&q)[4], uint32_t qsum, const uint32_t (&rank)[4], int p,
                                            uint4 (&out)[4], bool& bad) {
  const uint32_t lane = threadIdx.x & 63u;
  const int diff = (1 << p) - (int)qsum;
  if (diff > 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) q[j] += (uint32_t)(diff >> 8) + ((4u * lane + (uint32_t)j < (uint32_t)(diff & 255)) ? 1u : 0u);
  } else if (diff < 0) {
    int d = -diff;
    while (d > 0) {
      uint32_t gl = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) gl += q[j] > 1 ? 1u : 0u;
      const int g = (int)wave_sum32(gl);
      const int it = d < g ? d : g;
      if (it <= 0) {
        bad = true;
        break;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if ((int)rank[j] >= g - it && (int)rank[j] < g) q[j] -= 1;
      d -= it;
    }
  }
  // exclusive scan in symbol order: lane sums, then a wave scan
  const uint32_t ls = q[0] + q[1] + q[2] + q[3];
  uint32_t inc = ls;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(inc, o, 64);
    if (lane >= (uint32_t)o) inc += u;
  }
  uint32_t cdf = inc - ls;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t pdf = q[j];
    uint32_t shift = 0, magic = 0;
    if (pdf > 0) {
      shift = 32u - (uint32_t)__clz((int)(pdf - 1u));
      const uint64_t m = ((1ull << 32) * ((1ull << shift) - pdf)) / pdf + 1ull;
      magic = (uint32_t)m;
    }
    out[j] = make_uint4(pdf, cdf, magic, shift);
    cdf += pdf;
  }
}

// Normalises one plane with a single wavefront.  s_keys: 256 words of this
// wave's LDS (16-byte aligned).
__device__ inline void normalize_wave(const uint32_t (&count)[4], uint32_t total, int p, uint32_t* s_keys,
                                      uint4 (&out)[4], bool& bad) {
  const uint32_t lane = threadIdx.x & 63u;
  if (total == 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = make_uint4(0, 0, 0, 0);
    return;
  }
  uint32_t q[4], key[4], rank[4] = {0, 0, 0, 0};
  const uint32_t qsum = quantize_syms(count, total, p, q, key);
  if (qsum > (1u << p)) {  // (the ranks are needed only to take some away)
#pragma unroll
    for (int j = 0; j < 4; ++j) s_keys[4u * lane + (uint32_t)j] = key[j];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    rank_syms(key, s_keys, 0, kNumSymbols, rank);
  }
  settle_syms(q, qsum, rank, p, out, bad);
}

}  // namespace mans
