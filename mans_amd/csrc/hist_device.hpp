// hist_device.hpp -- byte histograms on the matrix cores, for the histogram
// launch (hist.hip) and the batched encoder's histogram phase.
//
// Let H[h][l] be the number of bytes with high nibble h and low nibble l, and
// g the value of an FP4 (e2m1) number in halves: g = 0 1 2 3 4 6 8 12 for
// codes 0-7, negated for 8-15.  One 16x16x128 FP4 matrix product whose A rows
// hold the high nibbles of 128 bytes, each ORed with its row number i, and
// whose B columns hold the low nibbles ORed with the column number j, adds
//   T[i][j] = sum over bytes of g(h | i) g(l | j) / 4
// and the 16 functions x -> g(x | m) are linearly independent, so H follows
// exactly from T (unmix16, along each axis).  Every term is a multiple of
// 1/4 of at most 36, so a float accumulator holds the exact sum of up to 2^24
// / 144 = 116,508 bytes; it is moved to an integer one long before
// (kTileFloats).
//
// Per 128 bytes and wavefront that is 8 vector operations (an OR with the
// DPP broadcast of one lane's nibbles to its row of 16 lanes) and one product,
// whatever the bytes.  (One LDS atomic a byte, even without conflicts, takes
// 5.0 cycles per 64 bytes and CU, 0.29 ms on 1 GiB; that loop with 64 KiB
// of counters a workgroup also left two workgroups per CU and had 64 KiB
// to clear and merge in every workgroup.)
#pragma once
#include "mans_internal.hpp"

namespace mans {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x8 __attribute__((ext_vector_type(8)));

// A tile is 4 KiB per wavefront: four 16-byte loads a lane.
constexpr uint32_t kTileU4 = 256;
// tiles between two moves to the integer accumulators (64 KiB a wavefront)
constexpr uint32_t kTileFloats = 16;
static_assert(kTileFloats * 4096u <= 116508u, "exact in float");
// tiles of a wavefront between two flushes: 144 per byte, and eight
// wavefronts' sums stay inside int32
constexpr uint32_t kTileFlush = 256;

// The OR of lane N's w (of this lane's row of 16 lanes) with m.
template <int N>
__device__ __forceinline__ int32_t row_or(uint32_t w, uint32_t m) {
  return (int32_t)((uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x150 + N, 0xf, 0xf, true) | m);
}
// The 32 bytes a row's lanes N and N + 1 hold as nibbles (hi, lo: two dwords
// of 8 nibbles each).
template <int N>
__device__ __forceinline__ void count_lanes(const uint32_t (&hi)[2], const uint32_t (&lo)[2], uint32_t m, f32x4& acc) {
  i32x8 a = {}, b = {};
  a[0] = row_or<N>(hi[0], m);
  a[1] = row_or<N>(hi[1], m);
  a[2] = row_or<N + 1>(hi[0], m);
  a[3] = row_or<N + 1>(hi[1], m);
  b[0] = row_or<N>(lo[0], m);
  b[1] = row_or<N>(lo[1], m);
  b[2] = row_or<N + 1>(lo[0], m);
  b[3] = row_or<N + 1>(lo[1], m);
  // formats 4, 4: FP4 both; zero scale operands: the product without scales
  acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, acc, 4, 4, 0, 0, 0, 0);
}
// Every lane's 16 bytes w of one plane (1 KiB of a wavefront).
__device__ __forceinline__ void count_16(const uint32_t (&w)[4], uint32_t m, f32x4& acc) {
  uint32_t hi[2], lo[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const uint32_t w0 = w[2 * q], w1 = w[2 * q + 1];
    hi[q] = ((w0 >> 4) & 0x0f0f0f0fu) | (w1 & 0xf0f0f0f0u);
    lo[q] = (w0 & 0x0f0f0f0fu) | ((w1 << 4) & 0xf0f0f0f0u);
  }
  count_lanes<0>(hi, lo, m, acc);
  count_lanes<2>(hi, lo, m, acc);
  count_lanes<4>(hi, lo, m, acc);
  count_lanes<6>(hi, lo, m, acc);
  count_lanes<8>(hi, lo, m, acc);
  count_lanes<10>(hi, lo, m, acc);
  count_lanes<12>(hi, lo, m, acc);
  count_lanes<14>(hi, lo, m, acc);
}
// A tile of S-byte elements (from an element boundary): byte b of each
// element counted in acc[b].
template <int S>
__device__ __forceinline__ void count_tile(const uint4 (&q)[4], uint32_t m, f32x4 (&acc)[S]) {
  const uint32_t w[16] = {q[0].x, q[0].y, q[0].z, q[0].w, q[1].x, q[1].y, q[1].z, q[1].w,
                          q[2].x, q[2].y, q[2].z, q[2].w, q[3].x, q[3].y, q[3].z, q[3].w};
  if constexpr (S == 1) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t p[4] = {w[4 * u], w[4 * u + 1], w[4 * u + 2], w[4 * u + 3]};
      count_16(p, m, acc[0]);
    }
  } else if constexpr (S == 2) {
    // bytes 0 and 2 (1 and 3) of two dwords
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        uint32_t p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          p[i] = __builtin_amdgcn_perm(w[8 * u + 2 * i + 1], w[8 * u + 2 * i], k ? 0x07050301u : 0x06040200u);
        count_16(p, m, acc[k]);
      }
  } else {
    // byte k of four dwords: pairs first, planes 0 / 1 and 2 / 3 together
    uint32_t p[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t a0 = w[4 * i], a1 = w[4 * i + 1], a2 = w[4 * i + 2], a3 = w[4 * i + 3];
      const uint32_t l0 = __builtin_amdgcn_perm(a1, a0, 0x05010400u), l1 = __builtin_amdgcn_perm(a3, a2, 0x05010400u);
      const uint32_t h0 = __builtin_amdgcn_perm(a1, a0, 0x07030602u), h1 = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
      p[0][i] = __builtin_amdgcn_perm(l1, l0, 0x05040100u);
      p[1][i] = __builtin_amdgcn_perm(l1, l0, 0x07060302u);
      p[2][i] = __builtin_amdgcn_perm(h1, h0, 0x05040100u);
      p[3][i] = __builtin_amdgcn_perm(h1, h0, 0x07060302u);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) count_16(p[k], m, acc[k]);
  }
}

// Tiles t0, t0 + step, ... below t1 of body, counted by one wavefront into
// the integer accumulators sum (element (i, j) of T at lane (i / 4) 16 + j,
// index i % 4).  The next tile's loads are in flight while a tile is counted.
template <int S>
__device__ __forceinline__ void count_tiles(const uint4* body, uint32_t t0, uint32_t t1, uint32_t step,
                                            int32_t (&sum)[S][4]) {
  if (t0 >= t1) return;
  const uint32_t lane = threadIdx.x & 63u, m = (lane & 15u) * 0x11111111u;
  auto load = [&](uint4 (&q)[4], uint32_t t) {
    // (a global pointer: a batch's comes from memory)
    const auto* p = (const __attribute__((address_space(1))) u32x4*)body + (uint64_t)t * kTileU4 + lane;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const u32x4 v = p[64 * u];
      q[u] = make_uint4(v.x, v.y, v.z, v.w);
    }
  };
  f32x4 acc[S];
#pragma unroll
  for (int k = 0; k < S; ++k) acc[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto to_int = [&]() {
#pragma unroll
    for (int k = 0; k < S; ++k) {
#pragma unroll
      for (int v = 0; v < 4; ++v) sum[k][v] += (int32_t)(acc[k][v] * 4.0f);
      acc[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  uint4 qa[4], qb[4];
  load(qa, t0);
  uint32_t held = 0;
  for (uint32_t t = t0;;) {
    // (past the last tile the same one is loaded again: straight-line code)
    load(qb, t + step < t1 ? t + step : t);
    count_tile<S>(qa, m, acc);
    t += step;
    if (t >= t1) break;
    load(qa, t + step < t1 ? t + step : t);
    count_tile<S>(qb, m, acc);
    t += step;
    if (t >= t1) break;
    held += 2;
    if (held >= kTileFloats) {
      to_int();
      held = 0;
    }
  }
  to_int();
}

// One axis of T back to counts, in place: t[m] = sum over x of g(x | m) h[x].
// With d[x] = h[x] - h[x + 8] and e[x] = h[x] + h[x + 8] (x < 8), t[m] = sum
// g(x | m) d[x] and t[m + 8] = -sum g(x | m) e[x].  In y = 7 - x and n = 7 -
// m, g(x | m) = k(y & n) with k = 12 8 6 4 3 2 1 0, and k(y & n) is the sum
// over subsets s of y & n of c[s] (c: k's differences over subsets, below), so
// the differences of t over subsets of n are c[s] times the sum of d[y] over
// y containing s: divided by c[s] exactly, and differenced over supersets,
// they give d.  Sums that wrap around 32 bits on the way come out right: every
// quotient's true value fits.
__device__ __forceinline__ void unmix16(int32_t (&t)[16]) {
  constexpr int32_t c[8] = {12, -4, -6, 2, -9, 3, 4, -2};
  int32_t r[2][8];
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    uint32_t a[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) a[n] = z ? 0u - (uint32_t)t[15 - n] : (uint32_t)t[7 - n];
#pragma unroll
    for (int b = 1; b < 8; b <<= 1)
#pragma unroll
      for (int n = 0; n < 8; ++n)
        if (n & b) a[n] -= a[n ^ b];
#pragma unroll
    for (int n = 0; n < 8; ++n) r[z][n] = (int32_t)a[n] / c[n];
#pragma unroll
    for (int b = 1; b < 8; b <<= 1)
#pragma unroll
      for (int n = 0; n < 8; ++n)
        if (!(n & b)) r[z][n] -= r[z][n | b];
  }
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const int32_t d = r[0][7 - x], e = r[1][7 - x];
    t[x] = (e + d) / 2;
    t[x + 8] = (e - d) / 2;
  }
}

// The workgroup's wavefronts' accumulators to byte counts, added to
// ghist[256 k + byte] for k < S; sum is left zeroed.  lds: S x 256 words, all
// zero or holding counts of single bytes (count_byte) at lds[1024 + ...]; both
// parts are left zeroed.  Every thread of the workgroup (T of them) calls it.
template <int S, int T>
__device__ __forceinline__ void flush_counts(int32_t (&sum)[S][4], uint32_t* lds, uint32_t* ghist) {
  const uint32_t t = threadIdx.x, lane = t & 63u;
#pragma unroll
  for (int k = 0; k < S; ++k)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      atomicAdd((int32_t*)lds + k * 256 + (4 * (lane >> 4) + v) * 16 + (lane & 15u), sum[k][v]);
      sum[k][v] = 0;
    }
  __syncthreads();
#pragma unroll
  for (int axis = 0; axis < 2; ++axis) {
    if (t < S * 16u) {
      int32_t* const row = (int32_t*)lds + (t >> 4) * 256 + (t & 15u) * (axis ? 1u : 16u);
      int32_t v[16];
#pragma unroll
      for (int x = 0; x < 16; ++x) v[x] = row[x * (axis ? 16 : 1)];
      unmix16(v);
#pragma unroll
      for (int x = 0; x < 16; ++x) row[x * (axis ? 16 : 1)] = v[x];
    }
    __syncthreads();
  }
  for (uint32_t i = t; i < S * 256u; i += T) {
    const uint32_t n = lds[i] + lds[1024u + i];
    lds[i] = 0;
    lds[1024u + i] = 0;
    if (n) atomicAdd(ghist + i, n);
  }
  __syncthreads();
}
// Words of LDS flush_counts needs.
constexpr uint32_t kFlushWords = 2048;
// A single byte of plane k.
__device__ __forceinline__ void count_byte(uint32_t* lds, uint32_t k, uint32_t byte) {
  atomicAdd(lds + 1024u + k * 256u + byte, 1u);
}

}  // namespace mans
