// lorenzo.hip -- dual-quantisation 3-D Lorenzo front end: the producer of
// uint16 quantisation codes for the codec, and its inverse.
//
// The reference has no such kernel; its mapping programs take the codes as
// given (mapping/cpu/mappingcpuV1.cpp reads a uint16 file).  This is the
// error-bounded step that makes them from a float32 field
// f[nz][ny][nx] with absolute error bound eb:
//   q = rint(f * (1 / (2 eb)))                    (prequantisation, float32)
//   L2(z, y, x) = q(z,y,x) - q(z,y-1,x) - q(z,y,x-1) + q(z,y-1,x-1)
//   r(z, y, x)  = L2(z, y, x) - L2(z-1, y, x)     (3-D Lorenzo residual; q = 0
//                                                 outside the field)
//   code = 32768 + r if |r| < radius, else 0 and (index, r) is an outlier.
// The inverse rebuilds q as the 3-D prefix sum of r and f' = q * (2 eb), so
// |f - f'| <= eb up to float rounding.
//
// Forward: a workgroup of 256 threads takes a tile of 256 x-columns x 16 rows
// x 16 planes (tiles taken by an atomic ticket, in ticket order).  A thread
// keeps its column's L2 of the previous plane for its 16 rows in registers,
// so each element's f is read once (plus one halo row and the plane below
// the tile), a plane's 17 rows loaded at once; q(z, y, x - 1) comes from the
// neighbouring lane.  Outliers are
// compacted in tile order (tile ticket, thread, plane, row) with a decoupled
// look-back over tiles; a thread holds up to kHold of them in registers, and
// a tile with more goes on a list, with each thread's offset inside the
// tile and its counts before planes 4, 8 and 12, for the fix-up launch to
// write (four plane groups of the tile at once).
#include "codec_device.hpp"

namespace mans {
namespace {

constexpr uint32_t kTX = 256, kTY = 16, kTZ = 16;
constexpr int kHold = kLorenzoHold;
constexpr int32_t kQLimit = 1 << 28;  // |q| bound: residuals stay inside int32

__device__ __forceinline__ int32_t quant(float f, float inv, bool& bad) {
  const float v = rintf(f * inv);
  if (!(fabsf(v) < (float)kQLimit)) {  // also NaN / inf
    bad = true;
    return 0;
  }
  return (int32_t)v;
}

struct TileGeom {
  uint32_t nxb, nyb, nzb;
};

__device__ __forceinline__ void tile_of(const LorenzoArgs& a, uint32_t t, uint32_t& x0, uint32_t& y0, uint32_t& z0) {
  const uint32_t nxb = (uint32_t)div_up(a.nx, kTX), nyb = (uint32_t)div_up(a.ny, kTY);
  x0 = (t % nxb) * kTX;
  y0 = ((t / nxb) % nyb) * kTY;
  z0 = (t / (nxb * nyb)) * kTZ;
}

// Codes of planes [dz0, dz1) of one tile (a thread per x-column: column
// threadIdx.x % 256); outliers go to `hold` (first kHold) and are counted in
// `cnt`, and `grp` gets the count before planes 4, 8 and 12 (a byte each;
// at most 192).  With WRITE_ALL, every outlier is written at a.out_idx /
// a.out_val from position `pos` on instead (the fix-up pass).  FULL: nx is a
// multiple of 256 and ny of 16, so every column and row of every tile is
// inside the field (only the row above the first row of tiles is not).
template <bool WRITE_ALL, bool FULL>
__device__ void code_tile(const LorenzoArgs& a, uint32_t x0, uint32_t y0, uint32_t z0, uint32_t dz0, uint32_t dz1,
                          uint32_t& cnt, uint32_t& grp, uint32_t (&hidx)[kHold], int32_t (&hval)[kHold], uint64_t pos,
                          bool& bad) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t x = x0 + threadIdx.x % kTX;
  const bool xin = FULL || x < a.nx;
  const uint64_t plane = (uint64_t)a.ny * a.nx;
  const float inv = a.inv2eb;
  const uint32_t ny1 = FULL ? kTY : (a.ny - y0 < kTY ? a.ny - y0 : kTY);
  const uint32_t nz0 = a.nz - z0 < kTZ ? a.nz - z0 : kTZ;
  const uint32_t nz1 = dz1 < nz0 ? dz1 : nz0;
  // q of plane z at rows y0 - 1 .. y0 + kTY - 1 (row j - 1 of the tile in
  // slot j; rows outside the field or the tile are 0) for this column and,
  // on lane 0, the column to its left (the other lanes take it from their
  // neighbour).  All of a plane's loads are issued before any is used.
  auto plane_q = [&](uint32_t z, int32_t (&qc)[kTY + 1], int32_t (&ql)[kTY + 1]) {
    float fc[kTY + 1], fl[kTY + 1];
#pragma unroll
    for (uint32_t j = 0; j <= kTY; ++j) {
      const int64_t y = (int64_t)y0 - 1 + (int64_t)j;
      const bool row = FULL ? (j > 0 || y0 > 0) : (y >= 0 && (j == 0 || j - 1 < ny1));
      const uint64_t r = row ? z * plane + (uint64_t)y * a.nx : 0u;
      fc[j] = row && xin ? a.field[r + x] : 0.0f;
      fl[j] = 0.0f;
      if (lane == 0 && row && x > 0 && (FULL || x - 1 < a.nx)) fl[j] = a.field[r + x - 1];
    }
#pragma unroll
    for (uint32_t j = 0; j <= kTY; ++j) {
      const int64_t y = (int64_t)y0 - 1 + (int64_t)j;
      const bool row = FULL ? (j > 0 || y0 > 0) : (y >= 0 && (j == 0 || j - 1 < ny1));
      qc[j] = row && xin ? quant(fc[j], inv, bad) : 0;
      int32_t nb = __shfl_up(qc[j], 1, 64);
      if (lane == 0) nb = row && x > 0 && (FULL || x - 1 < a.nx) ? quant(fl[j], inv, bad) : 0;
      ql[j] = nb;
    }
  };
  int32_t prev[kTY];
#pragma unroll
  for (uint32_t j = 0; j < kTY; ++j) prev[j] = 0;
  // the plane below the first one: its L2 per row
  if (z0 + dz0 > 0 && dz0 < nz1) {
    int32_t qc[kTY + 1], ql[kTY + 1];
    plane_q(z0 + dz0 - 1, qc, ql);
#pragma unroll
    for (uint32_t j = 0; j < kTY; ++j)
      if (j < ny1) prev[j] = qc[j + 1] - qc[j] - ql[j + 1] + ql[j];
  }
  for (uint32_t dz = dz0; dz < nz1; ++dz) {
    const uint32_t z = z0 + dz;
    if (!WRITE_ALL && dz > 0 && (dz & 3u) == 0) grp |= cnt << (8u * (dz / 4u - 1u));
    int32_t qc[kTY + 1], ql[kTY + 1];
    plane_q(z, qc, ql);
#pragma unroll
    for (uint32_t j = 0; j < kTY; ++j) {
      if (j < ny1) {
        const uint32_t y = y0 + j;
        const int32_t l2 = qc[j + 1] - qc[j] - ql[j + 1] + ql[j];
        const int32_t r = l2 - prev[j];
        prev[j] = l2;
        if (xin) {
          const uint64_t i = z * plane + (uint64_t)y * a.nx + x;
          const bool in = r > -(int32_t)a.radius && r < (int32_t)a.radius;
          if (!WRITE_ALL) a.codes[i] = in ? (uint16_t)(32768 + r) : (uint16_t)0;
          if (!in) {
            if (WRITE_ALL) {
              if (pos + cnt < a.out_cap) {
                a.out_idx[pos + cnt] = (uint32_t)i;
                a.out_val[pos + cnt] = r;
              }
            } else {
#pragma unroll
              for (int k = 0; k < kHold; ++k)
                if ((uint32_t)k == cnt) {
                  hidx[k] = (uint32_t)i;
                  hval[k] = r;
                }
            }
            ++cnt;
          }
        }
      }
    }
  }
}

// Exclusive scan of v over the workgroup's 256 threads; *total gets the sum.
__device__ __forceinline__ uint32_t block_scan256(uint32_t v, uint32_t* s_w, uint32_t& total) {
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  uint32_t inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(inc, o, 64);
    if (lane >= (uint32_t)o) inc += u;
  }
  if (lane == 63) s_w[w] = inc;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
  for (uint32_t k = 0; k < kTX / 64; ++k) {
    if (k < w) before += s_w[k];
    total += s_w[k];
  }
  __syncthreads();
  return before + inc - v;
}

template <bool FULL>
__global__ __launch_bounds__(kTX) void lorenzo_kernel(LorenzoArgs a) {
  __shared__ uint32_t s_t, s_k, s_w[kTX / 64];
  __shared__ uint64_t s_off;
  __shared__ int s_bad;
  if (threadIdx.x == 0) {
    s_t = atomicAdd(a.ticket, 1u);
    s_bad = 0;
  }
  __syncthreads();
  const uint32_t t = s_t;
  uint32_t x0, y0, z0;
  tile_of(a, t, x0, y0, z0);
  uint32_t cnt = 0, grp = 0;
  uint32_t hidx[kHold];
  int32_t hval[kHold];
  bool bad = false;
  code_tile<false, FULL>(a, x0, y0, z0, 0, kTZ, cnt, grp, hidx, hval, 0, bad);
  if (bad) s_bad = 1;
  uint32_t total = 0;
  const uint32_t mine = block_scan256(cnt, s_w, total);
  // wave 0: the tile's offset among the outliers of earlier tiles
  if (threadIdx.x < 64) {
    const uint64_t excl = look_back(a.status, t, total, (int)threadIdx.x);
    if (threadIdx.x == 0) {
      s_off = excl;
      a.tile_off[t] = excl;
      if (t + 1 == a.ntiles) *a.count = excl + total;
    }
  }
  __syncthreads();
  const uint64_t pos = s_off + mine;
#pragma unroll
  for (int k = 0; k < kHold; ++k)
    if ((uint32_t)k < cnt && pos + k < a.out_cap) {
      a.out_idx[pos + k] = hidx[k];
      a.out_val[pos + k] = hval[k];
    }
  // a thread with more outliers than it holds: the tile goes on the fix-up
  // list with every thread's offset inside the tile, and the fix-up launch
  // writes the tile's outliers; outliers past the capacity: flagged
  const uint32_t over = __syncthreads_or(cnt > (uint32_t)kHold);
  if (over) {  // uniform over the workgroup
    if (threadIdx.x == 0) s_k = atomicAdd(a.fix_list, 1u);
    __syncthreads();
    const uint32_t k = s_k;
    if (k < a.fix_cap) {
      if (threadIdx.x == 0) a.fix_list[1 + k] = t;
      a.fix_pos[(uint64_t)k * kTX + threadIdx.x] = mine;
      a.fix_grp[(uint64_t)k * kTX + threadIdx.x] = grp;
    } else if (threadIdx.x == 0) {
      // more than fix_cap tiles over kHold: more than out_cap outliers
      atomicOr(a.err, kErrCapacity);
    }
  }
  if (threadIdx.x == 0) {
    if (s_off + total > a.out_cap) atomicOr(a.err, kErrCapacity);
    if (s_bad) atomicOr(a.err, kErrAdmDomain);
  }
}

// Writes every outlier of the tiles on the fix-up list.  A workgroup of
// kFixGroups x 256 threads takes a listed tile, thread (g, column) codes
// planes [4g, 4g + 4) of its column from the offsets the main launch left:
// the column's first outlier in the tile plus its count before plane 4g.
constexpr uint32_t kFixGroups = kTZ / 4;
__global__ __launch_bounds__(kTX * kFixGroups) void lorenzo_fixup_kernel(LorenzoArgs a) {
  const uint32_t nfix = a.fix_list[0] < a.fix_cap ? a.fix_list[0] : a.fix_cap;
  const uint32_t col = threadIdx.x % kTX, g = threadIdx.x / kTX;
  for (uint32_t k = blockIdx.x; k < nfix; k += gridDim.x) {
    const uint32_t t = a.fix_list[1 + k];
    uint32_t x0, y0, z0;
    tile_of(a, t, x0, y0, z0);
    uint32_t cnt = 0, grp = 0, dummy_i[kHold];
    int32_t dummy_v[kHold];
    bool bad = false;
    const uint64_t e = (uint64_t)k * kTX + col;
    const uint32_t before = g ? (a.fix_grp[e] >> (8u * (g - 1u))) & 0xffu : 0u;
    const uint64_t pos = a.tile_off[t] + a.fix_pos[e] + before;
    code_tile<true, false>(a, x0, y0, z0, 4u * g, 4u * g + 4u, cnt, grp, dummy_i, dummy_v, pos, bad);
  }
}

// ---- inverse ---------------------------------------------------------------
// The outliers' residuals are scattered first.  Then either
//  * by tiles of `ty` rows x TZ planes x whole rows of x: the sums of the
//    residuals r over each tile's planes (per row), its rows (per plane) and
//    both; their prefixes over the tiles; then each tile from those, the
//    x-prefix last.  All sums are of 32-bit integers, so their order does not
//    matter.  The codes are read twice, the field is written once and the
//    sums take 0.4 bytes an element where tiles are 16 planes x 32 rows, 1.1
//    where they are 4 x 32 (rows over 2048) and up to 3.5 where they are
//    small (fields of few tiles); or
//  * (buffers that overlap, fields of few rows) per plane the x-prefix of each row plus the
//    y-prefix (running per column), then per column the z-prefix and
//    f' = q * 2 eb, with every q through memory.
// 500 x 499 x 900: by tiles 489 us, through q 820.
__global__ void lorenzo_scatter_kernel(LorenzoArgs a) {
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < a.n_out; k += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t i = a.in_idx[k];
    if ((uint64_t)i < (uint64_t)a.nx * a.ny * a.nz) a.q[i] = a.in_val[k];
    else atomicOr(a.err, kErrBlockWords);
  }
}

constexpr uint32_t kPlaneChunk = 1024;  // elements of a row a workgroup scans at a time
constexpr uint32_t kRowGroup = 8;       // rows of a plane loaded, scanned and synchronised together

// One workgroup per plane: per row, the x-prefix of r (wave scans, then the
// waves' totals through LDS), summed down each column (the y-prefix).  A
// thread takes E adjacent elements of a row (E = 2: one 4-byte load of two
// codes, one 8-byte store of two sums; needs an even row length and 4-byte
// aligned codes).  Rows go kRowGroup at a time: their loads are all issued
// before any is scanned, and one barrier serves the group (the wave totals
// alternate between two LDS buffers, so a buffer is rewritten only after the
// barrier that follows its last read).  Rows longer than kPlaneChunk go
// chunk by chunk with the row's running total carried between chunks.
template <uint32_t E>
__global__ __launch_bounds__(kPlaneChunk / E) __attribute__((amdgpu_waves_per_eu(8)))
void lorenzo_plane_kernel(LorenzoArgs a) {
  constexpr uint32_t kT = kPlaneChunk / E, kW = kT / 64;  // threads, waves
  constexpr uint32_t kMaxChunks = 8;                     // nx <= 8192
  static_assert(E == 1 || E == 2, "one or two elements a thread");
  __shared__ int32_t s_w[2][kRowGroup][kW];
  __shared__ int32_t s_col[kMaxChunks][kPlaneChunk];  // column sums of each chunk's elements
  const uint32_t z = blockIdx.x;
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const uint32_t wu = __builtin_amdgcn_readfirstlane(w);
  const uint32_t lw = lane & (kW - 1);
  const uint64_t plane = (uint64_t)a.ny * a.nx;
  const uint32_t nchunks = (uint32_t)div_up(a.nx, kPlaneChunk);
  for (uint32_t c = 0; c < nchunks; ++c)
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) s_col[c][threadIdx.x * E + e] = 0;
  uint32_t it = 0;
  for (uint32_t y0 = 0; y0 < a.ny; y0 += kRowGroup) {
    const uint32_t nrow = a.ny - y0 < kRowGroup ? a.ny - y0 : kRowGroup;
    int32_t carry[kRowGroup];
#pragma unroll
    for (uint32_t g = 0; g < kRowGroup; ++g) carry[g] = 0;
#pragma unroll 1
    for (uint32_t c = 0; c < nchunks; ++c) {
      // this thread's first element; with E = 2 the row length is even, so
      // x < nx means x + 1 < nx
      const uint32_t x = c * kPlaneChunk + threadIdx.x * E;
      const bool xin = x < a.nx;
      // row g of the group starts at element row0 + g * nx (uniform; the
      // lane adds x)
      const uint64_t row0 = z * plane + (uint64_t)y0 * a.nx;
      // cells outside the field or the group read as code 32768 (r = 0)
      uint32_t code[kRowGroup];
#pragma unroll
      for (uint32_t g = 0; g < kRowGroup; ++g) {
        const uint16_t* p = a.codes + row0 + (uint64_t)g * a.nx + x;
        if (E == 1) code[g] = xin && g < nrow ? *p : 32768u;
        else code[g] = xin && g < nrow ? *(const uint32_t*)p : 0x80008000u;
      }
      int32_t v[kRowGroup][E], inc[kRowGroup];
#pragma unroll
      for (uint32_t g = 0; g < kRowGroup; ++g) {
        inc[g] = 0;
#pragma unroll
        for (uint32_t e = 0; e < E; ++e) {
          const uint32_t ce = (code[g] >> (16 * e)) & 0xFFFFu;
          v[g][e] = ce ? (int32_t)ce - 32768 : (a.q + row0 + (uint64_t)g * a.nx)[x + e];
          inc[g] += v[g][e];
        }
      }
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
        for (uint32_t g = 0; g < kRowGroup; ++g) {
          const int32_t u = __shfl_up(inc[g], o, 64);
          if (lane >= (uint32_t)o) inc[g] += u;
        }
      }
      const uint32_t buf = it & 1u;
      ++it;
      if (lane == 63) {
#pragma unroll
        for (uint32_t g = 0; g < kRowGroup; ++g) s_w[buf][g][w] = inc[g];
      }
      __syncthreads();
      int32_t colsum[E];
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) colsum[e] = s_col[c][threadIdx.x * E + e];
#pragma unroll
      for (uint32_t g = 0; g < kRowGroup; ++g) {
        // scan of the kW wave totals over each kW-lane group of the wave
        int32_t t = s_w[buf][g][lw];
#pragma unroll
        for (uint32_t o = 1; o < kW; o <<= 1) {
          const int32_t u = __shfl_up(t, o, kW);
          if (lw >= o) t += u;
        }
        // all waves' total and the total of the waves before this one
        // (uniform: read from one lane)
        const int32_t all = __builtin_amdgcn_readlane(t, kW - 1);
        const int32_t prior = wu ? __builtin_amdgcn_readlane(t, wu - 1) : 0;
        int32_t run = carry[g] + prior + inc[g];  // x-prefix through this thread's last element
#pragma unroll
        for (uint32_t e = 0; e < E; ++e) run -= v[g][e];
#pragma unroll
        for (uint32_t e = 0; e < E; ++e) {
          run += v[g][e];
          colsum[e] += run;  // x-prefix of this row, summed over rows
        }
        carry[g] += all;
        if (xin && g < nrow) {
          int32_t* q = a.q + row0 + (uint64_t)g * a.nx + x;
          if (E == 1) *q = colsum[0];
          else *(int2*)q = make_int2(colsum[0], colsum[E - 1]);
        }
      }
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) s_col[c][threadIdx.x * E + e] = colsum[e];
    }
  }
}

constexpr uint32_t kColumnPlanes = 16;  // planes of a column loaded before any is summed

// Per (y, x) column: the z-prefix of the plane sums and f' = q * 2 eb.
__global__ __launch_bounds__(256) void lorenzo_column_kernel(LorenzoArgs a) {
  const uint64_t plane = (uint64_t)a.ny * a.nx;
  for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < plane; j += (uint64_t)gridDim.x * blockDim.x) {
    int32_t s = 0;
    for (uint32_t z0 = 0; z0 < a.nz; z0 += kColumnPlanes) {
      int32_t v[kColumnPlanes];
#pragma unroll
      for (uint32_t k = 0; k < kColumnPlanes; ++k)
        v[k] = z0 + k < a.nz ? a.q[(uint64_t)(z0 + k) * plane + j] : 0;
#pragma unroll
      for (uint32_t k = 0; k < kColumnPlanes; ++k) {
        s += v[k];
        if (z0 + k < a.nz) a.recon[(uint64_t)(z0 + k) * plane + j] = (float)s * a.twoeb;
      }
    }
  }
}

// The codes of planes z0 .. z0 + TZ - 1 at (y, x), and the residuals they
// stand for (FULL: every plane is in the field; else 0 past its end).
template <uint32_t TZ, bool FULL>
__device__ __forceinline__ void load_codes(const LorenzoArgs& a, uint32_t z0, uint32_t y, uint32_t x,
                                           uint32_t (&code)[TZ]) {
  const uint64_t plane = (uint64_t)a.ny * a.nx;
  const uint16_t* p = a.codes + z0 * plane + (uint64_t)y * a.nx + x;
#pragma unroll
  for (uint32_t k = 0; k < TZ; ++k) code[k] = FULL || z0 + k < a.nz ? p[k * plane] : 32768u;
}
template <uint32_t TZ>
__device__ __forceinline__ void residuals(const LorenzoArgs& a, uint32_t z0, uint32_t y, uint32_t x,
                                          const uint32_t (&code)[TZ], int32_t (&r)[TZ]) {
  const uint64_t plane = (uint64_t)a.ny * a.nx;
  const int32_t* q = a.q + z0 * plane + (uint64_t)y * a.nx + x;
#pragma unroll
  for (uint32_t k = 0; k < TZ; ++k) {
    r[k] = (int32_t)code[k] - 32768;
    if (code[k] == 0) r[k] = q[k * plane];
  }
}

// A tile's sums: over its planes for each row (slab), over its rows for each
// plane (band), over both (corner).  A thread per x, the next row's codes
// loaded ahead; the last slab's and the last band's are not needed.
// Memory bound: 154 us for 500 x 499 x 900.  (Workgroups of 256 columns, which
// share lines of a row across XCDs: 167.)
template <uint32_t TZ>
__global__ __launch_bounds__(1024) void lorenzo_sums_kernel(LorenzoArgs a) {
  const uint32_t nxc = (uint32_t)div_up(a.nx, 1024), nyt = gridDim.x / nxc, nzt = gridDim.y;
  const uint32_t yt = blockIdx.x / nxc, zt = blockIdx.y;
  const uint32_t y0 = yt * a.ty, y1 = a.ny - y0 < a.ty ? a.ny : y0 + a.ty, z0 = zt * TZ;
  auto columns = [&](uint32_t x, auto full) {
    constexpr bool FULL = decltype(full)::value;
    int32_t v[TZ];
#pragma unroll
    for (uint32_t k = 0; k < TZ; ++k) v[k] = 0;
    uint32_t code[TZ];
    load_codes<TZ, FULL>(a, z0, y0, x, code);
    for (uint32_t y = y0; y < y1; ++y) {
      uint32_t next[TZ];
      load_codes<TZ, FULL>(a, z0, y + 1 < y1 ? y + 1 : y, x, next);
      int32_t r[TZ], s = 0;
      residuals<TZ>(a, z0, y, x, code, r);
#pragma unroll
      for (uint32_t k = 0; k < TZ; ++k) {
        v[k] += r[k];
        s += r[k];
        code[k] = next[k];
      }
      if (zt + 1 < nzt) a.slab[((uint64_t)zt * a.ny + y) * a.nx + x] = s;
    }
    int32_t all = 0;
#pragma unroll
    for (uint32_t k = 0; k < TZ; ++k) {
      all += v[k];
      if (yt + 1 < nyt && (FULL || z0 + k < a.nz)) a.band[((uint64_t)yt * a.nz + z0 + k) * a.nx + x] = v[k];
    }
    if (zt + 1 < nzt && yt + 1 < nyt) a.corner[((uint64_t)zt * (nyt - 1) + yt) * a.nx + x] = all;
  };
  const uint32_t x = blockIdx.x % nxc * 1024u + threadIdx.x;
  if (x >= a.nx) return;
  if (z0 + TZ <= a.nz) columns(x, std::true_type{});
  else columns(x, std::false_type{});
}

// Prefixes over the tiles, a thread a column, all inclusive and in place: of
// slab over the slabs, of band over the bands, of corner over the bands and,
// once those are complete (AXIS 1, a launch of its own), over the slabs; of few
// slabs each tile sums them itself instead.  Every entry is read and written
// once an axis, whatever the shape.  (Each corner's
// prefix summed from all corners before it, in one launch: 502 us for 500 x 499
// x 900 against 489, 351 ms for 1 x 1,000,000 x 1000 against 14.)
constexpr uint32_t kCornerSlabs = 8;  // (48 x 29 x 246: 21.5 us with the launch, 20.4 without)
template <int AXIS>
__global__ __launch_bounds__(256) void lorenzo_prefix_kernel(LorenzoArgs a, uint32_t nzt, uint32_t nyt) {
  constexpr uint32_t B = 16;  // entries loaded before any is summed
  const uint64_t per_slab = (uint64_t)a.ny * a.nx, per_band = (uint64_t)a.nz * a.nx;
  const uint64_t per_row = (uint64_t)(nyt - 1) * a.nx;  // corners of a slab
  auto scan = [&](int32_t* p, uint64_t step, uint32_t n) {
    int32_t s = 0;
    for (uint32_t k0 = 0; k0 < n; k0 += B) {
      int32_t v[B];
#pragma unroll
      for (uint32_t k = 0; k < B; ++k) v[k] = k0 + k < n ? p[(k0 + k) * step] : 0;
#pragma unroll
      for (uint32_t k = 0; k < B; ++k) {
        s += v[k];
        if (k0 + k < n) p[(k0 + k) * step] = s;
      }
    }
  };
  const uint64_t nc = AXIS == 1 ? per_row : (nyt > 1 ? (uint64_t)(nzt - 1) * a.nx : 0);
  const uint64_t ns = AXIS == 0 && nzt > 1 ? per_slab : 0, nb = AXIS == 0 && nyt > 1 ? per_band : 0;
  for (uint64_t j = (uint64_t)blockIdx.x * 256 + threadIdx.x; j < nc + ns + nb; j += (uint64_t)gridDim.x * 256) {
    if (j < nc) {
      if (AXIS == 1) scan(a.corner + j, per_row, nzt - 1);
      else scan(a.corner + j / a.nx * per_row + j % a.nx, a.nx, nyt - 1);
    } else if (j < nc + ns) {
      scan(a.slab + (j - nc), per_slab, nzt - 1);
    } else {
      scan(a.band + (j - nc - ns), per_band, nyt - 1);
    }
  }
}

// Inclusive sum over the 64 lanes.
__device__ __forceinline__ int32_t wave_scan(int32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}
// Sum over each row of 16 lanes (every lane gets it).
__device__ __forceinline__ int32_t row_sum(int32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true);   // quad_perm [1,0,3,2]
  v += __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true);   // quad_perm [2,3,0,1]
  v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);  // row_half_mirror
  v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);  // row_mirror
  return v;
}

// A tile of the field.  A thread keeps, for its x of each 1024-column chunk
// and each of the tile's planes, the sum w of r over the planes and rows up
// to here; a row adds its r, summed over the planes so far, and its x-prefix
// is the row of q.  One barrier a row and chunk; the next row's codes are
// loaded before it and their outliers after it.  Threads past the end of a
// row repeat its last column: nothing reads their sums.  Memory bound: 307 us
// for 500 x 499 x 900 (1.43 GB, 4.7 TB/s; with every load waited for in its
// own row 413).
template <uint32_t C, uint32_t TZ, bool FULL>
__device__ __forceinline__ void write_tile(const LorenzoArgs& a, int32_t (&s_w)[2][TZ][16]) {
  static_assert(TZ % 4 == 0, "four planes a row sum");
  const uint32_t yt = blockIdx.x, zt = blockIdx.y, nyt = gridDim.x;
  const uint32_t y0 = yt * a.ty, y1 = a.ny - y0 < a.ty ? a.ny : y0 + a.ty, z0 = zt * TZ;
  const uint32_t t = threadIdx.x, lane = t & 63u, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint64_t plane = (uint64_t)a.ny * a.nx;
  auto column = [&](uint32_t c) {
    const uint32_t x = c * 1024u + t;
    return x < a.nx ? x : a.nx - 1u;
  };
  int32_t cz[C][TZ];
#pragma unroll
  for (uint32_t c = 0; c < C; ++c) {
    const uint32_t x = column(c);
    int32_t run = 0;
    if (yt > 0)
      for (uint32_t z = zt > 0 && gridDim.y > kCornerSlabs ? zt - 1 : 0; z < zt; ++z)
        run += a.corner[((uint64_t)z * (nyt - 1) + yt - 1) * a.nx + x];
#pragma unroll
    for (uint32_t k = 0; k < TZ; ++k) {
      if (yt > 0 && (FULL || z0 + k < a.nz)) run += a.band[((uint64_t)(yt - 1) * a.nz + z0 + k) * a.nx + x];
      cz[c][k] = run;
    }
  }
  uint32_t code[TZ];
  int32_t r[TZ], u = 0;
  auto load = [&](uint32_t y, uint32_t c) {
    load_codes<TZ, FULL>(a, z0, y, column(c), code);
    if (zt > 0) u = a.slab[((uint64_t)(zt - 1) * a.ny + y) * a.nx + column(c)];
  };
  load(y0, 0);
  residuals<TZ>(a, z0, y0, column(0), code, r);
  uint32_t buf = 0;
  for (uint32_t y = y0; y < y1; ++y) {
    int32_t carry[TZ];
#pragma unroll
    for (uint32_t k = 0; k < TZ; ++k) carry[k] = 0;
#pragma unroll
    for (uint32_t c = 0; c < C; ++c) {
      const uint32_t x = c * 1024u + t;
      int32_t inc[TZ], s = u;
#pragma unroll
      for (uint32_t k = 0; k < TZ; ++k) {
        s += r[k];
        cz[c][k] += s;
        inc[k] = wave_scan(cz[c][k]);
      }
      if (lane == 63) {
#pragma unroll
        for (uint32_t k = 0; k < TZ; ++k) s_w[buf][k][w] = inc[k];
      }
      // (the last row is loaded again after itself)
      const uint32_t cn = c + 1 < C ? c + 1 : 0u, yn = c + 1 < C || y + 1 == y1 ? y : y + 1;
      load(yn, cn);
      __syncthreads();
      float* const out = a.recon + z0 * plane + (uint64_t)y * a.nx + x;
#pragma unroll
      for (uint32_t k0 = 0; k0 < TZ; k0 += 4) {
        // lane 16 p + v: wavefront v's total of plane k0 + p
        const int32_t v = s_w[buf][k0 + (lane >> 4)][lane & 15u];
        const int32_t before = row_sum((lane & 15u) < w ? v : 0);
        const int32_t all = C > 1 ? row_sum(v) : 0;
#pragma unroll
        for (uint32_t p = 0; p < 4; ++p) {
          const uint32_t k = k0 + p;
          inc[k] += carry[k] + __builtin_amdgcn_readlane(before, 16 * p);
          if (C > 1) carry[k] += __builtin_amdgcn_readlane(all, 16 * p);
        }
      }
      // the next row's outliers, before this row is written: the threads past
      // the end of the row read their last column's from where its own thread
      // may be writing (and use none of them)
      residuals<TZ>(a, z0, yn, column(cn), code, r);
      if (x < a.nx) {
#pragma unroll
        for (uint32_t k = 0; k < TZ; ++k)
          if (FULL || z0 + k < a.nz) out[k * plane] = (float)inc[k] * a.twoeb;
      }
      buf ^= 1u;
    }
  }
}

template <uint32_t C, uint32_t TZ>
__global__ __launch_bounds__(1024) void lorenzo_tile_kernel(LorenzoArgs a) {
  __shared__ int32_t s_w[2][TZ][16];  // the wavefronts' row totals
  for (uint32_t i = threadIdx.x; i < 2 * TZ * 16; i += blockDim.x) ((int32_t*)s_w)[i] = 0;
  __syncthreads();
  if ((blockIdx.y + 1) * TZ <= a.nz) write_tile<C, TZ, true>(a, s_w);
  else write_tile<C, TZ, false>(a, s_w);
}

// Planes of a tile: as many as a thread's sums of all its columns fit in
// registers.
uint32_t tile_planes(uint32_t nx) { return nx <= 1024 ? 16u : (nx <= 2048 ? 8u : 4u); }
// Rows of a tile: those of 2 .. 32 with the least time, in rows: the rounds of
// resident tiles (16 wavefronts a compute unit, four tiles at most) times a
// tile's rows and two for its start, and a 32nd for each band, which the
// prefixes walk one after another (at most 256 bands under 32 rows).  Within 2 %
// of the best of the five over 105 shapes, where two tiles a compute unit
// whatever their size were 10 % (256 x 48 x 1024: 44 us against 60, through q
// 51; 500 x 100 x 900: 100 against 142).  More rows while a column has over
// 4096 bands and every compute unit would still have four tiles (1 x 1,000,000
// x 1000: 14.1 ms from 128 rows on, 16.2 with 32).
uint32_t tile_rows(uint32_t nz, uint32_t ny, uint32_t nx, int cu) {
  const uint64_t nzt = div_up(nz, tile_planes(nx)), chip = (uint64_t)std::max(cu, 1);
  const uint64_t waves = div_up(std::min(nx, 1024u), 64);
  const uint64_t held = chip * std::max<uint64_t>(1, std::min<uint64_t>(4, 16 / waves));
  uint32_t ty = 32;
  uint64_t least = ~0ull;
  for (uint32_t r = 32; r >= 2; r /= 2) {
    const uint64_t bands = div_up(ny, r);
    if (r < 32 && bands > 256) break;
    const uint64_t cost = 32 * div_up(nzt * bands, held) * (r + 2) + bands;
    if (cost < least) {
      least = cost;
      ty = r;
    }
  }
  while (div_up(ny, ty) > 4096 && nzt * div_up(ny, 2ull * ty) >= 4 * chip) ty *= 2;
  return ty;
}

template <uint32_t C, uint32_t TZ>
hipError_t launch_tiles(const LorenzoArgs& a, int cu, hipStream_t s) {
  const uint32_t nyt = (uint32_t)div_up(a.ny, a.ty), nzt = (uint32_t)div_up(a.nz, TZ);
  const uint32_t threads = a.nx > 1024 ? 1024u : (uint32_t)round_up(a.nx, 64);
  hipError_t e;
  if (nzt > 1 || nyt > 1) {  // (a single tile needs no sums)
    hipLaunchKernelGGL(lorenzo_sums_kernel<TZ>, dim3(nyt * (uint32_t)div_up(a.nx, 1024), nzt), dim3(threads), 0, s, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  auto grid = [&](uint64_t cols) { return dim3((uint32_t)std::min<uint64_t>(div_up(cols, 256), (uint64_t)cu * 16)); };
  if (nzt > 2 || nyt > 2) {  // (one entry is its own prefix)
    const uint64_t cols = ((uint64_t)nzt - 1 + a.ny + a.nz) * a.nx;
    hipLaunchKernelGGL(lorenzo_prefix_kernel<0>, grid(cols), dim3(256), 0, s, a, nzt, nyt);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (nzt > kCornerSlabs && nyt > 1) {
    hipLaunchKernelGGL(lorenzo_prefix_kernel<1>, grid((uint64_t)(nyt - 1) * a.nx), dim3(256), 0, s, a, nzt, nyt);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((lorenzo_tile_kernel<C, TZ>), dim3(nyt, nzt), dim3(threads), 0, s, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_lorenzo(const LorenzoArgs& a, hipStream_t s) {
  if (a.ntiles == 0) return hipSuccess;
  if (a.nx % kTX == 0 && a.ny % kTY == 0)
    hipLaunchKernelGGL(lorenzo_kernel<true>, dim3(a.ntiles), dim3(kTX), 0, s, a);
  else
    hipLaunchKernelGGL(lorenzo_kernel<false>, dim3(a.ntiles), dim3(kTX), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // the fix-up list is short (a tile is on it only with more than kHold
  // outliers in one thread): a small grid walks it
  const uint32_t g = a.fix_cap < 1024u ? a.fix_cap : 1024u;
  hipLaunchKernelGGL(lorenzo_fixup_kernel, dim3(g), dim3(kTX * kFixGroups), 0, s, a);
  return hipGetLastError();
}

uint32_t lorenzo_tiles(uint32_t nz, uint32_t ny, uint32_t nx) {
  return (uint32_t)(div_up(nx, kTX) * div_up(ny, kTY) * div_up(nz, kTZ));
}

// Whether the field goes through q, by what the two routes take (in 10 ns,
// fitted to 2092 shapes of up to 1024 planes and 64 rows on 256 compute units:
// within 5 % of the faster route on all but 59).  Through q are two launches
// whose time grows with the planes and, in steps of eight, with the rows; rows of
// odd length are taken an element a thread, rows over 1024 in two chunks.  By
// tiles are one launch (a single tile), two or three, of about the same time
// whatever the planes.  1 x 16 x 1024: 13 us through q, 21 by tiles; 64 x 8 x
// 512 13 and 22; 24 x 24 x 32 17 and 19; 256 x 16 x 1024 34 and 38; 1 x 64 x
// 64 35 and 16; 256 x 48 x 1024 51 and 44; 128 x 16 x 33 23 and 20.
static bool through_q(uint32_t nz, uint32_t ny, uint32_t nx) {
  const bool odd = nx % 2 != 0, one_slab = nz <= tile_planes(nx);
  if (nx > 2048 || ny > 64 || nz > 1024 || (ny == 1 && one_slab)) return false;
  const uint32_t groups = (ny + 7) / 8 - 1;  // beyond the first
  if (nx > 1024) {
    const uint32_t q = (odd ? 1450u : 1200u) + 10u * nz + (odd ? 900u : 750u) * groups;
    if (ny <= 2) return q < (one_slab ? 550u + nx / 4u : (ny == 1 ? 1300u : 1700u));
    return q < 2100u + 6u * nz;
  }
  const uint32_t q = (odd ? 1000u : 800u) + (odd ? 9u : 8u) * nz + (odd ? 550u : 420u) * groups;
  if (ny == 1) return q < 900u + nx / 2u;
  if (ny == 2) return q < (one_slab ? 550u + nx / 2u : 1100u + nx * 3u / 4u + nz);
  return q < (ny == 3 ? 1450u : 1740u) + nx * 3u / 4u + 3u * nz;
}

LorenzoScratch lorenzo_inverse_scratch(uint32_t nz, uint32_t ny, uint32_t nx, int cu) {
  LorenzoScratch l;
  l.ty = tile_rows(nz, ny, nx, cu);
  const uint64_t nzt = div_up(nz, tile_planes(nx)), nyt = div_up(ny, l.ty);
  // (65535: the grid's second dimension; tile_rows keeps the first small)
  l.tiles = nzt <= 65535 && !through_q(nz, ny, nx);
  l.band = (nzt - 1) * ny * nx;
  l.corner = l.band + (nyt - 1) * nz * nx;
  l.words = l.corner + (nzt - 1) * (nyt - 1) * nx;
  return l;
}

hipError_t launch_lorenzo_inverse(const LorenzoArgs& a, int cu, hipStream_t s) {
  const uint64_t n = (uint64_t)a.nx * a.ny * a.nz;
  if (n == 0) return hipSuccess;
  if (a.n_out) {
    const uint32_t g = (uint32_t)std::min<uint64_t>(div_up(a.n_out, 256), 4096);
    hipLaunchKernelGGL(lorenzo_scatter_kernel, dim3(g), dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (a.slab) {
    if (a.nx <= 1024) return launch_tiles<1, 16>(a, cu, s);
    if (a.nx <= 2048) return launch_tiles<2, 8>(a, cu, s);
    if (a.nx <= 4096) return launch_tiles<4, 4>(a, cu, s);
    return launch_tiles<8, 4>(a, cu, s);
  }
  // two elements a thread where rows are even and the codes 4-byte aligned
  // (the q scratch is a whole allocation)
  if (a.nx % 2 == 0 && ((uintptr_t)a.codes & 3u) == 0)
    hipLaunchKernelGGL(lorenzo_plane_kernel<2>, dim3(a.nz), dim3(kPlaneChunk / 2), 0, s, a);
  else
    hipLaunchKernelGGL(lorenzo_plane_kernel<1>, dim3(a.nz), dim3(kPlaneChunk), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const uint64_t plane = (uint64_t)a.ny * a.nx;
  const uint32_t g = (uint32_t)std::min<uint64_t>(div_up(plane, 256), (uint64_t)cu * 16);
  hipLaunchKernelGGL(lorenzo_column_kernel, dim3(g), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace mans
