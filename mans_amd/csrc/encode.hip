// encode.hip -- interleaved rANS encoder on gfx950 wavefronts.
//
// Reference: include/ans/GpuANSEncode.h:24-164 (encodeOne / ansEncodeBatch),
// :166-178 + BatchPrefixSum.h:29-187 (prefix of padded word counts) and
// :180-284 (ansEncodeCoalesceBatch).  The reference encodes each 4 KiB block
// into an uncoalesced staging buffer in HBM, scans the word counts with up to
// three launches (limit 512^2 blocks) and copies every block again into the
// final container.  Here one persistent launch does all of it
// (encode_mc_kernel):
//  * a workgroup takes a ticket (atomic counter) for a run of units, each
//    coding wavefront a few of them.  Each lane runs CH independent rANS
//    chains, one per unit, fed by the same element loads where units are byte
//    planes of one block, so the serial per-chain dependency is interleaved;
//  * elements arrive 16 bytes a lane, two chunks ahead, and pass through LDS;
//    the table entries of a step are read one step ahead;
//  * emitted 16-bit words are compacted in lane order within each step
//    (64-bit ballot + mbcnt) into a linear LDS stage of H + 256 words a
//    unit: at most every 4 steps, once H words are waiting, they go to a
//    spill slot in HBM and the rest moves to the front, so a wave needs a few
//    KiB of LDS and many waves stay resident;
//  * an extra wavefront per workgroup publishes each ticket's padded word
//    count and resolves its output offset by decoupled look-back over earlier
//    tickets (tickets are taken by running workgroups, so every ticket waited
//    on belongs to a resident one and finishes), while the others code on;
//  * the units' words then go from the slot straight to their final place, 16
//    bytes per lane per store.
// encode_kernel is the 32-lane coder without spill slots: units staged whole
// in LDS (bounded by lane_max_words), used by the allocation-free entry point
// and for concatenated planes.
// The arithmetic per symbol is the reference's: emit x & 0xffff when
// x >= pdf * 2^(31-p); q = x / pdf; x = q * 2^p + (x - q * pdf) + cdf,
// computed as x + q * (2^p - pdf) + cdf.
#include "codec_device.hpp"

namespace mans {
namespace {

constexpr int kBatch = 16;  // steps per prefetch batch
// encode_mc_kernel: spill slots of a coding wavefront (on 1 GiB of uint16
// codes 3 slots and more take the same time, 2 a third more: with one ticket
// of slack every workgroup waits for the slowest), and workgroups per CU (two
// chains: 5 take 0.59 ms, 4 0.61, more no less; four chains: 3 are enough.  In
// the 32-lane format 4 and 5 take the same; four chains 2 groups 0.157 ms on
// 128 MiB of uint32, 3 0.144, but each group has its slots, whose allocation
// a workspace pays for: 260 to 390 MB at p = 10 on 256 CUs, and 3 would make
// them half as large again as two slots of four chains were).
constexpr uint32_t kEncSlots = 3;
constexpr int enc_groups(int lanes, int chains) { return lanes == 32 ? (chains >= 4 ? 2 : 4) : (chains >= 4 ? 3 : 5); }

template <typename T>
using gptr = const __attribute__((address_space(1))) T*;
template <typename T>
using lds_ptr = __attribute__((address_space(3))) T*;
// 16 bytes as a native vector: arrays of it stay in registers
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct LanePlane {  // per-plane fields copied to LDS (dynamic index by lane)
  const uint8_t* src;
  uint64_t nsym;
  uint64_t section;
  uint64_t nb;
};

// The 32-lane reference format: L lanes per unit, PB probability bits, S
// element bytes, CH chains per lane, NW wavefronts per group; units are
// staged whole in LDS.  CH == S: the CH chains of a lane code the CH byte
// planes of the same elements (unit order 0 with P == S).  CH == 1, S == 1:
// one chain per lane on any unit (single streams, concatenated ADM planes).
template <int L, int PB, int S, int CH, int NW>
__global__ __launch_bounds__(64 * NW) void encode_kernel(EncodeArgs a) {
  constexpr uint32_t BLOCK = L == 32 ? 4096u : 8192u;
  constexpr uint32_t HALVES = L == 32 ? 2u : 1u;
  constexpr uint32_t UPW = CH * HALVES;  // units per ticket
  constexpr uint32_t CSTAGE = chain_stage_words<PB>();
  constexpr uint32_t REG = CSTAGE;  // LDS words per chain
  static_assert(CH == S, "chain c codes byte c of each element");
  extern __shared__ uint4 smem[];
  __shared__ LanePlane s_pl[kMaxPlanes];
  __shared__ uint64_t s_ubase[kMaxPlanes + 1];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int P = a.d.num_planes;

  uint4* s_tab = smem;  // [P][256] {thresh, magic, shift | cdf << 8, 2^PB - pdf}
  for (int i = t; i < P * (int)kNumSymbols; i += 64 * NW) {
    uint4 e = a.table[i];
    s_tab[i] = make_uint4(e.x << (31 - PB), e.z, e.w | (e.y << 8), (1u << PB) - e.x);
  }
  if (t < P) {
    s_pl[t].src = a.d.plane[t].src;
    s_pl[t].nsym = a.d.plane[t].nsym;
    s_pl[t].section = a.d.plane[t].section;
    s_pl[t].nb = a.d.plane[t].nb;
    s_ubase[t] = a.d.plane[t].unit_base;
  }
  if (t == 0) s_ubase[P] = a.d.total_units;
  __syncthreads();

  const uint32_t half = L == 32 ? (uint32_t)(lane >> 5) : 0u;
  const uint32_t lin = (uint32_t)lane & (L - 1);
  // staging: per wave, CH regions of REG words ([half] whole units), then
  // one dword-spaced dummy slot per lane
  const uint32_t wave_u = __builtin_amdgcn_readfirstlane((uint32_t)wave);
  uint16_t* wstage = (uint16_t*)(smem + P * kNumSymbols) + wave_u * (CH * REG + 128);
  const uint32_t doff = CH * REG + 2u * (uint32_t)lane;  // dummy slot, from wstage
  // words coded per plane by this wave (added to the section headers once,
  // at the end)
  uint32_t ptot[kMaxPlanes];
#pragma unroll
  for (int k = 0; k < kMaxPlanes; ++k) ptot[k] = 0;

  uint32_t tk = 0;
  if (lane == 0) tk = atomicAdd(a.ticket, UPW);
  tk = __builtin_amdgcn_readfirstlane(tk);
  while ((uint64_t)tk < a.d.total_units) {

    uint32_t x[CH], cnt[CH], n[CH];
    uint32_t soff[CH];  // chain region, from wstage
    const uint4* tab[CH];
    uint64_t blk[CH];
    int kp[CH];
    bool act[CH];
    const uint8_t* src[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const uint64_t unit = (uint64_t)tk + half * CH + c;
      act[c] = unit < a.d.total_units;
      int k = 0;
      uint64_t b = 0;
      if (act[c]) {
        if (a.d.order == 0) {  // planes of one element array: P is 1, 2 or 4
          k = (int)((uint32_t)unit & (uint32_t)(P - 1));
          b = unit >> (P == 4 ? 2 : (P == 2 ? 1 : 0));
        } else {
          while (k + 1 < P && unit >= s_ubase[k + 1]) ++k;
          b = unit - s_ubase[k];
        }
      }
      kp[c] = k;
      blk[c] = b;
      const LanePlane pl = s_pl[k];
      const uint64_t start = b * BLOCK;
      n[c] = act[c] ? (uint32_t)((pl.nsym - start) < BLOCK ? (pl.nsym - start) : BLOCK) : 0u;
      src[c] = pl.src;
      x[c] = kMinState;
      cnt[c] = 0;
      soff[c] = c * REG + half * (CSTAGE / HALVES);
      tab[c] = s_tab + k * kNumSymbols;
    }
    // wave-uniform step counts over all chains and halves
    uint32_t n_min = n[0], n_max = n[0];
#pragma unroll
    for (int c = 1; c < CH; ++c) {
      n_min = n[c] < n_min ? n[c] : n_min;
      n_max = n[c] > n_max ? n[c] : n_max;
    }
    if (L == 32) {
      const uint32_t a0 = __builtin_amdgcn_readlane(n_min, 0), a1 = __builtin_amdgcn_readlane(n_min, 32);
      const uint32_t b0 = __builtin_amdgcn_readlane(n_max, 0), b1 = __builtin_amdgcn_readlane(n_max, 32);
      n_min = a0 < a1 ? a0 : a1;
      n_max = b0 > b1 ? b0 : b1;
    } else {
      n_min = __builtin_amdgcn_readfirstlane(n_min);
      n_max = __builtin_amdgcn_readfirstlane(n_max);
    }
    const uint32_t all = (uint32_t)div_up(n_max, L);

    auto step = [&](int c, const uint4& e, bool v) {
      enc_step<L, 0xffffffffu>(x[c], cnt[c], wstage, soff[c], doff, e, v, half);
    };

    {
      // One element per lane per step feeds all CH chains (byte c -> chain
      // c).  Chain 0 of a ticket is plane 0 whenever CH > 1, so its plane
      // pointer is the element array; with CH == 1 it is the chain's own
      // byte stream (single streams, concatenated planes).
      const uint8_t* eb = src[0] + blk[0] * BLOCK * S;  // element block start (4-byte aligned)
      uint32_t s = 0;
      // Full blocks: each lane loads the aligned dword holding its element
      // and takes its bytes at a per-lane bit offset.  Two register buffers:
      // while one batch is coded the next is loading.  (Whole dwords keep the
      // compiler from narrowing the buffers and waiting on the next batch.)
      const gptr<uint32_t> dp = (gptr<uint32_t>)eb + ((lin * S) >> 2);
      const uint32_t sh = 8u * ((lin * S) & 3u);
      auto load = [&](uint32_t (&buf)[kBatch], uint32_t s0) {
        const gptr<uint32_t> bp = dp + (uint64_t)s0 * (L * S / 4);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) buf[j] = bp[j * (L * S / 4)];
      };
      // The table entries of step j + 1 are read before step j is coded:
      // they depend on the symbols only, not on the states.
      auto code = [&](const uint32_t (&buf)[kBatch]) {
        uint4 e[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) e[c] = tab[c][__builtin_amdgcn_ubfe(buf[0], sh + 8u * c, 8u)];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
          uint4 en[CH];
          if (j + 1 < kBatch) {
#pragma unroll
            for (int c = 0; c < CH; ++c) en[c] = tab[c][__builtin_amdgcn_ubfe(buf[j + 1], sh + 8u * c, 8u)];
          }
#pragma unroll
          for (int c = 0; c < CH; ++c) step(c, e[c], true);
          if (j + 1 < kBatch) {
#pragma unroll
            for (int c = 0; c < CH; ++c) e[c] = en[c];
          }
        }
      };
      // The prefetch is unconditional (the last batch reloads itself) so the
      // wait before each batch only covers that batch's loads.  Partial blocks
      // (one per plane) take the byte path below, which never reads past the
      // end of the input.
      const uint32_t nbatch = n_min == BLOCK ? BLOCK / L / kBatch : 0u;
      if (nbatch > 0) {
        const uint32_t last = (nbatch - 1) * kBatch;
        uint32_t bufA[kBatch], bufB[kBatch];
        load(bufA, 0);
        for (;;) {
          load(bufB, s + kBatch <= last ? s + kBatch : last);
          code(bufA);
          s += kBatch;
          if (s > last) break;
          load(bufA, s + kBatch <= last ? s + kBatch : last);
          code(bufB);
          s += kBatch;
          if (s > last) break;
        }
      }
      for (; s < all; ++s) {
        const uint32_t i = s * L + lin;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const bool v = i < n[c];
          const uint32_t sym = v ? (uint32_t)eb[(uint64_t)i * S + c] : 0u;
          step(c, tab[c][sym], v);
        }
      }
    }

    // ---- per chain: pad, states; wave aggregate over the ticket's units ---
    uint32_t padded[CH];
    uint64_t agg = 0;
    uint32_t a_lo[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      padded[c] = (uint32_t)round_up(cnt[c], 8);
      if (cnt[c] > CSTAGE / HALVES && lin == 0) atomicOr(a.err, kErrStageOverflow);
      if (lin < padded[c] - cnt[c]) wstage[soff[c] + cnt[c] + lin] = 0;
      if (act[c]) ((uint32_t*)(a.out + s_pl[kp[c]].section + kSectionFixed))[blk[c] * L + lin] = x[c];
      a_lo[c] = __builtin_amdgcn_readlane(padded[c], 0);
      agg += a_lo[c];
      if (L == 32) agg += __builtin_amdgcn_readlane(padded[c], 32);
    }

    const uint64_t excl = look_back(a.status, tk / UPW, agg, lane);

    // unit order inside the ticket: (half 0: chains 0..CH-1), (half 1: ...)
    uint64_t y = excl;
    if (half) {
#pragma unroll
      for (int c = 0; c < CH; ++c) y += a_lo[c];
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (act[c] && lin == 0) {
        uint8_t* sec = a.out + s_pl[kp[c]].section;
        uint32_t* bw = (uint32_t*)(sec + kSectionFixed + 4ull * L * s_pl[kp[c]].nb + 8ull * blk[c]);
        bw[0] = (n[c] << 16) | cnt[c];
        bw[1] = (uint32_t)y;
      }
      {
        // this chain's unit per half-wave (two units in the 32-lane format,
        // possibly of different planes when planes are concatenated)
        const uint32_t pa = act[c] ? padded[c] : 0u;
        const uint32_t k0 = __builtin_amdgcn_readlane((uint32_t)kp[c], 0), a0 = __builtin_amdgcn_readlane(pa, 0);
#pragma unroll
        for (int k = 0; k < kMaxPlanes; ++k) ptot[k] += k0 == (uint32_t)k ? a0 : 0u;
        if (L == 32) {
          const uint32_t k1 = __builtin_amdgcn_readlane((uint32_t)kp[c], 32), a1 = __builtin_amdgcn_readlane(pa, 32);
#pragma unroll
          for (int k = 0; k < kMaxPlanes; ++k) ptot[k] += k1 == (uint32_t)k ? a1 : 0u;
        }
      }
      uint4* dst = (uint4*)(a.out + a.d.data_off + 2ull * y);
      const uint4* st4 = (const uint4*)(wstage + soff[c]);
      for (uint32_t j = lin; j < padded[c] / 8; j += L) dst[j] = st4[j];
      y += padded[c];
    }

    if ((uint64_t)tk + UPW >= a.d.total_units && lane == 0) {
      const uint64_t total_words = excl + agg;
      const uint64_t size = a.d.data_off + 2ull * total_words;
      if (a.d_out_size32) *a.d_out_size32 = (uint32_t)size;
      if (a.d_out_size64) *a.d_out_size64 = size;
      if (a.frame) {
        ((uint64_t*)a.out)[6] = total_words;  // data_words at byte 48
        ((uint64_t*)a.out)[7] = size;         // total_size at byte 56
      }
    }
    __threadfence_block();
    // the next ticket only once this one is done: tickets start in ticket
    // order, so the tickets a look-back waits on are already being coded
    if (lane == 0) tk = atomicAdd(a.ticket, UPW);
    tk = __builtin_amdgcn_readfirstlane(tk);
  }
  // total coded words of each plane (the section headers start at 0)
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < kMaxPlanes; ++k)
      if (k < P && ptot[k]) atomicAdd((uint32_t*)(a.out + s_pl[k].section + 12), ptot[k]);
  }
}

// The multi-chain coder, for both formats.  A workgroup is NW coding
// wavefronts and one placing wavefront.  A ticket (one atomic, one look-back
// entry) is NW x NS consecutive units; a coding wavefront's NS units are BPT
// consecutive element blocks per unit half (CH = S * BPT chains a lane: the S
// planes of each block).  In the 64-lane format a wavefront codes CH units;
// in the 32-lane format 2 CH, lanes 0-31 the first CH and lanes 32-63 the
// next CH (the units of one chain are "streams" h * CH + c, h the half).  A
// stream's words go to a linear LDS stage of H + 256 words; once H are
// waiting (checked at most 4 steps apart) they go to the wave's spill slot
// in HBM and the rest moves to the front.  When the ticket is coded the
// stage's remainder follows them, so the slot holds all of the unit's words,
// padded.
//
// One barrier a ticket hands its padded word counts to the resolving
// wavefront, which publishes their sum, resolves the offsets of coded tickets
// in turn (decoupled look-back) and writes their units' block word offsets
// while the coding wavefronts code the next ticket into the next of NSLOT
// slots.  After each barrier a coding wavefront copies its units of the
// tickets resolved by then from their slots to their final place; a ticket
// has to be resolved only when its slot is needed again.
//
// What bounds it: memory.  A unit's words are written to the slot, read back
// and written out (2.6 GB for 1 GiB of codes of ratio 2.1, the 1.6 GB of input
// and output and twice the output): 0.58-0.59 ms, 4.6 TB/s against the 4.7 of a
// large copy; with every load and store taken out of the loop the steps take
// 0.39 ms.  (Before: a ticket per wavefront, its look-back and the next
// ticket's atomic in the coding wavefronts' way, the chains' steps one after
// another, table entries of 16 bytes: 0.69 ms.  Atomics on one address run at
// 11 ns each whatever their number.)
// (32 lanes: unit order 0 or single streams only, so both halves of a chain
// share its plane.)
template <int L, int PB, int S, int BPT, int NW, int HB>
__global__ __launch_bounds__(64 * (NW + 1), 5) void encode_mc_kernel(EncodeArgs a) {
  constexpr int CH = S * BPT;                     // chains per lane
  constexpr int HALVES = L == 32 ? 2 : 1;
  constexpr int NS = CH * HALVES;                 // streams (units) per coding wavefront
  constexpr int CK = 16 / S;          // steps per input chunk: a 16-byte load per lane and block
  constexpr int KB = CK < 8 ? CK : 8;  // steps per batch of symbols in registers
  constexpr int DP = 2;               // chunks loaded ahead
  constexpr uint32_t BLOCK = L == 32 ? 4096u : 8192u;
  constexpr uint32_t CSTAGE = chain_stage_words<PB>();
  constexpr uint32_t SSTAGE = CSTAGE / HALVES;    // a unit's words at most, rounded
  constexpr uint32_t H = 1u << HB;  // spill chunk words
  constexpr uint32_t H4 = H / 8;    // spill chunk uint4s
  constexpr uint32_t REG = H + 256u;  // LDS stage words per stream
  constexpr uint32_t SLOT = CH * CSTAGE;  // spill slot words of a coding wavefront
  constexpr uint32_t TU = NW * NS;        // units per ticket
  constexpr uint32_t NSLOT = kEncSlots;   // tickets coded and not yet placed, with the one being coded
  constexpr int NT = 64 * (NW + 1);
  constexpr int CB = 8;  // copy batch: uint4 loads per lane in flight
  constexpr int TP = L == 32 ? S : (S > 1 ? S : kMaxPlanes);  // tables held
  constexpr uint32_t IN = BPT * 1024u;  // LDS bytes of a chunk per wavefront
  static_assert(BLOCK / L % CK == 0, "whole chunks per block");
  static_assert(H >= 256 && H4 <= 64, "256 <= spill chunk <= 512 words");
  static_assert(CSTAGE % 16 == 0 && SSTAGE % 8 == 0 && REG % 8 == 0, "uint4-aligned areas");
  static_assert(TU <= 64 && TU % S == 0, "a lane of the resolving wavefront per unit");
  extern __shared__ uint4 smem[];
  __shared__ LanePlane s_pl[kMaxPlanes];
  __shared__ uint64_t s_ubase[kMaxPlanes + 1];
  // per slot, of the ticket in it: its number and each unit's padded words;
  // once resolved, its offset and each unit's within it
  __shared__ uint32_t s_tk[NSLOT], s_pad[NSLOT][TU], s_ex[NSLOT][TU];
  __shared__ uint64_t s_excl[NSLOT];
  // the next ticket and the group's tickets resolved so far (of two tickets
  // in turn); the ticket (counted from 1) whose coding is nearly done
  __shared__ uint32_t s_next[2], s_res[2], s_near;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int P = a.d.num_planes;
  const uint32_t half = L == 32 ? (uint32_t)(lane >> 5) : 0u;
  const uint32_t lin = (uint32_t)lane & (L - 1);

  // [P][256] entries of enc_entry, at a fixed LDS address so each chain's
  // base is an immediate offset of its reads
  __shared__ uint2 s_tab[TP * kNumSymbols];
  for (int i = t; i < P * (int)kNumSymbols; i += NT) s_tab[i] = enc_entry(a.table[i], PB);
  if (t < P) {
    s_pl[t].src = a.d.plane[t].src;
    s_pl[t].nsym = a.d.plane[t].nsym;
    s_pl[t].section = a.d.plane[t].section;
    s_pl[t].nb = a.d.plane[t].nb;
    s_ubase[t] = a.d.plane[t].unit_base;
  }
  if (t == 0) {
    s_ubase[P] = a.d.total_units;
    s_next[1] = atomicAdd(a.ticket, TU);
    s_near = 0;
  }
  __syncthreads();

  const uint32_t wave_u = __builtin_amdgcn_readfirstlane((uint32_t)wave);
  // the group's spill: per coding wavefront NSLOT slots of NS streams of
  // SSTAGE words
  uint16_t* const gspill = a.spill + (uint64_t)blockIdx.x * NW * (NSLOT * SLOT);
  // plane and block of a unit
  auto plane_of = [&](uint64_t unit, int& k, uint64_t& b) {
    if (a.d.order == 0) {  // planes of one element array: P is 1, 2 or 4
      k = (int)((uint32_t)unit & (uint32_t)(P - 1));
      b = unit >> (P == 4 ? 2 : (P == 2 ? 1 : 0));
    } else {
      k = 0;
      while (k + 1 < P && unit >= s_ubase[k + 1]) ++k;
      b = unit - s_ubase[k];
    }
  };

  uint32_t tk = __builtin_amdgcn_readfirstlane(s_next[1]);
  uint32_t it = 0;  // the group's tickets coded: ticket it goes to slot it % NSLOT

  if (wave_u == NW) {
    // ---- the resolving wavefront: lane u handles unit u of a ticket --------
    uint32_t ptot[kMaxPlanes];  // words of this lane's units per plane
#pragma unroll
    for (int k = 0; k < kMaxPlanes; ++k) ptot[k] = 0;
    auto tk_of = [&](uint32_t sl) { return (uint32_t)__builtin_amdgcn_readfirstlane(s_tk[sl]); };
    // the units' offsets within the ticket in slot sl and its words
    auto scan = [&](uint32_t sl, uint32_t& pw, uint32_t& ex) -> uint32_t {
      pw = (uint32_t)lane < TU ? s_pad[sl][lane] : 0u;
      uint32_t inc = pw;
#pragma unroll
      for (int o = 1; o < (int)TU; o <<= 1) {
        const uint32_t v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
      }
      ex = inc - pw;
      return __builtin_amdgcn_readlane(inc, TU - 1);
    };
    // resolves the ticket in slot sl; with TRY, returns false if one of its
    // predecessors has not yet published
    auto resolve = [&](uint32_t sl, auto try_) -> bool {
      constexpr bool TRY = decltype(try_)::value;
      const uint32_t p_tk = tk_of(sl);
      const uint64_t tix = p_tk / TU;
      uint32_t pw, ex;
      const uint32_t total = scan(sl, pw, ex);
      uint64_t excl = 0;
      if (tix > 0) {
        excl = look_back_window<8, TRY>(a.status, (int64_t)tix - 1, 0, kFlagPrefix, lane,
                                        [](uint64_t v, uint32_t& f, uint64_t& val) {
                                          f = (uint32_t)(v >> 62);
                                          val = v & kValueMask;
                                        });
        if (TRY && excl == ~0ull) return false;
        if (lane == 0)
          __hip_atomic_store(a.status + tix, kFlagPrefix | (excl + total), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if ((uint32_t)lane < TU) s_ex[sl][lane] = ex;
      if (lane == 0) s_excl[sl] = excl;
      const uint64_t unit = (uint64_t)p_tk + lane;
      if ((uint32_t)lane < TU && unit < a.d.total_units) {
        int k;
        uint64_t b;
        plane_of(unit, k, b);
        const LanePlane& pl = s_pl[k];
        ((uint32_t*)(a.out + pl.section + kSectionFixed + 4ull * L * pl.nb + 8ull * b))[1] = (uint32_t)(excl + ex);
#pragma unroll
        for (int q = 0; q < kMaxPlanes; ++q) ptot[q] += k == q ? pw : 0u;
      }
      if ((uint64_t)p_tk + TU >= a.d.total_units && lane == 0) {
        const uint64_t total_words = excl + total;
        const uint64_t size = a.d.data_off + 2ull * total_words;
        if (a.d_out_size32) *a.d_out_size32 = (uint32_t)size;
        if (a.d_out_size64) *a.d_out_size64 = size;
        if (a.frame) {
          ((uint64_t*)a.out)[6] = total_words;  // data_words at byte 48
          ((uint64_t*)a.out)[7] = size;         // total_size at byte 56
        }
      }
      return true;
    };
    auto publish = [&](uint32_t i) {
      uint32_t pw, ex;
      const uint32_t total = scan(i % NSLOT, pw, ex);
      publish_aggregate(a.status, tk_of(i % NSLOT) / TU, total, lane);
    };
    uint32_t res = 0;  // tickets resolved
    while ((uint64_t)tk < a.d.total_units) {
      if (lane == 0) s_tk[it % NSLOT] = tk;
      if (it > 0) publish(it - 1);
      // the ticket after this one goes to slot (it + 1) % NSLOT, whose
      // ticket must be resolved (the coding wavefronts place it after the
      // barrier); the others if they can be
      while (res + NSLOT < it + 2) {
        resolve(res % NSLOT, std::false_type{});
        ++res;
      }
      while (res < it && resolve(res % NSLOT, std::true_type{})) ++res;
      // the next ticket, taken shortly before it is needed: groups run at
      // different rates, and a ticket held long before it is coded keeps
      // those after it waiting.  (The launch drains: the lowest unpublished
      // ticket is being coded, or its group waits only for lower ones, all
      // of them published.)
      while (__hip_atomic_load(&s_near, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != it + 1)
        __builtin_amdgcn_s_sleep(4);
      if (lane == 0) {
        s_next[it & 1u] = atomicAdd(a.ticket, TU);
        s_res[it & 1u] = res;
      }
      __syncthreads();
      tk = __builtin_amdgcn_readfirstlane(s_next[it & 1u]);
      ++it;
    }
    if (it > 0) publish(it - 1);
    for (; res < it; ++res) resolve(res % NSLOT, std::false_type{});
    __syncthreads();
    // total coded words of each plane (the section headers start at 0)
#pragma unroll
    for (int k = 0; k < kMaxPlanes; ++k) {
      if (k < P) {
        const uint32_t v = wave_sum32(ptot[k]);
        if (lane == 0 && v) atomicAdd((uint32_t*)(a.out + s_pl[k].section + 12), v);
      }
    }
    return;
  }

  // ---- a coding wavefront: staging NS stages of REG words ------------------
  uint16_t* wstage = (uint16_t*)smem + wave_u * (NS * REG);
  const uint32_t win = lds_addr(smem) + NW * NS * REG * 2u + wave_u * IN;  // the chunk being coded (LDS address)
  uint16_t* const spill = gspill + wave_u * (NSLOT * SLOT);
  // Copies this wavefront's units of the resolved ticket in slot sl to their
  // final place, a batch of loads before any store.  (The slot was written
  // by other lanes of this wavefront, before a barrier.)
  auto place = [&](uint32_t sl) {
    const u32x4* s4 = (const u32x4*)(spill + sl * SLOT);
    uint32_t qb[NS + 1];  // first uint4 of each stream in the wavefront's output
    qb[0] = 0;
#pragma unroll
    for (int c = 0; c < NS; ++c)
      qb[c + 1] = qb[c] + __builtin_amdgcn_readfirstlane(s_pad[sl][wave_u * NS + c]) / 8;
    const uint32_t nq = qb[NS];
    u32x4* const dst = (u32x4*)(a.out + a.d.data_off + 2ull * (s_excl[sl] + s_ex[sl][wave_u * NS]));
    for (uint32_t j0 = 0; j0 < nq; j0 += CB * 64) {
      u32x4 q[CB];
#pragma unroll
      for (int u = 0; u < CB; ++u) {
        if (j0 + u * 64 < nq) {  // wave-uniform
          // lanes past the end load entry 0 (always in the slot)
          const uint32_t j = j0 + u * 64 + (uint32_t)lane;
          const uint32_t jj = j < nq ? j : 0u;
          // stream k's words sit at k * SSTAGE / 8 in the slot, at qb[k] here
          uint32_t d = 0;
#pragma unroll
          for (int k = 1; k < NS; ++k) d = jj >= qb[k] ? k * (SSTAGE / 8) - qb[k] : d;
          q[u] = s4[jj + d];
        }
      }
#pragma unroll
      for (int u = 0; u < CB; ++u) {
        const uint32_t j = j0 + u * 64 + (uint32_t)lane;
        if (j < nq) __builtin_nontemporal_store(q[u], dst + j);
      }
    }
  };
  uint32_t placed = 0;  // the group's tickets placed
  while ((uint64_t)tk < a.d.total_units) {
    const uint32_t slot = it % NSLOT;
    // per chain (this lane's half): unit, plane, block, symbols
    uint32_t x[CH], n[CH];
    const uint2* tab[CH];
    uint64_t blk[CH];
    int kp[CH];
    bool act[CH];
    const uint8_t* src[CH];
    // per stream: LDS byte address of the stage and of the next word, words
    // moved to the slot
    uint32_t cb[NS], sb[NS], fl[NS];
    uint16_t* const wslot = spill + slot * SLOT;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const uint64_t unit = (uint64_t)tk + wave_u * NS + half * CH + c;
      act[c] = unit < a.d.total_units;
      int k = 0;
      uint64_t b = 0;
      if (act[c]) plane_of(unit, k, b);
      kp[c] = k;
      blk[c] = b;
      const LanePlane pl = s_pl[k];
      const uint64_t start = b * BLOCK;
      n[c] = act[c] ? (uint32_t)((pl.nsym - start) < BLOCK ? (pl.nsym - start) : BLOCK) : 0u;
      if (L == 64) n[c] = __builtin_amdgcn_readfirstlane(n[c]);
      src[c] = pl.src;
      x[c] = kMinState;
      // S > 1 only on element arrays of S planes: chain c is plane c % S
      // (both halves: CH is a multiple of P)
      tab[c] = s_tab + (S > 1 ? c % S : (L == 32 ? 0 : k)) * kNumSymbols;
    }
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      fl[c] = 0;
      cb[c] = lds_addr(smem) + (wave_u * NS + (uint32_t)c) * REG * 2u;  // = wstage + c * REG
      sb[c] = cb[c];
    }
    uint32_t n_min = n[0], n_max = n[0];
#pragma unroll
    for (int c = 1; c < CH; ++c) {
      n_min = n[c] < n_min ? n[c] : n_min;
      n_max = n[c] > n_max ? n[c] : n_max;
    }
    if (L == 32) {
      const uint32_t a0 = __builtin_amdgcn_readlane(n_min, 0), a1 = __builtin_amdgcn_readlane(n_min, 32);
      const uint32_t b0 = __builtin_amdgcn_readlane(n_max, 0), b1 = __builtin_amdgcn_readlane(n_max, 32);
      n_min = a0 < a1 ? a0 : a1;
      n_max = b0 > b1 ? b0 : b1;
    }
    const uint32_t all = (uint32_t)div_up(n_max, L);

    // stage upkeep: a stream with H or more unspilled words moves its first
    // H to the slot and the rest (fewer than 256: at most 64 words per step,
    // at most 4 steps apart) to the front
    auto spill_full = [&]() {
#pragma unroll
      for (int c = 0; c < NS; ++c) {
        const uint32_t un = (sb[c] - cb[c]) >> 1;  // unspilled words
        if (un >= H) {
          uint16_t* st = wstage + c * REG;
          if ((uint32_t)lane < H4) ((uint4*)(wslot + c * SSTAGE + fl[c]))[lane] = ((const uint4*)st)[lane];
          if (4u * (uint32_t)lane < un - H) ((uint2*)st)[lane] = ((const uint2*)(st + H))[lane];
          fl[c] += H;
          sb[c] -= 2u * H;
        }
      }
    };
    auto steps = [&](const uint2 (&e)[CH], const bool (&v)[CH], auto full) {
      constexpr bool FULL = decltype(full)::value;
      if constexpr (L == 64) enc_steps64<PB, CH, FULL>(x, sb, e, v);
      else enc_steps32<PB, CH, FULL>(x, sb, half, e, v);
    };

    {
      // Per step each lane takes one element of each of the ticket's BPT
      // blocks (of its half); byte b of block d's element feeds chain
      // d * S + b.  With S > 1 the first chain of a block is its plane 0,
      // whose pointer is the element array; with S == 1 each chain has its
      // own byte stream (single streams, concatenated planes).
      const uint8_t* eb[BPT];
#pragma unroll
      for (int d = 0; d < BPT; ++d) eb[d] = src[d * S] + blk[d * S] * BLOCK * S;
      uint32_t s = 0;
      // Whole chunks: CK steps of each block are 1 KiB (512 B per half), read
      // with one 16-byte load per lane and passed through LDS, where each
      // lane then finds its element of every step.  (Elements loaded one by
      // one, 128 B a load and 8 steps ahead: 4 % slower on 1 GiB of uint16
      // codes.)
      using EL = typename ElemOf<S>::T;
      typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(4)));  // inputs are 4-byte aligned
      auto load = [&](u32x4 (&r)[BPT], uint32_t s0) {
#pragma unroll
        for (int d = 0; d < BPT; ++d)
          r[d] = __builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4a*)(eb[d] + (uint64_t)s0 * L * S + lin * 16u));
      };
      auto stash = [&](const u32x4 (&r)[BPT]) {
#pragma unroll
        for (int d = 0; d < BPT; ++d) *(lds_ptr<u32x4>)(uintptr_t)(win + d * 1024u + (uint32_t)lane * 16u) = r[d];
      };
      // steps j0 .. j0 + KB - 1 of the chunk in LDS
      auto unpack = [&](uint32_t (&buf)[BPT][KB], uint32_t j0) {
        const uint32_t at = win + half * 512u + (j0 * L + lin) * S;
#pragma unroll
        for (int d = 0; d < BPT; ++d)
#pragma unroll
          for (int j = 0; j < KB; ++j) buf[d][j] = *(lds_ptr<EL>)(uintptr_t)(at + d * 1024u + j * L * S);
      };
      // table entries of the chains for step j of a batch
      auto lookup = [&](uint2 (&e)[CH], const uint32_t (&buf)[BPT][KB], int j) {
#pragma unroll
        for (int d = 0; d < BPT; ++d) {
          const uint32_t w = buf[d][j];
          e[d * S] = *(const uint2*)((const char*)tab[d * S] + byte_x8<0>(w));
          if constexpr (S > 1) e[d * S + 1] = *(const uint2*)((const char*)tab[d * S + 1] + byte_x8<1>(w));
          if constexpr (S > 2) {
            e[d * S + 2] = *(const uint2*)((const char*)tab[d * S + 2] + byte_x8<2>(w));
            e[d * S + 3] = *(const uint2*)((const char*)tab[d * S + 3] + byte_x8<3>(w));
          }
        }
      };
      // The table entries of step j + 1 are read before step j is coded:
      // they depend on the symbols only, not on the states.  The stage is
      // checked every 4 steps: at most 4 * 64 words arrive in between.
      // FULL: every lane has a symbol at every step of the batch; else step
      // s0 + j of block d has one in the lanes below nb[d].
      auto code = [&](const uint32_t (&buf)[BPT][KB], uint32_t s0, auto full) {
        constexpr bool FULL = decltype(full)::value;
        uint2 e[CH];
        lookup(e, buf, 0);
#pragma unroll
        for (int j = 0; j < KB; ++j) {
          uint2 en[CH];
          if (j + 1 < KB) lookup(en, buf, j + 1);
          bool v[CH];
#pragma unroll
          for (int c = 0; c < CH; ++c) v[c] = FULL || (s0 + (uint32_t)j) * L + lin < n[c];
          steps(e, v, full);
          if ((j & 3) == 3) spill_full();
          if (j + 1 < KB) {
#pragma unroll
            for (int c = 0; c < CH; ++c) e[c] = en[c];
          }
        }
      };
      static_assert(KB % 4 == 0, "stage checks at batch-relative steps 3, 7, ...");
      // Chunks of CK steps where every lane of every chain has a symbol, DP of
      // them in flight.  (Loads past the last chunk reload it, so the wait
      // before each chunk only covers that chunk's loads.)
      const uint32_t nchunk = n_min / (L * CK);
      // three quarters through, the resolving wavefront takes the next ticket
      const uint32_t near_at = nchunk >= 8 ? nchunk * 3 / 4 : ~0u;
      auto near = [&]() {
        if (wave_u == 0 && lane == 0) __hip_atomic_store(&s_near, it + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      };
      if (nchunk < 8) near();
      if (nchunk > 0) {
        u32x4 r[DP][BPT];
#pragma unroll
        for (uint32_t k = 0; k < DP; ++k) load(r[k], (k < nchunk ? k : nchunk - 1) * CK);
        for (uint32_t c = 0; c < nchunk;) {
#pragma unroll
          for (uint32_t k = 0; k < DP; ++k) {
            stash(r[k]);
            load(r[k], (c + DP < nchunk ? c + DP : nchunk - 1) * CK);
            if (c == near_at) near();
#pragma unroll 1
            for (uint32_t j0 = 0; j0 < CK; j0 += KB) {
              uint32_t buf[BPT][KB];
              unpack(buf, j0);
              code(buf, c * CK + j0, std::true_type{});
            }
            if (++c == nchunk) break;
          }
        }
        s = nchunk * CK;
      }
      // The rest (a plane's last, partial block; the whole blocks beside it):
      // batches whose lanes past a block's end load nothing and keep their
      // state, also loaded one batch ahead.
      if (s < all) {
        auto load_part = [&](uint32_t (&buf)[BPT][KB], uint32_t s0) {
#pragma unroll
          for (int d = 0; d < BPT; ++d) {
            const gptr<EL> bp = (gptr<EL>)eb[d];
#pragma unroll
            for (int j = 0; j < KB; ++j) {
              const uint32_t i = (s0 + (uint32_t)j) * L + lin;
              buf[d][j] = i < n[d * S] ? (uint32_t)bp[i] : 0u;
            }
          }
        };
        uint32_t buf[BPT][KB], nxt[BPT][KB];
        load_part(buf, s);
        for (;;) {
          load_part(nxt, s + KB);
          code(buf, s, std::false_type{});
          s += KB;
          if (s >= all) break;
#pragma unroll
          for (int d = 0; d < BPT; ++d)
#pragma unroll
            for (int j = 0; j < KB; ++j) buf[d][j] = nxt[d][j];
        }
      }
    }

    // ---- per stream: pad, move the stage's remainder to the slot; per chain
    // and half: states and block words
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      const uint32_t rem = (sb[c] - cb[c]) >> 1;  // words still in the stage
      const uint32_t cnt = fl[c] + rem;
      const uint32_t padded = (uint32_t)round_up(cnt, 8);
      if (cnt > SSTAGE && lane == 0) atomicOr(a.err, kErrStageOverflow);
      uint16_t* st = wstage + c * REG;
      if ((uint32_t)lane < padded - cnt) st[rem + lane] = 0;
      const uint32_t nr = (padded - fl[c]) / 8;
      for (uint32_t j = lane; j < nr; j += 64) ((uint4*)(wslot + c * SSTAGE + fl[c]))[j] = ((const uint4*)st)[j];
      if (lane == 0) s_pad[slot][wave_u * NS + c] = padded;  // (0 for inactive units: they code nothing)
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const LanePlane& pl = s_pl[kp[c]];
      if (act[c]) ((uint32_t*)(a.out + pl.section + kSectionFixed))[blk[c] * L + lin] = x[c];
      // this lane's half: stream h * CH + c
      uint32_t cnt_h = 0;
#pragma unroll
      for (int h = 0; h < HALVES; ++h) {
        const int sidx = h * CH + c;
        const uint32_t cnt = fl[sidx] + ((sb[sidx] - cb[sidx]) >> 1);
        cnt_h = (uint32_t)h == half ? cnt : cnt_h;
      }
      if (act[c] && lin == 0)
        ((uint32_t*)(a.out + pl.section + kSectionFixed + 4ull * L * pl.nb + 8ull * blk[c]))[0] = (n[c] << 16) | cnt_h;
    }
    __syncthreads();
    for (const uint32_t res = __builtin_amdgcn_readfirstlane(s_res[it & 1u]); placed < res; ++placed)
      place(placed % NSLOT);
    tk = __builtin_amdgcn_readfirstlane(s_next[it & 1u]);
    ++it;
  }
  __syncthreads();
  for (; placed < it; ++placed) place(placed % NSLOT);
}

// The whole-unit staged 32-lane kernel (encode_kernel): CH == S chains, no
// spill areas.  The multi-chain kernel (encode_mc_kernel): BPT blocks per
// half-wave ticket, spill areas.
template <int L, int PB, int S, int CH, int NW>
hipError_t launch_staged(const EncodeArgs& a, int cu, hipStream_t s, SpillNeed* need_spill) {
  constexpr uint32_t CSTAGE = chain_stage_words<PB>();
  const size_t lds = (size_t)a.d.num_planes * kNumSymbols * sizeof(uint4) + (size_t)NW * (CH * CSTAGE + 128) * 2u;
  int per_cu = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, encode_kernel<L, PB, S, CH, NW>, 64 * NW, lds);
  if (e != hipSuccess) return e;
  if (per_cu < 1) per_cu = 1;
  const uint64_t waves = div_up(a.d.total_units, CH * 2u);
  uint64_t grid = div_up(waves, NW);
  const uint64_t cap = (uint64_t)cu * (uint64_t)per_cu;
  if (grid > cap) grid = cap;
  if (grid < 1) grid = 1;
  if (need_spill) {
    *need_spill = SpillNeed{};
    return hipSuccess;
  }
  hipLaunchKernelGGL((encode_kernel<L, PB, S, CH, NW>), dim3((uint32_t)grid), dim3(64 * NW), lds, s, a);
  return hipGetLastError();
}

template <int L, int PB, int S, int BPT, int NW, int HB>
hipError_t launch_mc(const EncodeArgs& a, int cu, hipStream_t s, SpillNeed* need_spill) {
  constexpr uint32_t CSTAGE = chain_stage_words<PB>();
  constexpr int CH = S * BPT, NS = CH * (L == 32 ? 2 : 1);
  constexpr uint32_t REG = (1u << HB) + 256u;
  // dynamic LDS: the stages and the input chunks (the tables are static)
  const size_t lds = (size_t)NW * (NS * REG * 2u + BPT * 1024u);
  int per_cu = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, encode_mc_kernel<L, PB, S, BPT, NW, HB>,
                                                              64 * (NW + 1), lds);
  if (e != hipSuccess) return e;
  if (per_cu < 1) per_cu = 1;
  if (per_cu > enc_groups(L, CH)) per_cu = enc_groups(L, CH);
  const uint64_t waves = div_up(a.d.total_units, NS);
  uint64_t grid = div_up(waves, NW);
  const uint64_t cap = (uint64_t)cu * (uint64_t)per_cu;
  if (grid > cap) grid = cap;
  if (grid < 1) grid = 1;
  // kEncSlots slots per coding wavefront of CH chains of 64 lanes
  const uint64_t group_bytes = (uint64_t)NW * kEncSlots * CH * CSTAGE * 2ull;
  if (need_spill) {
    *need_spill = SpillNeed{grid, group_bytes, (uint64_t)NW * kEncSlots * 4u * CSTAGE * 2ull};
    return hipSuccess;
  }
  // as many workgroups as the area holds (tickets go to any number of them)
  const uint64_t held = a.spill ? a.spill_bytes / group_bytes : 0;
  if (held < 1) return hipErrorInvalidValue;
  if (grid > held) grid = held;
  hipLaunchKernelGGL((encode_mc_kernel<L, PB, S, BPT, NW, HB>), dim3((uint32_t)grid), dim3(64 * (NW + 1)), lds, s, a);
  return hipGetLastError();
}

// staged: the 32-lane whole-unit kernel (no spill areas: the allocation-free
// entry point, and ADM planes concatenated at 32 lanes).
template <int L, int PB>
hipError_t launch_s(const EncodeArgs& a, int cu, hipStream_t s, SpillNeed* need_spill, bool staged) {
  const int P = a.d.num_planes;
  const uint32_t S = a.d.plane[0].stride;
  if constexpr (L == 64) {
    // two chains per lane (four for uint32: its planes share the element
    // loads), linear stages of 256 + 256 words; four coding wavefronts
    if (a.d.order == 0 && P == 2 && S == 2) return launch_mc<64, PB, 2, 1, 4, 8>(a, cu, s, need_spill);
    if (a.d.order == 0 && P == 4 && S == 4) return launch_mc<64, PB, 4, 1, 4, 8>(a, cu, s, need_spill);
    if (S == 1) return launch_mc<64, PB, 1, 2, 4, 8>(a, cu, s, need_spill);
  } else {
    if (!staged && a.d.order == 0) {
      // as above, two units per chain (one per half-wave)
      if (P == 2 && S == 2) return launch_mc<32, PB, 2, 1, 4, 8>(a, cu, s, need_spill);
      if (P == 4 && S == 4) return launch_mc<32, PB, 4, 1, 4, 8>(a, cu, s, need_spill);
      if (P == 1 && S == 1) return launch_mc<32, PB, 1, 2, 4, 8>(a, cu, s, need_spill);
    }
    if (a.d.order == 0 && P == 2 && S == 2) return launch_staged<L, PB, 2, 2, 2>(a, cu, s, need_spill);
    if (a.d.order == 0 && P == 4 && S == 4) return launch_staged<L, PB, 4, 4, 1>(a, cu, s, need_spill);
    if (S == 1) return launch_staged<L, PB, 1, 1, 4>(a, cu, s, need_spill);
  }
  return hipErrorInvalidValue;
}

template <int L>
hipError_t launch_p(const EncodeArgs& a, int cu, hipStream_t s, SpillNeed* need_spill, bool staged) {
  switch (a.d.prob_bits) {
    case 9: return launch_s<L, 9>(a, cu, s, need_spill, staged);
    case 10: return launch_s<L, 10>(a, cu, s, need_spill, staged);
    case 11: return launch_s<L, 11>(a, cu, s, need_spill, staged);
  }
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t encode_spill(const EncodeArgs& a, int cu, SpillNeed* need) {
  *need = SpillNeed{};
  if (a.d.total_units == 0) return hipSuccess;
  return a.d.lanes == 64 ? launch_p<64>(a, cu, nullptr, need, false) : launch_p<32>(a, cu, nullptr, need, false);
}

// a.spill == nullptr selects the 32-lane whole-unit kernel (no spill areas).
hipError_t launch_encode(const EncodeArgs& a, int cu, hipStream_t s) {
  if (a.d.total_units == 0) return hipSuccess;
  if (a.d.lanes == 64) return launch_p<64>(a, cu, s, nullptr, false);
  return launch_p<32>(a, cu, s, nullptr, a.spill == nullptr);
}

}  // namespace mans
