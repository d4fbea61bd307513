// Keccak-f[1600] with one state spread over 16 lanes (a DPP row), four states per wave:
// the latency form for long serial sponge chains when the GPU has SIMDs to spare.
//
// Lane (h, y) = (bit 3, bits 0..2 of the lane) holds the bit-interleaved half h (even /
// odd bits, keccak.cuh) of the five words of plane y; lanes y = 5..7 hold zeros.  Per
// round and lane:
//   theta  column parities by a butterfly over the 8 lanes of the half (3 DPP xors per
//          word; the zero lanes do not count), rot(C, 1) as a per-lane rotation fused with
//          the half swap (DPP row_ror:8);
//   rho    one 32-bit rotation by a per-lane amount; an odd rotation's change of half and
//   pi     are the address of an LDS write (the state's rows, [half][plane][x]);
//   chi    on the plane read back (one 16-byte and one 4-byte read), iota from a table that
//          is zero for the other planes.
// About 50 instructions per round and lane, where a lane pair takes 107 and a lone lane
// 180; a wave issues one every ~4.4 cycles, and the LDS round trip adds ~120 cycles.
// Measured on MI355X, us per permutation at one wave per SIMD: 3.3, against 4.9 for an
// unrolled interleaved lane pair, 6.3 for the rolled pair, 7.9 for one state per lane; at
// two waves per SIMD 4.8.  Its throughput is about a fifth of the one-state-per-lane form's
// (1.7 G permutations/s at two waves per SIMD, ~2.1 G at more, against 10.1 G).
#pragma once
#include <stddef.h>

#include <type_traits>

#include "keccak.cuh"

namespace pqc {
namespace wide {

// LDS image of a state: rows (half, plane) of words x = 0..3 at 4 row, word x = 4 at
// kCol4 + row.  With these strides and the zero lanes' places after the four states, a
// round's five writes and two reads meet ~40 bank cycles per wave; rows of 8 words took
// 50, and four waves on a CU ran 40% slower for it (116 permutations each: 551 against
// 388 us).
constexpr int kCol4 = 45, kStateWords = 80;

struct Maps {
  uint8_t amt[2][8][5];   // alignbit amount of the word about to move
  uint16_t dst[2][8][5];  // its place in the state's LDS rows
};
constexpr Maps make_maps() {
  Maps m{};
  for (int h = 0; h < 2; ++h)
    for (int y = 0; y < 5; ++y)
      for (int x = 0; x < 5; ++x) {
        // rot64 by 2k: both halves by k; by 2k + 1: the odd half by k + 1 into the even
        // one, the even half by k into the odd one
        const int o = kKeccakMaps.rho[x + 5 * y];
        const int rot = o / 2 + ((o & 1) && h ? 1 : 0);
        m.amt[h][y][x] = (uint8_t)((32 - rot) & 31);
        const int row = (h ^ (o & 1)) * 5 + (2 * x + 3 * y) % 5;
        m.dst[h][y][x] = (uint16_t)(y < 4 ? 4 * row + y : kCol4 + row);
      }
  return m;
}
static __device__ const Maps c_maps = make_maps();
static __device__ const IlRc c_rc = il_round_constants();

// Constants of a workgroup's waves, and one wave's states
struct Consts {
  uint32_t rc[2][24], none[24];
};
struct States {
  alignas(16) uint32_t w[4 * kStateWords];
  uint32_t trash[72];  // where the zero lanes write: a word each
  uint32_t zero[8];    // and read
};
static_assert(offsetof(States, zero) % 16 == 0, "16-byte read");

// every thread of the workgroup; a barrier must follow
__device__ __forceinline__ void init_consts(Consts& c) {
  const int t = threadIdx.x;
  if (t < 24) {
    c.rc[0][t] = c_rc.e[t];
    c.rc[1][t] = c_rc.o[t];
    c.none[t] = 0;
  }
}

__device__ __forceinline__ void sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kMirror8 = 0x141, kOtherHalf = 0x128;  // quad_perm, half mirror, row_ror:8

// A wave's four sponges.  a[x]: this lane's word of column x.
struct Sponge {
  uint32_t a[5];
  uint32_t amt[5];
  uint32_t* dst[5];
  const uint32_t *src, *src4;
  const uint32_t* rc;
  uint32_t rot1, sel_in, sel_out;
  int h, y, st;

  __device__ __forceinline__ void init(States& s, Consts& c) {
    const int l = (int)__lane_id();
    y = l & 7;
    h = (l >> 3) & 1;
    st = l >> 4;
    uint32_t* base = s.w + st * kStateWords;
#pragma unroll
    for (int x = 0; x < 5; ++x) {
      amt[x] = c_maps.amt[h][y][x];
      dst[x] = y < 5 ? base + c_maps.dst[h][y][x] : s.trash + l;
    }
    src = y < 5 ? base + 4 * (5 * h + y) : s.zero;
    src4 = y < 5 ? base + kCol4 + 5 * h + y : s.zero + 4;
    if (l < 8) s.zero[l] = 0;
    rc = y == 0 ? c.rc[h] : c.none;
    rot1 = h ? 31u : 0u;
    sel_in = h ? 0x03010705u : 0x06040200u;
    sel_out = h ? 0x03070206u : 0x05010400u;
    clear();
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int x = 0; x < 5; ++x) a[x] = 0;
  }

  // UNROLL rounds per loop trip: 24 (9 KB of code) for a kernel that is one long chain,
  // 3% faster than 4
  template <int UNROLL = 4>
  __device__ __forceinline__ void permute() {
#pragma unroll UNROLL
    for (int r = 0; r < 24; ++r) {
      const uint32_t k = rc[r];
      uint32_t C[5], S[5];
#pragma unroll
      for (int x = 0; x < 5; ++x) C[x] = a[x] ^ dpp<kXor1>(a[x]);
#pragma unroll
      for (int x = 0; x < 5; ++x) C[x] ^= dpp<kXor2>(C[x]);
#pragma unroll
      for (int x = 0; x < 5; ++x) C[x] ^= dpp<kMirror8>(C[x]);
#pragma unroll
      for (int x = 0; x < 5; ++x) S[x] = __builtin_amdgcn_alignbit(C[x], C[x], rot1);
#pragma unroll
      for (int x = 0; x < 5; ++x) {
        const uint32_t t = a[x] ^ (C[(x + 4) % 5] ^ dpp<kOtherHalf>(S[(x + 1) % 5]));
        *dst[x] = __builtin_amdgcn_alignbit(t, t, amt[x]);
      }
      sync();
      typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 q = *reinterpret_cast<const u32x4*>(src);
      const uint32_t B[5] = {q[0], q[1], q[2], q[3], *src4};
      sync();
#pragma unroll
      for (int x = 0; x < 5; ++x) a[x] = chi_32(B[x], B[(x + 1) % 5], B[(x + 2) % 5]);
      a[0] ^= k;
    }
  }

  // 32-bit halves of the 64-bit words <-> this lane's interleaved words.  Lane h handles
  // the low / high half of a word; the exchange with the other half's lane is one DPP
  // move, the byte order of both sides one v_perm_b32.
  __device__ __forceinline__ uint32_t interleave(uint32_t x) const {
    uint32_t t = (x ^ (x >> 1)) & 0x22222222u;
    x ^= t ^ (t << 1);
    t = (x ^ (x >> 2)) & 0x0C0C0C0Cu;
    x ^= t ^ (t << 2);
    t = (x ^ (x >> 4)) & 0x00F000F0u;
    x ^= t ^ (t << 4);
    return __builtin_amdgcn_perm(dpp<kOtherHalf>(x), x, sel_in);
  }
  __device__ __forceinline__ uint32_t join(uint32_t own) const {
    uint32_t x = __builtin_amdgcn_perm(dpp<kOtherHalf>(own), own, sel_out);
    uint32_t t = (x ^ (x >> 4)) & 0x00F000F0u;
    x ^= t ^ (t << 4);
    t = (x ^ (x >> 2)) & 0x0C0C0C0Cu;
    x ^= t ^ (t << 2);
    t = (x ^ (x >> 1)) & 0x22222222u;
    return x ^ t ^ (t << 1);
  }

  // xor a block of raw 32-bit halves into the state: m[x] belongs to word x + 5 y
  __device__ __forceinline__ void absorb(const uint32_t (&m)[5]) {
#pragma unroll
    for (int x = 0; x < 5; ++x) a[x] ^= interleave(m[x]);
  }
  // f(x, value): the raw 32-bit half h of word x + 5 y, for x in [0, COLS) of every plane
  template <int COLS, class F>
  __device__ __forceinline__ void squeeze(F&& f) const {
#pragma unroll
    for (int x = 0; x < COLS; ++x) f(x, join(a[x]));
  }
  __device__ __forceinline__ int word(int x) const { return x + 5 * y; }  // >= 25 on the zero lanes

  // Absorb blocks [b0, b1) (17 words each) of a message of nwords 64-bit words at the
  // 4-byte aligned p (the same for all states or one per state), SHA3-256 / SHAKE256 padding
  // included in the last one; the next block's words load during a permutation.  The words
  // stay as loaded until they are absorbed (a select on a loaded value waits for it where it
  // stands), and no branch goes around a load: lanes without a word read the message's
  // first one and drop it.
  template <int UNROLL = 4, class P>
  __device__ __forceinline__ void absorb17(P p, int nwords, uint32_t domain, int b0, int b1) {
    uint32_t raw[5];
    auto load = [&](int b) {
      const int rem = nwords - 17 * b, own = rem < 17 ? rem : 17;
#pragma unroll
      for (int x = 0; x < 5; ++x) raw[x] = p[word(x) < own ? 2 * (17 * b + word(x)) + h : h];
    };
    load(b0);
    for (int b = b0; b < b1; ++b) {
      const int rem = nwords - 17 * b, own = rem < 17 ? rem : 17;  // words left
      uint32_t m[5];
#pragma unroll
      for (int x = 0; x < 5; ++x) {
        const int w = word(x);
        uint32_t v = w < own ? raw[x] : 0u;
        v = (w < 17 && w == rem && h == 0) ? domain : v;
        v ^= (w == 16 && rem < 17 && h == 1) ? 0x80000000u : 0u;
        m[x] = v;
      }
      absorb(m);
      load(b + 1 < b1 ? b + 1 : b);
      permute<UNROLL>();
    }
  }
};

// ---- workgroups of the kernels with four chains per wave ----------------------------
// WG waves per workgroup.  Chains finish soonest on SIMDs that hold as few of them as
// possible.  The hardware spreads workgroups over CUs and a workgroup's waves over the
// CU's four SIMDs, but not the waves of several one-wave workgroups on one CU.  So a
// launch that needs a wave on most SIMDs takes four waves per workgroup, one of two waves
// per SIMD eight: a workgroup per CU.  Launches of up to two waves per CU take one-wave
// workgroups whose register allocation leaves no second place on a SIMD (as PQC_SIMD_WAVES
// in internal.h): they fill at most half of the SIMDs, and up to four of them side by side
// spread better than by workgroups (four calls of 500 FrodoKEM decapsulations 860 us,
// 1209 with four waves per workgroup).  A larger launch must not take whole SIMDs: it
// shuts out whatever runs beside it on other streams.  Measured, four contexts on four
// streams, us per round of calls, registers rounded up to one or two waves per SIMD ->
// this: FrodoKEM-976 encapsulation of 4096 5061 -> 2985 (one call 1295 -> 1260),
// decapsulation of 2048 2618 -> 1897 and of 4096 3418 -> 3162; NewHope-1024 CCA
// encapsulation of 3000 408 -> 320 and of 8000 836 -> 770.
#define PQC_WIDE_KERNEL(WG) \
  __launch_bounds__(64 * (WG)) __attribute__((amdgpu_waves_per_eu((WG) == 1 ? 1 : 4, (WG) == 1 ? 1 : 8)))

template <int WG>
__device__ __forceinline__ int wg_wave() {
  return WG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}
template <int WG>
__device__ __forceinline__ int wave_of() {
  return (int)blockIdx.x * WG + wg_wave<WG>();
}

// f(std::integral_constant<int, WG>) for a launch of `waves` waves on `cus` CUs
template <class F>
inline void with_wg(int cus, int waves, F&& f) {
  if (waves <= 2 * cus)
    f(std::integral_constant<int, 1>{});
  else if (waves <= 4 * cus)
    f(std::integral_constant<int, 4>{});
  else
    f(std::integral_constant<int, 8>{});
}
inline dim3 wg_grid(int waves, int wg) { return dim3((unsigned)((waves + wg - 1) / wg)); }

}  // namespace wide
}  // namespace pqc
