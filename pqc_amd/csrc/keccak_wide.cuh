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
// two waves per SIMD 4.8.  Its throughput is a fifth of the one-state-per-lane form's.
#pragma once
#include "keccak.cuh"

namespace pqc {
namespace wide {

constexpr int kRowWords = 8, kHalfWords = 5 * kRowWords, kStateWords = 2 * kHalfWords;

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
        m.dst[h][y][x] = (uint16_t)((h ^ (o & 1)) * kHalfWords + (2 * x + 3 * y) % 5 * kRowWords + y);
      }
  return m;
}
static __device__ const Maps c_maps = make_maps();
static __device__ const IlRc c_rc = il_round_constants();

// Constants of a workgroup's waves, and one wave's states
struct Consts {
  alignas(16) uint32_t zero[8];
  uint32_t trash[8];
  uint32_t rc[2][24], none[24];
};
struct States {
  alignas(16) uint32_t w[4 * kStateWords];
};

// every thread of the workgroup; a barrier must follow
__device__ __forceinline__ void init_consts(Consts& c) {
  const int t = threadIdx.x;
  if (t < 8) c.zero[t] = 0;
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
  const uint32_t* src;
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
      dst[x] = y < 5 ? base + c_maps.dst[h][y][x] : c.trash;
    }
    src = y < 5 ? base + h * kHalfWords + y * kRowWords : c.zero;
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

  __device__ __forceinline__ void permute() {
#pragma unroll 4
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
      const uint32_t B[5] = {q[0], q[1], q[2], q[3], src[4]};
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

  // this lane's halves of block b (17 words) of a message of nwords 64-bit words at the
  // 4-byte aligned p (the same one, or one per state), SHA3-256 / SHAKE256 padding included
  template <class P>
  __device__ __forceinline__ void load_block17(uint32_t (&m)[5], P p, int nwords, int b, uint32_t domain) const {
    const int rem = nwords - 17 * b;  // words left
#pragma unroll
    for (int x = 0; x < 5; ++x) {
      const int w = word(x);
      uint32_t v = 0;
      if (w < 17 && w < rem) v = p[2 * (17 * b + w) + h];
      if (w < 17 && w == rem && h == 0) v = domain;
      if (w == 16 && rem < 17 && h == 1) v ^= 0x80000000u;
      m[x] = v;
    }
  }
  // absorb blocks [b0, b1) of it, the next block's words loaded during a permutation
  template <class P>
  __device__ __forceinline__ void absorb17(P p, int nwords, uint32_t domain, int b0, int b1) {
    uint32_t m[5];
    load_block17(m, p, nwords, b0, domain);
    for (int b = b0; b < b1; ++b) {
      absorb(m);
      if (b + 1 < b1) load_block17(m, p, nwords, b + 1, domain);
      permute();
    }
  }
};

}  // namespace wide
}  // namespace pqc
