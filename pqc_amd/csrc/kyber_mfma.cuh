// Kyber polynomial arithmetic for 16 requests per wave, with the transforms on the
// matrix cores.
//
// The number-theoretic transform of a Kyber polynomial is two 128-point transforms,
// of its even and of its odd coefficients, by one matrix: X[f] = sum_j W[f][j] x[j],
// W[f][j] = zeta^((2 br7(f) + 1) j) mod q, and the inverse by V[j][f] = 128^-1
// zeta^(-(2 br7(f) + 1) j).  Both run as v_mfma_f32_16x16x32_f16 products that are
// exact: entries are centred (|w| <= 1664, exact in f16's 11 bits) and the data is
// small (noise, |x| <= 2) or split into two digits (x = 64 xh + xl), so that every
// sum of 128 products stays below 2^24 and FP32 accumulates it without rounding.
//
//   noise input        128 * 2 * 1664       = 0.43 M
//   residue, xh        128 * 26 * 1664      = 5.6 M     (|x| <= 1665 centred)
//   residue, xl        128 * 32 * 1664      = 6.9 M
//   12-bit value, xh   128 * 52 * 1664      = 11.1 M    (0 <= x < q, plain digits)
//   12-bit value, xl   128 * 63 * 1664      = 13.5 M    < 2^24 = 16.8 M
//
// A butterfly network on a wave (kyber_wavef.cuh) costs about 150 VALU instructions
// per polynomial, half of them lane swaps; here a polynomial's share is 20 to 45
// (operand conversion, digits, reduction of the sums) and the products run on the
// otherwise idle matrix cores.
//
// Layout.  Lane l = n + 16 g serves request n (0..15) of the wave's group.  A value
// index v (coefficient pair j, or frequency f, 0..127) sits in chunk t = v / 16 at
// 4 g + i: the accumulator layout of the 16 x 16 product (column n, rows 4 g + i).
// The product's K index may be permuted freely as long as both operands agree, so
// the constant operand is stored for the K order (t = 2s, 2s + 1; i) that the data
// already has: a transform's output is the next transform's input without a lane
// move.  Even and odd coefficients are two operands of the same lane, so chunk t of
// a lane is the 8 consecutive coefficients 8 c .. 8 c + 7, c = 4 t + g: every
// packing width reads and writes whole bytes per lane.
#pragma once
#include "kyber_f32.h"
#include "kyber_wave.cuh"
#include "kyber_wavef.cuh"

namespace pqc {
namespace kyber {
namespace mfma {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u3v __attribute__((ext_vector_type(3)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// f16 bit pattern of an integer |v| < 2048
constexpr uint16_t f16_bits(int v) {
  if (v == 0) return 0;
  const unsigned a = (unsigned)(v < 0 ? -v : v);
  int e = 0;
  while ((a >> e) > 1) ++e;
  return (uint16_t)((v < 0 ? 0x8000u : 0u) | (unsigned)(e + 15) << 10 | ((a << (10 - e)) & 0x3FFu));
}

// [tile of 16 output rows][step of 32 inputs][lane][8]: the constant operand's
// fragments in the order a wave reads them (16 bytes per lane, 1 KB per fragment).
struct DftTables {
  uint16_t fwd[8][4][64][8];
  uint16_t inv[8][4][64][8];
  float gamma[128];   // base multiplication twiddle of pair f, centred
  float gammaq[128];  // gamma / q
};
constexpr int kInv128 = 3303;
static_assert((128 * kInv128) % Q == 1, "128^-1");

constexpr DftTables make_dft_tables() {
  DftTables d{};
  int pw[256] = {};
  int x = 1;
  for (int i = 0; i < 256; ++i) {
    pw[i] = x;
    x = x * 17 % Q;
  }
  uint16_t wf[256] = {}, wi[256] = {};
  for (int i = 0; i < 256; ++i) {
    wf[i] = f16_bits(centred(pw[i]));
    wi[i] = f16_bits(centred(pw[(256 - i) & 255] * kInv128));
  }
  unsigned e[128] = {};
  for (unsigned f = 0; f < 128; ++f) {
    e[f] = 2 * brv7(f) + 1;
    d.gamma[f] = (float)centred(pw[e[f]]);
    d.gammaq[f] = d.gamma[f] / f32::kQf;
  }
  for (unsigned mt = 0; mt < 8; ++mt)
    for (unsigned s = 0; s < 4; ++s)
      for (unsigned l = 0; l < 64; ++l)
        for (unsigned i = 0; i < 8; ++i) {
          const unsigned m = 16 * mt + (l & 15), k = 16 * (2 * s + (i >> 2)) + 4 * (l >> 4) + (i & 3);
          d.fwd[mt][s][l][i] = wf[(e[m] * k) & 255];
          d.inv[mt][s][l][i] = wi[(e[k] * m) & 255];
        }
  return d;
}

// the LDS copy: which matrices a kernel needs
template <bool FWD, bool INV>
struct alignas(16) DftLds {
  u4v fwd[FWD ? 8 * 4 * 64 : 1];
  u4v inv[INV ? 8 * 4 * 64 : 1];
  float gamma[128], gammaq[128];
};

template <bool FWD, bool INV, int THREADS>
__device__ __forceinline__ void load_tables(DftLds<FWD, INV>& sh, const DftTables* __restrict__ d) {
  const u4v* f = reinterpret_cast<const u4v*>(d->fwd);
  const u4v* v = reinterpret_cast<const u4v*>(d->inv);
  for (int i = threadIdx.x; i < 8 * 4 * 64; i += THREADS) {
    if constexpr (FWD) sh.fwd[i] = f[i];
    if constexpr (INV) sh.inv[i] = v[i];
  }
  for (int i = threadIdx.x; i < 128; i += THREADS) {
    sh.gamma[i] = d->gamma[i];
    sh.gammaq[i] = d->gammaq[i];
  }
  __syncthreads();
}

// 128 + 128 values of one polynomial as packed f16 pairs: v[half][t][p] holds values
// i = 2p, 2p + 1 of chunk t (half 0: even coefficients, half 1: odd).
struct HPoly {
  uint32_t v[2][8][2];
};

__device__ __forceinline__ h8 operand(const HPoly& p, int half, int s) {
  u4v w = {p.v[half][2 * s][0], p.v[half][2 * s][1], p.v[half][2 * s + 1][0], p.v[half][2 * s + 1][1]};
  return __builtin_bit_cast(h8, w);
}

// Makes the packed values opaque: a loop that reads them must not keep their FP32
// conversions (twice the registers) across its iterations; v_fma_mix_f32 reads the
// halves directly.
__device__ __forceinline__ void keep_packed(HPoly& p) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < 8; ++t) asm volatile("" : "+v"(p.v[h][t][0]), "+v"(p.v[h][t][1]));
}

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));  // exact: integers below 2048
}
__device__ __forceinline__ uint32_t add_h2(uint32_t a, float c) {
  const h2 r = __builtin_bit_cast(h2, a) + (h2){(_Float16)c, (_Float16)c};
  return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ float h2_get(uint32_t a, int i) { return (float)__builtin_bit_cast(h2, a)[i]; }

// The products' fully unrolled loops would let the scheduler hoist every load to the
// front (and spill): a fence per tile keeps one tile's work together, with the next
// tile's constant fragments loaded behind this tile's products.
__device__ __forceinline__ void tile_fence() { __builtin_amdgcn_sched_barrier(0); }

// Two transforms in a row read the constant fragments from LDS each; without this the
// compiler keeps all 128 registers of them from one to the next.
__device__ __forceinline__ void fresh_fragments() { asm volatile("" ::: "memory"); }

struct Frags {
  u4v a[4];
  __device__ __forceinline__ void load(const u4v* __restrict__ m, int mt) {
#pragma unroll
    for (int s = 0; s < 4; ++s) a[s] = m[(mt * 4 + s) * 64 + lane_id()];
  }
};

// tile mt of M x for one-digit data: out(mt, even[4], odd[4]), the raw sums
template <class F>
__device__ __forceinline__ void dft1(const u4v* __restrict__ m, const HPoly& x, F&& out) {
  fresh_fragments();
  Frags f;
  f.load(m, 0);
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    f4v e = {0.f, 0.f, 0.f, 0.f}, o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const h8 a = __builtin_bit_cast(h8, f.a[s]);
      e = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, operand(x, 0, s), e, 0, 0, 0);
      o = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, operand(x, 1, s), o, 0, 0, 0);
    }
    tile_fence();
    if (mt + 1 < 8) f.load(m, mt + 1);
    out(mt, e, o);
    tile_fence();
  }
}

// the same for two-digit data x = 64 xh + xl: out gets the sums reduced (|.| <= 1665).
// pre(t) issues the loads that out(t) will need, two tiles ahead.
template <class Pre, class F>
__device__ __forceinline__ void dft2(const u4v* __restrict__ m, const HPoly& xh, const HPoly& xl, Pre&& pre, F&& out) {
  fresh_fragments();
  Frags f;
  f.load(m, 0);
  pre(0);
  pre(1);
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    if (mt + 2 < 8) pre(mt + 2);
    f4v hi[2], lo[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) hi[h] = lo[h] = (f4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const h8 a = __builtin_bit_cast(h8, f.a[s]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        hi[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, operand(xh, h, s), hi[h], 0, 0, 0);
        lo[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, operand(xl, h, s), lo[h], 0, 0, 0);
      }
    }
    tile_fence();
    if (mt + 1 < 8) f.load(m, mt + 1);
    // |64 red(hi) + lo| <= 64 * 1665 + 13.5 M < 2^24
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) hi[h][i] = f32::reduce_f(__builtin_fmaf(f32::reduce_f(hi[h][i]), 64.f, lo[h][i]));
    out(mt, hi[0], hi[1]);
    tile_fence();
  }
}

__device__ __forceinline__ void set_chunk(HPoly& p, int t, const f4v& e, const f4v& o) {
  p.v[0][t][0] = pack_h2(e[0], e[1]);
  p.v[0][t][1] = pack_h2(e[2], e[3]);
  p.v[1][t][0] = pack_h2(o[0], o[1]);
  p.v[1][t][1] = pack_h2(o[2], o[3]);
}

// chunk t of the two digits of reduced values: x = 64 xh + xl, |xh| <= 26, |xl| <= 32
__device__ __forceinline__ void set_digits(HPoly& ph, HPoly& pl, int t, const f4v& e, const f4v& o) {
  f4v eh, oh, el, ol;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    eh[i] = f32::round_mul(e[i], 1.f / 64.f);
    oh[i] = f32::round_mul(o[i], 1.f / 64.f);
    el[i] = __builtin_fmaf(eh[i], -64.f, e[i]);
    ol[i] = __builtin_fmaf(oh[i], -64.f, o[i]);
  }
  set_chunk(ph, t, eh, oh);
  set_chunk(pl, t, el, ol);
}

// ---- noise: 4 bytes (8 coefficients of 4 bits, cbd.cu:42-63) as f16 pairs ---------
// even[p] = coefficients 4p, 4p + 2 of the chunk, odd[p] = 4p + 1, 4p + 3
__device__ __forceinline__ void cbd_chunk(uint32_t (&even)[2], uint32_t (&odd)[2], uint32_t w) {
  const uint32_t d = (w & 0x55555555u) + ((w >> 1) & 0x55555555u);
  // nibble c: a - b + 4 in 2..6
  const uint32_t nib = ((d & 0x33333333u) | 0x44444444u) - ((d >> 2) & 0x33333333u);
  const uint32_t E = nib & 0x0F0F0F0Fu, O = (nib >> 4) & 0x0F0F0F0Fu;
  // bytes (n, 0x64) are f16 1024 + n
  constexpr uint32_t K64 = 0x64646464u;
  even[0] = add_h2(__builtin_amdgcn_perm(K64, E, 0x04010400u), -1028.f);
  even[1] = add_h2(__builtin_amdgcn_perm(K64, E, 0x04030402u), -1028.f);
  odd[0] = add_h2(__builtin_amdgcn_perm(K64, O, 0x04010400u), -1028.f);
  odd[1] = add_h2(__builtin_amdgcn_perm(K64, O, 0x04030402u), -1028.f);
}

// ---- 8 coefficients of D bits, chunk c of a polynomial -----------------------------
// The dwords that hold the chunk's D bytes, as loaded (no dword outside the ones
// with wanted bytes is read); the arithmetic on them comes where they are used.  Chunk
// c = 4 t + g starts 4 D t + D g bytes in: the lane's part is computed once per width
// (ChunkAt), the rest is an immediate offset.
template <int D>
struct Words {
  static constexpr int N = D == 12 ? 3 : D == 11 ? 4 : D == 10 ? 3 : D == 4 ? 1 : 2;
  uint32_t w[N];
};

template <int D>
struct ChunkAt {
  int off[Words<D>::N];  // byte offsets of the dwords of chunk g
  uint32_t sh;           // bits before the chunk in the first one
  __device__ __forceinline__ explicit ChunkAt(int g) {
    const int o = (D * g) & ~3, s = (D * g) & 3, nw = (s + D + 3) >> 2;  // dwords with wanted bytes
    sh = 8u * (uint32_t)s;
#pragma unroll
    for (int i = 0; i < Words<D>::N; ++i) off[i] = o + 4 * ((4 * i >= D && i >= nw) ? 0 : i);
  }
};

template <int D>
__device__ __forceinline__ void load_chunk(Words<D>& x, const uint8_t* poly, const ChunkAt<D>& at, int t) {
  if constexpr (D == 12) {
    const u3v v = *(const global_t<u3v>*)(poly + at.off[0] + 4 * D * t);
#pragma unroll
    for (int i = 0; i < 3; ++i) x.w[i] = v[i];
  } else {
#pragma unroll
    for (int i = 0; i < Words<D>::N; ++i) x.w[i] = *(const global_t<uint32_t>*)(poly + at.off[i] + 4 * D * t);
  }
}

template <int D>
__device__ __forceinline__ void unpack_chunk(uint32_t (&v)[8], const Words<D>& x, uint32_t sh) {
  constexpr int NW = (D + 3) / 4;  // dwords after alignment
  uint32_t a[NW + 1];
  if constexpr (D % 4 == 0) {
#pragma unroll
    for (int i = 0; i < NW; ++i) a[i] = x.w[i];
  } else {
#pragma unroll
    for (int i = 0; i < NW; ++i)
      a[i] = __builtin_amdgcn_alignbit(i + 1 < Words<D>::N ? x.w[i + 1] : 0u, x.w[i], sh);
  }
  a[NW] = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int b = D * k, wi = b >> 5, s = b & 31;
    const uint32_t r = s + D <= 32 ? a[wi] >> s : __builtin_amdgcn_alignbit(a[wi + 1], a[wi], s);
    v[k] = s + D == 32 ? r : r & ((1u << D) - 1);
  }
}

// D-bit values of a chunk to its D bytes at poly + D (4 t + g) (dword, then short / byte
// stores; unaligned global stores are single instructions on gfx950)
template <int D>
__device__ __forceinline__ void store_chunk(uint8_t* poly, int g, int t, const uint32_t (&v)[8]) {
  constexpr int NW = (D + 3) / 4;
  uint32_t a[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) a[i] = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int b = D * k, wi = b >> 5, s = b & 31;
    a[wi] |= v[k] << s;
    if (s + D > 32) a[wi + 1] |= v[k] >> (32 - s);
  }
  struct __attribute__((packed, aligned(1))) W4 { uint32_t v; };
  struct __attribute__((packed, aligned(1))) W2 { uint16_t v; };
  uint8_t* o = poly + D * g + 4 * D * t;
#pragma unroll
  for (int i = 0; i < D / 4; ++i) reinterpret_cast<W4*>(o + 4 * i)->v = a[i];
  if constexpr (D % 4 >= 2) reinterpret_cast<W2*>(o + (D & ~3))->v = (uint16_t)a[NW - 1];
  if constexpr (D % 2 == 1) o[D - 1] = (uint8_t)(a[NW - 1] >> (8 * ((D - 1) & 3)));
}

// ---- base multiplication (basemul2, poly.cu:204-225) ---------------------------------
// One chunk of sum_j a_j o b_j: even + gamma odd, and the cross sum, before reduction.
// With |a|, |b| <= 1665 up to kBasemulTerms products per odd coefficient accumulate
// exactly; the even coefficient's two sums take one product per j each.
struct ChunkSum {
  f4v s00, s11, s01;
};

__device__ __forceinline__ void chunk_zero(ChunkSum& s) {
  s.s00 = s.s11 = s.s01 = (f4v){0.f, 0.f, 0.f, 0.f};
}

// a[8]: the chunk's coefficients, reduced floats (even index: even coefficient)
__device__ __forceinline__ void chunk_mac(ChunkSum& s, const float (&a)[8], const HPoly& b, int t) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float b0 = h2_get(b.v[0][t][i >> 1], i & 1), b1 = h2_get(b.v[1][t][i >> 1], i & 1);
    s.s00[i] = __builtin_fmaf(a[2 * i], b0, s.s00[i]);
    s.s11[i] = __builtin_fmaf(a[2 * i + 1], b1, s.s11[i]);
    s.s01[i] = __builtin_fmaf(a[2 * i], b1, __builtin_fmaf(a[2 * i + 1], b0, s.s01[i]));
  }
}

// reduced (|.| <= 1665) pair values of the chunk
__device__ __forceinline__ void chunk_finish(const ChunkSum& s, const float* gamma, const float* gammaq, int t, int g,
                                             f4v& e, f4v& o) {
  const f4v z = *reinterpret_cast<const f4v*>(gamma + 16 * t + 4 * g);
  const f4v zq = *reinterpret_cast<const f4v*>(gammaq + 16 * t + 4 * g);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    e[i] = f32::reduce_f(s.s00[i] + f32::mulc(f32::reduce_f(s.s11[i]), z[i], zq[i]));
    o[i] = f32::reduce_f(s.s01[i]);
  }
}
static_assert(4 * f32::kOut * f32::kOut + f32::kOut < (1 << 24), "even sums of K = 4 terms stay exact");

}  // namespace mfma
}  // namespace kyber
}  // namespace pqc
