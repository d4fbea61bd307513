// NewHope CPA-PKE (N = 1024 and N = 512) as plain batched kernels
// (NewHope_NIST_GPU/cpapke.cu:265-476): one kernel per reference operation,
// and the NewHope CCA-KEM over them.  Polynomials are element-major (element
// x's N uint16 coefficients contiguous at x * N), and each kernel spreads an
// element over as many lanes as its data flow allows:
//   - NTT / inverse NTT: one wave per polynomial, N / 64 coefficients per lane
//     in VGPRs, the butterfly layers in register-resident groups (N = 1024:
//     index bits 0-3, 4-7, 8-9; N = 512: bits 0-2, 3-5, 6-8) with the
//     polynomial re-laid out through LDS between groups;
//   - poly_uniform / poly_sample: one lane per 64-coefficient SHAKE stream
//     (N / 64 per polynomial);
//   - pointwise, add/sub, (de)serialisation, (de)compression, message coding:
//     flat passes, one lane per 4 or 8 coefficients, 8- or 16-byte accesses.
//
// The 16-bit storage and 32-bit intermediate arithmetic of the reference are
// kept exactly (lazy even NTT levels stored as uint16, Barrett on a uint16
// argument at N = 1024 and % q at N = 512 on the odd levels, Montgomery with
// R = 2^18 in uint32), so results are identical for every input, including
// out-of-range ones.  N = 512 follows the reference's NEWHOPE_N == 512 branches
// (precomp.cu:75-190 tables, ntt.cu:130-180, poly.cu:244,279), which its
// batched GPU path never compiled.
#include <type_traits>

#include "internal.h"
#include "keccak_wide.cuh"
#include "newhope_f32.h"
#include "sponge.cuh"

namespace pqc {
namespace newhope {

constexpr uint32_t Q = 12289;
constexpr int SYM = 32;

// sizes of NewHope-N (params.h:26-39)
template <int N>
struct Par {
  static constexpr int POLYBYTES = 14 * N / 8;          // 1792 / 896
  static constexpr int CBYTES = 3 * N / 8;              // 384 / 192
  static constexpr int PK = POLYBYTES + SYM;            // 1824 / 928
  static constexpr int SK = POLYBYTES;                  // 1792 / 896
  static constexpr int CT = POLYBYTES + CBYTES;         // 2176 / 1088
  static constexpr int CCA_SK = SK + PK + 2 * SYM;      // 3680 / 1888: sk_cpa || pk || H(pk) || s
  static constexpr int CCA_CT = CT + SYM;               // 2208 / 1120: ct_cpa || d
  static constexpr int LOG = N == 1024 ? 10 : 9;
  static constexpr uint32_t G = N == 1024 ? 7 : 10968;  // precomp.cu: g = Mod(7 | 10968, q)
  static constexpr int STREAMS = N / 64;                // SHAKE streams per polynomial
  static constexpr int COPIES = N / 256;                // coefficients per message bit
};

// ---- tables: the Pari/GP definitions of precomp.cu:5-72 (mont = 2^18),
// evaluated at compile time ---------------------------------------------------
constexpr uint32_t powmod(uint32_t b, uint32_t e) {
  uint64_t r = 1, x = b % Q;
  while (e) {
    if (e & 1) r = r * x % Q;
    x = x * x % Q;
    e >>= 1;
  }
  return (uint32_t)r;
}

constexpr uint32_t bitrev(uint32_t i, int bits) {
  uint32_t r = 0;
  for (int b = 0; b < bits; b++) r |= ((i >> b) & 1u) << (bits - 1 - b);
  return r;
}

template <int N>
struct alignas(16) Tables {  // 16-byte aligned rows: read as uint4 by the NTT kernels
  uint16_t omegas_inv[N / 2];
  uint16_t gammas[N];
  uint16_t gammas_inv[N];
  uint16_t brv[N];
};

template <int N>
constexpr Tables<N> make_tables() {
  Tables<N> t{};
  constexpr int B = Par<N>::LOG;
  const uint32_t g = Par<N>::G, mont = (1u << 18) % Q;
  const uint32_t g2inv = powmod(g * g % Q, Q - 2), ginv = powmod(g, Q - 2), ninv = powmod(N, Q - 2);
  for (uint32_t k = 0; k < N / 2; k++) t.omegas_inv[k] = (uint16_t)((uint64_t)powmod(g2inv, bitrev(2 * k, B)) * mont % Q);
  for (uint32_t k = 0; k < N; k++) {
    t.gammas[k] = (uint16_t)((uint64_t)powmod(g, bitrev(k, B)) * mont % Q);
    t.gammas_inv[k] = (uint16_t)((uint64_t)powmod(ginv, k) * ninv % Q * mont % Q);
    t.brv[k] = (uint16_t)bitrev(k, B);
  }
  return t;
}

__constant__ Tables<1024> c_tab1024 = make_tables<1024>();
__constant__ Tables<512> c_tab512 = make_tables<512>();

template <int N>
__device__ __forceinline__ const Tables<N>& tab();
template <>
__device__ __forceinline__ const Tables<1024>& tab<1024>() { return c_tab1024; }
template <>
__device__ __forceinline__ const Tables<512>& tab<512>() { return c_tab512; }

// Plain centred twiddles of the bit-reversed-input, natural-output transforms whose layer
// L combines sub-transforms of 2^L points: entry 2^L + j belongs to output j of that layer.
// fwd holds g^((2 j + 1) N / 2^(L+1)): the products of the reference's gammas that its
// mul_coefficients and its layers apply one after another, as the powers they amount to.
// inv is the cyclic inverse's g^(-2 j N / 2^(L+1)), post its output scale g^-c / N.
template <int N>
constexpr float twiddle(bool inv, int L, int j) {
  const uint32_t e = (uint32_t)(N >> (L + 1)) * (uint32_t)(inv ? 2 * N - 2 * j : 2 * j + 1);
  const uint32_t v = powmod(Par<N>::G, e % (2 * N));
  return v > Q / 2 ? (float)((int)v - (int)Q) : (float)v;
}

template <int N>
struct alignas(16) TablesF {
  float fwd[N], inv[N], post[N];
};

template <int N>
constexpr TablesF<N> make_tables_f() {
  TablesF<N> t{};
  for (int L = 0; L < Par<N>::LOG; L++)
    for (int j = 0; j < (1 << L); j++) {
      t.fwd[(1 << L) + j] = twiddle<N>(false, L, j);
      t.inv[(1 << L) + j] = twiddle<N>(true, L, j);
    }
  const uint32_t ginv = powmod(Par<N>::G, Q - 2);
  uint32_t po = powmod(N, Q - 2);
  for (uint32_t k = 0; k < N; k++) {
    t.post[k] = po > Q / 2 ? (float)((int)po - (int)Q) : (float)po;
    po = (uint32_t)((uint64_t)po * ginv % Q);
  }
  return t;
}

__device__ const TablesF<1024> c_tabf1024 = make_tables_f<1024>();
__device__ const TablesF<512> c_tabf512 = make_tables_f<512>();

template <int N>
__device__ __forceinline__ const TablesF<N>& tabf() {
  if constexpr (N == 1024)
    return c_tabf1024;
  else
    return c_tabf512;
}

// floor(n / q) for n < 2^21: the high word of the 24-bit product n m with
// m = ceil(2^32 / q), one v_mul_hi_u32_u24 where the compiler's division by a
// constant takes five instructions.  Exact: n m / 2^32 = n / q + n e / (q 2^32)
// with e = m q - 2^32, and n e < 2^32.  Every operand here is below 2^17 (sums of
// two uint16 values, or of a uint16 value and 3q).  Written as the instruction
// itself because the compiler does not form it from C.
constexpr uint32_t kDivQM = (uint32_t)(((1ull << 32) + Q - 1) / Q);
static_assert(kDivQM < (1u << 24), "24-bit operand");
static_assert((((uint64_t)kDivQM * Q - (1ull << 32)) << 21) < (1ull << 32), "exact below 2^21");
static_assert(kDivQM == 0x55539u, "literal below");

__device__ __forceinline__ uint32_t div_q(uint32_t n) {
  uint32_t r;
  asm("v_mul_hi_u32_u24 %0, 0x55539, %1" : "=v"(r) : "v"(n));
  return r;
}

__device__ __forceinline__ uint32_t mod_q(uint32_t n) { return n - div_q(n) * Q; }

// reduce.cu:22-31
__device__ __forceinline__ uint32_t mont(uint32_t a) {
  uint32_t u = (a * 12287u) & ((1u << 18) - 1);
  u *= Q;
  a = a + u;
  return (a >> 18) & 0xFFFFu;
}

// reduce.cu:33-47 on a uint16 argument
__device__ __forceinline__ uint32_t barrett(uint32_t a16) {
  const uint32_t a = a16 & 0xFFFFu;
  const uint32_t u = ((a * 5) >> 16) * Q;
  return (a - u) & 0xFFFFu;
}

template <int N>
struct Pv {
  uint16_t* p;  // element x's coefficients at p + N x
  __device__ __forceinline__ uint16_t* el(int x) const { return p + (size_t)x * N; }
};

// ---- sponge kernels --------------------------------------------------------

// keypair seed expansion: z = SHAKE256(seed, 64) (cpapke.cu:283-298)
__global__ void k_seed_expand(int n, uint8_t* z, const uint8_t* seed, size_t seed_stride) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  uint64_t m[4], A[25];
#pragma unroll
  for (int w = 0; w < 4; ++w) m[w] = load_u64(seed + (size_t)x * seed_stride + 8 * w);
  absorb_fixed<kRateShake256, 4>(A, m, 0x1F);
#pragma unroll
  for (int w = 0; w < 8; ++w) store_u64(z + (size_t)x * 64 + 8 * w, A[w]);
}

// gen_a / poly_uniform (cpapke.cu:236-247, poly.cu:332-366): lane (x, i) runs
// SHAKE128(seed || i) and keeps 16-bit candidates < 5q for coefficients 64 i ..
// 64 i + 63.  Accepted values land at data-dependent positions, so each lane
// collects its 64 in its own LDS row (66 uint16: 33 words, rows on distinct
// banks) and then writes them out as eight 16-byte stores.  Fixed 128-lane
// workgroups (16.5 KB of LDS).
constexpr int kUniformBlock = 128;
constexpr int kUniformRow = 66;

template <int N>
__global__ __launch_bounds__(kUniformBlock) void k_uniform(int n, Pv<N> a, const uint8_t* seed, size_t stride) {
  constexpr int S = Par<N>::STREAMS;
  __shared__ uint16_t stage[kUniformBlock * kUniformRow];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int x = t / S, i = t % S;
  if (x >= n) return;  // no barrier below: every lane reads back only its own row
  uint16_t* row = stage + threadIdx.x * kUniformRow;
  uint64_t A[25];
#pragma unroll
  for (int w = 0; w < 25; ++w) A[w] = w < 4 ? load_u64(seed + (size_t)x * stride + 8 * w) : 0;
  A[4] = (uint64_t)i | (0x1Full << 8);
  A[kRateShake128 - 1] ^= 0x8000000000000000ull;
  int ctr = 0;
  for (int blk = 0; blk < 16 && ctr < 64; ++blk) {
    keccakf1600(A);
#pragma unroll
    for (int w = 0; w < kRateShake128; ++w) {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const uint32_t val = (uint32_t)(A[w] >> (16 * h)) & 0xFFFFu;
        if (val < 5 * Q && ctr < 64) row[ctr++] = (uint16_t)val;
      }
    }
  }
  const uint32_t* rw = reinterpret_cast<const uint32_t*>(row);
  uint4* dst = reinterpret_cast<uint4*>(a.el(x) + 64 * i);
#pragma unroll
  for (int q = 0; q < 8; ++q) dst[q] = make_uint4(rw[4 * q], rw[4 * q + 1], rw[4 * q + 2], rw[4 * q + 3]);
}

// poly_sample (poly.cu:396-444): lane (x, i) = coefficients 64 i .. 64 i + 63,
// hw(a) + q - hw(b) over SHAKE256(seed || nonce || i, 128)
template <int N>
__global__ void k_sample(int n, Pv<N> r, const uint8_t* seed, size_t stride, int nonce) {
  constexpr int S = Par<N>::STREAMS;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int x = t / S, i = t % S;
  if (x >= n) return;
  uint64_t s[4], A[25];
#pragma unroll
  for (int w = 0; w < 4; ++w) s[w] = load_u64(seed + (size_t)x * stride + 8 * w);
  absorb_fixed<kRateShake256, 4>(A, s, (uint64_t)nonce | ((uint64_t)i << 8) | (0x1Full << 16));
  uint4* dst = reinterpret_cast<uint4*>(r.el(x) + 64 * i);
#pragma unroll
  for (int w = 0; w < 16; w += 2) {
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint64_t word = A[w + (k >> 1)];
      const uint32_t ab0 = (uint32_t)(word >> (32 * (k & 1))) & 0xFFFFu;
      const uint32_t ab1 = (uint32_t)(word >> (32 * (k & 1) + 16)) & 0xFFFFu;
      const uint32_t c0 = (__popc(ab0 & 0xFF) + Q - __popc(ab0 >> 8)) & 0xFFFFu;
      const uint32_t c1 = (__popc(ab1 & 0xFF) + Q - __popc(ab1 >> 8)) & 0xFFFFu;
      o[k] = c0 | (c1 << 16);
    }
    dst[w >> 1] = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// ---- NTT kernels: one wave per polynomial ------------------------------------------

// One butterfly of ntt on 16-bit values: even layers keep the sum unreduced
// (stored as uint16), odd layers reduce it (MODE 1: Barrett, ntt.cu:195-234 at
// N = 1024; MODE 2: % q, ntt.cu:130-180 at N = 512); the difference is
// multiplied by W in Montgomery form.
template <int MODE>
__device__ __forceinline__ void bfly(uint32_t& a, uint32_t& b, uint32_t W) {
  const uint32_t t = a, h = b;
  a = MODE == 0 ? ((t + h) & 0xFFFFu) : MODE == 1 ? barrett(t + h) : mod_q(t + h);
  b = mont(W * (t + 3 * Q - h));
}

// Layer L (distance 2^L) on register pairs (r, r + 2^RB), RB the register bit
// that holds index bit L; the twiddle of index idx is omega[idx >> (L + 1)].
template <int R, int L, int RB, int ODD, typename IDX>
__device__ __forceinline__ void ntt_layer(uint32_t (&v)[R], const uint16_t* omega, IDX idx) {
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r & (1 << RB)) continue;
    const uint32_t W = omega[idx(r) >> (L + 1)];
    bfly<(L & 1) ? ODD : 0>(v[r], v[r + (1 << RB)], W);
  }
}

// ntt_core at N = 1024 on a polynomial that sits in LDS (sm) in ntt input
// order; returns the output in v with v[r] = coefficient 4 l + (r & 3) + 256 (r >> 2).
__device__ __forceinline__ void ntt_wave(uint32_t (&v)[16], uint16_t* sm, int l, const uint16_t* omega) {
  // layers 0-3: v[r] = index 16 l + r
  {
    const uint4 p0 = *reinterpret_cast<const uint4*>(sm + 16 * l), p1 = *reinterpret_cast<const uint4*>(sm + 16 * l + 8);
    const uint32_t w[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      v[2 * k] = w[k] & 0xFFFFu;
      v[2 * k + 1] = w[k] >> 16;
    }
  }
  auto ia = [l](int r) { return 16 * l + r; };
  ntt_layer<16, 0, 0, 1>(v, omega, ia);
  ntt_layer<16, 1, 1, 1>(v, omega, ia);
  ntt_layer<16, 2, 2, 1>(v, omega, ia);
  ntt_layer<16, 3, 3, 1>(v, omega, ia);
  {
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = v[2 * k] | (v[2 * k + 1] << 16);
    __syncthreads();
    *reinterpret_cast<uint4*>(sm + 16 * l) = make_uint4(w[0], w[1], w[2], w[3]);
    *reinterpret_cast<uint4*>(sm + 16 * l + 8) = make_uint4(w[4], w[5], w[6], w[7]);
    __syncthreads();
  }
  // layers 4-7: v[r] = index (l & 15) + 16 r + 256 (l >> 4)
  auto ib = [l](int r) { return (l & 15) + 16 * r + 256 * (l >> 4); };
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = sm[ib(r)];
  ntt_layer<16, 4, 0, 1>(v, omega, ib);
  ntt_layer<16, 5, 1, 1>(v, omega, ib);
  ntt_layer<16, 6, 2, 1>(v, omega, ib);
  ntt_layer<16, 7, 3, 1>(v, omega, ib);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) sm[ib(r)] = (uint16_t)v[r];
  __syncthreads();
  // layers 8-9: v[r] = index 4 l + (r & 3) + 256 (r >> 2)
  auto ic = [l](int r) { return 4 * l + (r & 3) + 256 * (r >> 2); };
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint2 p = *reinterpret_cast<const uint2*>(sm + 4 * l + 256 * q);
    v[4 * q] = p.x & 0xFFFFu;
    v[4 * q + 1] = p.x >> 16;
    v[4 * q + 2] = p.y & 0xFFFFu;
    v[4 * q + 3] = p.y >> 16;
  }
  ntt_layer<16, 8, 2, 1>(v, omega, ic);
  ntt_layer<16, 9, 3, 1>(v, omega, ic);
}

// ntt_core at N = 512 (nine layers): returns v[r] = coefficient l + 64 r.
__device__ __forceinline__ void ntt_wave(uint32_t (&v)[8], uint16_t* sm, int l, const uint16_t* omega) {
  // layers 0-2: v[r] = index 8 l + r
  {
    const uint4 p = *reinterpret_cast<const uint4*>(sm + 8 * l);
    const uint32_t w[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[2 * k] = w[k] & 0xFFFFu;
      v[2 * k + 1] = w[k] >> 16;
    }
  }
  auto ia = [l](int r) { return 8 * l + r; };
  ntt_layer<8, 0, 0, 2>(v, omega, ia);
  ntt_layer<8, 1, 1, 2>(v, omega, ia);
  ntt_layer<8, 2, 2, 2>(v, omega, ia);
  {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = v[2 * k] | (v[2 * k + 1] << 16);
    __syncthreads();
    *reinterpret_cast<uint4*>(sm + 8 * l) = make_uint4(w[0], w[1], w[2], w[3]);
    __syncthreads();
  }
  // layers 3-5: v[r] = index (l & 7) + 8 r + 64 (l >> 3)
  auto ib = [l](int r) { return (l & 7) + 8 * r + 64 * (l >> 3); };
#pragma unroll
  for (int r = 0; r < 8; ++r) v[r] = sm[ib(r)];
  ntt_layer<8, 3, 0, 2>(v, omega, ib);
  ntt_layer<8, 4, 1, 2>(v, omega, ib);
  ntt_layer<8, 5, 2, 2>(v, omega, ib);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 8; ++r) sm[ib(r)] = (uint16_t)v[r];
  __syncthreads();
  // layers 6-8: v[r] = index l + 64 r
  auto ic = [l](int r) { return l + 64 * r; };
#pragma unroll
  for (int r = 0; r < 8; ++r) v[r] = sm[ic(r)];
  ntt_layer<8, 6, 0, 2>(v, omega, ic);
  ntt_layer<8, 7, 1, 2>(v, omega, ic);
  ntt_layer<8, 8, 2, 2>(v, omega, ic);
}

// output position of register r of lane l after ntt_wave
template <int N>
__device__ __forceinline__ int out_index(int l, int r) {
  return N == 1024 ? 4 * l + (r & 3) + 256 * (r >> 2) : l + 64 * r;
}

template <int N>
__device__ __forceinline__ void store_out(const uint32_t (&v)[N / 64], uint16_t* el, int l) {
  if constexpr (N == 1024) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<uint2*>(el + 4 * l + 256 * q) =
          make_uint2(v[4 * q] | (v[4 * q + 1] << 16), v[4 * q + 2] | (v[4 * q + 3] << 16));
  } else {
#pragma unroll
    for (int r = 0; r < 8; ++r) el[l + 64 * r] = (uint16_t)v[r];
  }
}

// poly_ntt (poly.cu:519-527): mul_coefficients by gammas, then ntt with the same
// table.  Workgroup = one wave = one polynomial; lane l starts with
// coefficients (N / 64) l .. (N / 64) l + N / 64 - 1.
template <int N>
__global__ __launch_bounds__(64) void k_ntt(int n, Pv<N> r) {
  constexpr int C = N / 64;
  __shared__ __align__(16) uint16_t sm[N];
  const int x = blockIdx.x, l = threadIdx.x;
  if (x >= n) return;
  uint16_t* el = r.el(x);
  const uint4* src = reinterpret_cast<const uint4*>(el + C * l);
  const uint4* gam = reinterpret_cast<const uint4*>(tab<N>().gammas + C * l);
#pragma unroll
  for (int h = 0; h < C / 8; ++h) {
    const uint4 a = src[h], g = gam[h];
    const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, gw[4] = {g.x, g.y, g.z, g.w};
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      o[k] = mont((aw[k] & 0xFFFFu) * (gw[k] & 0xFFFFu)) | (mont((aw[k] >> 16) * (gw[k] >> 16)) << 16);
    *reinterpret_cast<uint4*>(sm + C * l + 8 * h) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  __syncthreads();
  uint32_t v[C];
  ntt_wave(v, sm, l, tab<N>().gammas);
  store_out<N>(v, el, l);
}

// poly_invntt (poly.cu:538-547): bitrev_vector, ntt with omegas_inv, then
// mul_coefficients by gammas_inv
template <int N>
__global__ __launch_bounds__(64) void k_invntt(int n, Pv<N> r) {
  constexpr int C = N / 64;
  __shared__ __align__(16) uint16_t sm[N];
  const int x = blockIdx.x, l = threadIdx.x;
  if (x >= n) return;
  uint16_t* el = r.el(x);
  const uint4* src = reinterpret_cast<const uint4*>(el + C * l);
  uint16_t raw[C];
#pragma unroll
  for (int h = 0; h < C / 8; ++h) {
    const uint4 a = src[h];
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      raw[8 * h + 2 * k] = (uint16_t)w[k];
      raw[8 * h + 2 * k + 1] = (uint16_t)(w[k] >> 16);
    }
  }
  // the coefficient at ntt input position i is the stored one at brv(i): write
  // stored coefficient c to position brv(c)
#pragma unroll
  for (int k = 0; k < C; ++k) sm[tab<N>().brv[C * l + k]] = raw[k];
  __syncthreads();
  uint32_t v[C];
  ntt_wave(v, sm, l, tab<N>().omegas_inv);
#pragma unroll
  for (int k = 0; k < C; ++k) v[k] = mont(v[k] * tab<N>().gammas_inv[out_index<N>(l, k)]);
  store_out<N>(v, el, l);
}

// ---- flat passes -------------------------------------------------------------------

// poly_mul_pointwise (poly.cu:455-468), 8 coefficients per lane
template <int N>
__global__ void k_pointwise(int n, Pv<N> r, Pv<N> a, Pv<N> b) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * (N / 8)) return;
  const uint4 av = reinterpret_cast<const uint4*>(a.p)[t], bv = reinterpret_cast<const uint4*>(b.p)[t];
  const uint32_t aw[4] = {av.x, av.y, av.z, av.w}, bw[4] = {bv.x, bv.y, bv.z, bv.w};
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t t0 = mont(3186u * (bw[k] & 0xFFFFu)), t1 = mont(3186u * (bw[k] >> 16));
    o[k] = mont((aw[k] & 0xFFFFu) * t0) | (mont((aw[k] >> 16) * t1) << 16);
  }
  reinterpret_cast<uint4*>(r.p)[t] = make_uint4(o[0], o[1], o[2], o[3]);
}

// poly_add / poly_sub (poly.cu:479-508), 8 coefficients per lane
template <int N>
__global__ void k_addsub(int n, Pv<N> r, Pv<N> a, Pv<N> b, int subtract) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * (N / 8)) return;
  const uint4 av = reinterpret_cast<const uint4*>(a.p)[t], bv = reinterpret_cast<const uint4*>(b.p)[t];
  const uint32_t aw[4] = {av.x, av.y, av.z, av.w}, bw[4] = {bv.x, bv.y, bv.z, bv.w};
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    uint32_t h[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t x = (aw[k] >> (16 * e)) & 0xFFFFu, y = (bw[k] >> (16 * e)) & 0xFFFFu;
      h[e] = mod_q(subtract ? x + 3 * Q - y : x + y);
    }
    o[k] = h[0] | (h[1] << 16);
  }
  reinterpret_cast<uint4*>(r.p)[t] = make_uint4(o[0], o[1], o[2], o[3]);
}

// ---- (de)serialisation --------------------------------------------------------

// coeff_freeze (poly.cu:21-33)
__device__ __forceinline__ uint32_t freeze(uint32_t x) {
  const uint32_t r = mod_q(x & 0xFFFFu);
  const uint32_t m = (r - Q) & 0xFFFFu;
  const uint32_t c = (uint32_t)((int32_t)(int16_t)m >> 15) & 0xFFFFu;
  return (m ^ ((r ^ m) & c)) & 0xFFFFu;
}

// flipabs (poly.cu:44-52)
__device__ __forceinline__ uint32_t flipabs(uint32_t x) {
  int32_t r = (int16_t)freeze(x);
  r = (int16_t)(r - (int32_t)(Q / 2));
  const int32_t m = (int16_t)(r >> 15);
  return (uint32_t)(uint16_t)((r + m) ^ m);
}

// poly_tobytes (poly.cu:105-127): lane (x, i) packs coefficients 4 i .. 4 i + 3
// into bytes 7 i .. 7 i + 6; lanes i < 4 also copy seed word i after the
// polynomial (encode_pk)
template <int N>
__global__ void k_tobytes(int n, uint8_t* dst, size_t stride, Pv<N> p, const uint8_t* seed, size_t seed_stride) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * (N / 4)) return;
  const int x = (int)(t / (N / 4)), i = (int)(t % (N / 4));
  const uint2 c = reinterpret_cast<const uint2*>(p.el(x))[i];
  const uint32_t t0 = freeze(c.x & 0xFFFFu), t1 = freeze(c.x >> 16), t2 = freeze(c.y & 0xFFFFu), t3 = freeze(c.y >> 16);
  uint8_t* r = dst + (size_t)x * stride + 7 * i;
  r[0] = (uint8_t)(t0 & 0xff);
  r[1] = (uint8_t)((t0 >> 8) | (t1 << 6));
  r[2] = (uint8_t)(t1 >> 2);
  r[3] = (uint8_t)((t1 >> 10) | (t2 << 4));
  r[4] = (uint8_t)(t2 >> 4);
  r[5] = (uint8_t)((t2 >> 12) | (t3 << 2));
  r[6] = (uint8_t)(t3 >> 6);
  if (seed && i < 4)
    store_u64(dst + (size_t)x * stride + Par<N>::POLYBYTES + 8 * i, load_u64(seed + (size_t)x * seed_stride + 8 * i));
}

// poly_frombytes (poly.cu:62-74): lane (x, i) unpacks bytes 7 i .. 7 i + 6;
// lanes i < 4 copy seed word i out (decode_pk)
template <int N>
__global__ void k_frombytes(int n, Pv<N> r, const uint8_t* src, size_t stride, uint8_t* seed_out) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * (N / 4)) return;
  const int x = (int)(t / (N / 4)), i = (int)(t % (N / 4));
  const uint8_t* a = src + (size_t)x * stride + 7 * i;
  const uint32_t c0 = a[0] | (((uint32_t)a[1] & 0x3f) << 8);
  const uint32_t c1 = (a[1] >> 6) | ((uint32_t)a[2] << 2) | (((uint32_t)a[3] & 0x0f) << 10);
  const uint32_t c2 = (a[3] >> 4) | ((uint32_t)a[4] << 4) | (((uint32_t)a[5] & 0x03) << 12);
  const uint32_t c3 = (a[5] >> 2) | ((uint32_t)a[6] << 6);
  reinterpret_cast<uint2*>(r.el(x))[i] = make_uint2((c0 & 0xFFFFu) | (c1 << 16), (c2 & 0xFFFFu) | ((c3 & 0xFFFFu) << 16));
  if (seed_out && i < 4)
    store_u64(seed_out + (size_t)x * 32 + 8 * i, load_u64(src + (size_t)x * stride + Par<N>::POLYBYTES + 8 * i));
}

// poly_compress (poly.cu:165-186): lane (x, g) packs coefficients 8 g .. 8 g + 7
// into ct + POLYBYTES + 3 g
template <int N>
__global__ void k_compress(int n, uint8_t* ct, size_t ct_stride, Pv<N> p) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * (N / 8)) return;
  const int x = (int)(t / (N / 8)), g = (int)(t % (N / 8));
  const uint4 c = reinterpret_cast<const uint4*>(p.el(x))[g];
  const uint32_t cw[4] = {c.x, c.y, c.z, c.w};
  uint32_t v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = div_q((freeze((cw[j >> 1] >> (16 * (j & 1))) & 0xFFFFu) << 3) + Q / 2) & 7;
  uint8_t* r = ct + (size_t)x * ct_stride + Par<N>::POLYBYTES + 3 * g;
  r[0] = (uint8_t)(v[0] | (v[1] << 3) | (v[2] << 6));
  r[1] = (uint8_t)((v[2] >> 2) | (v[3] << 1) | (v[4] << 4) | (v[5] << 7));
  r[2] = (uint8_t)((v[5] >> 1) | (v[6] << 2) | (v[7] << 5));
}

// poly_decompress (poly.cu:197-216): lane (x, g) = coefficients 8 g .. 8 g + 7
template <int N>
__global__ void k_decompress(int n, Pv<N> r, const uint8_t* ct, size_t ct_stride) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * (N / 8)) return;
  const int x = (int)(t / (N / 8)), g = (int)(t % (N / 8));
  const uint8_t* a = ct + (size_t)x * ct_stride + Par<N>::POLYBYTES + 3 * g;
  const uint32_t a0 = a[0], a1 = a[1], a2 = a[2];
  uint32_t v[8];
  v[0] = a0 & 7;
  v[1] = (a0 >> 3) & 7;
  v[2] = (a0 >> 6) | ((a1 << 2) & 4);
  v[3] = (a1 >> 1) & 7;
  v[4] = (a1 >> 4) & 7;
  v[5] = (a1 >> 7) | ((a2 << 1) & 6);
  v[6] = (a2 >> 2) & 7;
  v[7] = (a2 >> 5);
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    o[k] = (((v[2 * k] * Q + 4) >> 3) & 0xFFFFu) | ((((v[2 * k + 1] * Q + 4) >> 3) & 0xFFFFu) << 16);
  reinterpret_cast<uint4*>(r.el(x))[g] = make_uint4(o[0], o[1], o[2], o[3]);
}

// poly_frommsg_n (poly.cu:226-251): lane (x, i) spreads message byte i over
// coefficients 8 i + j + 256 q, q < N / 256
template <int N>
__global__ void k_frommsg(int n, Pv<N> r, const uint8_t* msg, size_t msg_stride) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * 32) return;
  const int x = t >> 5, i = t & 31;
  const uint32_t b = msg[(size_t)x * msg_stride + i];
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t v0 = (0u - ((b >> (2 * k)) & 1)) & (Q / 2), v1 = (0u - ((b >> (2 * k + 1)) & 1)) & (Q / 2);
    o[k] = v0 | (v1 << 16);
  }
#pragma unroll
  for (int q = 0; q < Par<N>::COPIES; ++q)
    reinterpret_cast<uint4*>(r.el(x) + 8 * i + 256 * q)[0] = make_uint4(o[0], o[1], o[2], o[3]);
}

// poly_tomsg_n (poly.cu:261-291): lane (x, i) decodes message byte i from the
// sum of flipabs over the N / 256 copies, compared with q (N = 1024) or q / 2
template <int N>
__global__ void k_tomsg(int n, uint8_t* msg, size_t msg_stride, Pv<N> p) {
  constexpr int CP = Par<N>::COPIES;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * 32) return;
  const int x = t >> 5, i = t & 31;
  uint32_t c[CP][8];
#pragma unroll
  for (int q = 0; q < CP; ++q) {
    const uint4 w = reinterpret_cast<const uint4*>(p.el(x) + 8 * i + 256 * q)[0];
    const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) c[q][j] = (ww[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
  }
  uint32_t byte = 0;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    uint32_t v = 0;
#pragma unroll
    for (int q = 0; q < CP; ++q) v += flipabs(c[q][j]);
    v = (v - (N == 1024 ? Q : Q / 2)) & 0xFFFFu;
    byte |= (v >> 15) << j;
  }
  msg[(size_t)x * msg_stride + i] = (uint8_t)byte;
}

// ---- fused per-element kernels: one wave per element ------------------------------
// Keypair, encryption and decryption each as one kernel.  The element's SHAKE
// streams run on the wave's lanes (one stream per lane), its polynomials stay in
// LDS or in VGPRs in ntt_wave's output layout, and HBM sees only the element's
// inputs and outputs.  The per-operation kernels above keep representatives below
// 2^16 of the residues mod q and lose none of them, these hold residues exactly in FP32,
// and every output is a function of residues alone: both paths give identical bytes.

// gen_a rows in LDS: 64 coefficients of one stream and the sampler's 4 spare slots, an odd
// number of words so that the lanes' stores fall on different banks
constexpr int kArow = 70;
static_assert(kArow >= 68 && kArow % 4 == 2, "spare slots, odd word count");

__device__ __forceinline__ int arow_index(int c) { return (c >> 6) * kArow + (c & 63); }

template <int N>
__device__ __forceinline__ int brv_index(int c) {
  return (int)(__builtin_bitreverse32((uint32_t)c) >> (32 - Par<N>::LOG));
}

// The fused kernels' transforms on FP32 values, in ntt_wave's register layouts, the
// exchanges between its register groups through an LDS buffer of floats.  Butterflies
// multiply first (a + z b, a - z b) and nothing is reduced on the way: a layer adds the
// bound of a product (the inverse's first register group, whose j = 0 butterflies take
// z = 1 without a product, doubles; newhope_f32.h has the bounds).  The weighting of the
// input is part of the twiddles, those of the first register group are literals and the
// others serve several butterflies, two polynomials at a time where there are two.  All of these kernels are
// bound by VALU issue (a wave's Keccak-f is 4320 of its ~7000 instructions).  Keypair,
// encryption and decryption of 16384 elements at N = 1024, us: 180, 215 and 50 with integer
// Montgomery layers and a branch per gen_a candidate; 160, 175 and 42 with these transforms
// and the branch-free sampler; keypair 136 with four elements per workgroup (below).
template <int N>
constexpr int kFxWords = N + N / 16;  // index i at i + i / 16: an exchange's lanes on different banks
__device__ __forceinline__ int fx(int i) { return i + (i >> 4); }

template <int R>
__device__ __forceinline__ void reduce_all(float (&v)[R]) {
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = fp::reduce(v[r]);
}

// layer L < log2(N / 64) on index (N / 64) l + r: the twiddle depends on r alone
template <int N, bool INV, int L, int P, int R = 0>
__device__ __forceinline__ void layer_low(float (&v)[P][N / 64]) {
  if constexpr (R < N / 64) {
    if constexpr ((R & (1 << L)) == 0) {
      constexpr float z = twiddle<N>(INV, L, R & ((1 << L) - 1));
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const float t = z == 1.0f ? v[p][R + (1 << L)] : fp::mul(v[p][R + (1 << L)], z, z * fp::kQinv);
        v[p][R + (1 << L)] = v[p][R] - t;
        v[p][R] += t;
      }
    }
    layer_low<N, INV, L, P, R + 1>(v);
  }
}

// layer L on index idx(r), whose bit L is register bit RB
template <int L, int RB, int P, int R, typename IDX>
__device__ __forceinline__ void layer_f(float (&v)[P][R], const float* __restrict__ tab, IDX idx) {
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r & (1 << RB)) continue;
    const float z = tab[(1 << L) + (idx(r) & ((1 << L) - 1))], zq = z * fp::kQinv;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const float t = fp::mul(v[p][r + (1 << RB)], z, zq);
      v[p][r + (1 << RB)] = v[p][r] - t;
      v[p][r] += t;
    }
  }
}

// orders one wave's LDS accesses: the wave's own are executed in program order, so only
// the compiler has to keep it
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// registers from index from(r) to index to(r), one polynomial after the other through buf
// (free before and after)
template <int P, int R, typename FROM, typename TO>
__device__ __forceinline__ void exchange(float (&v)[P][R], float* buf, FROM from, TO to) {
#pragma unroll
  for (int p = 0; p < P; ++p) {
#pragma unroll
    for (int r = 0; r < R; ++r) buf[fx(from(r))] = v[p][r];
    wave_sync();
#pragma unroll
    for (int r = 0; r < R; ++r) v[p][r] = buf[fx(to(r))];
    wave_sync();
  }
}

// P polynomials, v[p][r] = input index (N / 64) l + r -> v[p][r] = output coefficient
// out_index(l, r); buf is free before and after
template <int N, bool INV, int P>
__device__ __forceinline__ void transform_f(float (&v)[P][N / 64], float* buf, int l) {
  constexpr int C = N / 64;
  const float* tab = INV ? tabf<N>().inv : tabf<N>().fwd;
  auto ia = [l](int r) { return C * l + r; };
  auto ib = [l](int r) { return (l & (C - 1)) + C * r + C * C * (l / C); };
  auto ic = [l](int r) { return out_index<N>(l, r); };
  layer_low<N, INV, 0>(v);
  layer_low<N, INV, 1>(v);
  layer_low<N, INV, 2>(v);
  if constexpr (N == 1024) layer_low<N, INV, 3>(v);
  exchange(v, buf, ia, ib);
  if constexpr (N == 1024) {
    layer_f<4, 0>(v, tab, ib);
    layer_f<5, 1>(v, tab, ib);
    layer_f<6, 2>(v, tab, ib);
    layer_f<7, 3>(v, tab, ib);
  } else {
    layer_f<3, 0>(v, tab, ib);
    layer_f<4, 1>(v, tab, ib);
    layer_f<5, 2>(v, tab, ib);
  }
  exchange(v, buf, ib, ic);
  if constexpr (N == 1024) {
    layer_f<8, 2>(v, tab, ic);
    layer_f<9, 3>(v, tab, ic);
  } else {
    layer_f<6, 0>(v, tab, ic);
    layer_f<7, 1>(v, tab, ic);
    layer_f<8, 2>(v, tab, ic);
  }
}

// poly_ntt's input registers from the natural-order polynomial in sm
template <int N>
__device__ __forceinline__ void load_ntt(float (&v)[N / 64], const uint16_t* sm, int l) {
  constexpr int C = N / 64;
  const uint4* p = reinterpret_cast<const uint4*>(sm + C * l);
#pragma unroll
  for (int h = 0; h < C / 8; ++h) {
    const uint4 a = p[h];
    const uint32_t aw[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[8 * h + 2 * k] = (float)(aw[k] & 0xFFFFu);
      v[8 * h + 2 * k + 1] = (float)(aw[k] >> 16);
    }
  }
}

// poly_invntt of v[0][r] = coefficient out_index(l, r), |v| <= 2^14, in place
template <int N>
__device__ __forceinline__ void invntt_f(float (&v)[1][N / 64], float* buf, int l) {
  wave_sync();
  exchange(v, buf, [l](int r) { return brv_index<N>(out_index<N>(l, r)); }, [l](int r) { return (N / 64) * l + r; });
  transform_f<N, true>(v, buf, l);
#pragma unroll
  for (int r = 0; r < N / 64; ++r) v[0][r] = fp::mul(v[0][r], tabf<N>().post[out_index<N>(l, r)]);
}

// canonical residues to a natural-order uint16 polynomial
template <int N>
__device__ __forceinline__ void put_nat_f(uint16_t* sm, const float (&v)[N / 64], int l) {
#pragma unroll
  for (int r = 0; r < N / 64; ++r) sm[out_index<N>(l, r)] = (uint16_t)fp::canon(v[r]);
}

// One SHAKE stream on this lane: gen_a stream i (SHAKE128(seed || i), 16-bit
// candidates < 5q kept unreduced, poly.cu:332-366) when `uniform`, else
// poly_sample stream i (SHAKE256(seed || nonce || i, 128 bytes), hw(a) + q -
// hw(b), poly.cu:396-444).  Writes the stream's 64 coefficients to sm[off .. off + 63].
// Lanes that take no part pass active = false; every lane of the wave reaches
// the block loop's vote.
__device__ __forceinline__ void lane_stream(uint16_t* sm, uint32_t off, const uint64_t (&seed)[4], bool active,
                                            bool uniform, int nonce, int i) {
  uint64_t A[25];
#pragma unroll
  for (int w = 0; w < 25; ++w) A[w] = w < 4 ? seed[w] : 0;
  A[4] = uniform ? ((uint64_t)i | (0x1Full << 8)) : ((uint64_t)nonce | ((uint64_t)i << 8) | (0x1Full << 16));
  A[kRateShake128 - 1] ^= uniform ? 0x8000000000000000ull : 0;
  A[kRateShake256 - 1] ^= uniform ? 0 : 0x8000000000000000ull;
  keccakf1600_two(A);
  if (active && !uniform) {
#pragma unroll
    for (int w = 0; w < 16; w += 2) {
      uint32_t o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint64_t word = A[w + (k >> 1)];
        const uint32_t ab = (uint32_t)(word >> (32 * (k & 1)));
        const uint32_t c0 = __popc(ab & 0xFF) + Q - __popc(ab & 0xFF00);
        const uint32_t c1 = __popc(ab & 0xFF0000) + Q - __popc(ab & 0xFF000000);
        o[k] = c0 | (c1 << 16);
      }
      reinterpret_cast<uint4*>(sm + off)[w >> 1] = make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
  // branch-free: every candidate is written at the running position, which an accepted one
  // advances; the position is held at 64 after each word, so a row's slots 64..67 take what
  // comes after the 64th (a lane without a row has position 64 from the start)
  const uint32_t end = off + 64;
  uint32_t pos = (active && uniform) ? off : end;
  for (int blk = 0; blk < 16; ++blk) {
    if (blk > 0) {
      if (!__any(pos < end)) break;
      keccakf1600(A);
    }
    if (pos < end) {
#pragma unroll
      for (int w = 0; w < kRateShake128; ++w) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // two candidates per 32-bit half of the word
          const uint32_t val = (uint32_t)(A[w] >> (32 * h));
          sm[pos] = (uint16_t)val;
          pos += val << 16 < (5 * Q) << 16 ? 1 : 0;
          sm[pos] = (uint16_t)(val >> 16);
          pos += val < (5 * Q) << 16 ? 1 : 0;
        }
        pos = pos < end ? pos : end;
      }
    }
  }
}

// poly_frombytes of the 14-bit packing at src (8-byte aligned) into sm in
// natural order: group g (coefficients 4 g .. 4 g + 3) is bits 0..55 of the 7
// bytes at 7 g, read as one or two aligned words (never a word past the
// polynomial: only groups that straddle a word boundary read the next one)
template <int N>
__device__ __forceinline__ void unpack14(uint16_t* sm, const uint8_t* src, int l) {
  const uint64_t* s64 = reinterpret_cast<const uint64_t*>(src);
#pragma unroll
  for (int g = l; g < N / 4; g += 64) {
    const uint32_t bo = 7u * (uint32_t)g, sh = 8u * (bo & 7u);
    const uint64_t lo = s64[bo >> 3];
    const uint64_t hi = (bo & 7u) > 1u ? s64[(bo >> 3) + 1] : 0;
    const uint64_t w = sh ? (lo >> sh) | (hi << (64 - sh)) : lo;
    const uint32_t c0 = (uint32_t)w & 0x3FFFu, c1 = (uint32_t)(w >> 14) & 0x3FFFu;
    const uint32_t c2 = (uint32_t)(w >> 28) & 0x3FFFu, c3 = (uint32_t)(w >> 42) & 0x3FFFu;
    reinterpret_cast<uint2*>(sm)[g] = make_uint2(c0 | (c1 << 16), c2 | (c3 << 16));
  }
}

// poly_tobytes of the natural-order polynomial in sm (residues in [0, q)) into LDS bytes
// bb: lane l packs coefficients (N / 64) l .. (N / 64) (l + 1) - 1 into its 7 N / 256 bytes
template <int N>
__device__ __forceinline__ void pack14(uint8_t* bb, const uint16_t* sm, int l) {
  constexpr int C = N / 64;
  uint64_t g[C / 4];  // 56 bits of four coefficients each
#pragma unroll
  for (int h = 0; h < C / 4; ++h) {
    const uint2 c = reinterpret_cast<const uint2*>(sm + C * l)[h];
    const uint32_t lo = (c.x & 0xFFFFu) | (c.x >> 16 << 14), hi = (c.y & 0xFFFFu) | (c.y >> 16 << 14);
    g[h] = lo | ((uint64_t)hi << 28);
  }
  if constexpr (C == 16) {
    uint32_t* w = reinterpret_cast<uint32_t*>(bb) + 7 * l;
    w[0] = (uint32_t)g[0];
    w[1] = (uint32_t)(g[0] >> 32) | ((uint32_t)g[1] << 24);
    w[2] = (uint32_t)(g[1] >> 8);
    w[3] = (uint32_t)(g[1] >> 40) | ((uint32_t)g[2] << 16);
    w[4] = (uint32_t)(g[2] >> 16);
    w[5] = (uint32_t)(g[2] >> 48) | ((uint32_t)g[3] << 8);
    w[6] = (uint32_t)(g[3] >> 24);
  } else {
    uint16_t* w = reinterpret_cast<uint16_t*>(bb) + 7 * l;
    w[0] = (uint16_t)g[0];
    w[1] = (uint16_t)(g[0] >> 16);
    w[2] = (uint16_t)(g[0] >> 32);
    w[3] = (uint16_t)((uint32_t)(g[0] >> 48) | ((uint32_t)g[1] << 8));
    w[4] = (uint16_t)(g[1] >> 8);
    w[5] = (uint16_t)(g[1] >> 24);
    w[6] = (uint16_t)(g[1] >> 40);
  }
}

// poly_compress of the natural-order polynomial in sm (residues in [0, q)) into LDS bytes bb
template <int N>
__device__ __forceinline__ void compress3(uint8_t* bb, const uint16_t* sm, int l) {
#pragma unroll
  for (int g = l; g < N / 8; g += 64) {
    const uint4 c = reinterpret_cast<const uint4*>(sm)[g];
    const uint32_t cw[4] = {c.x, c.y, c.z, c.w};
    uint32_t v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = div_q((((cw[j >> 1] >> (16 * (j & 1))) & 0xFFFFu) << 3) + Q / 2) & 7;
    uint8_t* r = bb + 3 * g;
    r[0] = (uint8_t)(v[0] | (v[1] << 3) | (v[2] << 6));
    r[1] = (uint8_t)((v[2] >> 2) | (v[3] << 1) | (v[4] << 4) | (v[5] << 7));
    r[2] = (uint8_t)((v[5] >> 1) | (v[6] << 2) | (v[7] << 5));
  }
}

// poly_decompress of the 3-bit packing at src into sm in natural order
template <int N>
__device__ __forceinline__ void decompress3(uint16_t* sm, const uint8_t* src, int l) {
#pragma unroll
  for (int g = l; g < N / 8; g += 64) {
    const uint8_t* a = src + 3 * g;
    const uint32_t a0 = a[0], a1 = a[1], a2 = a[2];
    uint32_t v[8];
    v[0] = a0 & 7;
    v[1] = (a0 >> 3) & 7;
    v[2] = (a0 >> 6) | ((a1 << 2) & 4);
    v[3] = (a1 >> 1) & 7;
    v[4] = (a1 >> 4) & 7;
    v[5] = (a1 >> 7) | ((a2 << 1) & 6);
    v[6] = (a2 >> 2) & 7;
    v[7] = (a2 >> 5);
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      o[k] = (((v[2 * k] * Q + 4) >> 3) & 0xFFFFu) | ((((v[2 * k + 1] * Q + 4) >> 3) & 0xFFFFu) << 16);
    reinterpret_cast<uint4*>(sm)[g] = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// `bytes` (a multiple of 8) from LDS to global memory (8-byte aligned), one
// word per lane per step
__device__ __forceinline__ void copy_out(uint8_t* dst, const uint8_t* bb, int bytes, int l) {
  for (int w = l; w < bytes / 8; w += 64) store_u64(dst + 8 * w, reinterpret_cast<const uint64_t*>(bb)[w]);
}

// Keypair and encryption run in workgroups of four waves, four elements.  A wave's
// transforms are its own element's; the SHAKE streams of the four lie side by side on the
// workgroup's lanes, ordered by kind, so that a wave's lanes are all in use (alone, an
// element fills 48 or 64 of them at N = 1024, 24 or 32 at N = 512) and only the waves that
// hold gen_a streams step through its candidates.  The waves left without streams rotate
// with the workgroup, whose waves sit on the same SIMDs each time.
constexpr int kElems = 4;

// Runs the workgroup's streams: stream t is stream i of kind `kind` (0 gen_a, then the
// KINDS - 1 nonces) of element el, whose coefficients go to sm[el ES + off(kind, i)];
// seed(x, kind) is its seed.  Elements past n take part with the last one's seed and write
// nothing.
template <int N, int KINDS, int ES, typename SEED, typename OFF>
__device__ __forceinline__ void run_streams(uint16_t* sm, int n, SEED seed, OFF off) {
  constexpr int S = Par<N>::STREAMS, T = kElems * S * KINDS;
  const int t = (threadIdx.x + 64 * (blockIdx.x % kElems)) % (64 * kElems);
  if ((t & ~63) < T) {
    const int kind = t / (kElems * S), el = t / S % kElems, i = t % S;
    const int x = (int)blockIdx.x * kElems + el;
    const uint8_t* src = seed(x < n ? x : n - 1, kind < KINDS ? kind : 0);
    uint64_t sd[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) sd[w] = load_u64(src + 8 * w);
    lane_stream(sm, (uint32_t)(el * ES + off(kind, i)), sd, t < T && x < n, kind == 0, kind - 1, i);
  }
  __syncthreads();
}

// cpapke_keypair (cpapke.cu:265-338) for element kElems blockIdx.x + wave, from z =
// publicseed || noiseseed = SHAKE256(seed, 64) at z + 64 x (k_seed_expand: the one serial
// permutation stays on one lane per element).  Streams: gen_a, s (nonce 0), e (nonce 1).
template <int N>
__global__ __launch_bounds__(64 * kElems, 4) void k_keypair_fused(int n, uint8_t* pk, uint8_t* sk, size_t sk_stride,
                                                                  const uint8_t* z) {
  using P = Par<N>;
  constexpr int C = N / 64, S = P::STREAMS;
  // per element: gen_a rows | s | e; the transforms' buffer lies over s and e
  constexpr int ES = S * kArow + 2 * kFxWords<N>;
  static_assert(S * kArow % 8 == 0 && ES % 8 == 0, "16-byte rows");
  __shared__ __align__(16) uint16_t sm[kElems * ES];
  run_streams<N, 3, ES>(
      sm, n, [z](int x, int kind) { return z + (size_t)x * 64 + (kind ? 32 : 0); },
      [](int kind, int i) { return kind ? S * kArow + N * (kind - 1) + 64 * i : kArow * i; });
  const int l = threadIdx.x & 63, el = threadIdx.x >> 6, x = (int)blockIdx.x * kElems + el;
  if (x >= n) return;
  uint16_t *const sa = sm + el * ES, *const ss = sa + S * kArow, *const se = ss + N;
  float* const buf = reinterpret_cast<float*>(ss);
  float v[2][C];  // s, then e + s o a
  load_ntt<N>(v[0], ss, l);
  load_ntt<N>(v[1], se, l);
  wave_sync();
  transform_f<N, false>(v, buf, l);
  reduce_all(v[0]);
  // b = e + s o a (k_pointwise(AS, SHAT, AHAT), k_addsub(BHAT, EHAT, AS))
#pragma unroll
  for (int r = 0; r < C; ++r) v[1][r] += fp::mul((float)sa[arow_index(out_index<N>(l, r))], v[0][r]);
  put_nat_f<N>(ss, v[0], l);
  put_nat_f<N>(se, v[1], l);
  wave_sync();
  uint8_t* const bb = reinterpret_cast<uint8_t*>(sa);
  pack14<N>(bb, ss, l);
  wave_sync();
  copy_out(sk + (size_t)x * sk_stride, bb, P::POLYBYTES, l);
  wave_sync();
  pack14<N>(bb, se, l);
  wave_sync();
  uint8_t* pkx = pk + (size_t)x * P::PK;
  copy_out(pkx, bb, P::POLYBYTES, l);
  if (l < 4) store_u64(pkx + P::POLYBYTES + 8 * l, load_u64(z + (size_t)x * 64 + 8 * l));
}

// cpapke_enc (cpapke.cu:353-429) for element kElems blockIdx.x + wave.  Streams: gen_a of
// the public seed, then s', e', e'' (coin, nonces 0, 1, 2).
template <int N>
__global__ __launch_bounds__(64 * kElems, 4) void k_enc_fused(int n, uint8_t* ct, size_t ct_stride, const uint8_t* m,
                                                              size_t m_stride, const uint8_t* pk, size_t pk_stride,
                                                              const uint8_t* coin, size_t coin_stride) {
  using P = Par<N>;
  constexpr int C = N / 64, S = P::STREAMS;
  // per element: gen_a rows | e'' | s' | e'; the transforms' buffer lies over s' and e'
  constexpr int ES = S * kArow + N + 2 * kFxWords<N>;
  static_assert(S * kArow % 8 == 0 && ES % 8 == 0, "16-byte rows");
  __shared__ __align__(16) uint16_t sm[kElems * ES];
  run_streams<N, 4, ES>(
      sm, n,
      [=](int x, int kind) {
        return kind ? coin + (size_t)x * coin_stride : pk + (size_t)x * pk_stride + P::POLYBYTES;
      },
      [](int kind, int i) { return kind ? S * kArow + N * (kind % 3) + 64 * i : kArow * i; });
  const int l = threadIdx.x & 63, el = threadIdx.x >> 6, x = (int)blockIdx.x * kElems + el;
  if (x >= n) return;
  uint16_t *const sa = sm + el * ES, *const s3 = sa + S * kArow, *const s1 = s3 + N, *const s2 = s1 + N;
  float* const buf = reinterpret_cast<float*>(s1);
  float vv[1][C];
  {
    // u = a o s' + e' (k_pointwise(UHAT, AHAT, SP), k_addsub(UHAT, UHAT, EP)),
    // parked in natural order over the gen_a rows once every lane has read them
    float v[2][C];  // s', then u
    load_ntt<N>(v[0], s1, l);
    load_ntt<N>(v[1], s2, l);
    wave_sync();
    transform_f<N, false>(v, buf, l);
    reduce_all(v[0]);
#pragma unroll
    for (int r = 0; r < C; ++r) v[1][r] += fp::mul((float)sa[arow_index(out_index<N>(l, r))], v[0][r]);
    wave_sync();
    put_nat_f<N>(sa, v[1], l);
    unpack14<N>(s1, pk + (size_t)x * pk_stride, l);  // b (decode_pk)
    wave_sync();
    // v' = invntt(b o s') (k_pointwise(VP, BHAT, SP), k_invntt)
#pragma unroll
    for (int r = 0; r < C; ++r) vv[0][r] = fp::mul((float)s1[out_index<N>(l, r)], v[0][r]);
  }
  invntt_f<N>(vv, buf, l);
  // v = v' + e'' + frommsg(m) (k_addsub twice, k_frommsg)
  // Coefficient c takes message bit c mod 256: at N = 1024 a lane's bits are one nibble
  const uint8_t* mx = m + (size_t)x * m_stride;
  uint64_t mw[N == 1024 ? 1 : 4];
#pragma unroll
  for (int w = 0; w < (N == 1024 ? 1 : 4); ++w) mw[w] = load_u64(mx + 8 * (N == 1024 ? l >> 4 : w));
#pragma unroll
  for (int r = 0; r < C; ++r) {
    const int c = out_index<N>(l, r);
    const uint32_t bit = (uint32_t)(N == 1024 ? mw[0] >> (4 * (l & 15) + (r & 3)) : mw[r & 3] >> l) & 1u;
    vv[0][r] += (float)(s3[c] + ((0u - bit) & (Q / 2)));
  }
  wave_sync();
  put_nat_f<N>(s3, vv[0], l);
  wave_sync();
  pack14<N>(reinterpret_cast<uint8_t*>(s2), sa, l);
  compress3<N>(reinterpret_cast<uint8_t*>(s1), s3, l);
  wave_sync();
  uint8_t* ctx_ = ct + (size_t)x * ct_stride;
  copy_out(ctx_, reinterpret_cast<const uint8_t*>(s2), P::POLYBYTES, l);
  copy_out(ctx_ + P::POLYBYTES, reinterpret_cast<const uint8_t*>(s1), P::CBYTES, l);
}

// cpapke_dec (cpapke.cu:443-476) for element blockIdx.x
template <int N>
__global__ __launch_bounds__(64) void k_dec_fused(int n, uint8_t* m, size_t m_stride, const uint8_t* ct,
                                                  size_t ct_stride, const uint8_t* sk, size_t sk_stride) {
  using P = Par<N>;
  constexpr int C = N / 64;
  __shared__ __align__(16) float buf[kFxWords<N>];  // over s1 and s2
  __shared__ __align__(16) uint16_t s3[N];
  uint16_t *const s1 = reinterpret_cast<uint16_t*>(buf), *const s2 = s1 + N;
  const int x = blockIdx.x, l = threadIdx.x;
  if (x >= n) return;
  const uint8_t* ctx_ = ct + (size_t)x * ct_stride;
  unpack14<N>(s1, sk + (size_t)x * sk_stride, l);
  unpack14<N>(s2, ctx_, l);
  decompress3<N>(s3, ctx_ + P::POLYBYTES, l);
  __syncthreads();
  // tmp = invntt(s o u) - v (k_pointwise(TMP, SHAT, UHAT), k_invntt, k_addsub(TMP, TMP, VP, 1))
  float vt[1][C];
#pragma unroll
  for (int r = 0; r < C; ++r) {
    const int c = out_index<N>(l, r);
    vt[0][r] = fp::mul((float)s1[c], (float)s2[c]);
  }
  invntt_f<N>(vt, buf, l);
#pragma unroll
  for (int r = 0; r < C; ++r) vt[0][r] -= (float)s3[out_index<N>(l, r)];
  __syncthreads();
  put_nat_f<N>(s2, vt[0], l);
  __syncthreads();
  // poly_tomsg: byte i from the N / 256 copies of coefficients 8 i + j
  if (l < 32) {
    uint32_t byte = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      uint32_t v = 0;
#pragma unroll
      for (int q = 0; q < Par<N>::COPIES; ++q) v += flipabs(s2[8 * l + j + 256 * q]);
      v = (v - (N == 1024 ? Q : Q / 2)) & 0xFFFFu;
      byte |= (v >> 15) << j;
    }
    m[(size_t)x * m_stride + l] = (uint8_t)byte;
  }
}

// ---- CCA-KEM glue: one lane per element for the sponges, flat copies -------------

// out[x] = SHAKE256(in[x], 8 words bytes), first 8 OW bytes
template <int OW>
__global__ void k_shake256_words(int n, uint8_t* out, size_t out_stride, const uint8_t* in, size_t in_stride,
                                 int words) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  uint64_t A[25];
  sponge_absorb_words<kRateShake256>(A, reinterpret_cast<const uint64_t*>(in + (size_t)x * in_stride), words, 0x1F);
#pragma unroll
  for (int w = 0; w < OW; ++w) store_u64(out + (size_t)x * out_stride + 8 * w, A[w]);
}

// The same on a lane pair per element (lane 2x + h holds half h of every state
// word, keccakf1600_pair): the latency form for the long serial absorbs of a
// public key or a ciphertext (14 to 17 Keccak-f), with twice the lanes at work
template <int OW>
__global__ void k_shake256_pair(int n, uint8_t* out, size_t out_stride, const uint8_t* in, size_t in_stride,
                                int words) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int x = t >> 1;
  const uint32_t half = (uint32_t)(t & 1);
  if (x >= n) return;  // both lanes of a pair leave together (2n lanes, even)
  uint32_t S[25];
  absorb_range_pair(S, in + (size_t)x * in_stride, words, 0, words / kRateShake256 + 1, 0x1F, half);
  uint32_t* o = reinterpret_cast<uint32_t*>(out + (size_t)x * out_stride);
#pragma unroll
  for (int w = 0; w < OW; ++w) o[2 * w + half] = S[w];
}

// out[x] = SHAKE256(a[x] (32 bytes) || b[x] (32 bytes)), first 8 OW bytes
template <int OW>
__global__ void k_shake256_2x32(int n, uint8_t* out, size_t out_stride, const uint8_t* a, size_t a_stride,
                                const uint8_t* b, size_t b_stride) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  uint64_t m[8], A[25];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    m[w] = load_u64(a + (size_t)x * a_stride + 8 * w);
    m[4 + w] = load_u64(b + (size_t)x * b_stride + 8 * w);
  }
  absorb_fixed<kRateShake256, 8>(A, m, 0x1F);
#pragma unroll
  for (int w = 0; w < OW; ++w) store_u64(out + (size_t)x * out_stride + 8 * w, A[w]);
}

// dst[x][0 .. 8 words) = src[x][0 .. 8 words), one lane per word
__global__ void k_copy_words(int n, uint8_t* dst, size_t dst_stride, const uint8_t* src, size_t src_stride,
                             int words) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * words) return;
  const size_t x = t / words, w = t % words;
  store_u64(dst + x * dst_stride + 8 * w, load_u64(src + x * src_stride + 8 * w));
}

// fail[x] = 1 if a[x] and b[x] differ anywhere in `words` words, else 0: one wave
// per element, no early exit (verify.cu:15-28 without its data-dependent branch)
__global__ __launch_bounds__(64) void k_verify_words(int n, uint32_t* fail, size_t fail_stride, const uint8_t* a,
                                                    size_t a_stride, const uint8_t* b, size_t b_stride, int words) {
  const int x = blockIdx.x;
  if (x >= n) return;
  const uint64_t* pa = reinterpret_cast<const uint64_t*>(a + (size_t)x * a_stride);
  const uint64_t* pb = reinterpret_cast<const uint64_t*>(b + (size_t)x * b_stride);
  uint64_t d = 0;
  for (int w = threadIdx.x; w < words; w += 64) d |= pa[w] ^ pb[w];
  const bool any = __any(d != 0);
  if (threadIdx.x == 0) *reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(fail) + (size_t)x * fail_stride) = any;
}

// k[x] = fail ? z[x] : k[x], 32 bytes, by mask (verify.cu:40-50 cmov)
__global__ void k_cmov32(int n, uint8_t* k, size_t k_stride, const uint8_t* z, size_t z_stride, const uint32_t* fail,
                         size_t fail_stride) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * 4) return;
  const size_t x = t >> 2, w = t & 3;
  const uint64_t f = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(fail) + x * fail_stride);
  const uint64_t mask = 0ull - (f & 1);
  uint8_t* pk = k + x * k_stride + 8 * w;
  store_u64(pk, (load_u64(pk) & ~mask) | (load_u64(z + x * z_stride + 8 * w) & mask));
}

// Per-element CCA scratch row (one size for both N): mu or m' | H(pk) |
// K || coin || d | H(c) | fail | re-encrypted ct
constexpr int KM_MU = 0, KM_HPK = 32, KM_KCD = 64, KM_HC = 160, KM_FAIL = 192, KM_CT2 = 224;
static_assert(KM_CT2 + Par<1024>::CCA_CT == kNewhopeKemBytes, "scratch row size");

// ---- the CCA-KEM's hashes on 16 lanes per element (keccak_wide.cuh) ----------------
// Up to kWideMax elements the sponges above are serial chains on a few waves, and every
// step between two of them is a launch of its own.  Here four elements share a wave, and
// the copies, the comparison and the selection belong to the kernel that hashes next to
// them.  One encapsulation and decapsulation per element, us, lane-pair form -> this one:
// N = 512: 308 -> 141 (7 elements), 323 -> 161 (3001), 368 -> 274 (8192), 490 -> 548
// (16384: the pair form's 512 waves are still one per SIMD, these would be four);
// N = 1024: 506 -> 211, 530 -> 260, 585 -> 439, 753 -> 905.
constexpr int kWideMax = 8192;
// Decapsulation's H(c) runs beside the decryption and re-encryption.  Above this the
// lane-pair form still ends before they do and leaves them more of the chip: N = 1024, 8000
// elements, one call 189 us either way, two calls side by side 428 -> 344.
constexpr int kSideWideMax = 4096;

struct Wide4 {  // one wave's
  wide::States states;
  alignas(16) uint32_t dig[4][16];  // per element: the words of its next short message
};

// out[x] = SHAKE256(in[x], 8 words bytes), 32 bytes
template <int WG>
__global__ PQC_WIDE_KERNEL(WG) void k_shake256_wide(int n, uint8_t* out, size_t out_stride,
                                                                        const uint8_t* in, size_t in_stride,
                                                                        int words) {
  __shared__ wide::Consts consts;
  __shared__ Wide4 lds[WG];
  wide::init_consts(consts);
  __syncthreads();
  if (WG > 1 && 4 * wide::wave_of<WG>() >= n) return;
  Wide4& sh = lds[wide::wg_wave<WG>()];
  wide::Sponge s;
  s.init(sh.states, consts);
  const int rq = 4 * wide::wave_of<WG>() + s.st, r = rq < n ? rq : n - 1;
  s.absorb17<24>(reinterpret_cast<const uint32_t*>(in + (size_t)r * in_stride), words, 0x1F, 0, words / 17 + 1);
  uint32_t* o = reinterpret_cast<uint32_t*>(out + (size_t)r * out_stride);
  s.squeeze<4>([&](int x, uint32_t v) {
    if (rq < n && s.y == 0) o[2 * x + s.h] = v;
  });
}

// (K || coin || d) = SHAKE256(mu || H(pk), 96).  Encapsulation (ENC): mu = H(in[x], 32
// bytes), kept in the row, and H(pk) of the public key key[x] (words 64-bit words);
// decapsulation: m' of the row and the H(pk) that key[x] holds.
template <int WG, bool ENC>
__global__ PQC_WIDE_KERNEL(WG) void k_cca_open_wide(int n, uint8_t* km, const uint8_t* in,
                                                                        const uint8_t* key, size_t key_stride,
                                                                        int words) {
  __shared__ wide::Consts consts;
  __shared__ Wide4 lds[WG];
  wide::init_consts(consts);
  __syncthreads();
  if (WG > 1 && 4 * wide::wave_of<WG>() >= n) return;
  Wide4& sh = lds[wide::wg_wave<WG>()];
  wide::Sponge s;
  s.init(sh.states, consts);
  const int rq = 4 * wide::wave_of<WG>() + s.st, r = rq < n ? rq : n - 1;
  const bool act = rq < n;
  uint32_t* row = reinterpret_cast<uint32_t*>(km + (size_t)r * kNewhopeKemBytes);
  const uint32_t* kp = reinterpret_cast<const uint32_t*>(key + (size_t)r * key_stride);
  uint32_t* dig = sh.dig[s.st];
  if constexpr (ENC) {
    s.absorb17(reinterpret_cast<const uint32_t*>(in + (size_t)r * 32), 4, 0x1F, 0, 1);
    s.squeeze<4>([&](int x, uint32_t v) {
      if (s.y == 0) dig[2 * x + s.h] = v;
      if (act && s.y == 0) row[KM_MU / 4 + 2 * x + s.h] = v;
    });
    s.clear();
    s.absorb17<24>(kp, words, 0x1F, 0, words / 17 + 1);
    s.squeeze<4>([&](int x, uint32_t v) {
      if (s.y == 0) dig[8 + 2 * x + s.h] = v;
    });
    s.clear();
  } else {
    const int i = threadIdx.x & 15;
    dig[i] = i < 8 ? row[KM_MU / 4 + i] : kp[i - 8];
  }
  wide::sync();
  s.absorb17(dig, 8, 0x1F, 0, 1);
  s.squeeze<5>([&](int x, uint32_t v) {
    const int w = s.word(x);
    if (act && w < 12) row[KM_KCD / 4 + 2 * w + s.h] = v;
  });
}

// ss = SHAKE256(K || H(c), 32).  Encapsulation: d goes to the end of ct[x] and H(c) is made
// here.  Decapsulation: H(c) is in the row, and the element's 16 lanes compare ct[x] with
// the re-encryption and d, all of it (verify.cu:15-28 without its data-dependent branch);
// on any difference z[x] takes the place of K by mask (verify.cu:40-50).
template <int WG, bool ENC, int N>
__global__ PQC_WIDE_KERNEL(WG) void k_cca_close_wide(
    int n, uint8_t* ss, const uint8_t* km, std::conditional_t<ENC, uint8_t*, const uint8_t*> ct, const uint8_t* z,
    size_t z_stride) {
  using P = Par<N>;
  __shared__ wide::Consts consts;
  __shared__ Wide4 lds[WG];
  wide::init_consts(consts);
  __syncthreads();
  if (WG > 1 && 4 * wide::wave_of<WG>() >= n) return;
  Wide4& sh = lds[wide::wg_wave<WG>()];
  wide::Sponge s;
  s.init(sh.states, consts);
  const int rq = 4 * wide::wave_of<WG>() + s.st, r = rq < n ? rq : n - 1;
  const bool act = rq < n;
  const uint32_t* row = reinterpret_cast<const uint32_t*>(km + (size_t)r * kNewhopeKemBytes);
  const uint32_t* d = row + KM_KCD / 4 + 16;
  auto* c = reinterpret_cast<std::conditional_t<ENC, uint32_t*, const uint32_t*>>(ct + (size_t)r * P::CCA_CT);
  uint32_t* dig = sh.dig[s.st];
  const int i = threadIdx.x & 15;
  if constexpr (ENC) {
    static_assert(P::CT % 136 == 0, "d starts a block");
    if (act && i < 8) c[P::CT / 4 + i] = d[i];
    if (i < 8) dig[i] = row[KM_KCD / 4 + i];
    s.absorb17<24>((const uint32_t*)c, P::CT / 8, 0x1F, 0, P::CT / 136);
    s.absorb17(d, 4, 0x1F, 0, 1);
    s.squeeze<4>([&](int x, uint32_t v) {
      if (s.y == 0) dig[8 + 2 * x + s.h] = v;
    });
    s.clear();
  } else {
    const uint64_t* a = reinterpret_cast<const uint64_t*>(c);
    const uint64_t* b = reinterpret_cast<const uint64_t*>(row + KM_CT2 / 4);
    uint64_t diff = 0;
#pragma unroll 4
    for (int w = i; w < P::CT / 8; w += 16) diff |= a[w] ^ b[w];
    if (i < 4) diff |= a[P::CT / 8 + i] ^ reinterpret_cast<const uint64_t*>(d)[i];
    const uint64_t lanes = __ballot(diff != 0);
    const uint32_t mask = ((lanes >> (16 * s.st)) & 0xFFFFu) != 0 ? 0xFFFFFFFFu : 0u;
    const uint32_t kw = i < 8 ? row[KM_KCD / 4 + i] : row[KM_HC / 4 + i - 8];
    const uint32_t zw = reinterpret_cast<const uint32_t*>(z + (size_t)r * z_stride)[i & 7];
    dig[i] = i < 8 ? (kw & ~mask) | (zw & mask) : kw;
  }
  wide::sync();
  s.absorb17(dig, 8, 0x1F, 0, 1);
  uint32_t* o = reinterpret_cast<uint32_t*>(ss + (size_t)r * 32);
  s.squeeze<4>([&](int x, uint32_t v) {
    if (act && s.y == 0) o[2 * x + s.h] = v;
  });
}

// ---- orchestration (cpapke.cu:265-476) -------------------------------------------

template <int N>
struct Scratch {
  pqc_ctx* c;
  Pv<N> poly(int i) const { return Pv<N>{c->nhpolys + (size_t)i * N * c->ld}; }
};

// grid for `threads` lanes at the tuned block size
struct Launch {
  int block;
  dim3 grid(size_t threads) const { return dim3((unsigned)((threads + block - 1) / block)); }
};
inline dim3 elem_grid(int n) { return dim3((unsigned)((n + kElems - 1) / kElems)); }
#define LAUNCH(kern, threads, ...) hipLaunchKernelGGL(kern, L.grid(threads), dim3(L.block), 0, s, __VA_ARGS__)
#define LAUNCH_NTT(kern, ...) hipLaunchKernelGGL(kern, dim3(n), dim3(64), 0, s, __VA_ARGS__)

// kernel template NAME<WG, ...> on a wave per four elements
#define LAUNCH_WIDE(NAME, TARGS, st, ...)                                                                            \
  wide::with_wg(c->cu_count, (n + 3) / 4, [&](auto wg_) {                                                            \
    constexpr int WG = decltype(wg_)::value;                                                                         \
    hipLaunchKernelGGL((NAME<WG PQC_UNPAREN TARGS>), wide::wg_grid((n + 3) / 4, WG), dim3(64 * WG), 0, st, __VA_ARGS__); \
  })
#define PQC_UNPAREN(...) __VA_OPT__(,) __VA_ARGS__

// cpapke_keypair (cpapke.cu:265-338) with pk at stride PK and sk at sk_stride
// (the CCA-KEM's sk holds sk_cpa first), seeds at seed_stride
template <int N>
int keypair_impl(pqc_ctx* c, int n, uint8_t* pk, uint8_t* sk, size_t sk_stride, const uint8_t* seed,
                 size_t seed_stride, bool plain, hipStream_t s) {
  const Launch L{c->tune.newhope_block};
  if (!plain) {
    const size_t n1 = n;
    LAUNCH(k_seed_expand, n1, n, c->nhbytes, seed, seed_stride);
    hipLaunchKernelGGL(k_keypair_fused<N>, elem_grid(n), dim3(64 * kElems), 0, s, n, pk, sk, sk_stride,
                       (const uint8_t*)c->nhbytes);
    return hip_err(hipGetLastError());
  }
  const size_t n1 = n, nS = (size_t)Par<N>::STREAMS * n, n8 = (size_t)n * (N / 8), n4 = (size_t)n * (N / 4);
  Scratch<N> S{c};
  uint8_t* z = c->nhbytes;  // 64 bytes per element: publicseed || noiseseed
  const int AHAT = 0, EHAT = 1, AS = 2, BHAT = 3, SHAT = 4;
  LAUNCH(k_seed_expand, n1, n, z, seed, seed_stride);
  hipLaunchKernelGGL(k_uniform<N>, dim3((unsigned)((nS + kUniformBlock - 1) / kUniformBlock)), dim3(kUniformBlock), 0, s,
                     n, S.poly(AHAT), (const uint8_t*)z, (size_t)64);
  LAUNCH(k_sample<N>, nS, n, S.poly(SHAT), (const uint8_t*)z + 32, (size_t)64, 0);
  LAUNCH_NTT(k_ntt<N>, n, S.poly(SHAT));
  LAUNCH(k_sample<N>, nS, n, S.poly(EHAT), (const uint8_t*)z + 32, (size_t)64, 1);
  LAUNCH_NTT(k_ntt<N>, n, S.poly(EHAT));
  LAUNCH(k_pointwise<N>, n8, n, S.poly(AS), S.poly(SHAT), S.poly(AHAT));
  LAUNCH(k_addsub<N>, n8, n, S.poly(BHAT), S.poly(EHAT), S.poly(AS), 0);
  LAUNCH(k_tobytes<N>, n4, n, sk, sk_stride, S.poly(SHAT), (const uint8_t*)nullptr, (size_t)0);
  LAUNCH(k_tobytes<N>, n4, n, pk, (size_t)Par<N>::PK, S.poly(BHAT), (const uint8_t*)z, (size_t)64);
  return hip_err(hipGetLastError());
}

// cpapke_enc (cpapke.cu:353-429), every buffer at its own stride
template <int N>
int enc_impl(pqc_ctx* c, int n, uint8_t* ct, size_t ct_stride, const uint8_t* m, size_t m_stride, const uint8_t* pk,
             size_t pk_stride, const uint8_t* coin, size_t coin_stride, bool plain, hipStream_t s) {
  if (!plain) {
    hipLaunchKernelGGL(k_enc_fused<N>, elem_grid(n), dim3(64 * kElems), 0, s, n, ct, ct_stride, m, m_stride, pk, pk_stride,
                       coin, coin_stride);
    return hip_err(hipGetLastError());
  }
  const Launch L{c->tune.newhope_block};
  const size_t nS = (size_t)Par<N>::STREAMS * n, n32 = 32 * (size_t)n, n8 = (size_t)n * (N / 8), n4 = (size_t)n * (N / 4);
  Scratch<N> S{c};
  uint8_t* seed = c->nhbytes;  // publicseed copy, 32 bytes per element
  const int SP = 0, EP = 1, VP = 2, AHAT = 3, BHAT = 4, EPP = 5, UHAT = 6, V = 7;
  LAUNCH(k_frommsg<N>, n32, n, S.poly(V), m, m_stride);
  LAUNCH(k_frombytes<N>, n4, n, S.poly(BHAT), pk, pk_stride, seed);
  hipLaunchKernelGGL(k_uniform<N>, dim3((unsigned)((nS + kUniformBlock - 1) / kUniformBlock)), dim3(kUniformBlock), 0, s,
                     n, S.poly(AHAT), (const uint8_t*)seed, (size_t)32);
  LAUNCH(k_sample<N>, nS, n, S.poly(SP), coin, coin_stride, 0);
  LAUNCH(k_sample<N>, nS, n, S.poly(EP), coin, coin_stride, 1);
  LAUNCH(k_sample<N>, nS, n, S.poly(EPP), coin, coin_stride, 2);
  LAUNCH_NTT(k_ntt<N>, n, S.poly(SP));
  LAUNCH_NTT(k_ntt<N>, n, S.poly(EP));
  LAUNCH(k_pointwise<N>, n8, n, S.poly(UHAT), S.poly(AHAT), S.poly(SP));
  LAUNCH(k_addsub<N>, n8, n, S.poly(UHAT), S.poly(UHAT), S.poly(EP), 0);
  LAUNCH(k_pointwise<N>, n8, n, S.poly(VP), S.poly(BHAT), S.poly(SP));
  LAUNCH_NTT(k_invntt<N>, n, S.poly(VP));
  LAUNCH(k_addsub<N>, n8, n, S.poly(VP), S.poly(VP), S.poly(EPP), 0);
  LAUNCH(k_addsub<N>, n8, n, S.poly(VP), S.poly(VP), S.poly(V), 0);
  LAUNCH(k_tobytes<N>, n4, n, ct, ct_stride, S.poly(UHAT), (const uint8_t*)nullptr, (size_t)0);
  LAUNCH(k_compress<N>, n8, n, ct, ct_stride, S.poly(VP));
  return hip_err(hipGetLastError());
}

// cpapke_dec (cpapke.cu:443-476), every buffer at its own stride
template <int N>
int dec_impl(pqc_ctx* c, int n, uint8_t* m, size_t m_stride, const uint8_t* ct, size_t ct_stride, const uint8_t* sk,
             size_t sk_stride, bool plain, hipStream_t s) {
  if (!plain) {
    hipLaunchKernelGGL(k_dec_fused<N>, dim3((unsigned)n), dim3(64), 0, s, n, m, m_stride, ct, ct_stride, sk, sk_stride);
    return hip_err(hipGetLastError());
  }
  const Launch L{c->tune.newhope_block};
  const size_t n32 = 32 * (size_t)n, n8 = (size_t)n * (N / 8), n4 = (size_t)n * (N / 4);
  Scratch<N> S{c};
  const int VP = 0, UHAT = 1, TMP = 2, SHAT = 3;
  LAUNCH(k_frombytes<N>, n4, n, S.poly(SHAT), sk, sk_stride, (uint8_t*)nullptr);
  LAUNCH(k_frombytes<N>, n4, n, S.poly(UHAT), ct, ct_stride, (uint8_t*)nullptr);
  LAUNCH(k_decompress<N>, n8, n, S.poly(VP), ct, ct_stride);
  LAUNCH(k_pointwise<N>, n8, n, S.poly(TMP), S.poly(SHAT), S.poly(UHAT));
  LAUNCH_NTT(k_invntt<N>, n, S.poly(TMP));
  LAUNCH(k_addsub<N>, n8, n, S.poly(TMP), S.poly(TMP), S.poly(VP), 1);
  LAUNCH(k_tomsg<N>, n32, n, m, m_stride, S.poly(TMP));
  return hip_err(hipGetLastError());
}

// out[x] = SHAKE256(in[x], 8 words bytes), 32 bytes, of a public key or a ciphertext
inline void hash32(const pqc_ctx* c, int n, uint8_t* out, size_t out_stride, const uint8_t* in, size_t in_stride,
                   int words, hipStream_t s, int wide_max = kWideMax) {
  const Launch L{c->tune.newhope_block};
  if (n <= wide_max)
    LAUNCH_WIDE(k_shake256_wide, (), s, n, out, out_stride, in, in_stride, words);
  else
    LAUNCH(k_shake256_pair<4>, 2 * (size_t)n, n, out, out_stride, in, in_stride, words);
}

// NewHope CCA-KEM, the NewHope specification's transform over the CPA-PKE
// (SHAKE256 for every hash).  Keypair coins: CPA seed || s, 64 bytes.
template <int N>
int cca_keypair(pqc_ctx* c, size_t n_, uint8_t* pk, uint8_t* sk, const uint8_t* coins, bool plain, hipStream_t s) {
  using P = Par<N>;
  const Launch L{c->tune.newhope_block};
  const int n = (int)n_;
  int rc = keypair_impl<N>(c, n, pk, sk, P::CCA_SK, coins, 64, plain, s);
  if (rc) return rc;
  LAUNCH(k_copy_words, n_ * (P::PK / 8), n, sk + P::SK, (size_t)P::CCA_SK, (const uint8_t*)pk, (size_t)P::PK, P::PK / 8);
  hash32(c, n, sk + P::SK + P::PK, P::CCA_SK, pk, P::PK, P::PK / 8, s);
  LAUNCH(k_copy_words, n_ * 4, n, sk + P::CCA_SK - SYM, (size_t)P::CCA_SK, coins + SYM, (size_t)64, 4);
  return hip_err(hipGetLastError());
}

template <int N>
int cca_enc(pqc_ctx* c, size_t n_, uint8_t* ct, uint8_t* ss, const uint8_t* pk, const uint8_t* coins, bool plain,
            hipStream_t s) {
  using P = Par<N>;
  const Launch L{c->tune.newhope_block};
  const int n = (int)n_;
  uint8_t* km = c->nhkem;
  const size_t kb = kNewhopeKemBytes;
  const bool few = n <= kWideMax;
  if (few) {
    LAUNCH_WIDE(k_cca_open_wide, (true), s, n, km, coins, pk, (size_t)P::PK, P::PK / 8);
  } else {
    LAUNCH(k_shake256_words<4>, n_, n, km + KM_MU, kb, coins, (size_t)32, 4);  // mu = H(coins)
    hash32(c, n, km + KM_HPK, kb, pk, P::PK, P::PK / 8, s);
    LAUNCH(k_shake256_2x32<12>, n_, n, km + KM_KCD, kb, (const uint8_t*)km + KM_MU, kb, (const uint8_t*)km + KM_HPK,
           kb);
  }
  int rc = enc_impl<N>(c, n, ct, P::CCA_CT, km + KM_MU, kb, pk, P::PK, km + KM_KCD + SYM, kb, plain, s);
  if (rc) return rc;
  if (few) {
    LAUNCH_WIDE(k_cca_close_wide, (true, N), s, n, ss, (const uint8_t*)km, ct, (const uint8_t*)nullptr, (size_t)0);
  } else {
    LAUNCH(k_copy_words, n_ * 4, n, ct + P::CT, (size_t)P::CCA_CT, (const uint8_t*)km + KM_KCD + 2 * SYM, kb, 4);  // d
    hash32(c, n, km + KM_HC, kb, ct, P::CCA_CT, P::CCA_CT / 8, s);
    LAUNCH(k_shake256_2x32<4>, n_, n, ss, (size_t)32, (const uint8_t*)km + KM_KCD, kb, (const uint8_t*)km + KM_HC, kb);
  }
  return hip_err(hipGetLastError());
}

template <int N>
int cca_dec(pqc_ctx* c, size_t n_, uint8_t* ss, const uint8_t* ct, const uint8_t* sk, bool plain, hipStream_t s) {
  using P = Par<N>;
  const Launch L{c->tune.newhope_block};
  const int n = (int)n_;
  uint8_t* km = c->nhkem;
  const size_t kb = kNewhopeKemBytes;
  // H(c) depends only on the input ciphertext: it runs on the context's side
  // stream beside the decryption and re-encryption, and joins before the key selection
  if (hipEventRecord(c->nh_fork, s) != hipSuccess || hipStreamWaitEvent(c->nh_side, c->nh_fork, 0) != hipSuccess)
    return PQC_ERR_DEVICE;
  hash32(c, n, km + KM_HC, kb, ct, P::CCA_CT, P::CCA_CT / 8, c->nh_side, kSideWideMax);
  if (hipGetLastError() != hipSuccess || hipEventRecord(c->nh_join, c->nh_side) != hipSuccess) return PQC_ERR_DEVICE;
  int rc = dec_impl<N>(c, n, km + KM_MU, kb, ct, P::CCA_CT, sk, P::CCA_SK, plain, s);  // m'
  if (rc) {
    (void)hipStreamWaitEvent(s, c->nh_join, 0);
    return rc;
  }
  const uint8_t* hpk = sk + P::SK + P::PK;
  const bool few = n <= kWideMax;
  if (few)
    LAUNCH_WIDE(k_cca_open_wide, (false), s, n, km, (const uint8_t*)nullptr, hpk, (size_t)P::CCA_SK, 0);
  else
    LAUNCH(k_shake256_2x32<12>, n_, n, km + KM_KCD, kb, (const uint8_t*)km + KM_MU, kb, hpk, (size_t)P::CCA_SK);
  rc = enc_impl<N>(c, n, km + KM_CT2, kb, km + KM_MU, kb, sk + P::SK, P::CCA_SK, km + KM_KCD + SYM, kb, plain, s);
  if (rc) {
    (void)hipStreamWaitEvent(s, c->nh_join, 0);
    return rc;
  }
  if (few) {
    if (hipStreamWaitEvent(s, c->nh_join, 0) != hipSuccess) return PQC_ERR_DEVICE;
    LAUNCH_WIDE(k_cca_close_wide, (false, N), s, n, ss, (const uint8_t*)km, ct, sk + P::CCA_SK - SYM,
                (size_t)P::CCA_SK);
    return hip_err(hipGetLastError());
  }
  LAUNCH(k_copy_words, n_ * 4, n, km + KM_CT2 + P::CT, kb, (const uint8_t*)km + KM_KCD + 2 * SYM, kb, 4);  // d'
  hipLaunchKernelGGL(k_verify_words, dim3((unsigned)n), dim3(64), 0, s, n, reinterpret_cast<uint32_t*>(km + KM_FAIL),
                     kb, ct, (size_t)P::CCA_CT, (const uint8_t*)km + KM_CT2, kb, P::CCA_CT / 8);
  if (hipStreamWaitEvent(s, c->nh_join, 0) != hipSuccess) return PQC_ERR_DEVICE;
  LAUNCH(k_cmov32, n_ * 4, n, km + KM_KCD, kb, sk + P::CCA_SK - SYM, (size_t)P::CCA_SK,
         reinterpret_cast<const uint32_t*>(km + KM_FAIL), kb);
  LAUNCH(k_shake256_2x32<4>, n_, n, ss, (size_t)32, (const uint8_t*)km + KM_KCD, kb, (const uint8_t*)km + KM_HC, kb);
  return hip_err(hipGetLastError());
}

}  // namespace newhope

#define NH_DISPATCH(N, call) ((N) == 1024 ? newhope::call<1024> : newhope::call<512>)

int newhope_keypair(pqc_ctx* c, int N, size_t n, uint8_t* pk, uint8_t* sk, const uint8_t* seed, bool plain,
                    hipStream_t s) {
  if (N != 512 && N != 1024) return PQC_ERR_INVALID_ARG;
  const size_t sks = N == 1024 ? newhope::Par<1024>::SK : newhope::Par<512>::SK;
  return NH_DISPATCH(N, keypair_impl)(c, (int)n, pk, sk, sks, seed, 32, plain, s);
}

int newhope_enc(pqc_ctx* c, int N, size_t n, uint8_t* ct, const uint8_t* m, const uint8_t* pk, const uint8_t* coin,
                bool plain, hipStream_t s) {
  if (N != 512 && N != 1024) return PQC_ERR_INVALID_ARG;
  const size_t cts = N == 1024 ? newhope::Par<1024>::CT : newhope::Par<512>::CT;
  const size_t pks = N == 1024 ? newhope::Par<1024>::PK : newhope::Par<512>::PK;
  return NH_DISPATCH(N, enc_impl)(c, (int)n, ct, cts, m, 32, pk, pks, coin, 32, plain, s);
}

int newhope_dec(pqc_ctx* c, int N, size_t n, uint8_t* m, const uint8_t* ct, const uint8_t* sk, bool plain,
                hipStream_t s) {
  if (N != 512 && N != 1024) return PQC_ERR_INVALID_ARG;
  const size_t cts = N == 1024 ? newhope::Par<1024>::CT : newhope::Par<512>::CT;
  const size_t sks = N == 1024 ? newhope::Par<1024>::SK : newhope::Par<512>::SK;
  return NH_DISPATCH(N, dec_impl)(c, (int)n, m, 32, ct, cts, sk, sks, plain, s);
}

int newhope_cca_keypair(pqc_ctx* c, int N, size_t n, uint8_t* pk, uint8_t* sk, const uint8_t* coins, bool plain,
                        hipStream_t s) {
  if (N != 512 && N != 1024) return PQC_ERR_INVALID_ARG;
  return NH_DISPATCH(N, cca_keypair)(c, n, pk, sk, coins, plain, s);
}

int newhope_cca_enc(pqc_ctx* c, int N, size_t n, uint8_t* ct, uint8_t* ss, const uint8_t* pk, const uint8_t* coins,
                    bool plain, hipStream_t s) {
  if (N != 512 && N != 1024) return PQC_ERR_INVALID_ARG;
  return NH_DISPATCH(N, cca_enc)(c, n, ct, ss, pk, coins, plain, s);
}

int newhope_cca_dec(pqc_ctx* c, int N, size_t n, uint8_t* ss, const uint8_t* ct, const uint8_t* sk, bool plain,
                    hipStream_t s) {
  if (N != 512 && N != 1024) return PQC_ERR_INVALID_ARG;
  return NH_DISPATCH(N, cca_dec)(c, n, ss, ct, sk, plain, s);
}

int newhope_poly_sample(size_t n, uint16_t* polys, const uint8_t* seeds, size_t seed_stride, int nonce,
                        hipStream_t s) {
  using namespace newhope;
  if (nonce < 0 || nonce > 255 || seed_stride < 32 || seed_stride % 8) return PQC_ERR_INVALID_ARG;
  if (n == 0) return PQC_OK;
  if (n > (size_t)INT32_MAX / 16) return PQC_ERR_BATCH_TOO_LARGE;
  const size_t threads = 16 * n;
  hipLaunchKernelGGL(k_sample<1024>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, (int)n,
                     Pv<1024>{polys}, seeds, seed_stride, nonce);
  return hip_err(hipGetLastError());
}

int newhope_poly_transform(int op, size_t n, uint16_t* polys, hipStream_t s) {
  using namespace newhope;
  if (op != 0 && op != 1) return PQC_ERR_INVALID_ARG;
  if (n == 0) return PQC_OK;
  if (n > (size_t)INT32_MAX) return PQC_ERR_BATCH_TOO_LARGE;
  if (op == 0)
    hipLaunchKernelGGL(k_ntt<1024>, dim3((unsigned)n), dim3(64), 0, s, (int)n, Pv<1024>{polys});
  else
    hipLaunchKernelGGL(k_invntt<1024>, dim3((unsigned)n), dim3(64), 0, s, (int)n, Pv<1024>{polys});
  return hip_err(hipGetLastError());
}

}  // namespace pqc
