// Kyber key generation, encapsulation and decapsulation with one workgroup per request:
// small batches (the single-instance drop-ins, a serving loop's batches), where the time
// is that of one request's serial chain and the GPU has SIMDs to spare.
//
// The sponges run on 16 lanes per state (keccak_wide.cuh, 3.3 us per permutation against
// 7.9 on a lane of its own), the matrix entries four to a wave, the polynomial products
// one output polynomial per wave.  Decapsulation:
//   phase 1  wave 0: indcpa_dec, G, the noise streams; wave 1: H(ct), most of its blocks;
//            waves 2..: the entries of A^T;
//   phase 2  one wave per output polynomial: re-encryption and compare; wave 1: the rest
//            of H(ct), its state kept in registers across the barrier;
//   phase 3  wave 1: KDF.
// H(ct) (6, 9, 12 permutations) and the KDF are the longest chain: 33 us of Kyber-768's
// time.  Encapsulation and key generation: see their bodies.  Same bytes as every other
// path.
#include "internal.h"
#include "keccak_wide.cuh"
#include "kyber_coop.cuh"
#include "req_check.h"

namespace pqc {
namespace kyber {
namespace lowlat {

static __constant__ LaneTwiddlesF c_twf = kLaneTwF;

constexpr int kEntryStride = 260;  // int16 per matrix entry: 256 used, rows on different banks
constexpr int kMaxBlocks = 32;     // SHAKE128 blocks per entry before giving up (never reached)

template <int K>
struct Shape {
  static constexpr int matrix_waves = (K * K + 3) / 4;              // 1, 3, 4
  static constexpr int waves = K == 2 ? 4 : 2 + matrix_waves;       // 4, 5, 6
  static_assert(waves >= K + 2, "a wave per output polynomial beside wave 1");
};
constexpr int kMaxWaves = Shape<4>::waves;
// Waves per SIMD the registers are cut for.  K = 4's six waves fit a CU four times at 6
// (80 VGPRs, a few spills): 1000 decapsulations 124 us against 154 at 5 and 181 at 4, one
// 53 against 51.  K = 2, 3 decapsulation needs no more than 96
// VGPRs: 5, four workgroups per CU.
template <int K, bool DEC>
constexpr int simd_waves() {
  return K == 4 || !DEC ? 6 : 5;
}

template <int K>
struct alignas(16) Lds {
  wide::Consts consts;
  wide::States states[Shape<K>::waves];
  uint32_t block[Shape<K>::matrix_waves][4][42];       // a squeezed block of each entry in work
  alignas(16) uint8_t prf[(2 * K + 1) * 128];          // noise stream `nonce` at 128 nonce
  alignas(16) uint8_t msg[32];
  alignas(16) uint32_t gin[16];                        // G's and the KDF's 64-byte inputs
  uint32_t kbar[8], seed[8], rho[8];
  uint32_t fail[K + 1];                                // mismatch of each output polynomial
  alignas(16) uint8_t out[Params<K>::ct_bytes > Params<K>::pk_bytes ? Params<K>::ct_bytes : Params<K>::pk_bytes];
  alignas(16) int16_t a[K * K * kEntryStride];         // entry i K + j
};

// entries of one request in LDS, as the cooperative products read them
struct AtLds {
  const int16_t* a;
  int k;
  __device__ __forceinline__ void get(int i, int j, uint32_t& w0, uint32_t& w1) const {
    const uint32_t* e = reinterpret_cast<const uint32_t*>(a + (i * k + j) * kEntryStride + 4 * ntt_group(lane_id()));
    w0 = e[0];
    w1 = e[1];
  }
};

// Four matrix entries (4 aw .. 4 aw + 3, those below K^2) by one wave: SHAKE128(rho || x || y)
// on 16 lanes each; a block's 42 dwords per entry go through LDS and 42 lanes place their
// accepted candidates by a ballot's count (gen_matrix_n, indcpa.cu:339-403; the accepted
// 16-bit values themselves are kept, as everywhere here).  TRANS: A^T.
template <int K, bool TRANS>
__device__ __forceinline__ void sample_entries(Lds<K>& sh, const uint32_t* rho, int aw, int wave, uint32_t* status) {
  wide::Sponge s;
  s.init(sh.states[wave], sh.consts);
  const int l = lane_id();
  const int e = 4 * aw + s.st;
  const uint32_t x = TRANS ? e / K : e % K, y = TRANS ? e % K : e / K;
  {
    uint32_t m[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      const int w = s.word(c);
      m[c] = w < 4 ? rho[2 * (w & 3) + s.h] : 0;
      if (w == 4 && s.h == 0) m[c] = x | (y << 8) | (0x1Fu << 16);
      if (w == kRateShake128 - 1 && s.h == 1) m[c] = 0x80000000u;
    }
    s.absorb(m);
  }
  int have[4];
  bool more = false;
#pragma unroll
  for (int q = 0; q < 4; ++q) have[q] = 4 * aw + q < K * K ? 0 : N;
  uint32_t(&blk)[4][42] = sh.block[aw];
  for (int b = 0; b < kMaxBlocks; ++b) {
    s.permute();
    wide::sync();
    s.squeeze<5>([&](int c, uint32_t v) {
      const int w = s.word(c);
      if (w < kRateShake128) blk[s.st][2 * w + s.h] = v;
    });
    wide::sync();
    more = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (have[q] < N) {  // uniform
        const uint32_t d = blk[q][l < 42 ? l : 0];
        const uint32_t v0 = d & 0xFFFFu, v1 = d >> 16;
        const bool a0 = l < 42 && v0 < 19u * Q, a1 = l < 42 && v1 < 19u * Q;
        const uint64_t m0 = __ballot(a0), m1 = __ballot(a1);
        const uint64_t below = (1ull << l) - 1;
        const int p0 = have[q] + __popcll(m0 & below) + __popcll(m1 & below), p1 = p0 + (a0 ? 1 : 0);
        int16_t* ent = sh.a + (4 * aw + q) * kEntryStride;
        if (a0 && p0 < N) ent[p0] = (int16_t)v0;
        if (a1 && p1 < N) ent[p1] = (int16_t)v1;
        have[q] += __popcll(m0) + __popcll(m1);
        more |= have[q] < N;
      }
    }
    if (!more) break;
  }
  if (more && l == 0) atomicOr(status, 1u);
}

// (Kbar, seed) = SHA3-512(gin), 64 bytes in; NIN = 4: 32 bytes in (key generation's G),
// whose halves go to rho and seed
template <int K, int NIN>
__device__ __forceinline__ void hash_g(Lds<K>& sh, wide::Sponge& s, uint32_t* first) {
  s.clear();
  uint32_t m[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    const int w = s.word(c);
    m[c] = w < NIN ? sh.gin[2 * (w & 7) + s.h] : 0;
    if (w == NIN && s.h == 0) m[c] |= 0x06u;
    if (w == kRateSha3_512 - 1 && s.h == 1) m[c] |= 0x80000000u;
  }
  s.absorb(m);
  s.permute();
  s.squeeze<5>([&](int c, uint32_t v) {
    const int w = s.word(c);
    if (s.st == 0 && w < 4) first[2 * w + s.h] = v;
    if (s.st == 0 && w >= 4 && w < 8) sh.seed[2 * (w - 4) + s.h] = v;
  });
  wide::sync();
}

// noise streams 4 r .. 4 r + 3 below `count` from sh.seed
template <int K>
__device__ __forceinline__ void noise_streams(Lds<K>& sh, wide::Sponge& s, int r, int count) {
  s.clear();
  const int nonce = 4 * r + s.st;
  uint32_t m[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    const int w = s.word(c);
    m[c] = w < 4 ? sh.seed[2 * (w & 3) + s.h] : 0;
    if (w == 4 && s.h == 0) m[c] = (uint32_t)nonce | (0x1Fu << 8);
    if (w == kRateShake256 - 1 && s.h == 1) m[c] = 0x80000000u;
  }
  s.absorb(m);
  s.permute();
  uint32_t* o = reinterpret_cast<uint32_t*>(sh.prf + 128 * (nonce < count ? nonce : 0));
  s.squeeze<5>([&](int c, uint32_t v) {
    const int w = s.word(c);
    if (w < 16 && nonce < count) o[2 * w + s.h] = v;
  });
}

// ss = SHAKE256(gin, 32) by the calling wave
template <int K>
__device__ __forceinline__ void kdf(Lds<K>& sh, wide::Sponge& s, uint8_t* ss) {
  s.clear();
  s.absorb17(sh.gin, 8, 0x1F, 0, 1);
  uint32_t* o = reinterpret_cast<uint32_t*>(ss);
  s.squeeze<5>([&](int c, uint32_t v) {
    const int w = s.word(c);
    if (s.st == 0 && w < 4) o[2 * w + s.h] = v;
  });
}

// 32 bytes of a hash (words 0..3 of state 0) into gin's second half
template <int K>
__device__ __forceinline__ void hash_to_gin(Lds<K>& sh, const wide::Sponge& s) {
  s.squeeze<5>([&](int c, uint32_t v) {
    const int w = s.word(c);
    if (s.st == 0 && w < 4) sh.gin[8 + 2 * w + s.h] = v;
  });
}

// The (re-)encryption, one output polynomial per wave other than wave 1: row(i) runs it
// for i = 0..K.  Each wave makes r^ for itself (three transforms against the barrier and
// LDS trip of sharing them).
template <int K, bool DEC>
__device__ __forceinline__ void encrypt_rows(Lds<K>& sh, const uint8_t* pk, const uint8_t* c, const LaneZF& z, int wave,
                                             int l) {
  using P = Params<K>;
  if (wave == 1 || wave > K + 1) return;
  const int i = wave == 0 ? 0 : wave - 1;  // uniform
  const uint16_t* prf = reinterpret_cast<const uint16_t*>(sh.prf);
  uint32_t w[K], e, cw[3] = {0, 0, 0}, tw[K][2], bad;
  if (i == K) {
#pragma unroll
    for (int j = 0; j < K; ++j) load_h12(tw[j], pk + 384 * j, ntt_group(l));
  }
  if constexpr (DEC) {
    if (i < K)
      load_group<P::du>(cw, c + 32 * P::du * i, nat_group(l));
    else
      load_group<P::dv>(cw, c + P::polyvec_cbytes, nat_group(l));
  }
#pragma unroll
  for (int j = 0; j < K; ++j) w[j] = prf[64 * j + l];
  e = prf[64 * (K + i) + l];
  NoiseHat<K> sp;
  sp.make(w, z);
  if (i < K)
    bad = coop_row_u<K, DEC>(AtLds{sh.a, K}, i, sp, e, cw, sh.out, z);
  else
    bad = coop_row_v<K, DEC>(tw, sp, e, sh.msg, cw, sh.out, z);
  if constexpr (DEC) {
    const uint32_t f = __any(bad != 0) ? 1u : 0u;
    if (l == 0) sh.fail[i] = f;
  }
}

template <int K>
__device__ __forceinline__ void dec_body(uint8_t* ss, const uint8_t* c, const uint8_t* key, Lds<K>& sh, const LaneZF& z,
                                         int wave, int l, uint32_t* status) {
  using P = Params<K>;
  constexpr int HW = P::ct_bytes / 8;         // H(ct) message words
  constexpr int HB = HW / kRateSha3_256 + 1;  // H(ct) blocks, padding included
  constexpr int HB1 = (HB + 2) / 2;           // of them absorbed during phase 1
  const uint8_t* pk = key + P::sk_cpa_bytes;
  const uint32_t* c32 = reinterpret_cast<const uint32_t*>(c);
  wide::init_consts(sh.consts);
  DecIn<K> in;
  if (wave == 0) dec_load<K>(in, c, key);
  __syncthreads();
  // ---- phase 1
  wide::Sponge s;
  if (wave == 0) {
    if (l < 8) sh.gin[8 + l] = reinterpret_cast<const uint32_t*>(key + P::hpk_off)[l];
    coop_indcpa_dec_f<K>(in, z, sh.msg);
    wide::sync();
    if (l < 8) sh.gin[l] = reinterpret_cast<const uint32_t*>(sh.msg)[l];
    wide::sync();
    s.init(sh.states[0], sh.consts);
    hash_g<K, 8>(sh, s, sh.kbar);
    for (int r = 0; r < (2 * K + 1 + 3) / 4; ++r) noise_streams<K>(sh, s, r, 2 * K + 1);
  } else if (wave == 1) {
    s.init(sh.states[1], sh.consts);
    s.absorb17(c32, HW, 0x06, 0, HB1);
  } else if (wave < 2 + Shape<K>::matrix_waves) {
    sample_entries<K, true>(sh, reinterpret_cast<const uint32_t*>(pk + P::polyvec_bytes), wave - 2, wave, status);
  }
  __syncthreads();
  // ---- phase 2
  if (wave == 1) {
    s.absorb17(c32, HW, 0x06, HB1, HB);
    hash_to_gin<K>(sh, s);
  } else {
    encrypt_rows<K, true>(sh, pk, c, z, wave, l);
  }
  __syncthreads();
  // ---- phase 3: KDF(Kbar or z, H(ct)), z chosen by mask
  if (wave == 1) {
    uint32_t f = 0;
#pragma unroll
    for (int i = 0; i <= K; ++i) f |= sh.fail[i];
    const uint32_t mask = 0u - (f & 1u);
    if (l < 8) {
      const uint32_t zz = reinterpret_cast<const uint32_t*>(key + P::z_off)[l], kb = sh.kbar[l];
      sh.gin[l] = kb ^ (mask & (zz ^ kb));
    }
    wide::sync();
    kdf<K>(sh, s, ss);
  }
}

//   phase 1  wave 1: H(pk); wave 0: m = H(coins); waves 2..: A^T
//   phase 2  wave 0: G
//   phase 3  waves 0, 2, ..: the noise streams, four each
//   phase 4  one wave per output polynomial, into LDS
//   phase 5  wave 1: H(ct), KDF; the others: ct to memory
template <int K>
__device__ __forceinline__ void enc_body(uint8_t* ss, uint8_t* c, const uint8_t* pk, const uint8_t* coins, Lds<K>& sh,
                                         const LaneZF& z, int wave, int l, uint32_t* status) {
  using P = Params<K>;
  constexpr int PW = P::pk_bytes / 8, CW = P::ct_bytes / 8;
  wide::init_consts(sh.consts);
  __syncthreads();
  wide::Sponge s;
  if (wave == 0) {
    s.init(sh.states[0], sh.consts);
    s.absorb17(reinterpret_cast<const uint32_t*>(coins), 4, 0x06, 0, 1);  // "don't release system RNG output"
    s.squeeze<5>([&](int x, uint32_t v) {
      const int w = s.word(x);
      if (s.st == 0 && w < 4) {
        reinterpret_cast<uint32_t*>(sh.msg)[2 * w + s.h] = v;
        sh.gin[2 * w + s.h] = v;
      }
    });
  } else if (wave == 1) {
    s.init(sh.states[1], sh.consts);
    s.absorb17(reinterpret_cast<const uint32_t*>(pk), PW, 0x06, 0, PW / 17 + 1);
    hash_to_gin<K>(sh, s);
  } else if (wave < 2 + Shape<K>::matrix_waves) {
    sample_entries<K, true>(sh, reinterpret_cast<const uint32_t*>(pk + P::polyvec_bytes), wave - 2, wave, status);
  }
  __syncthreads();
  if (wave == 0) hash_g<K, 8>(sh, s, sh.kbar);
  __syncthreads();
  if (wave != 1) {
    const int r = wave == 0 ? 0 : wave - 1;
    if (4 * r < 2 * K + 1) {
      if (wave != 0) s.init(sh.states[wave], sh.consts);
      noise_streams<K>(sh, s, r, 2 * K + 1);
    }
  }
  __syncthreads();
  encrypt_rows<K, false>(sh, pk, nullptr, z, wave, l);
  if (wave == 1 && l < 8) sh.gin[l] = sh.kbar[l];
  __syncthreads();
  if (wave == 1) {
    s.clear();
    s.absorb17(reinterpret_cast<const uint32_t*>(sh.out), CW, 0x06, 0, CW / 17 + 1);
    hash_to_gin<K>(sh, s);
    wide::sync();
    kdf<K>(sh, s, ss);
  } else {
    const int t = (wave == 0 ? 0 : wave - 1) * 64 + l;  // the other waves' threads
    for (int w = t; w < CW; w += 64 * (Shape<K>::waves - 1))
      if (wave < Shape<K>::waves)
        reinterpret_cast<uint64_t*>(c)[w] = reinterpret_cast<const uint64_t*>(sh.out)[w];
  }
}

// Key generation (indcpa_keypair, indcpa.cu:474-533, and the KEM's H(pk), z):
//   phase 1  wave 0: (rho, sigma) = G(d)
//   phase 2  waves 2..: A; waves 0, 1: the noise streams
//   phase 3  one wave per row i: s_i^ into the secret key, t_i^ into LDS
//   phase 4  wave 1: H(pk) from LDS; the others: both copies of pk to memory
template <int K>
__device__ __forceinline__ void key_body(uint8_t* pk, uint8_t* sk, const uint8_t* coins, Lds<K>& sh, const LaneZF& z,
                                         int wave, int l, uint32_t* status) {
  using P = Params<K>;
  constexpr int PW = P::pk_bytes / 8;
  wide::init_consts(sh.consts);
  if (wave == 0 && l < 8) sh.gin[l] = reinterpret_cast<const uint32_t*>(coins)[l];
  if (wave == 1 && l < 8)
    reinterpret_cast<uint32_t*>(sk + P::z_off)[l] = reinterpret_cast<const uint32_t*>(coins + 32)[l];
  __syncthreads();
  wide::Sponge s;
  if (wave == 0) {
    s.init(sh.states[0], sh.consts);
    hash_g<K, 4>(sh, s, sh.rho);
    if (l < 8) reinterpret_cast<uint32_t*>(sh.out + P::polyvec_bytes)[l] = sh.rho[l];
  }
  __syncthreads();
  if (wave < 2) {
    if (wave == 1) s.init(sh.states[1], sh.consts);
    for (int r = wave; 4 * r < 2 * K; r += 2) noise_streams<K>(sh, s, r, 2 * K);
  } else if (wave < 2 + Shape<K>::matrix_waves) {
    sample_entries<K, false>(sh, sh.rho, wave - 2, wave, status);
  }
  __syncthreads();
  if (wave < K) {
    const int i = wave, gn = ntt_group(l);
    const uint16_t* prf = reinterpret_cast<const uint16_t*>(sh.prf);
    uint32_t w[K];
#pragma unroll
    for (int j = 0; j < K; ++j) w[j] = prf[64 * j + l];
    NoiseHat<K> sv;
    sv.make(w, z);
    P4 c;
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (j == i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) c.v[r] = (int32_t)f32::canon_f(sv.v[j].v[r]);
        store_poly12(sk + 384 * j, gn, c);
      }
    const AtLds at{sh.a, K};
    F4 acc = basemul_sum_f<K>(
        [&](int j) {
          uint32_t w0, w1;
          at.get(i, j, w0, w1);
          F4 a = {{(float)(w0 & 0xFFFF), (float)(w0 >> 16), (float)(w1 & 0xFFFF), (float)(w1 >> 16)}};
          reduce_f4(a);
          return a;
        },
        sv.v, sv.z);
    P4 e;
    cbd_group(e, prf[64 * (K + i) + l]);
    F4 ef = to_f4(e);
    ntt_f<2>(ef, z);
#pragma unroll
    for (int r = 0; r < 4; ++r) c.v[r] = (int32_t)f32::canon_f(acc.v[r] + ef.v[r]);
    store_poly12(sh.out + 384 * i, gn, c);
  }
  __syncthreads();
  if (wave == 1) {
    s.clear();
    s.absorb17(reinterpret_cast<const uint32_t*>(sh.out), PW, 0x06, 0, PW / 17 + 1);
    uint32_t* o = reinterpret_cast<uint32_t*>(sk + P::hpk_off);
    s.squeeze<5>([&](int x, uint32_t v) {
      const int w = s.word(x);
      if (s.st == 0 && w < 4) o[2 * w + s.h] = v;
    });
  } else {
    const int t = (wave == 0 ? 0 : wave - 1) * 64 + l;
    for (int w = t; w < PW; w += 64 * (Shape<K>::waves - 1)) {
      const uint64_t v = reinterpret_cast<const uint64_t*>(sh.out)[w];
      reinterpret_cast<uint64_t*>(pk)[w] = v;
      reinterpret_cast<uint64_t*>(sk + P::sk_cpa_bytes)[w] = v;
    }
  }
}

// Dense batches: request x at x * size in each buffer.  Measured on MI355X (Kyber-768, us),
// before (four waves per request, sponges on lanes and lane pairs) and now:
//   decapsulation 1 / 256 / 761 / 1000 requests: 102 / 122 / 124 / 145 -> 41 / 42 / 69 / 92
//   encapsulation 1 / 257 / 1000:                188 / 235 / 297 -> 82 / 92 / 124
//   key generation 1 / 300 / 1000 (was staged):  163 / 164 / 165 -> 57 / 66 / 89
template <int K, bool DEC>
__global__ __launch_bounds__(64 * Shape<K>::waves, (simd_waves<K, DEC>())) void k_lowlat(int n, uint8_t* __restrict__ ss,
                                                                    uint8_t* __restrict__ ct,
                                                                    const uint8_t* __restrict__ key,
                                                                    const uint8_t* __restrict__ coins,
                                                                    uint32_t* __restrict__ status) {
  using P = Params<K>;
  __shared__ Lds<K> sh;
  const size_t x = blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int l = threadIdx.x & 63;
  LaneZF z;
  load_lane_zf(z, &c_twf);
  if constexpr (DEC)
    dec_body<K>(ss + x * 32, ct + x * P::ct_bytes, key + x * P::sk_bytes, sh, z, wave, l, status);
  else
    enc_body<K>(ss + x * 32, ct + x * P::ct_bytes, key + x * P::pk_bytes, coins + x * 32, sh, z, wave, l, status);
}

template <int K>
__global__ __launch_bounds__(64 * Shape<K>::waves, 6) void k_lowlat_key(int n, uint8_t* __restrict__ pk,
                                                                        uint8_t* __restrict__ sk,
                                                                        const uint8_t* __restrict__ coins,
                                                                        uint32_t* __restrict__ status) {
  using P = Params<K>;
  __shared__ Lds<K> sh;
  const size_t x = blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  LaneZF z;
  load_lane_zf(z, &c_twf);
  key_body<K>(pk + x * P::pk_bytes, sk + x * P::sk_bytes, coins + x * 64, sh, z, wave, threadIdx.x & 63, status);
}

// Mixed batches: one descriptor per workgroup, checked as k_mixed_classify
// checks it (a rejected one sets status bit 1 and is skipped)
union LdsMixed {
  Lds<2> k2;
  Lds<3> k3;
  Lds<4> k4;
};

template <bool DEC>
__global__ __launch_bounds__(64 * kMaxWaves, 5) void k_lowlat_mixed(int n, unsigned alg_mask,
                                                                    const pqc_kem_req* __restrict__ reqs, uint8_t* ct,
                                                                    uint64_t ct_bytes, const uint8_t* key,
                                                                    uint64_t key_bytes, uint8_t* ss, uint64_t ss_bytes,
                                                                    const uint8_t* coins, uint64_t coins_bytes,
                                                                    uint32_t* __restrict__ status) {
  __shared__ LdsMixed sh;
  const pqc_kem_req d = reqs[blockIdx.x];
  const int k = pqc_req_k(d, DEC, alg_mask, ct_bytes, key_bytes, ss_bytes, coins_bytes);
  if (!k) {  // uniform: every lane read the same descriptor
    if (threadIdx.x == 0) atomicOr(status, 2u);
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int l = threadIdx.x & 63;
  LaneZF z;
  load_lane_zf(z, &c_twf);
  uint8_t* s_ = ss + d.ss_off;
  uint8_t* c_ = ct + d.ct_off;
  const uint8_t* k_ = key + d.key_off;
  const uint8_t* r_ = DEC ? nullptr : coins + d.coins_off;
  switch (k) {
    case 2:
      if constexpr (DEC) dec_body<2>(s_, c_, k_, sh.k2, z, wave, l, status);
      else enc_body<2>(s_, c_, k_, r_, sh.k2, z, wave, l, status);
      break;
    case 3:
      if constexpr (DEC) dec_body<3>(s_, c_, k_, sh.k3, z, wave, l, status);
      else enc_body<3>(s_, c_, k_, r_, sh.k3, z, wave, l, status);
      break;
    default:
      if constexpr (DEC) dec_body<4>(s_, c_, k_, sh.k4, z, wave, l, status);
      else enc_body<4>(s_, c_, k_, r_, sh.k4, z, wave, l, status);
      break;
  }
}

template <int K>
static int launch(int op, size_t n, uint8_t* ss, uint8_t* ct, const uint8_t* key, const uint8_t* coins,
                  uint32_t* status, hipStream_t s) {
  const dim3 grid((unsigned)n), wg(64 * Shape<K>::waves);
  if (op == 2)
    hipLaunchKernelGGL((k_lowlat<K, true>), grid, wg, 0, s, (int)n, ss, ct, key, coins, status);
  else
    hipLaunchKernelGGL((k_lowlat<K, false>), grid, wg, 0, s, (int)n, ss, ct, key, coins, status);
  return hip_err(hipGetLastError());
}

template <int K>
static int launch_key(size_t n, uint8_t* pk, uint8_t* sk, const uint8_t* coins, uint32_t* status, hipStream_t s) {
  hipLaunchKernelGGL((k_lowlat_key<K>), dim3((unsigned)n), dim3(64 * Shape<K>::waves), 0, s, (int)n, pk, sk, coins,
                     status);
  return hip_err(hipGetLastError());
}

}  // namespace lowlat
}  // namespace kyber

int kyber_lowlat_dec(int k, size_t n, uint8_t* ss, const uint8_t* ct, const uint8_t* sk, uint32_t* status,
                     hipStream_t s) {
  uint8_t* c = const_cast<uint8_t*>(ct);  // read-only in decapsulation
  switch (k) {
    case 2: return kyber::lowlat::launch<2>(2, n, ss, c, sk, nullptr, status, s);
    case 3: return kyber::lowlat::launch<3>(2, n, ss, c, sk, nullptr, status, s);
    case 4: return kyber::lowlat::launch<4>(2, n, ss, c, sk, nullptr, status, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

int kyber_lowlat_enc(int k, size_t n, uint8_t* ct, uint8_t* ss, const uint8_t* pk, const uint8_t* coins,
                     uint32_t* status, hipStream_t s) {
  switch (k) {
    case 2: return kyber::lowlat::launch<2>(1, n, ss, ct, pk, coins, status, s);
    case 3: return kyber::lowlat::launch<3>(1, n, ss, ct, pk, coins, status, s);
    case 4: return kyber::lowlat::launch<4>(1, n, ss, ct, pk, coins, status, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

int kyber_lowlat_keypair(int k, size_t n, uint8_t* pk, uint8_t* sk, const uint8_t* coins, uint32_t* status,
                         hipStream_t s) {
  switch (k) {
    case 2: return kyber::lowlat::launch_key<2>(n, pk, sk, coins, status, s);
    case 3: return kyber::lowlat::launch_key<3>(n, pk, sk, coins, status, s);
    case 4: return kyber::lowlat::launch_key<4>(n, pk, sk, coins, status, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

int kyber_lowlat_mixed(const pqc_ctx* c, int dec, size_t n, const pqc_kem_req* reqs, uint8_t* ct, size_t ct_bytes,
                       const uint8_t* key, size_t key_bytes, uint8_t* ss, size_t ss_bytes, const uint8_t* coins,
                       size_t coins_bytes, hipStream_t s) {
  using namespace kyber::lowlat;
  const dim3 grid((unsigned)n), wg(64 * kMaxWaves);
  if (dec)
    hipLaunchKernelGGL(k_lowlat_mixed<true>, grid, wg, 0, s, (int)n, c->alg_mask, reqs, ct, (uint64_t)ct_bytes, key,
                       (uint64_t)key_bytes, ss, (uint64_t)ss_bytes, coins, (uint64_t)coins_bytes, c->status);
  else
    hipLaunchKernelGGL(k_lowlat_mixed<false>, grid, wg, 0, s, (int)n, c->alg_mask, reqs, ct, (uint64_t)ct_bytes, key,
                       (uint64_t)key_bytes, ss, (uint64_t)ss_bytes, coins, (uint64_t)coins_bytes, c->status);
  return hip_err(hipGetLastError());
}

}  // namespace pqc
