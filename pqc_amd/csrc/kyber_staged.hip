// Batched Kyber encapsulation, decapsulation and key generation in stages.
//
// A batch runs as a short chain of launches, each with the shape its work wants:
//   sponge stages   one sponge chain per lane (H, G, PRF, KDF and the matrix entries
//                   A_ij, K^2 lanes per request), about 100 VGPRs and little LDS, so
//                   four waves share a SIMD and Keccak issues at its best rate;
//   product stages  16 requests per wave: transforms on the matrix cores, the rest of
//                   the polynomial arithmetic on FP32 values (kyber_mfma.cuh).
// Between them: the noise bytes, the sampled entries and 96 bytes per request, in the
// layouts the next stage reads (below).
//
//   decapsulation  k_open (indcpa_dec) -> k_dec_sponge (H(ct); G, PRF; A^T)
//                  -> k_dec_reencrypt (indcpa_enc, verify) -> k_dec_kdf
//   encapsulation  k_enc_sponge (H(pk), m, G; A^T) -> k_enc_prf -> k_enc_encrypt
//                  (indcpa_enc) -> k_enc_final (H(ct), KDF)
//   key generation k_key_seed (G) -> k_key_sponge (A; PRF) -> k_key_mul -> k_key_final (H(pk))
//   the ..._few and ..._pair kernels are the same stages for fewer requests
//
// Scratch, by group of 16 requests (request r of a bucket: group r / 16, slot r % 16;
// dense batches have one bucket, mixed batches three whose groups follow each other):
//   prf  [group][polynomial][chunk c][slot] 4 bytes: a wave's read of a chunk column is
//        4 x 64 contiguous bytes, the writing lanes' stores too
//   at   [group][entry][chunk c][slot] 16 bytes (8 coefficients)
//   row  [group][slot] 128 bytes: m, Kbar, H(ct) or the noise seed, mismatch
//
// The data flow and the reference functions are those of the 64-request tiles
// (kyber_fused.hip); every path gives the same bytes.
//
// Measured on MI355X, us per call, this path and the 32-request tiles (two waves per
// SIMD, butterfly transforms) or per-request workgroups it replaced:
//   Kyber-768 decapsulation, 65536 requests    610    712  (596 to 675 across boxes, 712 to 793)
//   Kyber-1024 decapsulation, 6000 requests    189    675 (a workgroup per request)
// At 65536 the sponge stage takes ~370 us (53 permutations per request at 9.4 G/s, the
// rate of the VALU on this mix), the product stages ~65 and ~140, the KDF ~15.
#include <algorithm>
#include <type_traits>

#include "internal.h"
#include "keccak_wide.cuh"
#include "kyber_mfma.cuh"
#include "kyber_src.cuh"
#include "sponge.cuh"

namespace pqc {
namespace kyber {
namespace staged {

using namespace mfma;

__device__ const DftTables c_dft = make_dft_tables();

constexpr int kMaxBlocks = 32;  // SHAKE128 blocks per entry before giving up (never reached)

struct Scratch {
  uint8_t* prf;
  size_t prf_group;  // bytes per group
  uint8_t* at;
  size_t at_group;  // bytes per group
  uint8_t* row;
  uint32_t* status;
  // chunk column (poly, 4 t + g) of a wave's group: uniform base + 32-bit lane offset
  __device__ __forceinline__ uint32_t prf_load(int grp, int poly, int t, uint32_t lane_off) const {
    const uint8_t* p = prf + (size_t)grp * prf_group + (poly * 32 + 4 * t) * 64;
    return *(const __attribute__((address_space(1))) uint32_t*)(p + lane_off);
  }
  __device__ __forceinline__ uint32_t* prf_word(int grp, int slot, int poly, int c) const {
    return reinterpret_cast<uint32_t*>(prf + (size_t)grp * prf_group) + (poly * 32 + c) * 16 + slot;
  }
  __device__ __forceinline__ uint8_t* at_chunk(int grp, int slot, int entry, int c) const {
    return at + (size_t)grp * at_group + ((size_t)(entry * 32 + c) * 16 + slot) * 16;
  }
  __device__ __forceinline__ uint8_t* row_of(int grp, int slot) const {
    return row + ((size_t)grp * 16 + slot) * 128;
  }
};
constexpr int kRowM = 0, kRowKbar = 32, kRowH = 64, kRowFail = 96;  // offsets inside a row

// One bucket of a batch: n requests of one parameter set, its groups from grp0 on.
struct Bucket {
  int n, grp0;
};

// ---- sponge pieces ---------------------------------------------------------------

__device__ __forceinline__ void load_words4(uint64_t (&w)[4], const uint8_t* p) {
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = load_u64_global(p + 8 * i);
}

__device__ __forceinline__ void store_words4(uint8_t* p, const uint64_t* w) {
#pragma unroll
  for (int i = 0; i < 4; ++i) store_u64(p + 8 * i, w[i]);
}

// PRF(seed, nonce): SHAKE256(seed || nonce), 128 bytes into the group's noise words
__device__ __forceinline__ void prf_store(const Scratch& sc, int grp, int slot, const uint64_t (&seed)[4], int nonce) {
  uint64_t A[25];
  absorb_fixed<kRateShake256, 4, true>(A, seed, (uint64_t)nonce | (0x1Full << 8));
  uint32_t* o = sc.prf_word(grp, slot, nonce, 0);
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    o[32 * w] = (uint32_t)A[w];
    o[32 * w + 16] = (uint32_t)(A[w] >> 32);
  }
}

// ---- matrix entries ----------------------------------------------------------------
// Sampling stage: one LDS row of 40 coefficients per lane.  A third of a block (28
// candidates) is written at the running position without a branch (an accepted
// candidate advances it, a rejected one is overwritten by the next); then whole chunks
// of 8 go to the entry with 16-byte stores and the 0..7 coefficients left move to the
// front of the row.  5 KB of LDS per wave leaves room for four waves per SIMD.
constexpr int kStageRow = 40;
constexpr int kPartWords = 7;
static_assert(kRateShake128 % kPartWords == 0 && 7 + 4 * kPartWords <= kStageRow && kStageRow % 8 == 0, "stage row");

struct SponLds {
  alignas(16) int16_t stage[64][kStageRow];
};

// SHAKE128(rho || x || y) rejection-sampled (gen_matrix_n, indcpa.cu:339-403) into the
// entry's chunks; as in the tiles the accepted candidates themselves (< 19 q) are kept.
__device__ __forceinline__ bool sample_entry(uint8_t* entry, int16_t* row, const uint64_t (&rho)[4], int x, int y,
                                             bool valid) {
  uint64_t A[25];
#pragma unroll
  for (int t = 0; t < 25; ++t) A[t] = (t < 4) ? rho[t] : 0;
  A[4] = (uint64_t)x | ((uint64_t)y << 8) | (0x1Full << 16);
  A[kRateShake128 - 1] ^= 0x8000000000000000ull;
  int left = 0;   // coefficients in the row
  int chunk = 0;  // chunks written
  for (int blk = 0; blk < kMaxBlocks; ++blk) {
    if (blk >= 4 && !__any(valid && chunk < 32)) break;
    keccakf1600_two(A);
#pragma unroll
    for (int part = 0; part < kRateShake128 / kPartWords; ++part) {
      int16_t* p = row + left;
#pragma unroll
      for (int w = kPartWords * part; w < kPartWords * (part + 1); ++w) {
        const uint32_t half[2] = {(uint32_t)A[w], (uint32_t)(A[w] >> 32)};
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const uint32_t val = (h & 1) ? (half[h >> 1] >> 16) : (half[h >> 1] & 0xFFFFu);
          *p = (int16_t)val;
          p += val < 19u * Q ? 1 : 0;
        }
      }
      const int have = (int)(p - row);
      const int whole = have >> 3;
#pragma unroll
      for (int c = 0; c < (7 + 4 * kPartWords) / 8; ++c)
        if (c < whole && chunk + c < 32 && valid)
          *(global_t<u4v>*)(entry + (size_t)(chunk + c) * 256) = *reinterpret_cast<const u4v*>(row + 8 * c);
      const u4v rest = *reinterpret_cast<const u4v*>(row + 8 * whole);
      *reinterpret_cast<u4v*>(row) = rest;
      left = have & 7;
      chunk += whole;
    }
  }
  return chunk >= 32;
}

// Matrix work of a bucket: wave w of matrix_waves, 4 (group, entry) pairs of 16 lanes.
// TRANS: entry (i, j) = XOF(rho, i, j) of A^T (encryption); else XOF(rho, j, i).
template <int K>
__host__ __device__ __forceinline__ int matrix_waves(int n) {
  return ((n + 15) / 16 * K * K + 3) / 4;
}

template <int K, bool TRANS, class RhoOf>
__device__ __forceinline__ void matrix_wave(const Scratch& sc, const Bucket& b, int w, SponLds& sh, RhoOf&& rho_of) {
  const int lane = threadIdx.x & 63;
  const int pair = 4 * w + (lane >> 4);
  const int grp = pair / (K * K), e = pair % (K * K);
  const int r = 16 * grp + (lane & 15);
  const bool valid = r < b.n;
  const int i = e / K, j = e % K;
  uint64_t rho[4];
  load_words4(rho, rho_of(valid ? r : b.n - 1));
  const bool ok = sample_entry(sc.at_chunk(b.grp0 + grp, lane & 15, e, 0), sh.stage[lane], rho, TRANS ? i : j,
                               TRANS ? j : i, valid);
  if (valid && !ok) atomicOr(sc.status, 1u);
}

// ---- decapsulation: sponge stage -------------------------------------------------------
// H(ct) of 64 requests
template <int K, class Src>
__device__ __forceinline__ void dec_hash_wave(const Src& src, const Scratch& sc, const Bucket& b, int w) {
  using P = Params<K>;
  const int r = 64 * w + (threadIdx.x & 63);
  const bool act = r < b.n;
  const ReqP q = src.template req<K, true>(act ? r : b.n - 1);
  uint64_t A[25];
  sponge_absorb_two<kRateSha3_256, P::ct_bytes / 8>(A, q.ct, 0x06);
  if (act) store_words4(sc.row_of(b.grp0 + r / 16, r % 16) + kRowH, A);
}

// (Kbar, coins) = G(m || H(pk)), then the 2K + 1 noise streams, of 64 requests
template <int K, class Src>
__device__ __forceinline__ void dec_prf_wave(const Src& src, const Scratch& sc, const Bucket& b, int w) {
  using P = Params<K>;
  const int r = 64 * w + (threadIdx.x & 63);
  const bool act = r < b.n;
  const int rc = act ? r : b.n - 1;
  const ReqP q = src.template req<K, true>(rc);
  uint8_t* row = sc.row_of(b.grp0 + rc / 16, rc % 16);
  uint64_t m[8], A[25], seed[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m[i] = load_u64_global(row + kRowM + 8 * i);
    m[4 + i] = load_u64_global(q.key + P::hpk_off + 8 * i);
  }
  absorb_fixed<kRateSha3_512, 8, true>(A, m, 0x06);
#pragma unroll
  for (int i = 0; i < 4; ++i) seed[i] = A[4 + i];
  if (act) {
    store_words4(row + kRowKbar, A);
    for (int nonce = 0; nonce < 2 * K + 1; ++nonce)
      prf_store(sc, b.grp0 + r / 16, r % 16, seed, nonce);
  }
}

// ---- encapsulation: sponge stages ---------------------------------------------------------
// H(pk), m = H(coins) ("don't release system RNG output"), (Kbar, coins') = G(m || H(pk))
// of 64 requests; coins' takes the row's hash place until the noise streams are drawn
template <int K, class Src>
__device__ __forceinline__ void enc_open_wave(const Src& src, const Scratch& sc, const Bucket& b, int w) {
  using P = Params<K>;
  const int r = 64 * w + (threadIdx.x & 63);
  const bool act = r < b.n;
  const int rc = act ? r : b.n - 1;
  const ReqP q = src.template req<K, false>(rc);
  uint64_t A[25], m[8], c4[4];
  sponge_absorb_two<kRateSha3_256, P::pk_bytes / 8>(A, q.key, 0x06);
#pragma unroll
  for (int i = 0; i < 4; ++i) m[4 + i] = A[i];
  load_words4(c4, q.coins);
  absorb_fixed<kRateSha3_256, 4, true>(A, c4, 0x06);
#pragma unroll
  for (int i = 0; i < 4; ++i) m[i] = A[i];
  absorb_fixed<kRateSha3_512, 8, true>(A, m, 0x06);
  if (act) {
    uint8_t* row = sc.row_of(b.grp0 + r / 16, r % 16);
    store_words4(row + kRowM, m);
    store_words4(row + kRowKbar, A);
    store_words4(row + kRowH, A + 4);
  }
}

// noise stream `nonce` of 64 requests, from the seeds in the rows
__device__ __forceinline__ void prf_wave(const Scratch& sc, const Bucket& b, int w, int nonce) {
  const int r = 64 * w + (threadIdx.x & 63);
  if (r >= b.n) return;
  uint64_t seed[4];
  load_words4(seed, sc.row_of(b.grp0 + r / 16, r % 16) + kRowH);
  prf_store(sc, b.grp0 + r / 16, r % 16, seed, nonce);
}

// ss = KDF(Kbar, H(ct)) of 64 requests
template <int K, class Src>
__device__ __forceinline__ void enc_final_wave(const Src& src, const Scratch& sc, const Bucket& b, int w) {
  using P = Params<K>;
  const int r = 64 * w + (threadIdx.x & 63);
  const bool act = r < b.n;
  const int rc = act ? r : b.n - 1;
  const ReqP q = src.template req<K, false>(rc);
  uint64_t A[25], m[8];
  sponge_absorb_two<kRateSha3_256, P::ct_bytes / 8>(A, q.ct, 0x06);
  const uint8_t* row = sc.row_of(b.grp0 + rc / 16, rc % 16);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m[i] = load_u64_global(row + kRowKbar + 8 * i);
    m[4 + i] = A[i];
  }
  absorb_fixed<kRateShake256, 8, true>(A, m, 0x1F);
  if (act) store_words4(q.ss, A);
}

// ---- key generation: sponge stages -----------------------------------------------------------
struct KeySrc {
  uint8_t* pk;
  uint8_t* sk;
  const uint8_t* coins;  // 64 bytes per request: d || z
};

// (rho, sigma) = G(d) of 64 requests: rho into both copies of the public key, sigma into
// the row, z into the secret key
template <int K>
__device__ __forceinline__ void key_seed_wave(const KeySrc& src, const Scratch& sc, int n, int w) {
  using P = Params<K>;
  const int r = 64 * w + (threadIdx.x & 63);
  if (r >= n) return;
  uint64_t d[4], z[4], A[25];
  load_words4(d, src.coins + (size_t)r * 64);
  load_words4(z, src.coins + (size_t)r * 64 + 32);
  absorb_fixed<kRateSha3_512, 4, true>(A, d, 0x06);
  uint8_t* sk = src.sk + (size_t)r * P::sk_bytes;
  store_words4(src.pk + (size_t)r * P::pk_bytes + P::polyvec_bytes, A);
  store_words4(sk + P::sk_cpa_bytes + P::polyvec_bytes, A);
  store_words4(sk + P::z_off, z);
  store_words4(sc.row_of(r / 16, r % 16) + kRowH, A + 4);
}

// H(pk) of 64 requests into the secret key
template <int K>
__device__ __forceinline__ void key_final_wave(const KeySrc& src, int n, int w) {
  using P = Params<K>;
  const int r = 64 * w + (threadIdx.x & 63);
  const int rc = r < n ? r : n - 1;
  uint64_t A[25];
  sponge_absorb_two<kRateSha3_256, P::pk_bytes / 8>(A, src.pk + (size_t)rc * P::pk_bytes, 0x06);
  if (r < n) store_words4(src.sk + (size_t)r * P::sk_bytes + P::hpk_off, A);
}

// ---- dense batches of at most kFewMax requests: the long chains shortened ------------------
// A stage lasts as long as its longest chain: on one lane the hash of a ciphertext or a
// public key (6 to 12 permutations at ~8 us) and decapsulation's G and 2K + 1 noise streams
// of a request.  With few requests the chip has room to shorten them: the hashes run on 16
// lanes per request (keccak_wide.cuh, 3.3 us per permutation), and every noise stream of
// decapsulation has a lane that makes its own G.  Decapsulation's H(ct) is not needed
// before the KDF and runs beside the re-encryption.  us per call, one lane per request ->
// this: Kyber-512 encapsulation 174 -> 109 (2501 requests), 182 -> 152 (8192), 205 -> 230
// (16384); Kyber-1024 decapsulation 217 -> 143 (2501), 218 -> 189 (6000), 259 -> 222 (8192),
// 309 -> 390 (16384); Kyber-768 key generation 168 -> 126 (2501), 187 -> 162 (8192).
constexpr int kFewMax = 8192;

struct WideLds {
  wide::Consts consts;
  wide::States states;
  alignas(16) uint32_t dig[4][16];  // per request: the words of its next short message
};

// this lane's request of wave w, four to a wave (past the batch's end: the last one)
struct WideReq {
  int r;
  bool act;
  uint8_t* row;
  __device__ __forceinline__ WideReq(const Scratch& sc, int n, int w, const wide::Sponge& s) {
    const int rq = 4 * w + s.st;
    act = rq < n;
    r = act ? rq : n - 1;
    row = sc.row_of(r / 16, r % 16);
  }
};

// the first 32 bytes of the state to o
__device__ __forceinline__ void wide_digest(const wide::Sponge& s, bool act, uint32_t* o) {
  s.squeeze<4>([&](int x, uint32_t v) {
    if (act && s.y == 0) o[2 * x + s.h] = v;
  });
}

__device__ __forceinline__ const uint32_t* words32(const uint8_t* p) { return reinterpret_cast<const uint32_t*>(p); }
__device__ __forceinline__ uint32_t* words32(uint8_t* p) { return reinterpret_cast<uint32_t*>(p); }

// SHA3-256 of NWORDS 64-bit words
template <int NWORDS>
__device__ __forceinline__ void wide_h(wide::Sponge& s, const uint32_t* p) {
  s.clear();
  s.absorb17<(NWORDS > 17 ? 24 : 4)>(p, NWORDS, 0x06, 0, NWORDS / 17 + 1);
}

template <int K>
__device__ __forceinline__ void dec_hash_wide(const DenseSrc& src, const Scratch& sc, int n, int w, wide::Sponge& s) {
  using P = Params<K>;
  const WideReq x(sc, n, w, s);
  wide_h<P::ct_bytes / 8>(s, words32(src.template req<K, true>(x.r).ct));
  wide_digest(s, x.act, words32(x.row + kRowH));
}

// G of 64 requests and noise stream `nonce`
template <int K>
__device__ __forceinline__ void dec_prf_one(const DenseSrc& src, const Scratch& sc, int n, int w, int nonce) {
  using P = Params<K>;
  const int r = 64 * w + (threadIdx.x & 63);
  if (r >= n) return;
  uint8_t* row = sc.row_of(r / 16, r % 16);
  uint64_t m[8], A[25], seed[4];
  load_words4(*reinterpret_cast<uint64_t(*)[4]>(m), row + kRowM);
  load_words4(*reinterpret_cast<uint64_t(*)[4]>(m + 4), src.template req<K, true>(r).key + P::hpk_off);
  absorb_fixed<kRateSha3_512, 8, true>(A, m, 0x06);
#pragma unroll
  for (int i = 0; i < 4; ++i) seed[i] = A[4 + i];
  if (nonce == 0) store_words4(row + kRowKbar, A);
  prf_store(sc, r / 16, r % 16, seed, nonce);
}

template <int K>
__device__ __forceinline__ void enc_open_wide(const DenseSrc& src, const Scratch& sc, int n, int w, wide::Sponge& s,
                                              WideLds& sh) {
  using P = Params<K>;
  const WideReq x(sc, n, w, s);
  const ReqP q = src.template req<K, false>(x.r);
  uint32_t* dig = sh.dig[s.st];
  wide_h<4>(s, words32(q.coins));
  wide_digest(s, true, dig);
  wide_digest(s, x.act, words32(x.row + kRowM));
  wide_h<P::pk_bytes / 8>(s, words32(q.key));
  wide_digest(s, true, dig + 8);
  wide::sync();
  s.clear();
  uint32_t m[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    const int word = s.word(c);
    m[c] = word < 8 ? dig[2 * (word & 7) + s.h] : 0;
    if (word == 8) m[c] = s.h ? 0x80000000u : 0x06u;  // the last word of SHA3-512's rate
  }
  wide::sync();
  s.absorb(m);
  s.permute();
  s.squeeze<5>([&](int c, uint32_t v) {  // Kbar, then the noise seed
    const int word = s.word(c);
    if (x.act && word < 8) words32(x.row + (word < 4 ? kRowKbar : kRowH - 32))[2 * word + s.h] = v;
  });
}

// ss = SHAKE256(first || second, 32), the two in dig
__device__ __forceinline__ void wide_kdf(wide::Sponge& s, const WideReq& x, const uint32_t* dig, uint8_t* ss) {
  wide::sync();
  s.clear();
  s.absorb17(dig, 8, 0x1F, 0, 1);
  wide::sync();
  wide_digest(s, x.act, words32(ss));
}

template <int K>
__device__ __forceinline__ void enc_final_wide(const DenseSrc& src, const Scratch& sc, int n, int w, wide::Sponge& s,
                                               WideLds& sh) {
  using P = Params<K>;
  const WideReq x(sc, n, w, s);
  const ReqP q = src.template req<K, false>(x.r);
  uint32_t* dig = sh.dig[s.st];
  wide_h<P::ct_bytes / 8>(s, words32(q.ct));
  wide_digest(s, true, dig + 8);
  const int i = threadIdx.x & 15;
  if (i < 8) dig[i] = words32(x.row + kRowKbar)[i];
  wide_kdf(s, x, dig, q.ss);
}

template <int K>
__device__ __forceinline__ void dec_kdf_wide(const DenseSrc& src, const Scratch& sc, int n, int w, wide::Sponge& s,
                                             WideLds& sh) {
  using P = Params<K>;
  const WideReq x(sc, n, w, s);
  const ReqP q = src.template req<K, true>(x.r);
  uint32_t* dig = sh.dig[s.st];
  const int i = threadIdx.x & 15;
  const uint32_t f = *words32(x.row + kRowFail), mask = 0u - ((f | (0u - f)) >> 31);
  const uint32_t v = words32(x.row + (i < 8 ? kRowKbar : kRowH - 32))[i];
  const uint32_t z = words32(q.key + P::z_off)[i & 7];
  dig[i] = i < 8 ? v ^ (mask & (z ^ v)) : v;
  wide_kdf(s, x, dig, q.ss);
}

template <int K>
__device__ __forceinline__ void key_final_wide(const KeySrc& src, const Scratch& sc, int n, int w, wide::Sponge& s) {
  using P = Params<K>;
  const WideReq x(sc, n, w, s);
  wide_h<P::pk_bytes / 8>(s, words32(src.pk + (size_t)x.r * P::pk_bytes));
  wide_digest(s, x.act, words32(src.sk + (size_t)x.r * P::sk_bytes + P::hpk_off));
}

// ---- dense batches of up to kPairMax requests: the last stage's hashes on lane pairs -------
// One lane per request would leave half of the SIMDs or more without a wave; a pair's chain
// is shorter (6.3 us per permutation against 7.65).  us per call, lane -> pair: Kyber-768
// encapsulation 302 -> 286 at 16384 requests, 378 -> 364 at 32768, 642 -> 666 at 65536;
// Kyber-1024 key generation 331 -> 321, 525 -> 524 and 922 -> 968.
constexpr int kPairMax = 32768;

__device__ __forceinline__ void digest_pair(const uint32_t (&S)[25], uint32_t half, uint8_t* o) {
#pragma unroll
  for (int i = 0; i < 4; ++i) words32(o)[2 * i + half] = S[i];
}

template <int K>
__device__ __forceinline__ void enc_final_pair(const DenseSrc& src, const Scratch& sc, int n, int w) {
  using P = Params<K>;
  const int r = 32 * w + ((threadIdx.x & 63) >> 1);
  const uint32_t half = threadIdx.x & 1;
  if (r >= n) return;  // both lanes of a pair
  const ReqP q = src.template req<K, false>(r);
  const uint32_t* kbar = words32(sc.row_of(r / 16, r % 16) + kRowKbar);
  uint32_t S[25], A[25];
  absorb_range_pair(S, q.ct, P::ct_bytes / 8, 0, P::ct_bytes / 136 + 1, 0x06, half);
#pragma unroll
  for (int i = 0; i < 25; ++i) A[i] = i < 4 ? kbar[2 * i + half] : i < 8 ? S[i - 4] : 0;
  A[8] = half ? 0u : 0x1Fu;
  A[kRateShake256 - 1] = half ? 0x80000000u : 0u;
  keccakf1600_pair(A, half);
  digest_pair(A, half, q.ss);
}

template <int K>
__device__ __forceinline__ void key_final_pair(const KeySrc& src, int n, int w) {
  using P = Params<K>;
  const int r = 32 * w + ((threadIdx.x & 63) >> 1);
  const uint32_t half = threadIdx.x & 1;
  if (r >= n) return;
  uint32_t S[25];
  absorb_range_pair(S, src.pk + (size_t)r * P::pk_bytes, P::pk_bytes / 8, 0, P::pk_bytes / 136 + 1, 0x06, half);
  digest_pair(S, half, src.sk + (size_t)r * P::sk_bytes + P::hpk_off);
}

// ---- product stages ----------------------------------------------------------------------
constexpr int kProdThreads = 256;  // 4 waves, 64 requests

// This lane's request of a 64-request tile: wave's group and slot (a slot past the
// batch's end repeats its last request and stores nothing)
struct Lane {
  int grp;  // wave-uniform
  int n, g, r;
  bool act;
  __device__ __forceinline__ uint32_t prf_off() const { return 64u * g + 4u * n; }   // in a column of 4 chunks
  __device__ __forceinline__ uint32_t at_off() const { return 256u * g + 16u * n; }  // the same, matrix entries
};
__device__ __forceinline__ Lane lane_of(const Bucket& b, int tile) {
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // computed per tile: nothing derived from it is worth registers across tiles
  const int l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  Lane x;
  x.n = l & 15;
  x.g = l >> 4;
  const int r = 64 * tile + 16 * w + x.n;
  x.act = r < b.n;
  x.r = x.act ? r : b.n - 1;
  x.grp = b.grp0 + 4 * tile + w;
  return x;
}

// a[8] of a chunk from 12-bit values (0..4095), reduced
__device__ __forceinline__ void chunk_from12(float (&a)[8], const Words<12>& x) {
  uint32_t v[8];
  unpack_chunk<12>(v, x, 0);
#pragma unroll
  for (int k = 0; k < 8; ++k) a[k] = f32::reduce_f((float)v[k]);
}
// and from sampled entries (16-bit, < 19 q)
__device__ __forceinline__ void chunk_from16(float (&a)[8], const u4v& x) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[2 * i] = f32::reduce_f((float)(x[i] & 0xFFFFu));
    a[2 * i + 1] = f32::reduce_f((float)(x[i] >> 16));
  }
}

// sum_j row_j o x_j, chunk by chunk: load(t) fetches chunk t's words of all j into a
// LOADED (issued PRE chunks ahead), conv(a, loaded, j, t) gives reduced coefficients,
// out(t, even, odd) takes the reduced sums.
template <int K, class LOADED, class Load, class Conv, class Out>
__device__ __forceinline__ void row_product(const HPoly (&x)[K], const float* gamma, const float* gammaq, int g,
                                            Load&& load, Conv&& conv, Out&& out) {
  constexpr int PRE = 2;
  LOADED q[PRE + 1];
#pragma unroll
  for (int t = 0; t < PRE; ++t) load(q[t], t);
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    if (t + PRE < 8) load(q[(t + PRE) % (PRE + 1)], t + PRE);
    ChunkSum s;
    chunk_zero(s);
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (j > 0 && j % f32::kBasemulTerms == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s.s01[i] = f32::reduce_f(s.s01[i]);
      }
      float a[8];
      conv(a, q[t % (PRE + 1)], j, t);
      chunk_mac(s, a, x[j], t);
    }
    f4v e, o;
    chunk_finish(s, gamma, gammaq, t, g, e, o);
    out(t, e, o);
    tile_fence();
  }
}

template <int K>
struct Loaded12 {
  Words<12> w[K];
};
template <int K>
struct Loaded16 {
  u4v w[K];
};

// r^ (or s^): noise polynomial p of the request, transformed and reduced
__device__ __forceinline__ void noise_ntt(HPoly& out, const Scratch& sc, const Lane& x, int p, const u4v* fwd) {
  HPoly c;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    uint32_t e[2], o[2];
    cbd_chunk(e, o, sc.prf_load(x.grp, p, t, x.prf_off()));
    c.v[0][t][0] = e[0];
    c.v[0][t][1] = e[1];
    c.v[1][t][0] = o[0];
    c.v[1][t][1] = o[1];
  }
  dft1(fwd, c, [&](int mt, f4v e, f4v o) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      e[i] = f32::reduce_f(e[i]);
      o[i] = f32::reduce_f(o[i]);
    }
    set_chunk(out, mt, e, o);
  });
}

// indcpa_dec of a tile (indcpa.cu:691-733): m' into the rows
template <int K, class Src>
__device__ __forceinline__ void open_tile(const Src& src, const Scratch& sc, const Bucket& b, int tile,
                                          const DftLds<true, true>& sh) {
  using P = Params<K>;
  const Lane x = lane_of(b, tile);
  const ReqP q = src.template req<K, true>(x.r);
  const ChunkAt<P::du> au(x.g);
  const ChunkAt<P::dv> av(x.g);
  const ChunkAt<12> as(x.g);
  HPoly u[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    Words<P::du> w[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) load_chunk<P::du>(w[t], q.ct + 32 * P::du * j, au, t);
    HPoly uh, ul;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      uint32_t v[8];
      unpack_chunk<P::du>(v, w[t], au.sh);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (uint32_t)decompress_d<P::du>(v[k]);  // [0, q)
      // digits v >> 6, v & 63 of two values as the f16 pairs 1024 + digit
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const uint32_t pr = v[4 * p + h] | (v[4 * p + 2 + h] << 16);
          uh.v[h][t][p] = add_h2(((pr >> 6) & 0x003F003Fu) | 0x64006400u, -1024.f);
          ul.v[h][t][p] = add_h2((pr & 0x003F003Fu) | 0x64006400u, -1024.f);
        }
    }
    dft2(sh.fwd, uh, ul, [](int) {}, [&](int mt, const f4v& e, const f4v& o) { set_chunk(u[j], mt, e, o); });
  }
  HPoly ph, pl;
  row_product<K, Loaded12<K>>(
      u, sh.gamma, sh.gammaq, x.g,
      [&](Loaded12<K>& l, int t) {
#pragma unroll
        for (int j = 0; j < K; ++j) load_chunk<12>(l.w[j], q.key + 384 * j, as, t);
      },
      [&](float (&a)[8], const Loaded12<K>& l, int j, int) { chunk_from12(a, l.w[j]); },
      [&](int t, const f4v& e, const f4v& o) { set_digits(ph, pl, t, e, o); });
  Words<P::dv> vw[3];
  uint8_t* m = sc.row_of(x.grp, x.n) + kRowM;
  auto pre = [&](int t) { load_chunk<P::dv>(vw[t % 3], q.ct + P::polyvec_cbytes, av, t); };
  dft2(sh.inv, ph, pl, pre, [&](int mt, const f4v& e, const f4v& o) {
    uint32_t v[8];
    unpack_chunk<P::dv>(v, vw[mt % 3], av.sh);
    uint32_t bits = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      bits |= f32::compress_f<1>((float)decompress_d<P::dv>(v[k]) - ((k & 1) ? o[k >> 1] : e[k >> 1])) << k;
    if (x.act) m[4 * mt + x.g] = (uint8_t)bits;
  });
}

// One output polynomial of indcpa_enc: inverse transform, + noise (+ message bits),
// compressed to D bits; compared with the ciphertext (DEC) or stored.
template <int D, bool DEC, bool MSG>
__device__ __forceinline__ uint32_t finish_poly(const u4v* inv, const HPoly& ph, const HPoly& pl, const Scratch& sc,
                                                int noise, const uint8_t* msg, uint8_t* ct, const Lane& x) {
  int g = x.g;
  asm volatile("" : "+v"(g));  // offsets per polynomial, not kept across the row products
  const ChunkAt<D> ac(g);
  Words<D> cw[DEC ? 3 : 1];
  uint32_t pw[3], mw[3];
  auto pre = [&](int t) {
    pw[t % 3] = sc.prf_load(x.grp, noise, t, x.prf_off());
    if constexpr (DEC) load_chunk<D>(cw[t % 3], ct, ac, t);
    if constexpr (MSG) mw[t % 3] = (uint32_t)*(const global_t<uint8_t>*)(msg + 4 * t + x.g);
  };
  uint32_t bad = 0;
  dft2(inv, ph, pl, pre, [&](int mt, const f4v& e, const f4v& o) {
    uint32_t ne[2], no[2], v[8];
    cbd_chunk(ne, no, pw[mt % 3]);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = k >> 1;
      float c = ((k & 1) ? o[i] : e[i]) + h2_get((k & 1) ? no[i >> 1] : ne[i >> 1], i & 1);
      if constexpr (MSG) c += ((mw[mt % 3] >> k) & 1) ? (float)((Q + 1) / 2) : 0.f;
      v[k] = f32::compress_f<D>(c);
    }
    if constexpr (DEC) {
      uint32_t t[8];
      unpack_chunk<D>(t, cw[mt % 3], ac.sh);
#pragma unroll
      for (int k = 0; k < 8; ++k) bad |= v[k] ^ t[k];
      asm volatile("" : "+v"(bad));  // this tile's compare ends here (else the values wait for the last tile)
    } else {
      if (x.act) store_chunk<D>(ct, x.g, mt, v);
    }
  });
  return bad;
}

// indcpa_enc of a tile (indcpa.cu:578-679).  DEC: compare, fail flags of the tile's 64
// requests into LDS.  Otherwise write the ciphertexts.
template <int K, bool DEC, class Src>
__device__ __forceinline__ void reencrypt_tile(const Src& src, const Scratch& sc, const Bucket& b, int tile,
                                               const DftLds<true, true>& sh) {
  using P = Params<K>;
  constexpr int PK_OFF = DEC ? P::sk_cpa_bytes : 0;  // public key inside the key buffer
  const Lane x = lane_of(b, tile);
  const ReqP q = src.template req<K, DEC>(x.r);
  HPoly r[K];
#pragma unroll
  for (int j = 0; j < K; ++j) noise_ntt(r[j], sc, x, j, sh.fwd);
  uint32_t bad = 0;
#pragma unroll 1
  for (int i = 0; i < K; ++i) {
#pragma unroll
    for (int j = 0; j < K; ++j) keep_packed(r[j]);
    HPoly ph, pl;
    const uint8_t* at = sc.at_chunk(x.grp, 0, i * K, 0);
    row_product<K, Loaded16<K>>(
        r, sh.gamma, sh.gammaq, x.g,
        [&](Loaded16<K>& l, int t) {
#pragma unroll
          for (int j = 0; j < K; ++j) l.w[j] = *(const global_t<u4v>*)(at + (j * 32 + 4 * t) * 256 + x.at_off());
        },
        [&](float (&a)[8], const Loaded16<K>& l, int j, int) { chunk_from16(a, l.w[j]); },
        [&](int t, const f4v& e, const f4v& o) { set_digits(ph, pl, t, e, o); });
    bad |= finish_poly<P::du, DEC, false>(sh.inv, ph, pl, sc, K + i, nullptr, q.ct + 32 * P::du * i, x);
  }
  {
    const ChunkAt<12> at12(x.g);
    HPoly ph, pl;
    row_product<K, Loaded12<K>>(
        r, sh.gamma, sh.gammaq, x.g,
        [&](Loaded12<K>& l, int t) {
#pragma unroll
          for (int j = 0; j < K; ++j) load_chunk<12>(l.w[j], q.key + PK_OFF + 384 * j, at12, t);
        },
        [&](float (&a)[8], const Loaded12<K>& l, int j, int) { chunk_from12(a, l.w[j]); },
        [&](int t, const f4v& e, const f4v& o) { set_digits(ph, pl, t, e, o); });
    bad |= finish_poly<P::dv, DEC, true>(sh.inv, ph, pl, sc, 2 * K, sc.row_of(x.grp, x.n) + kRowM,
                                         q.ct + P::polyvec_cbytes, x);
  }
  if constexpr (DEC) {
    bad |= (uint32_t)__shfl_xor((int)bad, 16);
    bad |= (uint32_t)__shfl_xor((int)bad, 32);
    if (x.g == 0 && x.act) *reinterpret_cast<uint32_t*>(sc.row_of(x.grp, x.n) + kRowFail) = bad;
  }
}

// Key generation of a tile (indcpa_keypair, indcpa.cu:474-533): s^ = NTT(s) into the
// secret key, t^ = A o s^ + NTT(e) into both copies of the public key, as canonical
// residues (the reference's frommont(A o s^) + e^, csubq'd; A o s^ carries no Montgomery
// factor here)
template <int K>
__device__ __forceinline__ void key_tile(const KeySrc& src, const Scratch& sc, const Bucket& b, int tile,
                                         const DftLds<true, false>& sh) {
  using P = Params<K>;
  const Lane x = lane_of(b, tile);
  uint8_t* sk = src.sk + (size_t)x.r * P::sk_bytes;
  uint8_t* pk = src.pk + (size_t)x.r * P::pk_bytes;
  HPoly sv[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    noise_ntt(sv[j], sc, x, j, sh.fwd);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      uint32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = f32::canon_f(h2_get(sv[j].v[k & 1][t][k >> 2], (k >> 1) & 1));
      if (x.act) store_chunk<12>(sk + 384 * j, x.g, t, v);
    }
  }
#pragma unroll 1
  for (int i = 0; i < K; ++i) {
#pragma unroll
    for (int j = 0; j < K; ++j) keep_packed(sv[j]);
    HPoly eh;
    noise_ntt(eh, sc, x, K + i, sh.fwd);
    const uint8_t* at = sc.at_chunk(x.grp, 0, i * K, 0);
    row_product<K, Loaded16<K>>(
        sv, sh.gamma, sh.gammaq, x.g,
        [&](Loaded16<K>& l, int t) {
#pragma unroll
          for (int j = 0; j < K; ++j) l.w[j] = *(const global_t<u4v>*)(at + (j * 32 + 4 * t) * 256 + x.at_off());
        },
        [&](float (&a)[8], const Loaded16<K>& l, int j, int) { chunk_from16(a, l.w[j]); },
        [&](int t, const f4v& e, const f4v& o) {
          uint32_t v[8];
#pragma unroll
          for (int k = 0; k < 8; ++k)
            v[k] = f32::canon_f(((k & 1) ? o[k >> 1] : e[k >> 1]) + h2_get(eh.v[k & 1][t][k >> 2], (k >> 1) & 1));
          if (x.act) {
            store_chunk<12>(pk + 384 * i, x.g, t, v);
            store_chunk<12>(sk + P::sk_cpa_bytes + 384 * i, x.g, t, v);
          }
        });
  }
}

// ss = KDF(Kbar or z, H(ct)) of 64 requests, one lane each
template <int K, class Src>
__device__ __forceinline__ void dec_kdf_wave(const Src& src, const Scratch& sc, const Bucket& b, int w) {
  using P = Params<K>;
  const int r = 64 * w + (threadIdx.x & 63);
  if (r >= b.n) return;
  const ReqP q = src.template req<K, true>(r);
  const uint8_t* row = sc.row_of(b.grp0 + r / 16, r % 16);
  const uint32_t f = *reinterpret_cast<const uint32_t*>(row + kRowFail);
  const uint64_t mask = 0 - (uint64_t)((f | (0u - f)) >> 31);
  uint64_t m[8], A[25];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint64_t kb = load_u64_global(row + kRowKbar + 8 * i), zz = load_u64_global(q.key + P::z_off + 8 * i);
    m[i] = kb ^ (mask & (zz ^ kb));
    m[4 + i] = load_u64_global(row + kRowH + 8 * i);
  }
  absorb_fixed<kRateShake256, 8, true>(A, m, 0x1F);
  store_words4(q.ss, A);
}

// ---- dense kernels ---------------------------------------------------------------------------
template <int K>
__global__ __launch_bounds__(kProdThreads, 2) void k_open(int n, DenseSrc src, Scratch sc) {
  __shared__ DftLds<true, true> sh;
  load_tables<true, true, kProdThreads>(sh, &c_dft);
  const Bucket b{n, 0};
  for (int tile = blockIdx.x; tile < (n + 63) / 64; tile += gridDim.x) open_tile<K>(src, sc, b, tile, sh);
}

// waves: H(ct), then G and PRF (the longest chains first), then the matrix entries
template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_dec_sponge(int n, DenseSrc src, Scratch sc) {
  using P = Params<K>;
  __shared__ SponLds sh;
  const Bucket b{n, 0};
  const int wr = (n + 63) / 64, total = 2 * wr + matrix_waves<K>(n);
  for (int w = blockIdx.x; w < total; w += gridDim.x) {
    if (w < wr)
      dec_hash_wave<K>(src, sc, b, w);
    else if (w < 2 * wr)
      dec_prf_wave<K>(src, sc, b, w - wr);
    else
      matrix_wave<K, true>(sc, b, w - 2 * wr, sh, [&](int r) {
        return src.template req<K, true>(r).key + P::sk_cpa_bytes + P::polyvec_bytes;
      });
  }
}

// at most kFewMax requests: a wave per 64 noise streams, then the matrix entries
template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_dec_sponge_few(int n, DenseSrc src, Scratch sc) {
  using P = Params<K>;
  __shared__ SponLds sh;
  const int wr = (n + 63) / 64, wp = wr * (2 * K + 1), total = wp + matrix_waves<K>(n);
  for (int w = blockIdx.x; w < total; w += gridDim.x) {
    if (w < wp)
      dec_prf_one<K>(src, sc, n, w % wr, w / wr);
    else
      matrix_wave<K, true>(sc, Bucket{n, 0}, w - wp, sh, [&](int r) {
        return src.template req<K, true>(r).key + P::sk_cpa_bytes + P::polyvec_bytes;
      });
  }
}

template <int K>
__global__ __launch_bounds__(kProdThreads, 2) void k_dec_reencrypt(int n, DenseSrc src, Scratch sc) {
  __shared__ DftLds<true, true> sh;
  load_tables<true, true, kProdThreads>(sh, &c_dft);
  const Bucket b{n, 0};
  for (int tile = blockIdx.x; tile < (n + 63) / 64; tile += gridDim.x) reencrypt_tile<K, true>(src, sc, b, tile, sh);
}

// at most kFewMax requests: the first `prod` workgroups re-encrypt, 64 requests each at a
// time, which leaves most CUs without work; the others hash ciphertexts, 16 requests each,
// for the KDF after this stage
template <int K>
__global__ __launch_bounds__(kProdThreads, 2) void k_dec_reencrypt_few(int n, int prod, DenseSrc src, Scratch sc) {
  constexpr int kWaves = kProdThreads / 64;
  __shared__ union {
    DftLds<true, true> dft;
    struct {
      wide::Consts consts;
      wide::States states[kWaves];
    } h;
  } sh;
  if ((int)blockIdx.x < prod) {
    load_tables<true, true, kProdThreads>(sh.dft, &c_dft);
    for (int tile = blockIdx.x; tile < (n + 63) / 64; tile += prod)
      reencrypt_tile<K, true>(src, sc, Bucket{n, 0}, tile, sh.dft);
    return;
  }
  wide::init_consts(sh.h.consts);
  __syncthreads();
  wide::Sponge s;
  const int wave = threadIdx.x >> 6;
  s.init(sh.h.states[wave], sh.h.consts);
  const int w = ((int)blockIdx.x - prod) * kWaves + wave;
  if (w < (n + 3) / 4) dec_hash_wide<K>(src, sc, n, w, s);
}

template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_dec_kdf(int n, DenseSrc src, Scratch sc) {
  for (int w = blockIdx.x; w < (n + 63) / 64; w += gridDim.x) dec_kdf_wave<K>(src, sc, Bucket{n, 0}, w);
}

// a kernel of one wave per four requests: NAME(n, source, scratch) runs the statement for
// each wave w of the batch
#define WIDE_KERNEL(NAME, SRC, ...)                                                                       \
  template <int K, int W>                                                                                 \
  __global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void NAME(int n, SRC src, Scratch sc) {              \
    __shared__ WideLds sh;                                                                                \
    wide::init_consts(sh.consts);                                                                         \
    __syncthreads();                                                                                      \
    wide::Sponge s;                                                                                       \
    s.init(sh.states, sh.consts);                                                                         \
    for (int w = blockIdx.x; w < (n + 3) / 4; w += gridDim.x) __VA_ARGS__;                                \
  }
WIDE_KERNEL(k_dec_kdf_few, DenseSrc, dec_kdf_wide<K>(src, sc, n, w, s, sh))
WIDE_KERNEL(k_enc_final_few, DenseSrc, enc_final_wide<K>(src, sc, n, w, s, sh))
WIDE_KERNEL(k_key_final_few, KeySrc, key_final_wide<K>(src, sc, n, w, s))
#undef WIDE_KERNEL

// encapsulation: H(pk), m, G (the longest chains first), then the matrix entries
template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_enc_sponge(int n, DenseSrc src, Scratch sc) {
  using P = Params<K>;
  __shared__ SponLds sh;
  const Bucket b{n, 0};
  const int wr = (n + 63) / 64, total = wr + matrix_waves<K>(n);
  for (int w = blockIdx.x; w < total; w += gridDim.x) {
    if (w < wr)
      enc_open_wave<K>(src, sc, b, w);
    else
      matrix_wave<K, true>(sc, b, w - wr, sh,
                           [&](int r) { return src.template req<K, false>(r).key + P::polyvec_bytes; });
  }
}

template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_enc_sponge_few(int n, DenseSrc src, Scratch sc) {
  using P = Params<K>;
  __shared__ union {
    SponLds m;
    WideLds h;
  } sh;
  const int wh = (n + 3) / 4, total = wh + matrix_waves<K>(n);
  for (int w = blockIdx.x; w < total; w += gridDim.x) {
    if (w < wh) {
      wide::Sponge s;
      __syncthreads();
      wide::init_consts(sh.h.consts);
      __syncthreads();
      s.init(sh.h.states, sh.h.consts);
      enc_open_wide<K>(src, sc, n, w, s, sh.h);
      __syncthreads();
    } else {
      matrix_wave<K, true>(sc, Bucket{n, 0}, w - wh, sh.m,
                           [&](int r) { return src.template req<K, false>(r).key + P::polyvec_bytes; });
    }
  }
}

template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_enc_prf(int n, Scratch sc) {
  const int wr = (n + 63) / 64;
  for (int w = blockIdx.x; w < wr * (2 * K + 1); w += gridDim.x) prf_wave(sc, Bucket{n, 0}, w % wr, w / wr);
}

template <int K>
__global__ __launch_bounds__(kProdThreads, 2) void k_enc_encrypt(int n, DenseSrc src, Scratch sc) {
  __shared__ DftLds<true, true> sh;
  load_tables<true, true, kProdThreads>(sh, &c_dft);
  const Bucket b{n, 0};
  for (int tile = blockIdx.x; tile < (n + 63) / 64; tile += gridDim.x) reencrypt_tile<K, false>(src, sc, b, tile, sh);
}

template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_enc_final(int n, DenseSrc src, Scratch sc) {
  for (int w = blockIdx.x; w < (n + 63) / 64; w += gridDim.x) enc_final_wave<K>(src, sc, Bucket{n, 0}, w);
}

// key generation
template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_key_seed(int n, KeySrc src, Scratch sc) {
  for (int w = blockIdx.x; w < (n + 63) / 64; w += gridDim.x) key_seed_wave<K>(src, sc, n, w);
}

template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_key_sponge(int n, KeySrc src, Scratch sc) {
  using P = Params<K>;
  __shared__ SponLds sh;
  const Bucket b{n, 0};
  const int mw = matrix_waves<K>(n), wr = (n + 63) / 64;
  for (int w = blockIdx.x; w < mw + 2 * K * wr; w += gridDim.x) {
    if (w < mw)
      matrix_wave<K, false>(sc, b, w, sh, [&](int r) { return src.pk + (size_t)r * P::pk_bytes + P::polyvec_bytes; });
    else
      prf_wave(sc, b, (w - mw) % wr, (w - mw) / wr);
  }
}

template <int K>
__global__ __launch_bounds__(kProdThreads, 2) void k_key_mul(int n, KeySrc src, Scratch sc) {
  __shared__ DftLds<true, false> sh;
  load_tables<true, false, kProdThreads>(sh, &c_dft);
  for (int tile = blockIdx.x; tile < (n + 63) / 64; tile += gridDim.x) key_tile<K>(src, sc, Bucket{n, 0}, tile, sh);
}

template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_key_final(int n, KeySrc src) {
  for (int w = blockIdx.x; w < (n + 63) / 64; w += gridDim.x) key_final_wave<K>(src, n, w);
}

// up to kPairMax requests
template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_enc_final_pair(int n, DenseSrc src, Scratch sc) {
  for (int w = blockIdx.x; w < (n + 31) / 32; w += gridDim.x) enc_final_pair<K>(src, sc, n, w);
}
template <int K, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_key_final_pair(int n, KeySrc src) {
  for (int w = blockIdx.x; w < (n + 31) / 32; w += gridDim.x) key_final_pair<K>(src, n, w);
}

// ---- mixed kernels ------------------------------------------------------------------------------
// The three buckets of k_mixed_classify, longest requests first.  Their sizes are known
// on the device only, so a launch has workgroups for the worst case and those without
// work leave.
struct Buckets {
  Bucket b2, b3, b4;
};
__device__ __forceinline__ Buckets buckets_of(const uint32_t* __restrict__ counts) {
  const int n2 = (int)counts[0], n3 = (int)counts[1], n4 = (int)counts[2];
  const int g4 = (n4 + 15) / 16, g3 = (n3 + 15) / 16;
  return Buckets{Bucket{n2, g4 + g3}, Bucket{n3, g4}, Bucket{n4, 0}};
}

// item w of the sequence [c4 items of K = 4][c3 of K = 3][c2 of K = 2]: f(K, bucket, item)
// for it; false when w is past them (then w is what is left)
template <class F>
__device__ __forceinline__ bool bucket_item(const Buckets& bs, int& w, int c4, int c3, int c2, F&& f) {
  if (w < c4) {
    f(std::integral_constant<int, 4>{}, bs.b4, w);
    return true;
  }
  w -= c4;
  if (w < c3) {
    f(std::integral_constant<int, 3>{}, bs.b3, w);
    return true;
  }
  w -= c3;
  if (w < c2) {
    f(std::integral_constant<int, 2>{}, bs.b2, w);
    return true;
  }
  w -= c2;
  return false;
}

template <class F>
__device__ __forceinline__ bool bucket_tile(const Buckets& bs, int& w, F&& f) {
  return bucket_item(bs, w, (bs.b4.n + 63) / 64, (bs.b3.n + 63) / 64, (bs.b2.n + 63) / 64, f);
}

template <bool DEC, class F>
__device__ __forceinline__ void mixed_matrix(const Buckets& bs, const MixedSrc& src, const Scratch& sc, int w, F& sh) {
  bucket_item(bs, w, matrix_waves<4>(bs.b4.n), matrix_waves<3>(bs.b3.n), matrix_waves<2>(bs.b2.n),
              [&](auto k, const Bucket& b, int i) {
                constexpr int K = decltype(k)::value;
                using P = Params<K>;
                matrix_wave<K, true>(sc, b, i, sh, [&](int r) {
                  return src.template req<K, DEC>(r).key + (DEC ? P::sk_cpa_bytes : 0) + P::polyvec_bytes;
                });
              });
}

__global__ __launch_bounds__(kProdThreads, 2) void k_mixed_open(const uint32_t* counts, MixedSrc src, Scratch sc) {
  __shared__ DftLds<true, true> sh;
  load_tables<true, true, kProdThreads>(sh, &c_dft);
  const Buckets bs = buckets_of(counts);
  for (int t = blockIdx.x;; t += gridDim.x) {
    int w = t;
    if (!bucket_tile(bs, w, [&](auto k, const Bucket& b, int i) { open_tile<decltype(k)::value>(src, sc, b, i, sh); }))
      break;
  }
}

__global__ __launch_bounds__(64, 4) void k_mixed_dec_sponge(const uint32_t* counts, MixedSrc src, Scratch sc) {
  __shared__ SponLds sh;
  const Buckets bs = buckets_of(counts);
  const int end = (bs.b4.n + 63) / 64 + (bs.b3.n + 63) / 64 + (bs.b2.n + 63) / 64;
  const int total = 2 * end + matrix_waves<4>(bs.b4.n) + matrix_waves<3>(bs.b3.n) + matrix_waves<2>(bs.b2.n);
  for (int t = blockIdx.x; t < total; t += gridDim.x) {
    int w = t;
    if (bucket_tile(bs, w, [&](auto k, const Bucket& b, int i) { dec_hash_wave<decltype(k)::value>(src, sc, b, i); }))
      continue;
    if (bucket_tile(bs, w, [&](auto k, const Bucket& b, int i) { dec_prf_wave<decltype(k)::value>(src, sc, b, i); }))
      continue;
    mixed_matrix<true>(bs, src, sc, w, sh);
  }
}

template <bool DEC>
__global__ __launch_bounds__(kProdThreads, 2) void k_mixed_encrypt(const uint32_t* counts, MixedSrc src, Scratch sc) {
  __shared__ DftLds<true, true> sh;
  load_tables<true, true, kProdThreads>(sh, &c_dft);
  const Buckets bs = buckets_of(counts);
  for (int t = blockIdx.x;; t += gridDim.x) {
    int w = t;
    if (!bucket_tile(bs, w, [&](auto k, const Bucket& b, int i) {
          reencrypt_tile<decltype(k)::value, DEC>(src, sc, b, i, sh);
        }))
      break;
  }
}

// KDF (DEC), or H(ct) and KDF
template <bool DEC, int W>
__global__ __launch_bounds__(64) PQC_SIMD_WAVES(W) void k_mixed_final(const uint32_t* counts, MixedSrc src, Scratch sc) {
  const Buckets bs = buckets_of(counts);
  for (int t = blockIdx.x;; t += gridDim.x) {
    int w = t;
    if (!bucket_tile(bs, w, [&](auto k, const Bucket& b, int i) {
          if constexpr (DEC)
            dec_kdf_wave<decltype(k)::value>(src, sc, b, i);
          else
            enc_final_wave<decltype(k)::value>(src, sc, b, i);
        }))
      break;
  }
}

__global__ __launch_bounds__(64, 4) void k_mixed_enc_sponge(const uint32_t* counts, MixedSrc src, Scratch sc) {
  __shared__ SponLds sh;
  const Buckets bs = buckets_of(counts);
  const int end = (bs.b4.n + 63) / 64 + (bs.b3.n + 63) / 64 + (bs.b2.n + 63) / 64;
  const int total = end + matrix_waves<4>(bs.b4.n) + matrix_waves<3>(bs.b3.n) + matrix_waves<2>(bs.b2.n);
  for (int t = blockIdx.x; t < total; t += gridDim.x) {
    int w = t;
    if (bucket_tile(bs, w, [&](auto k, const Bucket& b, int i) { enc_open_wave<decltype(k)::value>(src, sc, b, i); }))
      continue;
    mixed_matrix<false>(bs, src, sc, w, sh);
  }
}

__global__ __launch_bounds__(64, 4) void k_mixed_prf(const uint32_t* counts, Scratch sc) {
  const Buckets bs = buckets_of(counts);
  for (int t = blockIdx.x;; t += gridDim.x) {
    int w = t;
    if (!bucket_item(bs, w, 9 * ((bs.b4.n + 63) / 64), 7 * ((bs.b3.n + 63) / 64), 5 * ((bs.b2.n + 63) / 64),
                     [&](auto, const Bucket& b, int i) {
                       const int wr = (b.n + 63) / 64;
                       prf_wave(sc, b, i % wr, i / wr);
                     }))
      break;
  }
}

// ---- launchers ---------------------------------------------------------------------------------
static Scratch scratch_of(const pqc_ctx* c, int k) {
  return Scratch{c->kprf, (size_t)(2 * k + 1) * 2048, c->kat, (size_t)k * k * 16 * 512, c->krow, c->status};
}

// Product stages: persistent, two workgroups per CU (66 KB of tables each) at the default
// fused_waves_per_cu of 4.  Sponge stages: one workgroup per wave of work, handed out by
// the hardware in the order of their number; below 4, as many as fit that many per SIMD.
static int prod_grid(const pqc_ctx* c, int tiles) {
  const int g = c->fused_grid_override > 0 ? c->fused_grid_override : c->cu_count * c->tune.fused_waves_per_cu / 2;
  return std::max(1, std::min(g, tiles));
}
static int sponge_grid(const pqc_ctx* c, int waves) {
  int g = waves;
  if (c->fused_grid_override > 0)
    g = c->fused_grid_override;
  else if (c->tune.fused_waves_per_cu < 4)
    g = c->cu_count * 4 * c->tune.fused_waves_per_cu;
  return std::max(1, std::min(g, waves));
}

// one-wave workgroups of a kernel templated on the waves per SIMD it is compiled for
#define LAUNCH_WAVES(c, grid, s, KERNEL, ...)                                                 \
  with_simd_waves((c)->cu_count, grid, [&](auto w) {                                          \
    constexpr int W = decltype(w)::value;                                                     \
    hipLaunchKernelGGL((KERNEL), dim3(grid), dim3(64), 0, s, __VA_ARGS__);                    \
  })

template <int K>
static int dec(pqc_ctx* c, size_t n_all, uint8_t* ss, uint8_t* ct, const uint8_t* sk, hipStream_t s) {
  using P = Params<K>;
  const Scratch sc = scratch_of(c, K);
  for (size_t at = 0; at < n_all; at += c->kstage_max) {
    const int n = (int)std::min(n_all - at, c->kstage_max);
    const bool few = n <= kFewMax;
    const int tiles = (n + 63) / 64, fours = (n + 3) / 4;
    const int waves = tiles * (few ? 2 * K + 1 : 2) + matrix_waves<K>(n), prod = prod_grid(c, tiles);
    const DenseSrc src{ss + at * 32, ct + at * P::ct_bytes, sk + at * P::sk_bytes, nullptr, c->kprf};
    hipLaunchKernelGGL((k_open<K>), dim3(prod), dim3(kProdThreads), 0, s, n, src, sc);
    const int sg = sponge_grid(c, waves), kg = sponge_grid(c, few ? fours : tiles);
    if (few)
      LAUNCH_WAVES(c, sg, s, (k_dec_sponge_few<K, W>), n, src, sc);
    else
      LAUNCH_WAVES(c, sg, s, (k_dec_sponge<K, W>), n, src, sc);
    if (few)
      hipLaunchKernelGGL((k_dec_reencrypt_few<K>), dim3(prod + (fours + 3) / 4), dim3(kProdThreads), 0, s, n, prod, src,
                         sc);
    else
      hipLaunchKernelGGL((k_dec_reencrypt<K>), dim3(prod), dim3(kProdThreads), 0, s, n, src, sc);
    if (few)
      LAUNCH_WAVES(c, kg, s, (k_dec_kdf_few<K, W>), n, src, sc);
    else
      LAUNCH_WAVES(c, kg, s, (k_dec_kdf<K, W>), n, src, sc);
    const int rc = hip_err(hipGetLastError());
    if (rc) return rc;
  }
  return PQC_OK;
}

template <int K>
static int enc(pqc_ctx* c, size_t n_all, uint8_t* ss, uint8_t* ct, const uint8_t* pk, const uint8_t* coins,
               hipStream_t s) {
  using P = Params<K>;
  const Scratch sc = scratch_of(c, K);
  for (size_t at = 0; at < n_all; at += c->kstage_max) {
    const int n = (int)std::min(n_all - at, c->kstage_max);
    const bool few = n <= kFewMax;
    const int tiles = (n + 63) / 64, hash = few ? (n + 3) / 4 : tiles;
    const DenseSrc src{ss + at * 32, ct + at * P::ct_bytes, pk + at * P::pk_bytes, coins + at * 32, c->kprf};
    const int sg = sponge_grid(c, hash + matrix_waves<K>(n)), pg = sponge_grid(c, tiles * (2 * K + 1)),
              fg = sponge_grid(c, hash), qg = sponge_grid(c, (n + 31) / 32);
    if (few)
      LAUNCH_WAVES(c, sg, s, (k_enc_sponge_few<K, W>), n, src, sc);
    else
      LAUNCH_WAVES(c, sg, s, (k_enc_sponge<K, W>), n, src, sc);
    LAUNCH_WAVES(c, pg, s, (k_enc_prf<K, W>), n, sc);
    hipLaunchKernelGGL((k_enc_encrypt<K>), dim3(prod_grid(c, tiles)), dim3(kProdThreads), 0, s, n, src, sc);
    if (few)
      LAUNCH_WAVES(c, fg, s, (k_enc_final_few<K, W>), n, src, sc);
    else if (n <= kPairMax)
      LAUNCH_WAVES(c, qg, s, (k_enc_final_pair<K, W>), n, src, sc);
    else
      LAUNCH_WAVES(c, fg, s, (k_enc_final<K, W>), n, src, sc);
    const int rc = hip_err(hipGetLastError());
    if (rc) return rc;
  }
  return PQC_OK;
}

template <int K>
static int keypair(pqc_ctx* c, size_t n_all, uint8_t* pk, uint8_t* sk, const uint8_t* coins, hipStream_t s) {
  using P = Params<K>;
  const Scratch sc = scratch_of(c, K);
  for (size_t at = 0; at < n_all; at += c->kstage_max) {
    const int n = (int)std::min(n_all - at, c->kstage_max);
    const int tiles = (n + 63) / 64;
    const KeySrc src{pk + at * P::pk_bytes, sk + at * P::sk_bytes, coins + at * 64};
    const bool few = n <= kFewMax;
    const int sg = sponge_grid(c, matrix_waves<K>(n) + 2 * K * tiles), fg = sponge_grid(c, tiles),
              hg = sponge_grid(c, (n + 3) / 4), qg = sponge_grid(c, (n + 31) / 32);
    LAUNCH_WAVES(c, fg, s, (k_key_seed<K, W>), n, src, sc);
    LAUNCH_WAVES(c, sg, s, (k_key_sponge<K, W>), n, src, sc);
    hipLaunchKernelGGL((k_key_mul<K>), dim3(prod_grid(c, tiles)), dim3(kProdThreads), 0, s, n, src, sc);
    if (few)
      LAUNCH_WAVES(c, hg, s, (k_key_final_few<K, W>), n, src, sc);
    else if (n <= kPairMax)
      LAUNCH_WAVES(c, qg, s, (k_key_final_pair<K, W>), n, src);
    else
      LAUNCH_WAVES(c, fg, s, (k_key_final<K, W>), n, src);
    const int rc = hip_err(hipGetLastError());
    if (rc) return rc;
  }
  return PQC_OK;
}

// A mixed batch of at most kstage_max requests, already classified
static int mixed(pqc_ctx* c, int dec, size_t n, const MixedSrc& src, hipStream_t s) {
  const int kmax = (int)(c->kprf_per_elem / 128 - 1) / 2;  // largest K the context holds
  const Scratch sc = scratch_of(c, kmax);
  const uint32_t* counts = c->kmix_counts;
  const int tiles = (int)(n / 64) + 3;  // each bucket rounds up by itself
  const int mat = ((int)((n + 15) / 16) + 3) * kmax * kmax / 4 + 3;
  const int fg = sponge_grid(c, tiles);
  const dim3 prod(prod_grid(c, tiles)), prod_wg(kProdThreads), wg(64);
  if (dec) {
    hipLaunchKernelGGL(k_mixed_open, prod, prod_wg, 0, s, counts, src, sc);
    hipLaunchKernelGGL(k_mixed_dec_sponge, dim3(sponge_grid(c, 2 * tiles + mat)), wg, 0, s, counts, src, sc);
    hipLaunchKernelGGL(k_mixed_encrypt<true>, prod, prod_wg, 0, s, counts, src, sc);
    LAUNCH_WAVES(c, fg, s, (k_mixed_final<true, W>), counts, src, sc);
  } else {
    hipLaunchKernelGGL(k_mixed_enc_sponge, dim3(sponge_grid(c, tiles + mat)), wg, 0, s, counts, src, sc);
    hipLaunchKernelGGL(k_mixed_prf, dim3(sponge_grid(c, tiles * (2 * kmax + 1))), wg, 0, s, counts, sc);
    hipLaunchKernelGGL(k_mixed_encrypt<false>, prod, prod_wg, 0, s, counts, src, sc);
    LAUNCH_WAVES(c, fg, s, (k_mixed_final<false, W>), counts, src, sc);
  }
  return hip_err(hipGetLastError());
}

}  // namespace staged
}  // namespace kyber

size_t kyber_stage_at_bytes(int k) { return (size_t)k * k * 512; }

int kyber_staged_dec(pqc_ctx* c, int k, size_t n, uint8_t* ss, const uint8_t* ct, const uint8_t* sk, hipStream_t s) {
  uint8_t* ctm = const_cast<uint8_t*>(ct);
  switch (k) {
    case 2: return kyber::staged::dec<2>(c, n, ss, ctm, sk, s);
    case 3: return kyber::staged::dec<3>(c, n, ss, ctm, sk, s);
    case 4: return kyber::staged::dec<4>(c, n, ss, ctm, sk, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

int kyber_staged_enc(pqc_ctx* c, int k, size_t n, uint8_t* ct, uint8_t* ss, const uint8_t* pk, const uint8_t* coins,
                     hipStream_t s) {
  switch (k) {
    case 2: return kyber::staged::enc<2>(c, n, ss, ct, pk, coins, s);
    case 3: return kyber::staged::enc<3>(c, n, ss, ct, pk, coins, s);
    case 4: return kyber::staged::enc<4>(c, n, ss, ct, pk, coins, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

int kyber_staged_keypair(pqc_ctx* c, int k, size_t n, uint8_t* pk, uint8_t* sk, const uint8_t* coins, hipStream_t s) {
  switch (k) {
    case 2: return kyber::staged::keypair<2>(c, n, pk, sk, coins, s);
    case 3: return kyber::staged::keypair<3>(c, n, pk, sk, coins, s);
    case 4: return kyber::staged::keypair<4>(c, n, pk, sk, coins, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

int kyber_staged_mixed(pqc_ctx* c, int dec, size_t n, const kyber::MixedSrc& src, hipStream_t s) {
  return kyber::staged::mixed(c, dec, n, src, s);
}

}  // namespace pqc
