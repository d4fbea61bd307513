// Kyber dispatch, mixed-batch classification, and the fused persistent kernels over
// 64-request tiles (tuning.fused_*_tile = 64, the allocation-free entry above 8192 requests,
// contexts whose budget has no room for the staged path's scratch).
//
// One workgroup = one wave64; a persistent grid walks tiles of up to 64
// requests.  Inside a tile the work is split two ways:
//   * per-request sponge chains (H(ct), G, PRF, KDF, and for encaps H(seed),
//     H(pk), H(ct)) run one request per lane, the Keccak state in VGPRs;
//   * the matrix A^T is generated in rounds of up to 64 SHAKE128 entries, one
//     entry per lane, rejection-sampled straight from the state registers into
//     LDS, and consumed by the wave-cooperative polynomial arithmetic
//     (one request at a time, 4 coefficients per lane, NTT butterflies through
//     register/lane-bit swaps; kyber_wave.cuh).
// Keccak lanes stay >= 98% busy: every request contributes K*K entries per
// round and one lane per sequential chain.
//
// Data flow per request follows the round-2 FO decapsulation assembled from
// the reference's pieces: indcpa_dec (Kyber_GPU_Batched/indcpa.cu:691-733),
// G = sha3_512 (fips202.cu:672-689), indcpa_enc (indcpa.cu:578-679),
// verify + cmov (verify.cu:15-50, here a wave-wide OR of coefficient
// mismatches, no branch on it), H = sha3_256 (fips202.cu:615-632) and
// KDF = SHAKE256 (symmetric.h:33).  Comparing compressed coefficients is
// comparing ciphertext bytes: every width packs 256 coefficients into whole
// bytes with no unused bits.
#include <algorithm>
#include <mutex>

#include "internal.h"
#include "req_check.h"
#include "kyber_coop.cuh"
#include "kyber_src.cuh"
#include "kyber_wave.cuh"
#include "kyber_wavef.cuh"
#include "sponge.cuh"

namespace pqc {
namespace kyber {
namespace fused {

__constant__ LaneTwiddles c_lane_tw = make_lane_twiddles();
__constant__ LaneTwiddlesF c_lane_twf = kLaneTwF;

constexpr int kAStride = 262;   // int16 slots per A entry: 256 + guard, odd dword count
static_assert(kAStride >= N + 4, "guard slots for a word's four candidates past the 256th accept");
constexpr int kMaxBlocks = 32;  // SHAKE128 blocks per entry before giving up (never reached)

// A tile is 64 requests, one per lane in the per-request phases.  Its 64*K*K
// matrix entries are generated in K*K rounds of 64 (one per lane).  Entry
// E = t*K*K + i*K + j lives in ring slot E mod RING; a round's 64 entries plus
// the at most K*K-1 earlier entries of a request that straddles two rounds are
// exactly RING consecutive values of E, so no live slot is ever overwritten.
template <int K>
struct Tile {
  static constexpr int T = 64;                                  // requests per tile
  static constexpr int KK = K * K;
  static constexpr int NR = KK;                                 // rounds: 64*K*K / 64
  static constexpr int RING = (64 % KK == 0) ? 64 : 64 + KK - 1;  // 64, 72, 64 slots
  static constexpr int PRFB = (2 * K + 1) * 128;                // PRF bytes per request
};

template <int RING>
struct Lds {
  int16_t a[RING * kAStride];
  uint8_t msg[64][32];
  uint32_t fail[64];
};

// Sources of the A^T entries for the re-encryption: at.get(i, j, w0, w1) gives
// this lane's group of entry (i, j) as two words of two coefficients.
template <int K>
struct AtRing {  // the LDS ring of the 64-request tiles: entry e0 + i K + j in slot mod RING
  const int16_t* ring;
  int e0;
  __device__ __forceinline__ void get(int i, int j, uint32_t& w0, uint32_t& w1) const {
    const int slot = (e0 + i * K + j) % Tile<K>::RING;
    const uint32_t* e32 = reinterpret_cast<const uint32_t*>(ring + slot * kAStride + 4 * ntt_group(lane_id()));
    w0 = e32[0];
    w1 = e32[1];
  }
};

// ---- per-lane sponge pieces ---------------------------------------------------

// SHAKE128(rho || i || j) rejection-sampled into an LDS entry (gen_matrix_n,
// indcpa.cu:339-403, rej_uniform indcpa.cu:290-322).  The entry keeps the
// accepted 16-bit candidates themselves (< 19q): the reference stores
// v - (v >> 12) q, the same residue, and every consumer reduces the entry mod q
// when it converts it to FP32.  Every candidate is written without a branch:
// at the running position p, which advances past accepted ones only: a
// rejected candidate is overwritten by the next one, and whatever lies at or
// past the final count is never read.  p is clamped to slot 256 after each
// word's four candidates, so writes past the 256th land in slots 256..259
// (kAStride leaves 262).  Returns the accept count, clamped (256 unless the
// block cap was hit).
__device__ __forceinline__ int sample_entry(int16_t* dst, const uint64_t (&rho)[4], int x, int y, bool valid) {
  uint64_t A[25];
#pragma unroll
  for (int t = 0; t < 25; ++t) A[t] = (t < 4) ? rho[t] : 0;
  A[4] = (uint64_t)x | ((uint64_t)y << 8) | (0x1Full << 16);
  A[kRateShake128 - 1] ^= 0x8000000000000000ull;
  int16_t* p = dst;
  int16_t* const end = dst + N;
  for (int blk = 0; blk < kMaxBlocks; ++blk) {
    if (blk >= 4 && !__any(valid && p < end)) break;
    keccakf1600(A);
#pragma unroll
    for (int w = 0; w < kRateShake128; ++w) {
      const uint32_t half[2] = {(uint32_t)A[w], (uint32_t)(A[w] >> 32)};
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const uint32_t val = (h & 1) ? (half[h >> 1] >> 16) : (half[h >> 1] & 0xFFFFu);
        *p = (int16_t)val;
        p += val < 19u * Q ? 1 : 0;
      }
      p = p < end ? p : end;
    }
  }
  return (int)(p - dst);
}

// Request t of the tile, from the lane that holds it (t wave-uniform): no
// descriptor reload for the cooperative phases.
__device__ __forceinline__ ReqP lane_req(const ReqP& me, int t) {
  auto rd = [t](const void* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, t), hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), t);
    return reinterpret_cast<uint8_t*>(((uint64_t)hi << 32) | lo);
  };
  return ReqP{rd(me.ss), rd(me.ct), rd(me.key), rd(me.coins), rd(me.prf)};
}

// One tile of up to 64 requests (indices base .. base + 63 of the source, n of
// them valid) through the whole FO encapsulation (DEC false) or decapsulation.
// The cooperative phases load request t + 1's inputs while request t computes
// (one wave per SIMD: nothing else hides the loads' latency).
template <int K, bool DEC, class Src>
__device__ __forceinline__ void fused_tile(const Src& src, int base, int n, Lds<Tile<K>::RING>& sh, const LaneZF& z,
                                           uint32_t* __restrict__ status) {
  using P = Params<K>;
  using TL = Tile<K>;
  constexpr int PK_OFF = DEC ? P::sk_cpa_bytes : 0;  // public key inside the key buffer
  const int lane = threadIdx.x;
  const int r = base + lane;
  const bool active = lane < TL::T && r < n;
  const int rc = active ? r : min(base, n - 1);  // clamped request for address math
  const ReqP me = src.template req<K, DEC>(rc);
  uint64_t kbar[4], hct[4];

  if constexpr (DEC) {
    // ---- H(ct), one request per lane
    {
      uint64_t A[25];
      sponge_absorb_words_prefetch<kRateSha3_256>(A, reinterpret_cast<const uint64_t*>(me.ct), P::ct_bytes / 8, 0x06);
#pragma unroll
      for (int w = 0; w < 4; ++w) hct[w] = A[w];
    }
    // ---- indcpa_dec, wave-cooperative, one request at a time
    const int nt = min(TL::T, n - base);
    // request t's words were loaded during request t - 1: the copy at the top of
    // the iteration is the only wait for them, and the prefetch issued after it
    // is not waited for until the next iteration
    DecIn<K> cur, nxt;
    {
      const ReqP q = lane_req(me, 0);
      dec_load<K>(nxt, q.ct, q.key);
    }
    for (int t = 0; t < nt; ++t) {
      cur = nxt;
      if (t + 1 < nt) {
        const ReqP q = lane_req(me, t + 1);
        dec_load<K>(nxt, q.ct, q.key);
      }
      coop_indcpa_dec_f<K>(cur, z, sh.msg[t]);
    }
    __syncthreads();
  } else {
    // ---- m = H(seed) ("don't release system RNG output"), H(pk)
    uint64_t A[25];
    uint64_t c4[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) c4[w] = load_u64(me.coins + 8 * w);
    absorb_fixed<kRateSha3_256, 4>(A, c4, 0x06);
    if (active) {
#pragma unroll
      for (int w = 0; w < 4; ++w) store_u64(sh.msg[lane] + 8 * w, A[w]);
    }
    sponge_absorb_words_prefetch<kRateSha3_256>(A, reinterpret_cast<const uint64_t*>(me.key), P::pk_bytes / 8, 0x06);
#pragma unroll
    for (int w = 0; w < 4; ++w) hct[w] = A[w];  // holds H(pk) until G
    __syncthreads();
  }

  // ---- (Kbar, coins) = G(m || H(pk)); PRF(coins, 0..2K) -> scratch
  {
    uint64_t m[8], A[25];
    const uint8_t* msg = sh.msg[lane < TL::T ? lane : 0];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      m[w] = load_u64(msg + 8 * w);
      m[4 + w] = DEC ? load_u64_global(me.key + P::hpk_off + 8 * w) : hct[w];
    }
    absorb_fixed<kRateSha3_512, 8>(A, m, 0x06);
    uint64_t rc4[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      kbar[w] = A[w];
      rc4[w] = A[4 + w];
    }
    for (int nonce = 0; nonce < 2 * K + 1; ++nonce) {
      absorb_fixed<kRateShake256, 4>(A, rc4, (uint64_t)nonce | (0x1Full << 8));
      if (active) {
#pragma unroll
        for (int w = 0; w < 16; ++w) store_u64(me.prf + 128 * nonce + 8 * w, A[w]);
      }
    }
  }
  __syncthreads();

  // ---- A^T rounds + re-encryption
  const int nt = min(TL::T, n - base);
  int t_done = 0;  // requests whose re-encryption is finished
  EncIn<K, DEC> cur, nxt;
  // rho of this lane's entry in round g: the public seed of request E / KK, its
  // key pointer taken from the lane that holds it (invalid entries use lane 0's)
  auto load_rho = [&](uint64_t (&rho)[4], int g) {
    const int t = (64 * g + lane) / TL::KK;
    const uint8_t* key = reinterpret_cast<const uint8_t*>(__shfl((long long)me.key, t < nt ? t : 0));
#pragma unroll
    for (int w = 0; w < 4; ++w) rho[w] = load_u64_global(key + PK_OFF + P::polyvec_bytes + 8 * w);
  };
  uint64_t rho_next[4];
  load_rho(rho_next, 0);
  // a partial tile needs only the rounds that hold its nt * K^2 entries (a lone
  // request: one round instead of K^2, each at least 4 Keccak-f)
  const int ng = min(TL::NR, (nt * TL::KK + 63) / 64);
  for (int g = 0; g < ng; ++g) {
    // requests all of whose entries are sampled by the end of this round
    const int t_end = min(nt, (64 * (g + 1)) / TL::KK);
    if (t_done < t_end) {  // the round's first request loads during the sampling
      const ReqP q = lane_req(me, t_done);
      enc_load<K, DEC>(cur, q.prf, q.key + PK_OFF, q.ct);
    }
    {
      const int E = 64 * g + lane;
      const int t = E / TL::KK;
      const int ij = E % TL::KK;
      const bool valid = t < nt;
      uint64_t rho[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) rho[w] = rho_next[w];
      const int got = sample_entry(sh.a + (E % TL::RING) * kAStride, rho, ij / K, ij % K, valid);
      if (valid && got < N) atomicOr(status, 1u);
    }
    __syncthreads();
    // the next round's rho loads during this round's re-encryptions
    if (g + 1 < ng) load_rho(rho_next, g + 1);
    for (int t = t_done; t < t_end; ++t) {
      if (t + 1 < t_end) {
        const ReqP q = lane_req(me, t + 1);
        enc_load<K, DEC>(nxt, q.prf, q.key + PK_OFF, q.ct);
      }
      const ReqP q = lane_req(me, t);
      const uint32_t mm = coop_reencrypt_f<K, DEC>(AtRing<K>{sh.a, t * TL::KK}, cur, sh.msg[t], q.ct, z);
      cur = nxt;
      if constexpr (DEC) {
        const uint32_t f = __any(mm != 0) ? 1u : 0u;
        if (lane == 0) sh.fail[t] = f;
      }
    }
    t_done = max(t_done, t_end);
    __syncthreads();
  }

  // ---- KDF
  {
    uint64_t m[8], A[25];
    if constexpr (DEC) {
      const uint64_t mask = 0 - (uint64_t)(sh.fail[lane < TL::T ? lane : 0] & 1u);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint64_t zz = load_u64_global(me.key + P::z_off + 8 * w);
        m[w] = kbar[w] ^ (mask & (zz ^ kbar[w]));
        m[4 + w] = hct[w];
      }
    } else {
      sponge_absorb_words_prefetch<kRateSha3_256>(A, reinterpret_cast<const uint64_t*>(me.ct), P::ct_bytes / 8, 0x06);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        m[w] = kbar[w];
        m[4 + w] = A[w];
      }
    }
    absorb_fixed<kRateShake256, 8>(A, m, 0x1F);
    if (active) {
#pragma unroll
      for (int w = 0; w < 4; ++w) store_u64(me.ss + 8 * w, A[w]);
    }
  }
  __syncthreads();
}

// ---- key generation -----------------------------------------------------------------
// indcpa_keypair (Kyber_GPU_Batched/indcpa.cu:474-564) + the KEM tail: (rho, sigma)
// = G(d); s_j = CBD(PRF(sigma, j)), e_i = CBD(PRF(sigma, K + i)), both through
// poly_ntt (ntt + Barrett); t_i = frommont(sum_j A[i][j] o s_j) + e_i, Barrett;
// pk = t || rho, sk = s || pk || H(pk) || z, polynomials packed 12 bits per
// coefficient after csubq (polyvec_tobytes).  A is not transposed:
// A[i][j] = SHAKE128(rho || j || i) (gen_matrix_n with transposed = 0).

template <int K>
struct KeyIn {
  uint32_t prf[2 * K];
};

template <int K>
__device__ __forceinline__ void key_load(KeyIn<K>& in, const uint8_t* prf) {
  const uint16_t* prf16 = reinterpret_cast<const uint16_t*>(prf);
#pragma unroll
  for (int j = 0; j < 2 * K; ++j) in.prf[j] = prf16[64 * j + lane_id()];
}

// one request's s and t, written into sk_cpa, pk and sk's copy of pk, on the
// exact FP32 arithmetic (kyber_wavef.cuh).  The reference computes
// t = frommont(A o s) + e (basemul carries R^-1, frommont multiplies by R^2 R^-1)
// and packs csubq'd residues; here A o s carries no factor, and canon_f gives
// the same residues in [0, q).
template <int K, class AT>
__device__ __forceinline__ void coop_keypair(const AT& at, const KeyIn<K>& in, uint8_t* pk, uint8_t* sk,
                                             const LaneZF& z) {
  using P = Params<K>;
  const int gn = ntt_group(lane_id());
  F4 sv[K];
  Bz svz[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    P4 c;
    cbd_group(c, in.prf[j]);  // [-2, 2]
    sv[j] = to_f4(c);
    ntt_f<2>(sv[j], z);
    reduce_f4(sv[j]);
    svz[j] = basemul_twist(sv[j], z);
#pragma unroll
    for (int r = 0; r < 4; ++r) c.v[r] = (int32_t)f32::canon_f(sv[j].v[r]);
    store_poly12(sk + 384 * j, gn, c);
  }
#pragma unroll
  for (int i = 0; i < K; ++i) {
    F4 acc = basemul_sum_f<K>(
        [&](int j) {
          uint32_t w0, w1;
          at.get(i, j, w0, w1);  // A[i][j]: accepted candidates, [0, 19q)
          F4 a = {{(float)(w0 & 0xFFFF), (float)(w0 >> 16), (float)(w1 & 0xFFFF), (float)(w1 >> 16)}};
          reduce_f4(a);
          return a;
        },
        sv, svz);
    P4 e;
    cbd_group(e, in.prf[K + i]);
    F4 ef = to_f4(e);
    ntt_f<2>(ef, z);
    static_assert(f32::fwd_out_bound(2) + f32::kOut <= f32::kCanonMax, "t = A o s + e within canon_f's range");
    P4 c;
#pragma unroll
    for (int r = 0; r < 4; ++r) c.v[r] = (int32_t)f32::canon_f(acc.v[r] + ef.v[r]);
    store_poly12(pk + 384 * i, gn, c);
    store_poly12(sk + P::sk_cpa_bytes + 384 * i, gn, c);
  }
}

struct KeySrc {
  uint8_t* pk;
  uint8_t* sk;
  const uint8_t* coins;  // 64 bytes per request: d || z
  uint8_t* prf;
};

template <int K>
__device__ __forceinline__ void fused_keypair_tile(const KeySrc& src, int base, int n, Lds<Tile<K>::RING>& sh,
                                                   const LaneZF& z, uint32_t* __restrict__ status) {
  using P = Params<K>;
  using TL = Tile<K>;
  const int lane = threadIdx.x;
  const int r = base + lane;
  const bool active = r < n;
  const int rc = active ? r : base;  // clamped request for address math
  uint8_t* pk = src.pk + (size_t)rc * P::pk_bytes;
  uint8_t* sk = src.sk + (size_t)rc * P::sk_bytes;
  uint8_t* prf = src.prf + (size_t)rc * TL::PRFB;
  const uint8_t* coins = src.coins + (size_t)rc * 64;
  // ---- (rho, sigma) = G(d); PRF(sigma, 0 .. 2K-1) -> scratch; rho -> LDS and both pk copies
  {
    uint64_t d[4], A[25], sg[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) d[w] = load_u64(coins + 8 * w);
    absorb_fixed<kRateSha3_512, 4>(A, d, 0x06);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      sg[w] = A[4 + w];
      store_u64(sh.msg[lane] + 8 * w, A[w]);
      if (active) {
        store_u64(pk + P::polyvec_bytes + 8 * w, A[w]);
        store_u64(sk + P::sk_cpa_bytes + P::polyvec_bytes + 8 * w, A[w]);
      }
    }
    for (int nonce = 0; nonce < 2 * K; ++nonce) {
      absorb_fixed<kRateShake256, 4>(A, sg, (uint64_t)nonce | (0x1Full << 8));
      if (active) {
#pragma unroll
        for (int w = 0; w < 16; ++w) store_u64(prf + 128 * nonce + 8 * w, A[w]);
      }
    }
  }
  __syncthreads();
  // ---- A rounds + t, s
  const int nt = min(TL::T, n - base);
  int t_done = 0;
  KeyIn<K> cur, nxt;
  const int ng = min(TL::NR, (nt * TL::KK + 63) / 64);  // rounds that hold the tile's entries
  for (int g = 0; g < ng; ++g) {
    const int t_end = min(nt, (64 * (g + 1)) / TL::KK);
    if (t_done < t_end) key_load<K>(cur, src.prf + (size_t)(base + t_done) * TL::PRFB);
    {
      const int E = 64 * g + lane;
      const int t = E / TL::KK;
      const int ij = E % TL::KK;
      const bool valid = t < nt;
      uint64_t rho[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) rho[w] = load_u64(sh.msg[valid ? t : 0] + 8 * w);
      const int got = sample_entry(sh.a + (E % TL::RING) * kAStride, rho, ij % K, ij / K, valid);
      if (valid && got < N) atomicOr(status, 1u);
    }
    __syncthreads();
    for (int t = t_done; t < t_end; ++t) {
      if (t + 1 < t_end) key_load<K>(nxt, src.prf + (size_t)(base + t + 1) * TL::PRFB);
      coop_keypair<K>(AtRing<K>{sh.a, t * TL::KK}, cur, src.pk + (size_t)(base + t) * P::pk_bytes,
                      src.sk + (size_t)(base + t) * P::sk_bytes, z);
      cur = nxt;
    }
    t_done = max(t_done, t_end);
    __syncthreads();
  }
  // ---- H(pk) over the packed key (written by the whole wave), z
  {
    uint64_t A[25];
    sponge_absorb_words_prefetch<kRateSha3_256>(A, reinterpret_cast<const uint64_t*>(pk), P::pk_bytes / 8, 0x06);
    if (active) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        store_u64(sk + P::hpk_off + 8 * w, A[w]);
        store_u64(sk + P::z_off + 8 * w, load_u64(coins + 32 + 8 * w));
      }
    }
  }
  __syncthreads();
}

template <int K>
__global__ __launch_bounds__(64) void k_fused_keypair(int n, int ntiles, KeySrc src, uint32_t* __restrict__ status) {
  __shared__ Lds<Tile<K>::RING> sh;
  LaneZF z;
  load_lane_zf(z, &c_lane_twf);
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) fused_keypair_tile<K>(src, tile * 64, n, sh, z, status);
}

template <int K, bool DEC>
__global__ __launch_bounds__(64) void k_fused(int n, int ntiles, DenseSrc src, uint32_t* __restrict__ status) {
  __shared__ Lds<Tile<K>::RING> sh;
  LaneZF z;
  load_lane_zf(z, &c_lane_twf);
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) fused_tile<K, DEC>(src, tile * 64, n, sh, z, status);
}

// ---- mixed parameter sets ------------------------------------------------------
// Bucket n descriptors by K (Kyber-512/768/1024 -> K 2/3/4) into order[(K-2) * cap
// + slot], counts[K-2] = bucket sizes.  One wave-aggregated global atomic per
// bucket per wave; the order inside a bucket is whatever the atomics give (the
// results do not depend on it).  Descriptors with another algorithm id, an
// unaligned offset, a buffer outside its arena or a parameter set the context
// was not created for are skipped and set status bit 1.
__global__ void k_mixed_zero(uint32_t* counts) {
  if (threadIdx.x < 3) counts[threadIdx.x] = 0;
}

// One thread per descriptor, 1024 per workgroup.  A request's place inside its
// bucket does not matter, so each workgroup reserves its places with one atomic
// per K (the same three counters taken once per wave made the launch ~26 us at
// 65536 descriptors), and each wave's share follows from the waves before it.
constexpr int kClassifyBlock = 1024;
__global__ __launch_bounds__(kClassifyBlock) void k_mixed_classify(
    int n, int cap, int dec, unsigned alg_mask, const pqc_kem_req* __restrict__ reqs, uint64_t ct_bytes,
    uint64_t key_bytes, uint64_t ss_bytes, uint64_t coins_bytes, uint32_t* __restrict__ order,
    uint32_t* __restrict__ counts, uint32_t* __restrict__ status) {
  constexpr int kWaves = kClassifyBlock / 64;
  __shared__ uint32_t wcount[3][kWaves], wbase[3][kWaves];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int k = 0;
  if (i < n) {
    const pqc_kem_req d = reqs[i];
    k = pqc_req_k(d, dec != 0, alg_mask, ct_bytes, key_bytes, ss_bytes, coins_bytes);
    if (!k) atomicOr(status, 2u);
  }
  uint64_t mine = 0;  // the ballot of this lane's K
#pragma unroll
  for (int kk = 2; kk <= 4; ++kk) {
    const uint64_t mask = __ballot(k == kk);
    if (k == kk) mine = mask;
    if (lane == 0) wcount[kk - 2][wave] = (uint32_t)__popcll(mask);
  }
  __syncthreads();
  if (threadIdx.x < 3) {  // thread j: bucket K = j + 2
    const int j = threadIdx.x;
    uint32_t run = 0;
    for (int w = 0; w < kWaves; ++w) {
      wbase[j][w] = run;
      run += wcount[j][w];
    }
    const uint32_t g = run ? atomicAdd(&counts[j], run) : 0u;
    for (int w = 0; w < kWaves; ++w) wbase[j][w] += g;
  }
  __syncthreads();
  if (k) {
    const uint32_t below = (uint32_t)__popcll(mine & ((1ull << lane) - 1));
    order[(size_t)(k - 2) * cap + wbase[k - 2][wave] + below] = (uint32_t)i;
  }
}

// Tile i of a mixed batch -> (K, tile index inside the K bucket).  order 0:
// K = 4, 3, 2 (longest tiles first keeps the tail short); 1: K = 2, 3, 4;
// 2: round-robin over the buckets that still have tiles, in the order 4, 3, 2.
struct TilePick {
  int k, idx;
};

__device__ __forceinline__ TilePick pick_tile(int i, int order, int t4, int t3, int t2) {
  if (order == 0) {
    if (i < t4) return {4, i};
    if (i < t4 + t3) return {3, i - t4};
    return {2, i - t4 - t3};
  }
  if (order == 1) {
    if (i < t2) return {2, i};
    if (i < t2 + t3) return {3, i - t2};
    return {4, i - t2 - t3};
  }
  // round-robin: phases in which 3, 2, then 1 buckets remain
  int ks[3] = {4, 3, 2}, ts[3] = {t4, t3, t2};
  int done = 0;  // tiles per bucket consumed by earlier phases
  int live = (t4 > 0) + (t3 > 0) + (t2 > 0);
  while (live > 0) {
    int m = 1 << 30;  // rounds in this phase: the smallest remaining bucket
    for (int b = 0; b < 3; ++b)
      if (ts[b] > done && ts[b] - done < m) m = ts[b] - done;
    if (m == (1 << 30)) break;
    if (i < live * m) {
      const int round = i / live, pos = i % live;
      int seen = 0;
      for (int b = 0; b < 3; ++b)
        if (ts[b] > done) {
          if (seen == pos) return {ks[b], done + round};
          ++seen;
        }
    }
    i -= live * m;
    done += m;
    live = 0;
    for (int b = 0; b < 3; ++b) live += ts[b] > done ? 1 : 0;
  }
  return {0, 0};  // not reached for i below t4 + t3 + t2
}

// Persistent walk over the tiles of the three buckets.  LDS is sized for the
// largest ring (K = 3).
union LdsMixed {
  Lds<Tile<2>::RING> k2;
  Lds<Tile<3>::RING> k3;
  Lds<Tile<4>::RING> k4;
};

// Requests per tile of each bucket.  Order 3 (split) halves the K = 4 and K = 2
// tiles and walks K 4, 3, 2: with one tile per wave the launch lasts as long as
// its heaviest tile, and a K = 4 half tile plus a K = 2 half tile on one wave is
// about one K = 3 tile (the per-request sponges of a half tile run on half the
// lanes, its Aᵀ rounds and cooperative work halve).  The autotuner measures it
// against the other orders; a tile of fewer requests is a partial tile.
__host__ __device__ __forceinline__ int mixed_tile_req(int order, int k) { return (order == 3 && k != 3) ? 32 : 64; }

template <bool DEC>
__global__ __launch_bounds__(64) void k_fused_mixed(MixedSrc src, const uint32_t* __restrict__ counts, int order,
                                                    uint32_t* __restrict__ status) {
  __shared__ LdsMixed sh;
  LaneZF z;
  load_lane_zf(z, &c_lane_twf);
  const int n2 = (int)counts[0], n3 = (int)counts[1], n4 = (int)counts[2];
  const int s4 = mixed_tile_req(order, 4), s3 = mixed_tile_req(order, 3), s2 = mixed_tile_req(order, 2);
  const int t4 = (n4 + s4 - 1) / s4, t3 = (n3 + s3 - 1) / s3, t2 = (n2 + s2 - 1) / s2;
  const int walk = order == 3 ? 0 : order;
  for (int tile = blockIdx.x; tile < t4 + t3 + t2; tile += gridDim.x) {
    const TilePick p = pick_tile(tile, walk, t4, t3, t2);
    if (p.k == 4)
      fused_tile<4, DEC>(src, p.idx * s4, min(n4, (p.idx + 1) * s4), sh.k4, z, status);
    else if (p.k == 3)
      fused_tile<3, DEC>(src, p.idx * s3, min(n3, (p.idx + 1) * s3), sh.k3, z, status);
    else if (p.k == 2)
      fused_tile<2, DEC>(src, p.idx * s2, min(n2, (p.idx + 1) * s2), sh.k2, z, status);
  }
}

// ---- component kernels -------------------------------------------------------

// poly_ntt / poly_invntt on polynomials in coefficient order, one per wave.
__global__ __launch_bounds__(64) void k_poly_transform(int op, int n, int16_t* polys) {
  const int l = threadIdx.x;
  LaneZ z;
  load_lane_z(z, &c_lane_tw);
  for (int p = blockIdx.x; p < n; p += gridDim.x) {
    int16_t* poly = polys + (size_t)p * N;
    const int gin = op == 0 ? nat_group(l) : ntt_group(l);
    const int gout = op == 0 ? ntt_group(l) : nat_group(l);
    P4 x;
#pragma unroll
    for (int r = 0; r < 4; ++r) x.v[r] = poly[4 * gin + r];
    if (op == 0)
      ntt(x, z);
    else
      invntt(x, z);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) poly[4 * gout + r] = (int16_t)x.v[r];
    __syncthreads();
  }
}

// n fixed-length messages, one per lane: SHA3-256 / SHA3-512 / SHAKE128 / SHAKE256.
template <int RATE>
__device__ void keccak_one(uint8_t* out, size_t outlen, const uint8_t* in, int words, uint8_t domain) {
  uint64_t A[25];
  sponge_absorb_words<RATE>(A, reinterpret_cast<const uint64_t*>(in), words, domain);
  size_t done = 0;
  while (true) {
#pragma unroll
    for (int w = 0; w < RATE; ++w) {
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const size_t o = done + 8 * w + b;
        if (o < outlen) out[o] = (uint8_t)(A[w] >> (8 * b));
      }
    }
    done += 8 * RATE;
    if (done >= outlen) break;
    keccakf1600(A);
  }
}

__global__ void k_keccak_batch(int op, int n, uint8_t* out, size_t outlen, const uint8_t* in, size_t inlen) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  const uint8_t* m = in + (size_t)x * inlen;
  uint8_t* o = out + (size_t)x * outlen;
  const int words = (int)(inlen / 8);
  switch (op) {
    case 0: keccak_one<kRateSha3_256>(o, outlen, m, words, 0x06); break;
    case 1: keccak_one<kRateSha3_512>(o, outlen, m, words, 0x06); break;
    case 2: keccak_one<kRateShake128>(o, outlen, m, words, 0x1F); break;
    default: keccak_one<kRateShake256>(o, outlen, m, words, 0x1F); break;
  }
}

template <int K, bool DEC>
static int launch_fused(pqc_ctx* c, size_t n, uint8_t* ss, uint8_t* ct, const uint8_t* key, const uint8_t* coins,
                        hipStream_t s) {
  if (n == 0) return PQC_OK;
  const int ntiles = (int)((n + Tile<K>::T - 1) / Tile<K>::T);
  int grid = c->fused_grid_override > 0 ? c->fused_grid_override : c->cu_count * c->tune.fused_waves_per_cu;
  if (grid > ntiles) grid = ntiles;
  if (grid < 1) grid = 1;
  const DenseSrc src{ss, ct, key, coins, c->kprf};
  hipLaunchKernelGGL((k_fused<K, DEC>), dim3(grid), dim3(64), 0, s, (int)n, ntiles, src, c->status);
  return hip_err(hipGetLastError());
}

// Kyber batches of at most this many requests take the one-workgroup-per-request kernels
// (kyber_lowlat.hip), larger ones the stages (kyber_staged.hip).  A request's workgroup of
// four to six waves brings the time up in steps of one workgroup per CU (256 requests); the
// line is the last step at which the stages are slower.  Measured on MI355X, per-request /
// staged, us: Kyber-512 encapsulation 101 / 104 at 1280; Kyber-768 decapsulation 91 / 102 at
// 1024 and 127 / 104 at 1280, encapsulation 121 / 123 and 170 / 128, key generation 91 / 116
// and 122 / 118; Kyber-1024 decapsulation 122 / 126 and 172 / 135, key generation 134 / 150
// and 171 / 154, encapsulation 132 / 159 at 768 and 198 / 158 at 1024.  Mixed batches, whose
// stages hash on one lane per request: decapsulation 181 / 213 at 1536 (1:2:1; Kyber-512
// alone 109 / 116 at 1500) and 230 / 220 at 2048, encapsulation 253 / 308 at 1281 and 323 /
// 311 at 1800, but Kyber-512 alone 174 / 179 and 193 / 178 at 1500.
// tuning.lowlat_max overrides them all (-1 = never).
constexpr int lowlat_mixed(bool dec) { return dec ? 1536 : 1280; }
constexpr int lowlat_limit(int k, bool enc) { return k == 2 ? 1280 : k == 4 && enc ? 768 : 1024; }

// Larger batches run in stages unless `tile` (a fused_*_tile knob) says 64-request tiles or
// the context's budget left no scratch for the stages, or so little that the batch would
// take many passes of them: a pass lasts ~95 (Kyber-512) to ~160 us however short it is, 230
// to 320 mixed, where one tile launch does up to 65536 requests in 510, 880, 1290 us (mixed
// 1320).  Measured on MI355X, us, 2 / 4 / 8 passes and tiles: 65536 Kyber-768
// encapsulations 746 / 1147 / 1664 and 885, 16384 of them 418 / 597 / 1061 and 871; Kyber-512
// 501 / 764 / 1192 and 508, 298 / 481 / 855 and 496; mixed 970 / 1403 / 2566 and 1313, 643 /
// 1280 / 2513 and 1293.
inline bool use_stages(const pqc_ctx* c, size_t n, int tile) {
  if (!c->kat || tile == 64 || n == 0) return false;
  const size_t block = std::min<size_t>(n, 65536);  // no pass is longer
  return (block + c->kstage_max - 1) / c->kstage_max <= (block <= 16384 ? 4 : 2);
}

inline bool use_lowlat(const pqc_ctx* c, size_t n, int dflt) {
  const int lim = c->tune.lowlat_max != 0 ? c->tune.lowlat_max : dflt;
  return n > 0 && (long long)n <= (long long)lim;
}

template <int K>
static int launch_fused_keypair(pqc_ctx* c, size_t n, uint8_t* pk, uint8_t* sk, const uint8_t* coins, hipStream_t s) {
  if (n == 0) return PQC_OK;
  const int ntiles = (int)((n + Tile<K>::T - 1) / Tile<K>::T);
  int grid = c->fused_grid_override > 0 ? c->fused_grid_override : c->cu_count * c->tune.fused_waves_per_cu;
  if (grid > ntiles) grid = ntiles;
  if (grid < 1) grid = 1;
  const KeySrc src{pk, sk, coins, c->kprf};
  hipLaunchKernelGGL((k_fused_keypair<K>), dim3(grid), dim3(64), 0, s, (int)n, ntiles, src, c->status);
  return hip_err(hipGetLastError());
}

}  // namespace fused
}  // namespace kyber

int kyber_fused_keypair(pqc_ctx* c, int k, size_t n, uint8_t* pk, uint8_t* sk, const uint8_t* coins, hipStream_t s) {
  if (c->tune.fused_key_tile != 64 && kyber::fused::use_lowlat(c, n, kyber::fused::lowlat_limit(k, false)))
    return kyber_lowlat_keypair(k, n, pk, sk, coins, c->status, s);
  if (kyber::fused::use_stages(c, n, c->tune.fused_key_tile)) return kyber_staged_keypair(c, k, n, pk, sk, coins, s);
  switch (k) {
    case 2: return kyber::fused::launch_fused_keypair<2>(c, n, pk, sk, coins, s);
    case 3: return kyber::fused::launch_fused_keypair<3>(c, n, pk, sk, coins, s);
    case 4: return kyber::fused::launch_fused_keypair<4>(c, n, pk, sk, coins, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

int kyber_fused_dec(pqc_ctx* c, int k, size_t n, uint8_t* ss, const uint8_t* ct, const uint8_t* sk, hipStream_t s) {
  uint8_t* ctm = const_cast<uint8_t*>(ct);  // read-only in the decaps instantiation
  if (kyber::fused::use_lowlat(c, n, kyber::fused::lowlat_limit(k, false))) return kyber_lowlat_dec(k, n, ss, ct, sk, c->status, s);
  if (kyber::fused::use_stages(c, n, c->tune.fused_dec_tile)) return kyber_staged_dec(c, k, n, ss, ct, sk, s);
  switch (k) {
    case 2: return kyber::fused::launch_fused<2, true>(c, n, ss, ctm, sk, nullptr, s);
    case 3: return kyber::fused::launch_fused<3, true>(c, n, ss, ctm, sk, nullptr, s);
    case 4: return kyber::fused::launch_fused<4, true>(c, n, ss, ctm, sk, nullptr, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

int kyber_fused_enc(pqc_ctx* c, int k, size_t n, uint8_t* ct, uint8_t* ss, const uint8_t* pk, const uint8_t* coins,
                    hipStream_t s) {
  if (kyber::fused::use_lowlat(c, n, kyber::fused::lowlat_limit(k, true)))
    return kyber_lowlat_enc(k, n, ct, ss, pk, coins, c->status, s);
  if (kyber::fused::use_stages(c, n, c->tune.fused_enc_tile)) return kyber_staged_enc(c, k, n, ct, ss, pk, coins, s);
  switch (k) {
    case 2: return kyber::fused::launch_fused<2, false>(c, n, ss, ct, pk, coins, s);
    case 3: return kyber::fused::launch_fused<3, false>(c, n, ss, ct, pk, coins, s);
    case 4: return kyber::fused::launch_fused<4, false>(c, n, ss, ct, pk, coins, s);
    default: return PQC_ERR_UNSUPPORTED;
  }
}

// Mixed Kyber-512/768/1024 batch: classify into buckets, then the stages (or one persistent
// launch over 64-request tiles).  Every launch has a fixed shape (the bucket sizes are read on the
// device), so the sequence can be captured into a graph and replayed.
int kyber_fused_mixed(pqc_ctx* c, int dec, size_t n, const pqc_kem_req* reqs, uint8_t* ct, size_t ct_bytes,
                      const uint8_t* key, size_t key_bytes, uint8_t* ss, size_t ss_bytes, const uint8_t* coins,
                      size_t coins_bytes, hipStream_t s) {
  using namespace kyber::fused;
  if (n == 0) return PQC_OK;
  if (!c->kmix_order || !c->kprf) return PQC_ERR_UNSUPPORTED;
  if (use_lowlat(c, n, lowlat_mixed(dec != 0)))  // one workgroup per descriptor, no bucketing
    return kyber_lowlat_mixed(c, dec, n, reqs, ct, ct_bytes, key, key_bytes, ss, ss_bytes, coins, coins_bytes, s);
  const int cap = (int)c->max_batch;
  auto classify = [&](const pqc_kem_req* r, size_t m) {
    hipLaunchKernelGGL(k_mixed_zero, dim3(1), dim3(64), 0, s, c->kmix_counts);
    hipLaunchKernelGGL(k_mixed_classify, dim3((unsigned)((m + kClassifyBlock - 1) / kClassifyBlock)),
                       dim3(kClassifyBlock), 0, s, (int)m, cap, dec, c->alg_mask, r, (uint64_t)ct_bytes,
                       (uint64_t)key_bytes, (uint64_t)ss_bytes, (uint64_t)coins_bytes, c->kmix_order, c->kmix_counts,
                       c->status);
  };
  kyber::MixedSrc src{reqs, c->kmix_order, cap, ss, ct, key, coins, c->kprf, c->kprf_per_elem};
  if (use_stages(c, n, dec ? c->tune.fused_dec_tile : c->tune.fused_enc_tile)) {
    // in stages, kstage_max requests at a time (their scratch)
    for (size_t at = 0; at < n; at += c->kstage_max) {
      const size_t m = std::min(n - at, c->kstage_max);
      classify(reqs + at, m);
      src.reqs = reqs + at;
      const int rc = kyber_staged_mixed(c, dec, m, src, s);
      if (rc) return rc;
    }
    return PQC_OK;
  }
  classify(reqs, n);
  const int max_tiles = (int)((n + 31) / 32) + 2;  // half tiles at most; buckets round up separately
  int grid = c->fused_grid_override > 0 ? c->fused_grid_override : c->cu_count * c->tune.fused_waves_per_cu;
  if (grid > max_tiles) grid = max_tiles;
  if (grid < 1) grid = 1;
  if (dec)
    hipLaunchKernelGGL(k_fused_mixed<true>, dim3(grid), dim3(64), 0, s, src, (const uint32_t*)c->kmix_counts,
                       c->tune.mixed_order, c->status);
  else
    hipLaunchKernelGGL(k_fused_mixed<false>, dim3(grid), dim3(64), 0, s, src, (const uint32_t*)c->kmix_counts,
                       c->tune.mixed_order, c->status);
  return hip_err(hipGetLastError());
}

// ---- allocation-free decapsulation ------------------------------------------------
// pqc_kyber_dec_batch_noalloc gives the bytes of crypto_kem_dec_batch by the two forms
// that need no context's scratch: the per-request kernels up to 8192 requests, where the
// context path has been in stages for long, and 64-request tiles above.  The tile
// kernel's PRF rows and the status word are in `scratch`, a file-scope device array (one
// copy per GPU, held until the process ends).  The host never names `scratch`
// directly (in host code it is only a stand-in symbol): the device address is
// looked up once per device with hipGetSymbolAddress and that address is what
// the kernels receive.  Nothing in the scratch must start at zero: every PRF
// row is written by the same tile before it is read, and the status word only
// collects bits for callers that pass no status word of their own.
constexpr size_t kNoAllocMax = PQC_NOALLOC_MAX_BATCH;
constexpr size_t kNoAllocPrf = kNoAllocMax * kyber::fused::Tile<4>::PRFB;  // K = 4 rows are the largest
constexpr size_t kNoAllocBytes = 256 + kNoAllocPrf;                        // status word, then the PRF rows
static __device__ __align__(256) uint8_t scratch[kNoAllocBytes];

namespace {
constexpr int kMaxDevices = 64;
struct NoAllocDev {
  uint8_t* ptr = nullptr;  // device address of `scratch` on this device
  int cus = 0;
  bool ready = false;
};
std::mutex g_noalloc_mu;
NoAllocDev g_noalloc[kMaxDevices];

// Set-up on the first call on a device, with that device current.
int noalloc_device(NoAllocDev* out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return PQC_ERR_NO_DEVICE;
  if (dev < 0 || dev >= kMaxDevices) return PQC_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  NoAllocDev& d = g_noalloc[dev];
  if (!d.ready) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return PQC_ERR_DEVICE;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      return PQC_ERR_DEVICE;
    d.ptr = static_cast<uint8_t*>(p);
    d.cus = cus;
    d.ready = true;
  }
  *out = d;
  return PQC_OK;
}

template <int K>
int noalloc_dec(const NoAllocDev& d, size_t n, uint8_t* ss, uint8_t* ct, const uint8_t* sk, uint32_t* status,
                hipStream_t s) {
  using namespace kyber::fused;
  // a workgroup per request up to 8192; a 64-request tile launch is as long for any batch:
  // us at 8192 / in tiles 276 / 502, 666 / 853, 846 / 1255 for K = 2, 3, 4
  if (n <= 8192) {
    return kyber_lowlat_dec(K, n, ss, ct, sk, status, s);
  } else {
    const int ntiles = (int)((n + Tile<K>::T - 1) / Tile<K>::T);
    const int grid = std::max(1, std::min(ntiles, d.cus * 4));  // the default fused_waves_per_cu
    const kyber::DenseSrc src{ss, ct, sk, nullptr, d.ptr + 256};
    hipLaunchKernelGGL((k_fused<K, true>), dim3(grid), dim3(64), 0, s, (int)n, ntiles, src, status);
  }
  return hip_err(hipGetLastError());
}
}  // namespace

int kyber_poly_transform(int op, size_t n, int16_t* polys, hipStream_t s) {
  if (op != 0 && op != 1) return PQC_ERR_INVALID_ARG;
  if (n == 0) return PQC_OK;
  const int grid = (int)(n < 4096 ? n : 4096);
  hipLaunchKernelGGL(kyber::fused::k_poly_transform, dim3(grid), dim3(64), 0, s, op, (int)n, polys);
  return hip_err(hipGetLastError());
}

int keccak_batch(int op, size_t n, uint8_t* out, size_t outlen, const uint8_t* in, size_t inlen, hipStream_t s) {
  if (op < 0 || op > 3 || (inlen % 8) != 0) return PQC_ERR_INVALID_ARG;
  if ((op == 0 && outlen != 32) || (op == 1 && outlen != 64) || outlen == 0) return PQC_ERR_INVALID_ARG;
  if (n == 0) return PQC_OK;
  const int grid = (int)((n + 255) / 256);
  hipLaunchKernelGGL(kyber::fused::k_keccak_batch, dim3(grid), dim3(256), 0, s, op, (int)n, out, outlen, in, inlen);
  return hip_err(hipGetLastError());
}

}  // namespace pqc

extern "C" int pqc_kyber_dec_batch_noalloc(int alg, size_t n, uint8_t* ss, const uint8_t* ct, const uint8_t* sk,
                                           uint32_t* status, void* stream) {
  if (alg != PQC_ALG_KYBER512 && alg != PQC_ALG_KYBER768 && alg != PQC_ALG_KYBER1024) return PQC_ERR_UNSUPPORTED;
  if (n > pqc::kNoAllocMax) return PQC_ERR_BATCH_TOO_LARGE;
  if (n == 0) return PQC_OK;
  if (!ss || !ct || !sk || (((uintptr_t)ss | (uintptr_t)ct | (uintptr_t)sk) & 7) || ((uintptr_t)status & 3))
    return PQC_ERR_INVALID_ARG;
  pqc::NoAllocDev d;
  const int rc = pqc::noalloc_device(&d);
  if (rc) return rc;
  uint32_t* st = status ? status : reinterpret_cast<uint32_t*>(d.ptr);
  uint8_t* ctm = const_cast<uint8_t*>(ct);  // read-only in the decapsulation kernels
  hipStream_t s = (hipStream_t)stream;
  switch (alg) {
    case PQC_ALG_KYBER512: return pqc::noalloc_dec<2>(d, n, ss, ctm, sk, st, s);
    case PQC_ALG_KYBER768: return pqc::noalloc_dec<3>(d, n, ss, ctm, sk, st, s);
    default: return pqc::noalloc_dec<4>(d, n, ss, ctm, sk, st, s);
  }
}
