// One Kyber request by one wave: indcpa_dec, the (re-)encryption and the packings, 4
// coefficients of a polynomial per lane on the exact FP32 arithmetic (kyber_wavef.cuh).
// Used by the 64-request tiles (kyber_fused.hip) and the per-request workgroups
// (kyber_lowlat.hip).
#pragma once
#include "kyber_wave.cuh"
#include "kyber_wavef.cuh"

namespace pqc {
namespace kyber {

// indcpa_dec inputs of one request, as this lane's words: the ciphertext's u and v
// groups and the secret key's 12-bit groups.
template <int K>
struct DecIn {
  uint32_t u[K][3], s[K][2], v[3];
};

template <int K>
__device__ __forceinline__ void dec_load(DecIn<K>& in, const uint8_t* ct, const uint8_t* sk) {
  using P = Params<K>;
  const int l = lane_id();
#pragma unroll
  for (int i = 0; i < K; ++i) {
    load_group<P::du>(in.u[i], ct + 32 * P::du * i, nat_group(l));
    load_h12(in.s[i], sk + 384 * i, ntt_group(l));
  }
  load_group<P::dv>(in.v, ct + P::polyvec_cbytes, nat_group(l));
}

// Pack the lane's 4 D-bit values with its odd neighbour's: even lanes write D bytes.
template <int D>
__device__ __forceinline__ void pack_pair(uint8_t* dst, const uint32_t (&t)[4]) {
  const int l = lane_id();
  uint64_t mine = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) mine |= (uint64_t)t[r] << (D * r);
  const uint64_t nb = (uint64_t)__shfl_xor((long long)mine, 1);
  if ((l & 1) == 0) {
    // 8 values, 8*D bits: low 4*D bits mine, next 4*D bits the neighbour's
    const uint64_t lo = mine | (nb << (4 * D));
    const uint64_t hi = (4 * D + 4 * D > 64) ? (nb >> (64 - 4 * D)) : 0;
    uint8_t* o = dst + D * (l >> 1);
#pragma unroll
    for (int b = 0; b < D; ++b) o[b] = (uint8_t)(b < 8 ? (lo >> (8 * b)) : (hi >> (8 * (b - 8))));
  }
}

// Re-encryption inputs of one request, as this lane's words: its 16-bit PRF
// groups (2K+1 noise polynomials), the public key's 12-bit groups and, for
// decapsulation, the ciphertext's u and v groups to compare with.
template <int K, bool DEC>
struct EncIn {
  uint32_t prf[2 * K + 1];
  uint32_t t[K][2];
  uint32_t cu[DEC ? K : 1][3], cv[3];
};

// PRF_LDS: the PRF rows are in LDS (the per-request kernels); otherwise in the
// global scratch, read through a global-address-space pointer.
template <int K, bool DEC, bool PRF_LDS = false>
__device__ __forceinline__ void enc_load(EncIn<K, DEC>& in, const uint8_t* prf, const uint8_t* pk, const uint8_t* ct) {
  using P = Params<K>;
  const int l = lane_id();
  if constexpr (PRF_LDS) {
    const uint16_t* prf16 = reinterpret_cast<const uint16_t*>(prf);
#pragma unroll
    for (int j = 0; j < 2 * K + 1; ++j) in.prf[j] = prf16[64 * j + l];
  } else {
    const global_t<uint16_t>* prf16 = gptr(reinterpret_cast<const uint16_t*>(prf));
#pragma unroll
    for (int j = 0; j < 2 * K + 1; ++j) in.prf[j] = prf16[64 * j + l];
  }
#pragma unroll
  for (int j = 0; j < K; ++j) load_h12(in.t[j], pk + 384 * j, ntt_group(l));
  if constexpr (DEC) {
#pragma unroll
    for (int i = 0; i < K; ++i) load_group<P::du>(in.cu[i], ct + 32 * P::du * i, nat_group(l));
    load_group<P::dv>(in.cv, ct + P::polyvec_cbytes, nat_group(l));
  }
}

// ---- indcpa_dec and the re-encryption on exact FP32 values (kyber_wavef.cuh) -----
// Every polynomial value equals the reference's int16 value mod q (the
// reference's arithmetic never leaves the int16 range, so its values are exact
// residues too), and the outputs leave through compress_f, which reads only the
// residue: the message bits, the ciphertext and the mismatch bits are the
// reference's.

// indcpa_dec (indcpa.cu:691-733, poly_tomsg) for one request; the message is written to
// msg (LDS, 32 bytes).
template <int K>
__device__ __forceinline__ void coop_indcpa_dec_f(const DecIn<K>& in, const LaneZF& z, uint8_t* msg) {
  using P = Params<K>;
  const int l = lane_id();
  F4 u[K];
  Bz uz[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    uint32_t t[4];
    unpack_loaded<P::du>(t, in.u[i], nat_group(l));
#pragma unroll
    for (int r = 0; r < 4; ++r) u[i].v[r] = (float)decompress_d<P::du>(t[r]);  // [0, q)
    ntt_f<Q>(u[i], z);
    reduce_f4(u[i]);
    uz[i] = basemul_twist(u[i], z);
  }
  F4 mp = basemul_sum_f<K>(
      [&](int i) {
        P4 s;
        poly12_loaded(s, in.s[i], ntt_group(l));  // 12-bit, unreduced
        F4 sf = to_f4(s);
        reduce_f4(sf);
        return sf;
      },
      u, uz);
  invntt_f(mp, z);
  uint32_t tv[4];
  unpack_loaded<P::dv>(tv, in.v, nat_group(l));
  uint32_t nib = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) nib |= f32::compress_f<1>((float)decompress_d<P::dv>(tv[r]) - mp.v[r]) << r;
  const uint32_t other = (uint32_t)__shfl_xor((int)nib, 1);
  if ((l & 1) == 0) msg[l >> 1] = (uint8_t)(nib | (other << 4));
}

// r^ of one request: the K noise polynomials transformed, with their base-multiplication
// twists (the first K PRF words of the lane)
template <int K>
struct NoiseHat {
  F4 v[K];
  Bz z[K];
  __device__ __forceinline__ void make(const uint32_t* prf, const LaneZF& z_) {
#pragma unroll
    for (int j = 0; j < K; ++j) {
      P4 c;
      cbd_group(c, prf[j]);  // [-2, 2]
      v[j] = to_f4(c);
      ntt_f<2>(v[j], z_);
      reduce_f4(v[j]);
      z[j] = basemul_twist(v[j], z_);
    }
  }
};

// u_i of the re-encryption: A^T's row i, noise word e.  DEC: compare with the ciphertext
// words cu and return the lane's mismatch bits.  ENC: write the packed polynomial.
template <int K, bool DEC, class AT>
__device__ __forceinline__ uint32_t coop_row_u(const AT& at, int i, const NoiseHat<K>& sp, uint32_t e16,
                                               const uint32_t (&cu)[3], uint8_t* ct, const LaneZF& z) {
  using P = Params<K>;
  F4 acc = basemul_sum_f<K>(
      [&](int j) {
        uint32_t w0, w1;
        at.get(i, j, w0, w1);  // accepted candidates, [0, 19q)
        F4 a = {{(float)(w0 & 0xFFFF), (float)(w0 >> 16), (float)(w1 & 0xFFFF), (float)(w1 >> 16)}};
        reduce_f4(a);
        return a;
      },
      sp.v, sp.z);
  invntt_f(acc, z);
  P4 e;
  cbd_group(e, e16);
  uint32_t c[4], mismatch = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) c[r] = f32::compress_f<P::du>(acc.v[r] + (float)e.v[r]);
  if constexpr (DEC) {
    uint32_t t[4];
    unpack_loaded<P::du>(t, cu, nat_group(lane_id()));
#pragma unroll
    for (int r = 0; r < 4; ++r) mismatch |= c[r] ^ t[r];
  } else {
    pack_pair<P::du>(ct + 32 * P::du * i, c);
  }
  return mismatch;
}

// v of the re-encryption: the public key's words t, noise word e, the message
template <int K, bool DEC>
__device__ __forceinline__ uint32_t coop_row_v(const uint32_t (&tw)[K][2], const NoiseHat<K>& sp, uint32_t e16,
                                               const uint8_t* msg, const uint32_t (&cv)[3], uint8_t* ct,
                                               const LaneZF& z) {
  using P = Params<K>;
  const int l = lane_id(), gn = ntt_group(l);
  F4 acc = basemul_sum_f<K>(
      [&](int j) {
        P4 t;
        poly12_loaded(t, tw[j], gn);
        F4 tf = to_f4(t);
        reduce_f4(tf);
        return tf;
      },
      sp.v, sp.z);
  invntt_f(acc, z);
  P4 e;
  cbd_group(e, e16);
  const uint32_t nib = (msg[l >> 1] >> (4 * (l & 1))) & 0xF;
  uint32_t c[4], mismatch = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float kq = ((nib >> r) & 1) ? (float)((Q + 1) / 2) : 0.f;
    c[r] = f32::compress_f<P::dv>(acc.v[r] + (float)e.v[r] + kq);
  }
  if constexpr (DEC) {
    uint32_t t[4];
    unpack_loaded<P::dv>(t, cv, nat_group(l));
#pragma unroll
    for (int r = 0; r < 4; ++r) mismatch |= c[r] ^ t[r];
  } else {
    pack_pair<P::dv>(ct + P::polyvec_cbytes, c);
  }
  return mismatch;
}

// Re-encryption of one request (indcpa_enc from sp-sampling on) by one wave.  DEC: compare
// with ct and return the lane's mismatch bits.  ENC: write ct.
template <int K, bool DEC, class AT>
__device__ __forceinline__ uint32_t coop_reencrypt_f(const AT& at, const EncIn<K, DEC>& in, const uint8_t* msg,
                                                     uint8_t* ct, const LaneZF& z) {
  NoiseHat<K> sp;
  sp.make(in.prf, z);
  uint32_t mismatch = 0;
#pragma unroll
  for (int i = 0; i < K; ++i) mismatch |= coop_row_u<K, DEC>(at, i, sp, in.prf[K + i], in.cu[DEC ? i : 0], ct, z);
  return mismatch | coop_row_v<K, DEC>(in.t, sp, in.prf[2 * K], msg, in.cv, ct, z);
}

// 12-bit pack of a group in its NTT-order slot (the inverse of load_poly12)
__device__ __forceinline__ void store_poly12(uint8_t* base, int g, const P4& p) {
  uint16_t* h = reinterpret_cast<uint16_t*>(base + 6 * g);
  const uint32_t c0 = (uint32_t)p.v[0], c1 = (uint32_t)p.v[1], c2 = (uint32_t)p.v[2], c3 = (uint32_t)p.v[3];
  h[0] = (uint16_t)(c0 | (c1 << 12));
  h[1] = (uint16_t)((c1 >> 4) | (c2 << 8));
  h[2] = (uint16_t)((c2 >> 8) | (c3 << 4));
}

}  // namespace kyber
}  // namespace pqc
