// Where the requests of a Kyber batch live.  DenseSrc: element-contiguous arrays
// of one parameter set (element r at r * size).  MixedSrc: requests of mixed
// parameter sets named by descriptors (pqc_kem_req: alg + byte offsets into four
// arenas), bucketed by K into `order` by k_mixed_classify; index r of the K
// bucket is request order[(K - 2) * cap + r].
#pragma once
#include "internal.h"
#include "kyber_arith.cuh"

namespace pqc {
namespace kyber {

struct ReqP {
  uint8_t* ss;
  uint8_t* ct;
  const uint8_t* key;
  const uint8_t* coins;
  uint8_t* prf;
};

struct DenseSrc {
  uint8_t* ss;
  uint8_t* ct;
  const uint8_t* key;
  const uint8_t* coins;
  uint8_t* prf;
  template <int K, bool DEC>
  __device__ __forceinline__ ReqP req(int r) const {
    using P = Params<K>;
    return ReqP{ss + (size_t)r * 32, ct + (size_t)r * P::ct_bytes,
                key + (size_t)r * (DEC ? P::sk_bytes : P::pk_bytes), coins ? coins + (size_t)r * 32 : nullptr,
                prf + (size_t)r * ((2 * K + 1) * 128)};
  }
};

struct MixedSrc {
  const pqc_kem_req* reqs;
  const uint32_t* order;
  int cap;
  uint8_t* ss;
  uint8_t* ct;
  const uint8_t* key;
  const uint8_t* coins;
  uint8_t* prf;       // prf_stride bytes per request index
  size_t prf_stride;  // >= (2K+1) * 128 of every K the context holds
  template <int K, bool DEC>
  __device__ __forceinline__ ReqP req(int r) const {
    const uint32_t idx = order[(size_t)(K - 2) * cap + r];
    const pqc_kem_req d = reqs[idx];
    return ReqP{ss + d.ss_off, ct + d.ct_off, key + d.key_off, coins ? coins + d.coins_off : nullptr,
                prf + (size_t)idx * prf_stride};
  }
};

}  // namespace kyber

// a classified mixed batch in stages (kyber_staged.hip); n <= ctx->kstage_max
int kyber_staged_mixed(pqc_ctx* c, int dec, size_t n, const kyber::MixedSrc& src, hipStream_t s);

}  // namespace pqc
