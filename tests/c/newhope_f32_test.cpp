// CPU check of NewHope's exact FP32 arithmetic mod q (pqc_amd/csrc/newhope_f32.h): fma,
// multiply and add in round-to-nearest-even give the same bits on the host as on the GPU.
//   - mul: every twiddle by every |x| <= 20000, by a stride over the transforms' whole range
//     and by its ends; every packed value by every packed value; gen_a candidates by centred
//     values; and the ends of |x z| <= kMulMax q;
//   - reduce and canon: every value of their ranges;
//   - the transforms' layers by simulation on extreme and random inputs, against exact
//     modular arithmetic, every intermediate against its bound.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../pqc_amd/csrc/newhope_f32.h"

using namespace pqc::newhope::fp;

constexpr int Q = 12289;
static int fails = 0;
#define CHECK(c, ...)                          \
  do {                                         \
    if (!(c) && fails++ < 20) {                \
      std::fprintf(stderr, "line %d: ", __LINE__); \
      std::fprintf(stderr, __VA_ARGS__);       \
      std::fprintf(stderr, "\n");              \
    }                                          \
  } while (0)

static int64_t modq(int64_t a) { return ((a % Q) + Q) % Q; }

static inline bool mul_good(int x, int z, float zq) {
  const float r = mul((float)x, (float)z, zq);
  const int64_t ri = (int64_t)r;
  return (float)ri == r && ri <= kOut && ri >= -kOut && (ri - (int64_t)x * z) % Q == 0;
}

static void check_mul() {
  const int top = inv_bound(1024) > fwd_bound(1024) ? inv_bound(1024) : fwd_bound(1024);
  for (int z = -kTwiddle; z <= kTwiddle; ++z) {
    const float zq = (float)z * kQinv;
    for (int x = -20000; x <= 20000; x += 3) CHECK(mul_good(x, z, zq), "mul(%d, %d)", x, z);
    for (int x = -top; x <= top; x += 997) CHECK(mul_good(x, z, zq), "mul(%d, %d)", x, z);
    CHECK(mul_good(top, z, zq) && mul_good(-top, z, zq), "mul(+-%d, %d)", top, z);
    if (z != 0) {
      const int64_t lim = (int64_t)kMulMax * Q / std::abs(z);
      const int x = (int)(lim < (1 << 24) ? lim : (1 << 24));
      CHECK(mul_good(x, z, zq) && mul_good(-x, z, zq), "mul(+-%d, %d)", x, z);
    }
  }
  for (int z = 0; z < kIn; ++z)
    for (int x = 0; x < kIn; x += 5) CHECK(mul_good(x, z, (float)z * kQinv), "mul(%d, %d)", x, z);
  for (int z = -kCentred; z <= kCentred; z += 7)
    for (int x = 0; x < 5 * Q; ++x) CHECK(mul_good(x, z, (float)z * kQinv), "mul(%d, %d)", x, z);
}

static void check_reduce() {
  for (int x = -kReduceMax; x <= kReduceMax; ++x) {
    const float r = reduce((float)x);
    const int ri = (int)r;
    CHECK((float)ri == r && std::abs(ri) <= kCentred && (ri - x) % Q == 0, "reduce(%d) = %f", x, r);
  }
  for (int x = -kCanonMax; x <= kCanonMax; ++x)
    CHECK(canon((float)x) == (uint32_t)modq(x), "canon(%d) = %u", x, canon((float)x));
}

static int64_t pw(int64_t b, int64_t e) {
  int64_t r = 1;
  for (b = modq(b); e; e >>= 1, b = b * b % Q)
    if (e & 1) r = r * b % Q;
  return r;
}

// bit-reversed input, natural output: layer L combines sub-transforms of 2^L points
static void simulate(int n, bool inv, const std::vector<int>& in) {
  const int64_t g = n == 1024 ? 7 : 10968;
  const int lg = log2n(n), bound = inv ? inv_bound(n) : fwd_bound(n);
  std::vector<float> f(in.begin(), in.end());
  std::vector<int64_t> e(in.begin(), in.end());
  for (int L = 0; L < lg; ++L)
    for (int j = 0; j < (1 << L); ++j) {
      const int64_t ex = (int64_t)(n >> (L + 1)) * (inv ? 2 * n - 2 * j : 2 * j + 1);
      const int64_t w = pw(g, ex % (2 * n));
      const int z = (int)(w > Q / 2 ? w - Q : w);
      for (int a = j; a < n; a += 2 << L) {
        const int b = a + (1 << L);
        const bool plain = L < lg - 6 && z == 1;  // the first register group multiplies by literals
        const float t = plain ? f[b] : mul(f[b], (float)z, (float)z * kQinv);
        f[b] = f[a] - t;
        f[a] += t;
        const int64_t te = modq(e[b] * z);
        e[b] = modq(e[a] - te);
        e[a] = modq(e[a] + te);
        CHECK(std::fabs(f[a]) <= bound && std::fabs(f[b]) <= bound, "N %d inv %d layer %d: %f, %f over %d", n, inv, L,
              f[a], f[b], bound);
      }
    }
  for (int i = 0; i < n; ++i) CHECK(modq((int64_t)f[i]) == e[i], "N %d inv %d output %d", n, inv, i);
}

int main() {
  check_mul();
  check_reduce();
  std::mt19937 rng(5);
  for (int n : {512, 1024})
    for (bool inv : {false, true}) {
      const int lo = inv ? -kIn : 0;  // the inverse takes products of either sign
      for (int v : {lo, 0, kIn}) simulate(n, inv, std::vector<int>(n, v));
      for (int rep = 0; rep < 200; ++rep) {
        std::vector<int> in(n);
        for (int& x : in) x = rep & 1 ? (rng() & 1 ? kIn : lo) : lo + (int)(rng() % (unsigned)(kIn - lo + 1));
        simulate(n, inv, in);
      }
    }
  if (fails) {
    std::fprintf(stderr, "%d checks failed\n", fails);
    return 1;
  }
  std::printf("NewHope f32 arithmetic mod q: all checks hold\n");
  return 0;
}
