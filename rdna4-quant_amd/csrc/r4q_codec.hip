// Weight dequantisation and FP8 KV codec kernels.
//
// dequant_int4 replaces the reference's dequant_int4_kernel (hip:3568-3603),
// fp16_to_fp8 its fp16_to_fp8_kernel (hip:3606-3618).  The dequantised value
// is fp16(float(q - zp) * float(scale)): the fp32 product is exact (at most
// 9 + 11 significant bits) so the single fp16 rounding makes the result
// bit-identical to the reference's torch path (int4_quant_v2.py:105-127).
#include <algorithm>

#include "r4q_device.hpp"
#include "r4q_host.hpp"

namespace r4q {
namespace {

// Eight consecutive elements (16 bytes of fp16) per thread and turn: loads and
// stores of a wave are contiguous.  kTurns turns of a workgroup apart, so that
// several loads are in flight.  Bound by HBM, three quarters of it writes at INT4
// (2 of 2.625 bytes per element): 17408 x 5120 INT4 61 -> 35 us (6.6 TB/s), INT8 67 ->
// 43; before, a 32-element block per thread wrote 16 bytes of every 64 per store
// instruction.
constexpr int kTurns = 4;
template <int WBITS>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ w,
                                                      const uint32_t* __restrict__ sz,
                                                      uint16_t* __restrict__ out, int64_t n8) {
  const int64_t p0 = (int64_t)blockIdx.x * (256 * kTurns) + threadIdx.x;
  uint32_t q[kTurns][2], s2[kTurns];
#pragma unroll
  for (int i = 0; i < kTurns; ++i) {
    const int64_t p = min(p0 + 256 * i, n8 - 1);
    if constexpr (WBITS == 4) {
      q[i][0] = reinterpret_cast<const uint32_t*>(w)[p];
    } else {
      const u2_t v = reinterpret_cast<const u2_t*>(w)[p];
      q[i][0] = v[0];
      q[i][1] = v[1];
    }
    s2[i] = sz[p >> 2];
  }
#pragma unroll
  for (int i = 0; i < kTurns; ++i) {
    const int64_t p = p0 + 256 * i;
    const float scale = h2f((uint16_t)(s2[i] & 0xFFFFu)), zp = h2f((uint16_t)(s2[i] >> 16));
    u4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t a, b;
      if constexpr (WBITS == 4) {
        a = (q[i][0] >> (8 * e)) & 0xFu;
        b = (q[i][0] >> (8 * e + 4)) & 0xFu;
      } else {
        a = (q[i][e >> 1] >> (16 * (e & 1))) & 0xFFu;
        b = (q[i][e >> 1] >> (16 * (e & 1) + 8)) & 0xFFu;
      }
      const float lo = ((float)a - zp) * scale, hi = ((float)b - zp) * scale;  // exact in fp32
      o[e] = (uint32_t)f2h(lo) | ((uint32_t)f2h(hi) << 16);
    }
    if (p < n8) reinterpret_cast<u4_t*>(out)[p] = o;
  }
}

// E4M3 codes of a pair of fp16 patterns (in the low byte of each half), the
// recipe of fp8_encode on the fp16 fields: t = the exponent and top 3 mantissa
// bits rounded up on bit 6; E4M3 has 8 binades less at the bottom, so the code
// is t - 64, zero below 8 (E <= 0) and 126 from 120 on (E >= 15, infinities
// included); a NaN gives +126.
__device__ __forceinline__ uint32_t fp8_encode_pair(uint32_t h) {
  typedef uint16_t us2_t __attribute__((ext_vector_type(2)));
  const us2_t mag = __builtin_bit_cast(us2_t, h & 0x7FFF7FFFu);
  const us2_t one = {1, 1};
  const us2_t t = (mag + (us2_t){0x40, 0x40}) >> 7;
  us2_t c = __builtin_elementwise_sub_sat(
      __builtin_elementwise_min(t, (us2_t){184, 184}), (us2_t){64, 64});     // 0 .. 120
  c += __builtin_elementwise_sub_sat(c, (us2_t){119, 119}) * (uint16_t)6;    // 120 -> 126
  c *= __builtin_elementwise_min(__builtin_elementwise_sub_sat(c, (us2_t){7, 7}), one);
  const us2_t nan =
      __builtin_elementwise_min(__builtin_elementwise_sub_sat(mag, (us2_t){0x7C00, 0x7C00}), one);
  const us2_t sign = __builtin_elementwise_sub_sat(
      __builtin_bit_cast(us2_t, (h >> 8) & 0x00800080u), nan * (uint16_t)0x80);
  return __builtin_bit_cast(uint32_t, c) | __builtin_bit_cast(uint32_t, sign);
}

// Turns of the FP8 codecs.  Up to kOneTurn elements one turn each: that many
// workgroups fit the chip at once, and the time is that of a thread's own work
// (encode, one turn / four: 64 K values 2.3 / 2.9 us, 1 M 2.5 / 3.0, 8.4 M 5.8 / 6.1, 33.5 M
// 20.0 / 18.9; decode on 8 codes 2.2 / 2.7, 2.5 / 2.9, 5.1 / 5.5, 16.2 / 15.7).
constexpr int64_t kOneTurn = (int64_t)1 << 23;

// Four elements per thread and turn.  The scalar recipe's ~22 instructions per
// element were as long as the stream: 33.5 M values 27 -> 19.5 us (5.2 TB/s).
// Eight elements (16-byte loads where src is so aligned) measured the same.
template <int TURNS>
__global__ __launch_bounds__(256) void fp16_to_fp8_kernel(const uint16_t* __restrict__ src,
                                                          uint8_t* __restrict__ dst, int64_t n) {
  const int64_t p0 = (int64_t)blockIdx.x * (256 * TURNS) + threadIdx.x, np = n / 4;
  u2_t v[TURNS];
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const int64_t p = p0 + 256 * i;
    if (p < np) v[i] = reinterpret_cast<const u2_t*>(src)[p];
  }
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const int64_t p = p0 + 256 * i;
    if (p < np)  // bytes 0 and 2 of the two pairs
      reinterpret_cast<uint32_t*>(dst)[p] = __builtin_amdgcn_perm(
          fp8_encode_pair(v[i][1]), fp8_encode_pair(v[i][0]), 0x06040200u);
  }
  if (blockIdx.x == 0 && threadIdx.x < n % 4)  // the last n % 4 elements
    dst[np * 4 + threadIdx.x] = (uint8_t)fp8_encode_pair(src[np * 4 + threadIdx.x]);
}

// VEC = 8 codes per thread and turn where src is 8-byte and dst 16-byte
// aligned, else 1 (four turns at every size: one was as fast up to 512 K codes and
// slower from 1 M on).  33.5 M codes: 16 us (6.3 TB/s) with 8, 25 with 1; 40 with 1
// code per thread in all.
template <int VEC, int TURNS>
__global__ __launch_bounds__(256) void fp8_to_fp16_kernel(const uint8_t* __restrict__ src,
                                                          uint16_t* __restrict__ dst, int64_t n) {
  const h2_t k256 = as_h2(0x5C005C00u);  // (256, 256): exact, subnormals included
  const int64_t p0 = (int64_t)blockIdx.x * (256 * TURNS) + threadIdx.x, np = n / VEC;
  u2_t c[TURNS];
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const int64_t p = p0 + 256 * i;
    if (p >= np) continue;
    if constexpr (VEC == 8) c[i] = reinterpret_cast<const u2_t*>(src)[p];
    else c[i][0] = src[p];
  }
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const int64_t p = p0 + 256 * i;
    if (p >= np) continue;
    u4_t o;
#pragma unroll
    for (int e = 0; e < VEC / 2; ++e)
      o[e] = as_u32(as_h2(fp8x2_to_h2_div256(c[i][e >> 1] >> (16 * (e & 1)))) * k256);
    if constexpr (VEC == 8)
      reinterpret_cast<u4_t*>(dst)[p] = o;
    else
      dst[p] = (uint16_t)(as_u32(as_h2(fp8x2_to_h2_div256(c[i][0])) * k256) & 0xFFFFu);
  }
  if (blockIdx.x == 0 && threadIdx.x < n % VEC) {
    const int64_t j = np * VEC + threadIdx.x;
    dst[j] = (uint16_t)(as_u32(as_h2(fp8x2_to_h2_div256(src[j])) * k256) & 0xFFFFu);
  }
}

// workgroups for n pieces of work; at least one (it also does the remainder)
unsigned turn_grid(int64_t n, int turns = kTurns) {
  return (unsigned)std::max<int64_t>(1, (n + 256 * turns - 1) / (256 * turns));
}

bool aligned(const void* p, int a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

template <int WBITS>
int dequant(const void* w, const void* sz, void* out, int64_t N, int64_t K, void* stream) {
  R4Q_REQUIRE(w && sz && out, "dequant_int%d: null pointer", WBITS);
  R4Q_REQUIRE(N > 0 && K > 0 && K % 32 == 0,
              "dequant_int%d: need N > 0 and K %% 32 == 0 (N=%lld K=%lld)", WBITS,
              (long long)N, (long long)K);
  R4Q_REQUIRE(aligned(w, 16) && aligned(sz, 4) && aligned(out, 16),
              "dequant_int%d: misaligned pointer", WBITS);
  const int64_t n8 = N * (K / 8);
  hipLaunchKernelGGL((dequant_kernel<WBITS>), dim3(turn_grid(n8)), dim3(256), 0, as_stream(stream),
                     static_cast<const uint8_t*>(w), static_cast<const uint32_t*>(sz),
                     static_cast<uint16_t*>(out), n8);
  return launch_status(WBITS == 4 ? "dequant_int4" : "dequant_int8");
}

}  // namespace
}  // namespace r4q

extern "C" int r4q_dequant_int4(const void* packed, const void* sz, void* out, int64_t N,
                                int64_t K, void* stream) {
  return r4q::dequant<4>(packed, sz, out, N, K, stream);
}

extern "C" int r4q_dequant_int8(const void* q, const void* sz, void* out, int64_t N,
                                int64_t K, void* stream) {
  return r4q::dequant<8>(q, sz, out, N, K, stream);
}

extern "C" int r4q_fp16_to_fp8(const void* src, void* dst, int64_t n, void* stream) {
  R4Q_REQUIRE(n >= 0, "fp16_to_fp8: negative size");
  if (n == 0) return R4Q_OK;
  R4Q_REQUIRE(src && dst, "fp16_to_fp8: null pointer");
  R4Q_REQUIRE(r4q::aligned(src, 8) && r4q::aligned(dst, 4), "fp16_to_fp8: misaligned pointer");
  const auto* sp = static_cast<const uint16_t*>(src);
  auto* dp = static_cast<uint8_t*>(dst);
  const hipStream_t st = r4q::as_stream(stream);
  if (n <= r4q::kOneTurn)
    hipLaunchKernelGGL(r4q::fp16_to_fp8_kernel<1>, dim3(r4q::turn_grid(n / 4, 1)), dim3(256), 0, st,
                       sp, dp, n);
  else
    hipLaunchKernelGGL(r4q::fp16_to_fp8_kernel<r4q::kTurns>, dim3(r4q::turn_grid(n / 4)), dim3(256),
                       0, st, sp, dp, n);
  return r4q::launch_status("fp16_to_fp8");
}

extern "C" int r4q_fp8_to_fp16(const void* src, void* dst, int64_t n, void* stream) {
  R4Q_REQUIRE(n >= 0, "fp8_to_fp16: negative size");
  if (n == 0) return R4Q_OK;
  R4Q_REQUIRE(src && dst, "fp8_to_fp16: null pointer");
  const auto* sp = static_cast<const uint8_t*>(src);
  auto* dp = static_cast<uint16_t*>(dst);
  const hipStream_t st = r4q::as_stream(stream);
  if (!r4q::aligned(src, 8) || !r4q::aligned(dst, 16))
    hipLaunchKernelGGL((r4q::fp8_to_fp16_kernel<1, r4q::kTurns>), dim3(r4q::turn_grid(n)), dim3(256),
                       0, st, sp, dp, n);
  else if (n <= r4q::kOneTurn)
    hipLaunchKernelGGL((r4q::fp8_to_fp16_kernel<8, 1>), dim3(r4q::turn_grid(n / 8, 1)), dim3(256), 0,
                       st, sp, dp, n);
  else
    hipLaunchKernelGGL((r4q::fp8_to_fp16_kernel<8, r4q::kTurns>), dim3(r4q::turn_grid(n / 8)),
                       dim3(256), 0, st, sp, dp, n);
  return r4q::launch_status("fp8_to_fp16");
}
