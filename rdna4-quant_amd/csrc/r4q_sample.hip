// Temperature + top-p (nucleus) sampling of the next token on the device.
//
// Semantics of the reference's Python sampler (int4_engine_v5.py:387-399):
//   z = float(logits) / temperature;
//   if top_p < 1: sort z descending, drop every token whose cumulative
//                 softmax probability *before* it is >= top_p;
//   draw one token from softmax over the kept tokens.
// temperature <= 0 is the greedy argmax (int4_engine_v5.py:352-353), served
// by the argmax kernels of the decode step.
//
// gfx950 design.  fp16 logits take at most 65,536 distinct values, and the
// order-preserving 16-bit key of a value ranks it exactly, so
//  * sample_hist_kernel builds an integer histogram of the keys, one
//    65,536-bin table per row: 4 workgroups per row, each counting a quarter
//    of the keys in LDS over the whole row and writing its bins (integer
//    counts are order-independent, so every result below is deterministic);
//  * sample_select_kernel (one 1024-thread workgroup per row) scans the bins
//    from the largest key down: per-bin mass = count * exp(z_b - z_max), the
//    top-p cutoff per bin (tokens tied in a bin are ranked by index, like a
//    stable descending sort), the kept mass, and the draw: u * kept mass
//    lands in one bin at one tie rank;
//  * sample_pick_kernel finds the token with that key and tie rank (lowest
//    index first), writes its id and, for the decode loop, gathers its
//    embedding row into the next step's hidden state.
// u is a counter-based uniform draw: x = splitmix64(seed ^ counter), then
// splitmix64(x ^ row), u = top 24 bits / 2^24 -- reproducible from (seed,
// position, row) without any RNG state.
#include <math.h>

#include "r4q_ctx.hpp"
#include "r4q_device.hpp"
#include "r4q_host.hpp"
#include "r4q_kernels.hpp"

namespace r4q {
namespace {

constexpr int kBins = 65536;
constexpr int kSelThreads = 1024;
constexpr int kBinsPerThread = kBins / kSelThreads;  // 64
constexpr int kHistParts = 4;                       // workgroups per row
constexpr int kPartBins = kBins / kHistParts;       // 16,384
constexpr int kPartChunks = kPartBins / kBinsPerThread;
// Workspace layout, independent of B: the selection words of up to kMaxRows
// rows first, then one table per row.
constexpr int kMaxRows = 1024;
constexpr size_t kSelBytes = (size_t)kMaxRows * 8;

// Descending rank of an fp16 bit pattern among all of them: r = 65535 - key with
// key the order-preserving 16-bit key (larger value, larger key).  A pair of
// patterns in one word: positive h -> 0x7FFF - h, negative h -> h.  Here -0
// (rank 0x8000) still follows +0 (0x7FFF); the two share a key, which the
// histogram and the pick see to (NaN is not a valid logit).
__device__ __forceinline__ uint32_t rank_pair(uint32_t h) {
  const uint32_t neg = (h >> 15) & 0x00010001u;
  return h ^ (0x7FFF7FFFu - neg * 0x7FFFu);  // 0 where negative
}
__device__ __forceinline__ uint32_t unkey16(uint32_t k) {
  return (k & 0x8000u) ? (k & 0x7FFFu) : (~k & 0xFFFFu);
}

// splitmix64 finalizer (S. Vigna, public domain).
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// Rows are walked in 16-byte groups of 8 logits from the aligned address at or
// before their start.  f(i0, v, valid) for the groups at i0, i0 + step, ...
// below end: v the logits i0 .. i0 + 7, the bits of `valid` those inside [0, V).
// kBatch loads are in flight where a batch lies inside the row.
constexpr int kBatch = 5;
__device__ __forceinline__ int64_t group_start(const uint16_t* row) {
  return -(int64_t)((reinterpret_cast<uintptr_t>(row) & 15) / 2);
}
__device__ __forceinline__ uint32_t load_group(const uint16_t* __restrict__ row, int64_t V,
                                               int64_t i0, u4_t& v) {
  if (i0 >= 0 && i0 + 8 <= V) {
    v = *reinterpret_cast<const u4_t*>(row + i0);
    return 0xFFu;
  }
  uint32_t valid = 0;
  v = u4_t{0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (i0 + e >= 0 && i0 + e < V) {
      v[e >> 1] |= (uint32_t)row[i0 + e] << (16 * (e & 1));
      valid |= 1u << e;
    }
  return valid;
}
template <class F>
__device__ __forceinline__ void for_groups(const uint16_t* __restrict__ row, int64_t V, int64_t i0,
                                           int64_t end, int step, F f) {
  while (i0 < end) {
    u4_t v[kBatch];
    if (i0 >= 0 && i0 + (kBatch - 1) * step < end && i0 + (kBatch - 1) * step + 8 <= V) {
#pragma unroll
      for (int b = 0; b < kBatch; ++b) v[b] = *reinterpret_cast<const u4_t*>(row + i0 + b * step);
#pragma unroll
      for (int b = 0; b < kBatch; ++b) f(i0 + b * step, v[b], 0xFFu);
      i0 += kBatch * step;
    } else {
      const uint32_t valid = load_group(row, V, i0, v[0]);
      f(i0, v[0], valid);
      i0 += step;
    }
  }
}

// Table of a row: the count of the bin at descending rank r = 64 t + j is word
// j % 4 of the 16-byte piece (j / 4) * 1024 + t, so that the select kernel's
// thread t reads its 64 bins with coalesced loads.  Part p of a row holds the
// ranks r with (r + 0x2000) / 0x4000 = p (mod 4): +0 and -0 in one part, whose
// counts are added.  LDS chunks of 64 bins are padded to 68 words
// (conflict-free 16-byte reads).  The counts are LDS atomics: global ones ran
// at ~24 G/s (8 rows of 151,936: 50 us).  Bound by the vector instructions per
// logit of a part's one CU (13.5 us for 8 rows of 151,936).
__device__ __forceinline__ int bin_word(uint32_t i) { return (int)(i + (i >> 6) * 4); }
__global__ __launch_bounds__(1024) void sample_hist_kernel(const uint16_t* __restrict__ logits,
                                                           int64_t V, int64_t stride,
                                                           uint32_t* __restrict__ hist) {
  constexpr uint32_t kShift = kPartBins / 2;
  __shared__ __align__(16) uint32_t cnt[kPartChunks * 68];
  const uint32_t part = blockIdx.x, t = threadIdx.x;
  const uint16_t* row = logits + blockIdx.y * stride;
  for (int i = t; i < kPartChunks * 68; i += 1024) cnt[i] = 0u;
  __syncthreads();
  for_groups(row, V, group_start(row) + 8 * t, V, 8 * 1024, [&](int64_t, u4_t v, uint32_t valid) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t r = rank_pair(v[e >> 1]) >> (16 * (e & 1));
      const uint32_t i = ((r + kShift) & 0xFFFFu) - part * kPartBins;
      if (i < kPartBins && (valid >> e & 1u)) atomicAdd(&cnt[bin_word(i)], 1u);
    }
  });
  __syncthreads();
  if (t == 0 && part == (0x8000u + kShift) / kPartBins) {
    const uint32_t i = 0x8000u + kShift - part * kPartBins;  // -0 counts as +0
    cnt[bin_word(i - 1)] += cnt[bin_word(i)];
    cnt[bin_word(i)] = 0u;
  }
  __syncthreads();
  u4_t* out = reinterpret_cast<u4_t*>(hist + (int64_t)blockIdx.y * kBins);
  for (int i = t; i < kPartBins / 4; i += 1024) {
    const int c = i % kPartChunks, q = i / kPartChunks;
    const int chunk = (part * kPartChunks + c + kSelThreads - kPartChunks / 2) % kSelThreads;
    out[q * kSelThreads + chunk] = *reinterpret_cast<const u4_t*>(cnt + c * 68 + 4 * q);
  }
}

// Exclusive scan of one float per thread in a fixed order (thread order),
// returning the prefix and setting *total (buf: two rows of kSelThreads, read
// and written in turn: one barrier a step).
__device__ float block_exclusive_scan(float v, float (*buf)[kSelThreads], float* total) {
  const int t = threadIdx.x;
  float x = v;
  int cur = 0;
  buf[0][t] = x;
  __syncthreads();
  // Hillis-Steele over 1024 entries; each step's adds happen in a fixed order
  for (int off = 1; off < kSelThreads; off <<= 1) {
    x += t >= off ? buf[cur][t - off] : 0.f;
    cur ^= 1;
    buf[cur][t] = x;
    __syncthreads();
  }
  *total = buf[cur][kSelThreads - 1];
  __syncthreads();
  return x - v;
}

// Per row: cutoff, kept mass, the draw.  sel[b] = {key, tie rank}.  Thread
// t owns bins r = 64t .. 64t+63 in descending key order (key = 65535 - r),
// four counts per coalesced load, the next load in flight.  The sums run over a
// thread's bins in order; four bins at a time are computed without branches
// (their weights are independent), groups empty across the wave are skipped.
// Bound by the serial work of one workgroup per row and the scans' barriers
// (28 us, hardly depending on the vocabulary; counts held in registers over
// unrolled passes measured the same); 139 us when every pass read its counts one
// uncoalesced word at a time.
__global__ __launch_bounds__(kSelThreads) void sample_select_kernel(
    const uint32_t* __restrict__ hist, float temperature, float top_p, uint64_t seed,
    const int* __restrict__ counter_dev, int64_t counter_host, int* __restrict__ sel) {
  const int b = blockIdx.x, t = threadIdx.x;
  __shared__ float buf[2][kSelThreads];
  __shared__ float own_before, own_kbefore;
  __shared__ int kmax_s, owner;
  const int r0 = kBinsPerThread * t;
  const u4_t* h4 = reinterpret_cast<const u4_t*>(hist + (int64_t)b * kBins);
  // f(bins' counts, first of the four descending ranks) over this thread's bins
  auto for_bins = [&](auto f) {
    u4_t next = h4[t];
#pragma unroll 1
    for (int q = 0; q < kBinsPerThread / 4; ++q) {
      const u4_t c = next;
      next = h4[min(q + 1, kBinsPerThread / 4 - 1) * kSelThreads + t];
      if (__any((c[0] | c[1] | c[2] | c[3]) != 0u)) f(c, r0 + 4 * q);
    }
  };
  auto zval = [&](int r) {  // logit / temperature of the bin at descending rank r
    return h2f((uint16_t)unkey16((uint32_t)(kBins - 1 - r))) / temperature;
  };
  // largest occupied key (the logits are finite: some bin is occupied)
  int first = kBins;
#pragma unroll
  for (int q = kBinsPerThread / 4 - 1; q >= 0; --q) {
    const u4_t c = h4[q * kSelThreads + t];
#pragma unroll
    for (int i = 3; i >= 0; --i)
      if (c[i]) first = r0 + 4 * q + i;
  }
  if (t == 0) {
    kmax_s = kBins;
    owner = -1;
  }
  __syncthreads();
  if (first < kBins) atomicMin(&kmax_s, first);
  __syncthreads();
  if (t == 0) {  // greedy: the largest value at tie rank 0 (lowest index)
    sel[2 * b] = kBins - 1 - kmax_s;
    sel[2 * b + 1] = 0;
  }
  if (temperature <= 0.f) return;
  const float zmax = zval(kmax_s);
  // pass 1: this thread's softmax mass (unnormalised) and the row total Z
  float mass = 0.f;
  for_bins([&](u4_t c, int r) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float m = __builtin_fmaf((float)c[i], __expf(zval(r + i) - zmax), mass);
      mass = c[i] ? m : mass;  // (an empty bin's value may be a NaN pattern)
    }
  });
  float Z;
  const float before = block_exclusive_scan(mass, buf, &Z);
  // pass 2: tokens kept by top-p.  The token at tie rank k of a bin with
  // per-token mass w and mass S before the bin is kept iff S + k w < top_p Z.
  const bool cut = top_p < 1.0f;
  const float lim = top_p * Z;
  auto kept_in = [&](uint32_t c, float w, float S) {
    if (w == 0.f) return 0;  // underflowed: no mass to draw
    if (!cut) return (int)c;
    const float r = (lim - S) / w;  // ranks k < r are kept
    return r <= 0.f ? 0 : (r >= (float)c ? (int)c : (int)ceilf(r));
  };
  // (everything is kept without a cut, nothing once the mass before is past it)
  float S = before, kept = cut ? 0.f : mass;
  if (cut && __any(before < lim))
    for_bins([&](u4_t c, int r) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float w = __expf(zval(r + i) - zmax);
        const float k = __builtin_fmaf((float)kept_in(c[i], w, S), w, kept);
        const float s = __builtin_fmaf((float)c[i], w, S);
        kept = c[i] ? k : kept;
        S = c[i] ? s : S;
      }
    });
  float K = Z, kbefore = before;
  if (cut) kbefore = block_exclusive_scan(kept, buf, &K);
  // pass 3: the draw, target = u * K in kept mass, walked in descending key
  // order and, inside a bin, by tie rank
  const uint64_t ctr = counter_dev ? (uint64_t)(int64_t)*counter_dev : (uint64_t)counter_host;
  const uint64_t x = mix64(mix64(seed ^ ctr) ^ (uint64_t)b);
  const float u = (float)(x >> 40) * (1.0f / 16777216.0f);
  const float target = u * K;
  // owner: the last thread with kept mass whose range starts at or below the
  // target (rounding at a range end falls to that thread's last kept token)
  if (kept > 0.f && kbefore <= target) atomicMax(&owner, t);
  __syncthreads();
  if (t == owner) {
    own_before = before;
    own_kbefore = kbefore;
  }
  __syncthreads();
  // wave 0, lane j: bin j of the owner; the two running sums go along the lanes
  if (t >= 64 || owner < 0) return;
  const uint32_t c = hist[(int64_t)b * kBins + 4 * (t / 4 * kSelThreads + owner) + t % 4];
  const float w = c ? __expf(zval(kBinsPerThread * owner + t) - zmax) : 0.f;
  auto running = [&](float v0, float n) {  // lane j: v0 + sum over bins below j of n w, in order
    float v = v0, mine = v0;
#pragma unroll
    for (int j = 0; j < kBinsPerThread; ++j) {
      if (t == j) mine = v;
      v = __builtin_fmaf(readlane_f(n, j), readlane_f(w, j), v);
    }
    return mine;
  };
  const float Sj = running(own_before, (float)c);
  const int k = c ? kept_in(c, w, Sj) : 0;
  const float Cj = running(own_kbefore, (float)k);
  const uint64_t any = __ballot(k > 0);
  const uint64_t hit = __ballot(k > 0 && target < __builtin_fmaf((float)k, w, Cj));
  // past the last kept bin by rounding: its last token
  const int j = hit ? __ffsll((unsigned long long)hit) - 1
                    : 63 - __clzll((long long)any);
  if (any && t == j) {
    const int q = (int)floorf((target - Cj) / w);
    sel[2 * b] = kBins - 1 - (kBinsPerThread * owner + j);
    sel[2 * b + 1] = !hit ? k - 1 : q < 0 ? 0 : (q >= k ? k - 1 : q);
  }
}

// The token of key sel[b].x with tie rank sel[b].y (lowest index first).  Each
// wave counts the matches in a contiguous sixteenth of the row, two logits per
// packed instruction; the one holding the rank walks its part again.  88 ->
// 16 us for 8 rows of 151,936 (before: 2-byte loads of a contiguous part per thread).
__global__ __launch_bounds__(kSelThreads) void sample_pick_kernel(
    const uint16_t* __restrict__ logits, int64_t V, int64_t stride, const int* __restrict__ sel,
    int64_t* __restrict__ ids, const uint16_t* __restrict__ embed, int D, uint16_t* __restrict__ h,
    int64_t* __restrict__ tokens_out, const int* __restrict__ state, int step_host, int B) {
  constexpr int kWaves = kSelThreads / 64;
  const int b = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t key = (uint32_t)sel[2 * b];
  const int rank = sel[2 * b + 1];
  const uint16_t* row = logits + (int64_t)b * stride;
  const int64_t g0 = group_start(row);
  const int64_t per = (V - g0 + 512 * kWaves - 1) / (512 * kWaves) * 512;  // elements of a wave
  const int64_t lo = g0 + wave * per;
  // the key's pattern in both halves; a zero matches either sign
  const uint32_t pat = unkey16(key) * 0x10001u;
  const uint32_t mask = pat == 0u ? 0x7FFF7FFFu : 0xFFFFFFFFu;
  auto matches = [&](u4_t v, uint32_t valid) {  // bit e: element e of the group has the key
    uint32_t m = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      m |= (uint32_t)((((v[e >> 1] ^ pat) & mask) >> (16 * (e & 1)) & 0xFFFFu) == 0u) << e;
    return m & valid;
  };
  typedef uint16_t us2_t __attribute__((ext_vector_type(2)));
  us2_t differ = {0, 0};  // elements of whole groups that differ, per half
  int n = 0, groups = 0;
  for_groups(row, V, lo + 8 * lane, lo + per, 512, [&](int64_t, u4_t v, uint32_t valid) {
    if (valid == 0xFFu) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const us2_t d = __builtin_bit_cast(us2_t, (v[i] ^ pat) & mask);
        differ += __builtin_elementwise_min(d, us2_t{1, 1});
      }
      if (++groups == 4096) {  // before a half can overflow
        n += 8 * groups - differ[0] - differ[1];
        groups = 0;
        differ = us2_t{0, 0};
      }
    } else {
      n += __popc(matches(v, valid));
    }
  });
  n += 8 * groups - differ[0] - differ[1];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
  __shared__ int total[kWaves], tok;
  if (lane == 0) total[wave] = n;
  if (t == 0) tok = 0;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < wave; ++w) before += total[w];
  if (before <= rank && rank < before + n) {  // wave-uniform
    for (int64_t i = 0; i < per && before <= rank; i += kBatch * 512) {
      u4_t v[kBatch];
      uint32_t valid[kBatch];
#pragma unroll
      for (int g = 0; g < kBatch; ++g)
        valid[g] = load_group(row, V, lo + i + g * 512 + 8 * lane, v[g]) &
                   (i + g * 512 < per ? 0xFFu : 0u);
#pragma unroll
      for (int g = 0; g < kBatch; ++g) {
        uint32_t m = matches(v[g], valid[g]);
        const int c = __popc(m);
        int all = 0, below = 0;  // of the wave, of the lanes before this one
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint64_t bit = __ballot(c >> q & 1);
          all += __popcll(bit) << q;
          below += __popcll(bit & ((1ull << lane) - 1)) << q;
        }
        const int at = rank - before - below;
        if (at >= 0 && at < c) {
          for (int q = 0; q < at; ++q) m &= m - 1u;
          tok = (int)(lo + i + g * 512 + 8 * lane + __ffs(m) - 1);
        }
        before += all;
      }
    }
  }
  __syncthreads();
  if (t == 0) {
    ids[b] = tok;
    const int step = state ? state[kStep] : step_host;
    if (tokens_out) tokens_out[(int64_t)step * B + b] = tok;
  }
  if (embed) {
    const u4_t* src = reinterpret_cast<const u4_t*>(embed + (int64_t)tok * D);
    u4_t* dst = reinterpret_cast<u4_t*>(h + (int64_t)b * D);
    for (int i = t; i < D / 8; i += kSelThreads) dst[i] = src[i];
  }
}

}  // namespace

size_t sample_ws_bytes(int64_t B) { return kSelBytes + (size_t)B * kBins * 4; }

int sample_reserve(r4q_ctx* ctx, int64_t B, void** ws) {
  R4Q_TRY(ctx->sample.reserve(sample_ws_bytes(B)));
  *ws = ctx->sample.ptr;
  return R4Q_OK;
}

int launch_sample(const void* logits, int64_t B, int64_t V, int64_t stride, const SampleCfg& cfg,
                  const int* counter_dev, int64_t counter_host, void* ws, int64_t* ids,
                  const void* embed, int64_t D, void* h, int64_t* tokens_out, const int* state,
                  int step_host, hipStream_t st) {
  R4Q_REQUIRE(cfg.top_p > 0.f, "sample: top_p must be > 0");
  R4Q_REQUIRE(V >= 1 && V < (1LL << 31) && stride >= V, "sample: bad vocabulary size / stride");
  R4Q_REQUIRE(!embed || (D % 8 == 0), "sample: embedding width must be a multiple of 8");
  R4Q_REQUIRE(B <= kMaxRows, "sample: at most %d rows per call (got %lld)", kMaxRows,
              (long long)B);
  int* sel = static_cast<int*>(ws);
  uint32_t* hist = reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(ws) + kSelBytes);
  const auto* lg = static_cast<const uint16_t*>(logits);
  hipLaunchKernelGGL(sample_hist_kernel, dim3(kHistParts, (unsigned)B), dim3(1024), 0, st, lg, V,
                     stride, hist);
  R4Q_TRY(launch_status("sample_hist"));
  hipLaunchKernelGGL(sample_select_kernel, dim3((unsigned)B), dim3(kSelThreads), 0, st, hist,
                     cfg.temperature, cfg.top_p, cfg.seed, counter_dev, counter_host, sel);
  R4Q_TRY(launch_status("sample_select"));
  hipLaunchKernelGGL(sample_pick_kernel, dim3((unsigned)B), dim3(kSelThreads), 0, st, lg, V,
                     stride, sel, ids, static_cast<const uint16_t*>(embed), (int)D,
                     static_cast<uint16_t*>(h), tokens_out, state, step_host, (int)B);
  return launch_status("sample_pick");
}

}  // namespace r4q

extern "C" int r4q_sample(r4q_ctx* ctx, const void* logits, int64_t B, int64_t V, int64_t stride,
                          float temperature, float top_p, uint64_t seed, int64_t counter,
                          int64_t* ids_out, void* stream) {
  R4Q_REQUIRE(ctx && logits && ids_out, "sample: null argument");
  R4Q_REQUIRE(B >= 1, "sample: B must be >= 1");
  R4Q_REQUIRE((reinterpret_cast<uintptr_t>(logits) & 1) == 0, "sample: logits must be fp16");
  const hipStream_t st = r4q::as_stream(stream);
  void* ws = nullptr;
  R4Q_TRY(r4q::sample_reserve(ctx, B, &ws));
  return r4q::launch_sample(logits, B, V, stride, r4q::SampleCfg{temperature, top_p, seed}, nullptr,
                            counter, ws, ids_out, nullptr, 0, nullptr, nullptr, nullptr, 0, st);
}
