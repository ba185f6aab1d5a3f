// Kernels of the prompt (prefill) pass that the decode step does not have:
// the embedding gather and causal self-attention over the prompt's own
// fp16 Q/K/V.
//
// Reference: int4_prefill_logits (hip:2127-2320) gathers embeddings with
// torch::embedding (:2172) and runs causal SDPA with GQA on the fp16
// head-normed, RoPE'd Q/K and raw V (:2254-2265), followed by the FWHT-32
// of the attention output (:2269).  Here the FWHT runs in the attention
// kernel's epilogue, before the single fp16 rounding.
#include <math.h>

#include "r4q_device.hpp"
#include "r4q_host.hpp"
#include "r4q_kernels.hpp"

namespace r4q {
namespace {

// out[m, :] = table[ids[m], :] (fp16 rows of D elements, D % 8 == 0).
// ids are range-checked on the host before launch.
__global__ __launch_bounds__(256) void embed_gather_kernel(const int64_t* __restrict__ ids,
                                                           const uint16_t* __restrict__ table,
                                                           uint16_t* __restrict__ out, int D) {
  const int64_t m = blockIdx.x;
  const u4_t* src = reinterpret_cast<const u4_t*>(table + ids[m] * (int64_t)D);
  u4_t* dst = reinterpret_cast<u4_t*>(out + m * (int64_t)D);
  for (int i = threadIdx.x; i < D / 8; i += blockDim.x) dst[i] = src[i];
}

// Causal GQA flash attention on the matrix cores (v_mfma_f32_16x16x32_f16).
// A workgroup (4 waves) takes 64 query rows of one query head; wave w owns
// rows q0 + 16w .. +15.  Rows of `qkv` (stride `stride` elements) hold q
// heads at h*128, k heads at (H + kh)*128 and v heads at (H + Hk + kh)*128,
// kh = h / (H/Hk).  out[m, h*128 + d] =
//   FWHT32(softmax_{j <= m}(q_m . k_j / sqrt(128)) V)[d].
// Keys go in blocks of 32 through LDS, two stages each for K and for V filled by
// direct copies.  Both tiles are row major, 256 bytes a key, the 16-byte pieces of
// row r at piece ^ (r & 15) for K and piece ^ 2 (r & 7) for V, which spreads each
// read below over all banks.  In turn kb a wave takes S of block kb + 1 (matrix
// cores) and the softmax and P V of block kb, two chains that do not depend on
// each other; K of kb + 2 and V of kb + 1 are in flight.
// Per block and wave (lane l: column n = l % 16, group g = l / 16):
//  * S^T = K Q^T for two 16-key halves: A = K (lane: key n of the half,
//    dims 32k + 8g .. over the 4 k-steps), B = Q^T (lane: query row n, the
//    same dims, held in registers for the whole loop).  C: lane holds query
//    n at keys 4g .. 4g+3 of the half;
//  * online softmax per query across the 4 lanes holding it, probabilities
//    rounded to fp16, keys past the query masked (in the diagonal block only);
//  * O += P V: A = P (lane: query n; k-slots = its 8 keys 4g + r and
//    16 + 4g + r), B = V (lane: dim 16j + n of N-block j, the same keys: two
//    transposing LDS reads).  C: lane holds dim 16j + n of queries 4g .. 4g+3.
//    O is rescaled only where some row's maximum moved (a factor of 1 is exact).
// Epilogue: O / l, FWHT-32 per 32-dim chunk (the 16-dim step inside the
// lane, steps 1 .. 8 across lanes xor 1 .. 8), one fp16 rounding.
//
// Bound by the softmax's vector instructions with the waves that one CU holds (four
// workgroups, 128 VGPRs).  40 heads over 8 K/V heads, 2000 rows: 191 -> 76-79 us; 512
// rows: 31 -> 19 us, a chain of 16 turns in the longest workgroup.  Before, V was
// transposed by 2-byte LDS stores that conflicted 4 ways, K, softmax and V of a
// block were one chain, and the tiles with the fewest keys came first.  32 query
// rows per wave (half the LDS reads per row) measured 93 and 27 us.
constexpr int kFaRows = 64;        // query rows of a workgroup
constexpr int kFaTile = 32 * 256;  // bytes of a block's K (or V) in LDS: K, K, V, V

typedef short s4_t __attribute__((ext_vector_type(4)));

// maximum over the lanes n, n + 16, n + 32, n + 48, in all of them
__device__ __forceinline__ float max_groups(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = fmaxf(__builtin_bit_cast(float, (uint32_t)a[0]), __builtin_bit_cast(float, (uint32_t)a[1]));
  const uint32_t w = __builtin_bit_cast(uint32_t, v);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)b[0]),
               __builtin_bit_cast(float, (uint32_t)b[1]));
}

__global__ __launch_bounds__(256, 4) void prefill_fa_kernel(const uint16_t* __restrict__ qkv,
                                                            int64_t stride,
                                                            uint16_t* __restrict__ out,
                                                            int64_t out_stride, int M, int H,
                                                            int Hk) {
  __shared__ __align__(1024) uint8_t smem[4 * kFaTile];
  lds8* const lds = (lds8*)smem;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int col = lane & 15, g = lane >> 4;
  // workgroup -> (head, query tile): the tiles with the most keys first, and a
  // run of heads (which share K/V heads) per XCD where the head count allows
  int h, qt;
  {
    const int S = H % 8 == 0 ? 8 : 1, id = blockIdx.x, j = id / S, hc = H / S;
    h = (id % S) * hc + j % hc;
    qt = (int)(gridDim.x / H) - 1 - j / hc;
  }
  const int q0 = qt * kFaRows;
  const int kh = h / (H / Hk);
  const uint16_t* kbase = qkv + (int64_t)(H + kh) * 128;
  const int r0 = q0 + 16 * wave;                     // this wave's first query row
  const int nkb = (min(q0 + kFaRows, M) + 31) / 32;  // blocks of keys of the workgroup
  const int nwb = min(nkb, r0 / 32 + 1);             // and of this wave; the last one masked

  // staging: 512 16-byte slots per tile (slot 16 row + place), two copies per
  // thread, the source pieces swizzled as above; keys past the prompt clamped.
  // kp, vp: this thread's first piece of the next K and V block to load
  const int srow = 4 * wave + g;
  const uint16_t* kp = kbase + srow * stride + 8 * (col ^ srow);
  const uint16_t* vp = kbase + Hk * 128 + srow * stride + 8 * (col ^ (2 * (srow & 7)));
  auto load_tile = [&](const uint16_t*& p, int kb, int tile) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint16_t* src = p + 16 * i * stride;
      if (32 * kb + 32 > M)  // rows past the prompt: its last one
        src -= max(32 * kb + 16 * i + srow - (M - 1), 0) * stride;
      copy16(src, lds + tile * kFaTile + 4096 * i + 1024 * wave);
    }
    p += 32 * stride;
  };
  load_tile(kp, 0, 0);
  load_tile(vp, 0, 2);
  if (nkb > 1) load_tile(kp, 1, 1);

  // Q^T fragments: qb[k] = Q[row r0 + col][32k + 8g .. +7] (rows past M clamped)
  u4_t qb[4];
  {
    const uint16_t* qr = qkv + (int64_t)min(r0 + col, M - 1) * stride + h * 128 + 8 * g;
#pragma unroll
    for (int k = 0; k < 4; ++k) qb[k] = *reinterpret_cast<const u4_t*>(qr + 32 * k);
  }
  int ka[4], va[4];  // LDS offsets of the reads: stage 0, first 16 keys, j < 4
#pragma unroll
  for (int k = 0; k < 4; ++k) ka[k] = 256 * col + 16 * ((4 * k + g) ^ col);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = 4 * g + (col >> 2);
    va[j] = 2 * kFaTile + 256 * row + 16 * ((2 * j + ((col & 3) >> 1)) ^ (2 * (row & 7))) +
            8 * (col & 1);
  }

  const float sscale = 0.08838834764831845f;  // 1 / sqrt(128)
  const uint32_t ones = 0x3C003C00u;           // fp16 (1, 1)
  float m_run = -INFINITY, l_run = 0.f;        // query col; l over this lane's keys
  f4_t o[8], s0[2], s1[2];                      // s0, s1: scores of even and odd blocks
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = f4_t{0.f, 0.f, 0.f, 0.f};
  auto kpos = [&](int e) { return e < 4 ? 4 * g + e : 16 + 4 * g + (e - 4); };

  // S^T = K Q^T of the block in K stage `stage`
  auto scores = [&](f4_t(&s)[2], int stage) {
#pragma unroll
    for (int bb = 0; bb < 2; ++bb) {
      s[bb] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const h8_t kf = *(const __attribute__((address_space(3))) h8_t*)(lds + ka[k] + 4096 * bb +
                                                                         stage * kFaTile);
        s[bb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, __builtin_bit_cast(h8_t, qb[k]), s[bb],
                                                       0, 0, 0);
      }
    }
  };
  // online softmax for query r0 + col over block kb's keys 32 kb + kpos(e), O += P V
  auto attend = [&](const f4_t(&s)[2], int kb, int stage, bool masked) {
    // scores are rounded before the maximum is subtracted, in every block alike
#pragma clang fp contract(off)
    float sv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sv[e] = s[e >> 2][e & 3] * sscale;
      if (masked && 32 * kb + kpos(e) > r0 + col) sv[e] = -INFINITY;
    }
    float mx = sv[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mx = fmaxf(mx, sv[e]);
    const float mn = fmaxf(m_run, max_groups(mx));  // finite: key 32 kb is unmasked
    const float alpha = __expf(m_run - mn);         // 0 in the first block
    u4_t pa;                                        // fp16 probabilities, k-slot e = key kpos(e)
    float lp = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p0 = __expf(sv[2 * i] - mn), p1 = __expf(sv[2 * i + 1] - mn);
      pa[i] = cvt_pk_h(p0, p1);
      lp = __builtin_amdgcn_fdot2(as_h2(pa[i]), as_h2(ones), lp, false);
    }
    l_run = __builtin_fmaf(l_run, alpha, lp);
    m_run = mn;
    if (__any(!(alpha == 1.0f))) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {  // query 4g + r of C's rows: lane 4g + r holds its alpha
        const float ar = __shfl(alpha, 4 * g + r);
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j][r] *= ar;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      typedef __attribute__((address_space(3))) s4_t lds_s4;
      lds8* const v = lds + (va[j & 3] ^ (j < 4 ? 0 : 128)) + stage * kFaTile;
      const u2_t lo = __builtin_bit_cast(u2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)v));
      const u2_t hi =
          __builtin_bit_cast(u2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(v + 4096)));
      const h8_t vb = __builtin_bit_cast(h8_t, (u4_t{lo[0], lo[1], hi[0], hi[1]}));
      o[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, pa), vb, o[j], 0, 0,
                                                    0);
    }
  };
  // this wave's copies so far have landed, after the barrier everyone's, and
  // everyone's LDS reads of the turn before are done
  auto sync = [] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto begin = [&](int kb, int st) {  // st = kb & 1
    sync();
    if (kb + 2 < nkb) load_tile(kp, kb + 2, st);
    if (kb + 1 < nkb) load_tile(vp, kb + 1, 3 - st);
  };
  sync();
  scores(s0, 0);
  int kb = 0;
  for (; kb + 2 < nwb; kb += 2) {
    begin(kb, 0);
    scores(s1, 1);
    attend(s0, kb, 0, false);
    begin(kb + 1, 1);
    scores(s0, 0);
    attend(s1, kb + 1, 1, false);
  }
  begin(kb, 0);
  if (kb + 1 < nwb) {
    scores(s1, 1);
    attend(s0, kb, 0, false);
    begin(++kb, 1);
    s0[0] = s1[0];
    s0[1] = s1[1];
  }
  attend(s0, kb, kb & 1, true);
  for (++kb; kb < nkb; ++kb) begin(kb, kb & 1);  // the other waves' last blocks
  // ---- O / l, FWHT-32, fp16 out (rows 4g + r of the wave's 16)
  float lsum = l_run + __shfl_xor(l_run, 16);
  lsum += __shfl_xor(lsum, 32);
  float inv[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) inv[r] = 1.0f / __shfl(lsum, 4 * g + r);
#pragma unroll
  for (int c = 0; c < 4; ++c) {  // 32-dim chunk c = N-blocks 2c, 2c+1
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float a = o[2 * c][r] * inv[r], b = o[2 * c + 1][r] * inv[r];
      {  // element bit 4 (dims 16 apart) inside the lane
        const float t0 = a + b, t1 = a - b;
        a = t0;
        b = t1;
      }
#pragma unroll
      for (int bit = 1; bit <= 8; bit <<= 1) {  // element bits 0..3 across lanes
        const float oa = __shfl_xor(a, bit), ob = __shfl_xor(b, bit);
        if (col & bit) {
          a = oa - a;
          b = ob - b;
        } else {
          a = a + oa;
          b = b + ob;
        }
      }
      const int row = r0 + 4 * g + r;
      if (row < M) {
        uint16_t* dst = out + (int64_t)row * out_stride + h * 128 + 32 * c + col;
        dst[0] = f2h(a * kInvSqrt32);
        dst[16] = f2h(b * kInvSqrt32);
      }
    }
  }
}

}  // namespace

int launch_embed_gather(const int64_t* ids, const void* table, void* out, int64_t M, int64_t D,
                        hipStream_t st) {
  if (M == 0) return R4Q_OK;
  hipLaunchKernelGGL(embed_gather_kernel, dim3((unsigned)M), dim3(256), 0, st, ids,
                     static_cast<const uint16_t*>(table), static_cast<uint16_t*>(out), (int)D);
  return launch_status("embed_gather");
}

int launch_prefill_attention(const void* qkv, int64_t stride, void* out, int64_t out_stride,
                             int64_t M, int64_t H, int64_t Hk, hipStream_t st) {
  if (M == 0) return R4Q_OK;
  hipLaunchKernelGGL(prefill_fa_kernel, dim3((unsigned)(H * ((M + kFaRows - 1) / kFaRows))),
                     dim3(256), 0, st, static_cast<const uint16_t*>(qkv), stride,
                     static_cast<uint16_t*>(out), out_stride, (int)M, (int)H, (int)Hk);
  return launch_status("prefill_attention");
}

}  // namespace r4q

extern "C" int r4q_prefill_attention(const void* qkv, int64_t stride, void* out,
                                     int64_t out_stride, int64_t M, int64_t H, int64_t Hk,
                                     void* stream) {
  R4Q_REQUIRE(qkv && out, "prefill_attention: null pointer");
  R4Q_REQUIRE(M >= 1 && M < (1LL << 31), "prefill_attention: bad row count");
  R4Q_REQUIRE(H >= 1 && Hk >= 1 && H % Hk == 0, "prefill_attention: bad head counts");
  R4Q_REQUIRE(stride >= (H + 2 * Hk) * 128 && stride % 8 == 0 && out_stride >= H * 128 &&
                  (reinterpret_cast<uintptr_t>(qkv) & 15) == 0,
              "prefill_attention: rows must be 16-byte aligned and hold H + 2 Hk heads of 128");
  return r4q::launch_prefill_attention(qkv, stride, out, out_stride, M, H, Hk,
                                       r4q::as_stream(stream));
}
