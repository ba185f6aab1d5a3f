// Prefill GEMM Y[M,N] = X[M,K] W[N,K]^T with the weight dequantised on the
// fly (INT4 / INT8 block-32 asymmetric, or FP16) and multiplied on the
// matrix cores with v_mfma_f32_16x16x32_f16 (fp32 accumulate).
//
// Replaces the reference's prefill projection dequant_matmul_out
// (hip:1973-1988), which materialises the whole fp16 weight with
// dequant_int4_kernel and then calls rocBLAS through at::mm_out: here each
// weight byte is read from HBM once per M-tile and never written back.
//
// Two kernels, by shape:
//  * gemm_tile_kernel (M >= 17): tiles of 32 .. 128 rows x 128 columns or 256 x
//    256, X and the raw weights copied global -> LDS through a ring, the
//    weights dequantised per wave in registers (FP16: read as they are), the
//    K steps of the tiles shared evenly by the CUs (deterministic reduce over
//    a caller workspace);
//  * gemm_skinny_kernel (2 <= M <= 16): weights streamed once for all rows
//    through an LDS ring (split along K for narrow N).
// Dequantised values equal r4q_dequant_int4/8 bit-for-bit (fp16((q - zp) * scale)
// from an exact product, one rounding): between 17 and 255 rows for every
// zero-point, elsewhere for whole numbers up to 1024 (others are rounded to the
// nearest one: zp + 1024 is a fp16 number there).
#include <stdint.h>
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "r4q_device.hpp"
#include "r4q_gemv.hpp"
#include "r4q_host.hpp"

namespace r4q {
namespace {

// (1024 + q_2p, 1024 + q_2p+1) as an fp16 pair from byte p of a packed INT4
// word w (w4 = w >> 4): v_perm puts byte p of w in byte 0 and byte p of w4 in
// byte 2, one v_and_or keeps the low nibbles and sets the 0x64 exponent bytes
// (written out: with two literal operands, which VOP3 cannot encode on this
// target, the compiler emits a separate AND and OR).
__device__ __forceinline__ uint32_t nib_pair(uint32_t w, uint32_t w4, int p) {
  const uint32_t t = __builtin_amdgcn_perm(w4, w, (uint32_t)(p | (p + 4) << 16));
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(t), "s"(0x000F000Fu), "v"(0x64006400u));
  return r;
}

// ---------------------------------------------------------------------
// Weight fragments of the skinny GEMM (below).  The MFMA contraction index k
// is only a label: lane group g's 8 k-slots of an MFMA carry 8 weight
// elements, and the A fragment of that lane group holds the activation
// values of exactly those elements.  Because the weights are fully
// dequantised before the MFMA -- fp16((q - zp) * s) by an exact packed fp16
// subtraction and one rounded packed multiply, bit-identical to the dequant
// kernel -- the accumulation may run across blocks.
//   INT4: 4 MFMAs per 16 weight bytes; the nibble pair (q_2j, q_2j+1) of
//         byte j of a word w is byte j of w and of w >> 4 (v_perm), masked
//         and tagged 0x6400 in one v_and_or: natural k order, so the
//         activation is used as loaded;
//   INT8: 2 MFMAs per 16 bytes; byte pairs by v_perm, natural order;
//   FP16: 1 MFMA per 16 bytes.
// B fragment of MFMA d from 16 weight bytes w and the block's (scale, zero) s2.
template <int WBITS>
__device__ __forceinline__ h8_t skinny_b(const u4_t w, uint32_t s2, int d) {
  if constexpr (WBITS == 16) {
    return __builtin_bit_cast(h8_t, w);
  } else {
    const uint32_t sb = s2 & 0xFFFFu;
    const h2_t sc = as_h2(sb | (sb << 16));
    const uint32_t zb = s2 >> 16;
    // -(1024 + zp) as an fp16 pair (exact: an integer below 2048)
    const h2_t nz = -(as_h2(0x64006400u) + as_h2(zb | (zb << 16)));
    uint32_t pr[4];
    if constexpr (WBITS == 4) {
      const uint32_t wd = w[d], wd4 = wd >> 4;
#pragma unroll
      for (int p = 0; p < 4; ++p) pr[p] = nib_pair(wd, wd4, p);
    } else {
      const uint32_t w0 = w[2 * d], w1 = w[2 * d + 1];
      pr[0] = __builtin_amdgcn_perm(w0, 0x64646464u, 0x00050004u);
      pr[1] = __builtin_amdgcn_perm(w0, 0x64646464u, 0x00070006u);
      pr[2] = __builtin_amdgcn_perm(w1, 0x64646464u, 0x00050004u);
      pr[3] = __builtin_amdgcn_perm(w1, 0x64646464u, 0x00070006u);
    }
    u4_t o;
#pragma unroll
    for (int p = 0; p < 4; ++p) o[p] = as_u32((as_h2(pr[p]) + nz) * sc);
    return __builtin_bit_cast(h8_t, o);
  }
}

template <class T>
__device__ __forceinline__ T lds_ld(const lds8* p) {
  return *(const __attribute__((address_space(3))) T*)p;
}

template <int N>
__device__ __forceinline__ void wait_copies() {  // at most N of this wave's copies outstanding
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Workgroup barrier that, unlike __syncthreads, does not first wait for
// every outstanding global access (the copies still in flight): only for
// this wave's LDS accesses.
__device__ __forceinline__ void ring_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Stream-K bookkeeping shared by the GEMM and the reduce: first unit of
// workgroup w, and the workgroup holding unit u.
__device__ __forceinline__ int64_t sk_lo(int w, int64_t TU, int sk) {
  return (int64_t)w * TU / sk;
}
__device__ __forceinline__ int sk_owner(int64_t u, int64_t TU, int sk) {
  int w = (int)(u * sk / TU);
  while (w + 1 < sk && sk_lo(w + 1, TU, sk) <= u) ++w;
  while (w > 0 && sk_lo(w, TU, sk) > u) --w;
  return w;
}

// ---------------------------------------------------------------------
// Tile GEMM (M >= 17): 16 MT MG rows of X x 64 NF weight rows per workgroup of
// MG groups of 4 waves; wave w of a group owns its 16 MT rows and weight rows
// 16 NF w .. of the tile.
//  * M < 256: MT = 2 .. 8, NF = 1 or 2, MG = 1: 32 x 64 .. 128 x 128, each tile
//    over all of K; tile_shape picks the one that loads the CUs most evenly.
//  * M >= 256: 256 x 256 (MT = 8, NF = 4, MG = 2), each wave 128 x 64: the
//    fewest bytes copied and LDS reads per MFMA that two waves per SIMD (256
//    VGPRs, 128 of them accumulators) allow.  The second wave's MFMAs run while
//    the first reads LDS, dequantises or issues copies.
// X, the raw weights and their (scale, zero) words of a K step (KS = 64 or 128
// k) arrive by global->LDS copies through a ring of D stages, D - 1 steps in
// flight, one barrier per step, the copies spread over the step's MFMAs.
// Longer steps mean fewer barriers, which measured more than a shorter step's
// deeper ring (512 x 151936 x 5120 FP16: 64 k and 2 stages 782 us, 32 k and 5
// stages 812); a step less in flight costs more than reading ahead across the
// barrier gains (FP16, 32768 outputs: 224 against 169 us).
// Every output is one chain of 16x16x32 MFMAs over its k in natural order (per
// segment), whatever the tile: the shapes give the same bits.  MFMA k-step j
// covers block j of the step, lane group g its k labels 32 j + 8 g .. + 7.  The
// weights are the MFMA's A operand, so that a lane's results are consecutive
// outputs of one row of Y; LDS slots are swizzled against bank conflicts (wsw,
// xsw).  A scale or zero-point is broadcast to a pair by the operand selects
// of the packed instructions (dqp): 2.4 vector instructions per MFMA at INT4.
// Work split (M >= 256): a tile is a K loop of U units; blocks [0, dp) compute
// whole tiles, the sk others share the units of the remaining tiles evenly
// (split_plan): workgroup w takes units [floor(w TU / sk), floor((w + 1) TU / sk))
// of the TU = (T - dp) U flattened ones.  A tile shared by several workgroups
// gets one fp16 partial per workgroup (segment), summed in fp32 in segment
// order by gemm_tile_reduce_kernel: the result does not depend on timing.
// What bounds it: M >= 256, the work of a step that its MFMAs do not cover: at 512 x
// 32768 x 5120 INT4 the matrix cores are busy 48% of the cycles at the 2.0 GHz (of
// 2.4) that the power limit leaves, 57% without the dequantisation.  Timing
// builds of that shape, us with everything / without the copies / without the
// steps' barriers too: INT4 160 / 144 / 133, INT8 158 / 148 / 135, FP16 (2 stages,
// every step opens with a wait for its copies) 163 / 121 / 119 -- on what the LDS
// happens to hold, which also draws less power.  The rest, the LDS reads and the
// dequantisation ahead of a step's first MFMA among it, is not taken apart.
// M < 256, the serial chain of K steps (0.34 us per 128 k for a 32 x 64 tile),
// whose parts are not taken apart either.
// Measured (us, graph replays on one box, weights not evicted between them;
// before: a 128 x 128 kernel with one 32-wide step in flight for M < 256, 256 x
// 256 tiles with one wave per SIMD for M >= 256): INT4 17 x 7168 x 5120 116 -> 20,
// 96 x 7168 x 5120 122 -> 23, 128 x 5120 x 17408 420 -> 71, 96 x 34816 x 5120 139 -> 70,
// 24 x 151936 x 5120 FP16 396 -> 282; 512 x 17408 x 5120 INT4 126 -> 112, 512 x 5120 x
// 17408 109 -> 102, 512 x 34816 x 5120 198 -> 187, 1999 x 34816 x 5120 INT8 796 -> 707 (1.01
// PFLOP/s), 512 x 151936 x 5120 FP16 958 -> 804.  Another box, and less heat, moves
// them by up to 15%.
template <int WBITS, int MT, int NF, int MG>
struct Tile {
  static constexpr int kMG = MG;
  static constexpr int kOut = NF > 1 ? 8 : 4;  // outputs per store
  static constexpr int kThreads = 256 * MG;
  static constexpr int KS = MG == 2 || NF > 1 || WBITS == 16 ? 64 : 128;
  // K of a stream-K unit, in whole steps: a unit that ends inside a step costs its
  // segment a partly empty step and clear_tail (FP16, 256 x 34816 x 5120: 145 us with
  // units of 32 k, 125 of 64; 1300 x 9000 x 3008 109 and 100; 256 x 256 x 4096 46 and 28)
  static constexpr int kUnit = WBITS == 4 ? 256 : WBITS == 8 ? 128 : 64;
  static_assert(kUnit % KS == 0, "units of whole steps");
  static constexpr int BM = 16 * MT * MG, BN = 64 * NF;
  static constexpr int J = KS / 32;  // MFMA k-steps, one quantisation block each
  static constexpr int XRow = KS * 2, WRow = KS * WBITS / 8;  // bytes of a row per step
  static constexpr int SW = WBITS == 16 ? 0 : J;              // scale words of a row per step
  static constexpr int kX = BM * XRow, kW = BN * WRow, kS = BN * SW * 4;
  static constexpr int kStage = kX + kW + kS;
  static constexpr int kFit = (MG == 2 ? 160 : 80) * 1024 / kStage;
  static constexpr int D = kFit < 8 ? kFit : 8;  // ring stages: one in use, the others in flight
  // copies per wave and step
  static constexpr int CX = kX / (4096 * MG), CW = kW / (4096 * MG), CS = kS / (1024 * MG);
  static constexpr int kPer = CX + CW + CS;
  static constexpr int WD = WBITS / 4;  // weight words of a lane per fragment and MFMA k-step
  static constexpr int Q = J * MT;  // X fragments of a wave per step
  static constexpr int P = Q % 4 == 0 ? 4 : Q % 3 == 0 ? 3 : 2;  // of which are read ahead
  static constexpr int kWPieces = WRow / 16;
  static_assert(kX % (4096 * MG) == 0 && kW % (4096 * MG) == 0 && kS % (1024 * MG) == 0,
                "copies split evenly");
  static_assert(D >= 2 && (D - 2) * kPer <= 63 && Q % P == 0, "ring");
  // 16-byte piece p of a row sits in slot p ^ swizzle of the row, so that the
  // 16 rows of a fragment read fall on 16 different 16-byte groups of the 256
  // bytes of banks: X fragments read 16 consecutive rows, weight fragments
  // rows 4 NF (c / 4) + 4 f + c % 4 (c = 0 .. 15; the same slots for every f)
  static constexpr int kSh = NF == 4 ? 4 : NF == 2 ? 3 : 2;
  static __device__ __forceinline__ int wsw(int r) {
    const int h = (r >> kSh) & 3;
    return kWPieces >= 16 ? (r & 3) | (h << 2)
           : kWPieces == 8 ? ((r >> 1) & 1) | (h << 1)
           : kWPieces == 4 ? h : h & 1;
  }
  static __device__ __forceinline__ int xsw(int r) {
    return XRow / 16 >= 16 ? r & 15 : XRow / 16 == 8 ? (r >> 1) & 7 : (r >> 2) & 3;
  }
};

template <int WBITS, int MT, int NF, int MG>
struct TileSeg {
  using T = Tile<WBITS, MT, NF, MG>;
  static constexpr bool kAnyZp = MG == 1 && WBITS != 16;  // exact for every zero-point
  lds8* ring;
  const uint8_t *X, *W, *SZ;  // first row of the tile
  int K, ka, ke, nk, wave, col, g, mg, ws;  // k range [ka, ke) in nk steps
  uint32_t xo[T::CX], wo[T::CW], so[T::CS > 0 ? T::CS : 1];  // this lane's copies: byte offsets
  uint32_t ox[T::J], ow, os;                                  // LDS offsets within a stage
  // 0x000F000F and 0x64006400 in registers: as literals the compiler would
  // need two instructions for x & mask | tag
  uint32_t nmask, ntag;

  struct Raw {
    uint32_t w[NF][T::J][T::WD];
    uint32_t s2[NF][T::J];
  };

  __device__ __forceinline__ void init(const uint16_t* x, const uint8_t* w, const uint32_t* sz,
                                       int M, int N, int K_, int m0, int n0, int t) {
    const int lane = t & 63;
    nmask = 0x000F000Fu;
    ntag = 0x64006400u;
    asm volatile("" : "+s"(nmask), "+v"(ntag));
    K = K_;
    const uint32_t xb = 2u * K, wb = (uint32_t)K * WBITS / 8, sb = K / 8;  // bytes per row
    X = reinterpret_cast<const uint8_t*>(x) + (int64_t)m0 * xb;
    W = w + (int64_t)n0 * wb;
    SZ = reinterpret_cast<const uint8_t*>(sz) + (int64_t)n0 * sb;
    col = lane & 15;
    g = lane >> 4;
    mg = MG == 2 ? wave >> 2 : 0;
    // (the min within a row only matters when a row is shorter than a step)
#pragma unroll
    for (int i = 0; i < T::CX; ++i) {
      const int off = 1024 * (T::CX * wave + i) + 16 * lane, r = off / T::XRow;
      xo[i] = (uint32_t)min(r, M - 1 - m0) * xb +
              min(16u * (((off % T::XRow) / 16) ^ T::xsw(r)), xb - 16);
    }
#pragma unroll
    for (int i = 0; i < T::CW; ++i) {
      const int off = 1024 * (T::CW * wave + i) + 16 * lane, r = off / T::WRow;
      wo[i] = (uint32_t)min(r, N - 1 - n0) * wb +
              min(16u * (((off % T::WRow) / 16) ^ T::wsw(r)), wb - 16);
    }
    if constexpr (T::CS > 0) {
#pragma unroll
      for (int i = 0; i < T::CS; ++i) {
        const int off = 256 * (T::CS * wave + i) + 4 * lane, r = off / (T::SW * 4);
        so[i] = (uint32_t)min(r, N - 1 - n0) * sb + min((uint32_t)off % (T::SW * 4), sb - 4);
      }
    }
    // fragment reads: X rows 16 m + col (the swizzle of col for every m);
    // weight rows 16 NF wq + wrow + 4 f
    const int wrow = 4 * NF * (col >> 2) + (col & 3);
    ws = T::wsw(wrow);
    const int wq = wave & 3;
#pragma unroll
    for (int j = 0; j < T::J; ++j)
      ox[j] = T::XRow * (16 * MT * mg + col) + 16 * ((4 * j + g) ^ T::xsw(col));
    ow = T::kX + T::WRow * (16 * NF * wq + wrow);
    os = T::kX + T::kW + T::SW * 4 * (16 * NF * wq + wrow);
  }

  // first k that the stage of step i holds: a step that would reach past K
  // holds the KS before K instead (clear_tail drops the others)
  __device__ __forceinline__ int first_k(int i) const {
    return max(min(ka + min(i, nk - 1) * T::KS, K - T::KS), 0);
  }
  // copy c of the kPer a wave makes of step i (clamped to the segment's last)
  // into stage st
  struct Src {
    const uint8_t *x, *w, *s;
    lds8 *dx, *dw, *ds;
  };
  __device__ __forceinline__ Src src(int i, lds8* st) const {
    const int k = first_k(i);
    return Src{X + 2 * (int64_t)k, W + (int64_t)k * WBITS / 8, SZ + k / 8,
               st + 1024 * T::CX * wave, st + T::kX + 1024 * T::CW * wave,
               st + T::kX + T::kW + 256 * T::CS * wave};
  }
  // (offsets added in the copy's own instruction below 256 rows: 0-3% faster there,
  // 1999 x 34816 x 5120 INT8 1% slower)
  template <int C>
  __device__ __forceinline__ void copy(const Src& s) const {
    constexpr bool kX = C < T::CX, kW = !kX && C < T::CX + T::CW;
    constexpr int kOff = kX ? 1024 * C : kW ? 1024 * (C - T::CX) : 256 * (C - T::CX - T::CW);
    constexpr int kIn = MG == 1 ? kOff : 0, kOut = kOff - kIn;
    if constexpr (kX) copy16s<kIn>(s.x, xo[C], s.dx + kOut);
    else if constexpr (kW) copy16s<kIn>(s.w, wo[C - T::CX], s.dw + kOut);
    else copy4s<kIn>(s.s, so[C - T::CX - T::CW], s.ds + kOut);
  }
  // the copies c >= C for which f(c)
  template <int C = 0, class F>
  __device__ __forceinline__ void copies(const Src& s, F f) const {
    if constexpr (C < T::kPer) {
      if (f(C)) copy<C>(s);
      copies<C + 1>(s, f);
    }
  }
  __device__ __forceinline__ void issue(int i, lds8* st) const {
    const Src s = src(i, st);
    copies(s, [](int) { return true; });
  }

  // zeroes what the stage of a last step i holds outside its own k (before
  // them, or past the segment's end), once its copies have landed: X, and the
  // scale words (FP16: the weights)
  __device__ __forceinline__ void clear_tail(int i, lds8* st, int t) const {
    typedef __attribute__((address_space(3))) u4_t lds_u4;
    typedef __attribute__((address_space(3))) uint32_t lds_u1;
    const int lo = ka + i * T::KS - first_k(i), hi = ke - first_k(i);  // the step's own k
    for (int e = t; e < T::kX / 16; e += T::kThreads) {
      const int r = e / (T::XRow / 16), p = e % (T::XRow / 16);
      if (8 * p < lo || 8 * p >= hi)
        *(lds_u4*)(st + r * T::XRow + 16 * (p ^ T::xsw(r))) = u4_t{0u, 0u, 0u, 0u};
    }
    if constexpr (WBITS == 16) {
      for (int e = t; e < T::kW / 16; e += T::kThreads) {
        const int r = e / T::kWPieces, p = e % T::kWPieces;
        if (8 * p < lo || 8 * p >= hi)
          *(lds_u4*)(st + T::kX + r * T::WRow + 16 * (p ^ T::wsw(r))) = u4_t{0u, 0u, 0u, 0u};
      }
    } else {
      for (int e = t; e < T::BN * T::SW; e += T::kThreads) {
        const int k = 32 * (e % T::SW);
        if (k < lo || k >= hi) *(lds_u1*)(st + T::kX + T::kW + 4 * e) = 0u;
      }
    }
    ring_barrier();
  }

  __device__ __forceinline__ void load_raw(const lds8* st, Raw& r) const {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const lds8* wb = st + ow + 4 * f * T::WRow;
#pragma unroll
      for (int j = 0; j < T::J; ++j) {  // k labels 32 j + 8 g .. + 7
        const int b = 4 * WBITS * j + WBITS * g;
        const lds8* q = wb + (((b >> 4) ^ ws) << 4) + (b & 15);
        if constexpr (WBITS == 4) {
          r.w[f][j][0] = lds_ld<uint32_t>(q);
        } else if constexpr (WBITS == 8) {
          const u2_t v = lds_ld<u2_t>(q);
          r.w[f][j][0] = v[0];
          r.w[f][j][1] = v[1];
        } else {
          const u4_t v = lds_ld<u4_t>(q);
#pragma unroll
          for (int e = 0; e < 4; ++e) r.w[f][j][e] = v[e];
        }
      }
      if constexpr (WBITS != 16) {
        const lds8* q = st + os + 4 * f * T::SW * 4;
        if constexpr (T::J == 4) {
          const u4_t v = lds_ld<u4_t>(q);
#pragma unroll
          for (int j = 0; j < 4; ++j) r.s2[f][j] = v[j];
        } else {
          const u2_t v = lds_ld<u2_t>(q);
          r.s2[f][0] = v[0];
          r.s2[f][1] = v[1];
        }
      }
    }
  }

  // Pair k (labels 2k, 2k + 1) of B fragment f of MFMA k-step j: fp16((q - zp)
  // * scale), bit-identical to the dequant kernel for zero-points that are whole
  // numbers from 0 to 1024, which is what checkpoints hold (q - zp is a difference
  // of fp16 numbers).  One pair at a time, so that the arithmetic can be spread
  // between MFMAs; nz / sc / w4: the fragment's constants, set by its pair-0 call.
  __device__ __forceinline__ uint32_t dqp(const Raw& r, int f, int j, int k, h2_t& nz, h2_t& sc,
                                          uint32_t& w4) const {
    if constexpr (WBITS == 16) {
      return r.w[f][j][k];
    } else {
      if (k == 0) {
        const h2_t s = as_h2(r.s2[f][j]);  // broadcasts: operand selects of the packed ops
        sc = __builtin_shufflevector(s, s, 0, 0);
        nz = -(as_h2(0x64006400u) + __builtin_shufflevector(s, s, 1, 1));  // -(1024 + zp), exact
        if constexpr (WBITS == 4) w4 = r.w[f][j][0] >> 4;
      }
      uint32_t pr;
      if constexpr (WBITS == 4)
        pr = (__builtin_amdgcn_perm(w4, r.w[f][j][0], (uint32_t)(k | (k + 4) << 16)) & nmask) | ntag;
      else
        pr = __builtin_amdgcn_perm(r.w[f][j][k >> 1], 0x64646464u,
                                   (k & 1) ? 0x00070006u : 0x00050004u);
      return as_u32((as_h2(pr) + nz) * sc);
    }
  }
  // The same for any zero-point, as the dequant kernel computes it.
  __device__ __forceinline__ h8_t dqx(const Raw& r, int f, int j) const {
    const float scale = h2f((uint16_t)(r.s2[f][j] & 0xFFFFu)), zp = h2f((uint16_t)(r.s2[f][j] >> 16));
    u4_t o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint32_t q[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        q[e] = WBITS == 4 ? (r.w[f][j][0] >> (8 * k + 4 * e)) & 0xFu
                          : (r.w[f][j][k >> 1] >> (16 * (k & 1) + 8 * e)) & 0xFFu;
      const float lo = ((float)q[0] - zp) * scale, hi = ((float)q[1] - zp) * scale;
      o[k] = (uint32_t)f2h(lo) | ((uint32_t)f2h(hi) << 16);
    }
    return __builtin_bit_cast(h8_t, o);
  }

  // Zero-points that dqp rounds, in the (scale, zero) words that a lane looks at
  // in a step (lane group g: weight row + 4 (g / J), MFMA k-step g % J): the OR of
  // their fractions and their maximum, as patterns (1024 is 0x6400, a negative
  // number is larger; a NaN is one either way).
  struct Zp {
    uint32_t frac = 0, top = 0;
    __device__ __forceinline__ void look(uint32_t w) {
      typedef uint16_t us2_t __attribute__((ext_vector_type(2)));
      const _Float16 z = __builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
      frac |= __builtin_bit_cast(uint16_t, (_Float16)__builtin_amdgcn_fracth(z));
      top = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2_t, top),
                                                                   __builtin_bit_cast(us2_t, w)));
    }
    __device__ __forceinline__ bool found() const { return frac != 0 || (top >> 16) > 0x6400u; }
  };
  __device__ __forceinline__ uint32_t zp_word(const lds8* st) const {
    static_assert(!kAnyZp || NF * T::J == 4, "a wave looks at every word of its rows");
    return lds_ld<uint32_t>(st + os + T::SW * 16 * (g / T::J) + 4 * (g % T::J));
  }

  __device__ __forceinline__ h8_t dq(const Raw& r, int f, int j) const {
    u4_t o;
    h2_t nz, sc;
    uint32_t w4 = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = dqp(r, f, j, k, nz, sc, w4);
    return __builtin_bit_cast(h8_t, o);
  }

  // X fragment q of a step's Q = J MT from its stage
  __device__ __forceinline__ h8_t xfrag(const lds8* st, int q) const {
    return lds_ld<h8_t>(st + ox[q / MT] + 16 * (q % MT) * T::XRow);
  }

  __device__ __forceinline__ lds8* next(lds8* st) const {  // the ring's stage after st
    return st + T::kStage == ring + T::D * T::kStage ? ring : st + T::kStage;
  }

  // the segment's first copies
  __device__ __forceinline__ void start() const {
#pragma unroll
    for (int s = 0; s < T::D - 1; ++s) issue(s, ring + s * T::kStage);
  }

  // the segment's K loop, after start(); stores issued since then only make
  // the first wait stricter (copies retire in order among themselves).
  // kAnyZp: a tile with zero-points that dqp rounds is computed again, with dqx:
  // 96 x 7168 x 5120 INT4 21 us, with such zero-points 51.  Without the look / with it,
  // us: 96 x 7168 x 5120 INT4 20.6 / 21.0, 64 x 5120 x 17408 52.3 / 53.9, 128 x 34816 x 5120
  // 78.3 / 81.3; INT8 18.9 / 19.6, 51.5 / 48.2, 255 x 34816 x 5120 133 / 132 (with the copies'
  // LDS addresses taken in one instruction, which gave 0-3% back).  A branch in every
  // step took the first two to 25.2 and 62.8, a fifth wave that looks the first three
  // to 23.1, 57.1 and 98.6.
  __device__ __forceinline__ void run(f4_t (&acc)[NF][MT], int t) const {
    Zp zp;
    loop(acc, t, zp);
    if constexpr (kAnyZp) {
      // the waves' findings, in the one stage that start() does not fill
      typedef __attribute__((address_space(3))) uint32_t lds_u1;
      lds8* const found = ring + (T::D - 1) * T::kStage;
      *(lds_u1*)(found + 4 * wave) = __any(zp.found());
      ring_barrier();
      const u4_t f = lds_ld<u4_t>(found);
      if (__builtin_amdgcn_readfirstlane(f[0] | f[1] | f[2] | f[3])) {
        start();
        loop_any_zp(acc, t);
      }
    }
  }
  __device__ __forceinline__ void loop_any_zp(f4_t (&acc)[NF][MT], int t) const {
    const bool tail = ka + nk * T::KS > ke;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[f][m] = f4_t{0.f, 0.f, 0.f, 0.f};
    lds8 *cur = ring, *far = ring + (T::D - 1) * T::kStage;
    for (int i = 0; i < nk; ++i) {
      Raw raw;
      wait_copies<(T::D - 2) * T::kPer>();
      ring_barrier();
      if (tail && i + 1 == nk) clear_tail(nk - 1, cur, t);
      issue(i + T::D - 1, far);
      load_raw(cur, raw);
#pragma unroll
      for (int j = 0; j < T::J; ++j) {
        h8_t b[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) b[f] = dqx(raw, f, j);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const h8_t a = xfrag(cur, j * MT + m);
#pragma unroll
          for (int f = 0; f < NF; ++f)
            acc[f][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[f], a, acc[f][m], 0, 0, 0);
        }
      }
      far = cur;
      cur = next(cur);
    }
    wait_copies<0>();
    ring_barrier();
  }
  __device__ __forceinline__ void loop(f4_t (&acc)[NF][MT], int t, Zp& zp) const {
    const bool tail = ka + nk * T::KS > ke;
    Raw raw;
    uint32_t zw = 0;
    h8_t a[T::P], b[NF];
    lds8 *cur = ring, *far = ring + (T::D - 1) * T::kStage;
    for (int i = 0; i < nk; ++i) {
      wait_copies<(T::D - 2) * T::kPer>();
      ring_barrier();
      if (tail && i + 1 == nk) clear_tail(nk - 1, cur, t);
      load_raw(cur, raw);
      // the word to look at, read ahead of the X fragments or after them, and looked
      // at in the next step or in this one's last MFMAs, as measured: us of 17 x 7168 x
      // 5120 INT4 next / this step 18.8 / 18.2, INT8 ahead 17.0, after them 17.7; 128 x
      // 5120 x 17408 (48-row tiles) INT4 61.0 / 63.8, INT8 ahead 57.3, after them 55.3
      constexpr bool kTuned = kAnyZp && NF == 1 && MT != 3;
      constexpr bool kAhead = kTuned && WBITS == 8, kLate = kTuned && WBITS == 4;
      uint32_t zn = 0;
      if constexpr (kAhead) zn = zp_word(cur);
#pragma unroll
      for (int q = 0; q < T::P; ++q) a[q] = xfrag(cur, q);
      if constexpr (kAnyZp && !kLate) zp.look(zw);
      if constexpr (kAnyZp) zw = kAhead ? zn : zp_word(cur);
#pragma unroll
      for (int f = 0; f < NF; ++f) b[f] = dq(raw, f, 0);
      const Src sc0 = src(i + T::D - 1, far);
#pragma unroll
      for (int j = 0; j < T::J; ++j) {
        // NF MFMAs of X fragment m, its refill P fragments ahead, a share of
        // the step's copies and of the next B fragments' pairs
        u4_t bn[NF];
        h2_t nz, sc;
        uint32_t w4 = 0;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int q = j * MT + m;
          copies(sc0, [q](int c) { return c * T::Q / T::kPer == q; });
#pragma unroll
          for (int f = 0; f < NF; ++f)
            acc[f][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[f], a[q % T::P], acc[f][m], 0, 0, 0);
          if (q + T::P < T::Q) a[q % T::P] = xfrag(cur, q + T::P);
          if constexpr (kLate) {
            if (q == T::Q - 2) {
              asm volatile("" : "+v"(zw));  // not earlier
              zp.look(zw);
              zw = 0;
            }
          }
#pragma unroll
          for (int e = m * 4 * NF / MT; e < (m + 1) * 4 * NF / MT; ++e) {
            if (j + 1 < T::J) bn[e / 4][e % 4] = dqp(raw, e / 4, j + 1, e % 4, nz, sc, w4);
          }
        }
#pragma unroll
        for (int f = 0; f < NF; ++f) if (j + 1 < T::J) b[f] = __builtin_bit_cast(h8_t, bn[f]);
      }
      far = cur;
      cur = next(cur);
    }
    if constexpr (kAnyZp) zp.look(zw);
    wait_copies<0>();  // no copy may land once the ring is reused
    ring_barrier();
  }
};

// Blocks are dealt to the 8 XCDs in turn: block b of n takes place
// xcd_order(b, n) of an order whose neighbours share an XCD and its L2.
__device__ __forceinline__ int xcd_order(int b, int n) {
  const int x = b & 7, q = n >> 3, r = n & 7;
  return x * q + min(x, r) + (b >> 3);
}

// Tiles are numbered along N first.  Place o of the first dp tiles, visited
// along M first: tiles of the same weights are neighbours.
__device__ __forceinline__ int tile_place(int o, int dp, int ntn) {
  const int rows = dp / ntn, rem = dp % ntn;  // columns below rem hold one tile more
  if (o < rem * (rows + 1)) return o % (rows + 1) * ntn + o / (rows + 1);
  o -= rem * (rows + 1);
  return o % rows * ntn + rem + o / rows;
}

template <int WBITS, int MT, int NF, int MG>
__global__ __launch_bounds__(256 * MG, 2) void gemm_tile_kernel(
    const uint16_t* __restrict__ X, const uint8_t* __restrict__ W,
    const uint32_t* __restrict__ SZ, uint16_t* __restrict__ Y, uint16_t* __restrict__ part, int M,
    int N, int K, int dp, int sk, int U, int unit, int maxseg, int vec) {
  using T = Tile<WBITS, MT, NF, MG>;
  __shared__ __align__(16) uint8_t ring[T::D * T::kStage];
  const int t = threadIdx.x;
  TileSeg<WBITS, MT, NF, MG> sg;
  sg.ring = (lds8*)ring;
  sg.wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int ntm = (M + T::BM - 1) / T::BM, ntn = (N + T::BN - 1) / T::BN;
  const int tiles = ntm * ntn, b = blockIdx.x;
  int64_t lo, hi, TU = 0;
  int w = 0;
  if (b < dp) {
    lo = (int64_t)tile_place(xcd_order(b, dp), dp, ntn) * U;
    hi = lo + U;
  } else {
    w = xcd_order(b - dp, sk);
    TU = (int64_t)(tiles - dp) * U;
    lo = (int64_t)dp * U + sk_lo(w, TU, sk);
    hi = (int64_t)dp * U + sk_lo(w + 1, TU, sk);
  }
  int64_t u = lo, ue = lo;
  int tile = 0, m0 = 0, n0 = 0, ua = 0, ub = 0;
  auto begin = [&]() {  // the segment starting at unit u: its part of a tile, its first copies
    tile = __builtin_amdgcn_readfirstlane((int)(u / U));  // (uniform: kept in SGPRs)
    ue = min(hi, (int64_t)(tile + 1) * U);
    m0 = (tile / ntn) * T::BM;
    n0 = (tile % ntn) * T::BN;
    ua = __builtin_amdgcn_readfirstlane((int)(u - (int64_t)tile * U));
    ub = __builtin_amdgcn_readfirstlane((int)(ue - (int64_t)tile * U));
    sg.ka = ua * unit;
    sg.ke = min(ub * unit, K);
    sg.nk = (sg.ke - sg.ka + T::KS - 1) / T::KS;
    sg.init(X, W, SZ, M, N, K, m0, n0, t);
    sg.start();
  };
  if (u < hi) begin();
  while (u < hi) {
    f4_t acc[NF][MT];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[f][m] = f4_t{0.f, 0.f, 0.f, 0.f};
    sg.run(acc, t);
    // the next segment's first copies go out before this one's results
    const int ctile = tile, cm0 = m0, cn0 = n0;
    const bool whole = ua == 0 && ub == U;
    u = ue;
    if (u < hi) begin();
    const int wc = sg.wave & 3;
    // C fragment f: the lane holds weight rows 4 NF g + 4 f .. + 3 of the
    // wave's 16 NF (4 NF consecutive outputs over its NF fragments) for row
    // col of M-block m
    const int n = cn0 + 16 * NF * wc + 4 * NF * sg.g;
    if (whole) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = cm0 + 16 * (MT * sg.mg + m) + sg.col;
        uint16_t* y = Y + (int64_t)row * N + n;
        if (row < M) {
#pragma unroll
          for (int f = 0; f < NF; f += T::kOut / 4) {
            if (vec && n + 4 * f < N) {
              if constexpr (T::kOut == 8) {
                *reinterpret_cast<u4_t*>(y + 4 * f) =
                    u4_t{cvt_pk_h(acc[f][m][0], acc[f][m][1]), cvt_pk_h(acc[f][m][2], acc[f][m][3]),
                         cvt_pk_h(acc[f + 1][m][0], acc[f + 1][m][1]),
                         cvt_pk_h(acc[f + 1][m][2], acc[f + 1][m][3])};
              } else {
                *reinterpret_cast<u2_t*>(y + 4 * f) =
                    u2_t{cvt_pk_h(acc[f][m][0], acc[f][m][1]), cvt_pk_h(acc[f][m][2], acc[f][m][3])};
              }
            } else if (!vec) {
#pragma unroll
              for (int e = 0; e < T::kOut; ++e)
                if (n + 4 * f + e < N) y[4 * f + e] = f2h(acc[f + e / 4][m][e % 4]);
            }
          }
        }
      }
    } else {
      // fp16 partials in 16-byte pieces, outputs 8 h .. 8 h + 7 of the lane's 4 NF
      // at piece ((wc MTT + M-block) NF / 2 + h) 64 + lane: a store instruction
      // of a wave covers whole lines
      if constexpr (MG == 2) {
        const int tl = ctile - dp, j = w - sk_owner((int64_t)tl * U, TU, sk);
        u4_t* pt = reinterpret_cast<u4_t*>(part + ((int64_t)tl * maxseg + j) * (T::BM * T::BN));
        pt += (wc * MT * MG + MT * sg.mg) * (NF / 2 * 64) + 16 * sg.g + sg.col;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
          for (int h = 0; h < NF / 2; ++h)
            pt[(m * (NF / 2) + h) * 64] = u4_t{
                cvt_pk_h(acc[2 * h][m][0], acc[2 * h][m][1]),
                cvt_pk_h(acc[2 * h][m][2], acc[2 * h][m][3]),
                cvt_pk_h(acc[2 * h + 1][m][0], acc[2 * h + 1][m][1]),
                cvt_pk_h(acc[2 * h + 1][m][2], acc[2 * h + 1][m][3])};
        }
      }
    }
  }
}

// Y = fp16(sum of the segments of each shared tile, in segment order, in
// fp32).  A thread takes a 16-byte piece of every segment and writes that many
// outputs of one row; 2 NF consecutive threads a row of a wave's 16 NF outputs.
// Blocks are placed as the GEMM's are, so that a tile is summed on the XCD that
// wrote its segments.  Read on any XCD, the partials of a following GEMM into the
// same workspace took up to 14 us to be accepted (its kernel's own clock; the less
// it had read before them, the longer), it seems for the copies that the other L2s
// held: 1024 x 4096 x 1024 INT4 36 us, with whole lines per store 35, with the
// placement 27; 512 x 1024 x 1024 INT8 21, 19 and 14; 512 x 17408 x 5120 INT4 108, 107.
template <class T>
__global__ __launch_bounds__(256) void gemm_tile_reduce_kernel(const uint16_t* __restrict__ part,
                                                               uint16_t* __restrict__ Y, int M,
                                                               int N, int dp, int sk, int U,
                                                               int maxseg, int vec) {
  constexpr int NF = T::BN / 64, MTT = T::BM / 16, E = T::kOut, kPerTile = T::BM * T::BN / E;
  const int64_t gt = (int64_t)xcd_order(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  const int ntm = (M + T::BM - 1) / T::BM, ntn = (N + T::BN - 1) / T::BN;
  const int tl = (int)(gt / kPerTile), x = (int)(gt % kPerTile);
  if (tl >= ntm * ntn - dp) return;
  const int64_t TU = (int64_t)(ntm * ntn - dp) * U;
  const int w0 = sk_owner((int64_t)tl * U, TU, sk), w1 = sk_owner((int64_t)tl * U + U - 1, TU, sk);
  const int nseg = w1 - w0 + 1;
  if (nseg == 1) return;  // computed whole: written by the GEMM
  const int tile = dp + tl;
  constexpr int G = 2 * NF;  // threads of a row of a wave's 16 NF outputs
  const int q = x % G, col = x / G % 16, wm = x / (16 * G);  // wm = wc MTT + M-block
  const int row = (tile / ntn) * T::BM + 16 * (wm % MTT) + col;
  const int n = (tile % ntn) * T::BN + 16 * NF * (wm / MTT) + E * q;
  if (row >= M || n >= N) return;
  const u4_t* p = reinterpret_cast<const u4_t*>(part + (int64_t)tl * maxseg * (T::BM * T::BN)) +
                  (wm * (NF / 2) + q % (NF / 2)) * 64 + 16 * (q / (NF / 2)) + col;
  float v[E];
  auto add = [&](u4_t x, bool first) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float lo = h2f((uint16_t)(x[i] & 0xFFFFu)), hi = h2f((uint16_t)(x[i] >> 16));
      v[2 * i] = first ? lo : v[2 * i] + lo;
      v[2 * i + 1] = first ? hi : v[2 * i + 1] + hi;
    }
  };
  add(p[0], true);
  for (int s0 = 1; s0 < nseg; s0 += 4) {  // up to 4 segments in flight, added in order
    u4_t x[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = p[(int64_t)min(s0 + s, nseg - 1) * kPerTile];
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (s0 + s < nseg) add(x[s], false);
  }
  uint16_t* y = Y + (int64_t)row * N + n;
  if (vec) {
    *reinterpret_cast<u4_t*>(y) = u4_t{cvt_pk_h(v[0], v[1]), cvt_pk_h(v[2], v[3]),
                                       cvt_pk_h(v[4], v[5]), cvt_pk_h(v[6], v[7])};
  } else {
#pragma unroll
    for (int l = 0; l < E; ++l)
      if (n + l < N) y[l] = f2h(v[l]);
  }
}

// ---------------------------------------------------------------------
// Skinny GEMM for 2 <= M <= 16 rows (batched decode) through an LDS ring.
// A workgroup (4 waves) owns 64 weight rows (16 per wave) and a range of K
// steps; each step stages, by global->LDS copies, 128 bytes of every weight
// row (8 rows x 128 B per copy instruction: whole cache lines, which reads
// the weights at ~5.6-6 TB/s where 16 rows x 64 B per instruction -- the
// MFMA B-fragment layout loaded straight into registers -- measured
// 4.4-4.9 TB/s), the rows' (scale, zero) words and the matching slice of the
// MR activation rows.  kSkStages ring stages, stages - 1 steps in flight
// (kSkDeepStages stages when the grid has at most one workgroup per CU, whose
// LDS then allows it); one barrier per step
// (the ring of gemm_tile_kernel).  Per step each wave runs KS/32 MFMA
// 16x16x32 tiles: B = its 16 weight rows dequantised from LDS (skinny_b),
// A = the activation rows (in the k labels below), C = 16 activation
// rows x 16 weight rows.  Lane group g of MFMA j holds the k labels
// k0 + (KS/4) g + 8 j .. +7 in both operands, so each lane reads its 32
// weight bytes of the step with two 16-byte LDS reads.  The 16-byte pieces
// of a row sit in LDS slot piece ^ (row & 7) (bank spread).
// Split-K (S > 1): the workgroup covers steps [s kps, (s+1) kps) and writes
// fp32 partials part[s][m][n]; gemm_skinny_reduce_kernel sums them in order.
// SiLU epilogue (SILU, unsplit, M <= 8; W = [gate; up] over 2I rows): tile t
// holds gate rows 32t .. 32t+31 (waves 0, 1) and the up rows I + 32t ..
// of the same indices (waves 2, 3); its fp16-rounded results meet in LDS
// and each of the 256 threads finishes one (activation row, element):
// y[m][32t + i] = fp16(FWHT32(silu(g) * u)) with the butterflies across 32
// lanes -- the arithmetic of silu_kernel<true>.  A weight row's MFMA chain
// does not depend on the tile it sits in, so the result equals the unsplit
// GEMM followed by that kernel bit for bit.
constexpr int kSkTile = 64;   // weight rows per workgroup
constexpr int kSkStages = 3;      // ring stages (stages - 1 steps in flight)
// at most one workgroup per CU; against 3 stages the batch-8 step measured
// -19 us with 4, +44 us with 5 and +100 us with 6
constexpr int kSkDeepStages = 4;
constexpr int kSkMaxSplits = 8;

template <int WBITS, int MR>
struct SkRing {
  static constexpr int kKS = 1024 / WBITS;          // k per step: 128 B of each weight row
  static constexpr int kSteps = kKS / 32;           // MFMA k-steps per step
  static constexpr int kW = kSkTile * 128;          // weights: 8 KB
  static constexpr int kSRow = WBITS == 16 ? 0 : (kKS / 32) * 4;  // (scale, zero) bytes per row
  static constexpr int kS = kSkTile * kSRow;        // 2 KB (INT4) / 1 KB (INT8) / 0
  static constexpr int kXRow = kKS * 2;             // activation bytes per row per step
  static constexpr int kX = MR * kXRow;
  static constexpr int kStage = kW + kS + kX;
  static constexpr bool kX16 = kX >= 4096;          // activation as 1 KB copies (else 256 B)
  static constexpr int kCX = kX16 ? kX / 4096 : kX / 1024;  // activation copies per wave
  static constexpr int kCS = WBITS == 4 ? 2 : WBITS == 8 ? 1 : 0;  // scale copies (256 B) per wave
  static constexpr int kPer = 2 + kCS + kCX;        // copies per wave per step
  static_assert(kX % (kX16 ? 4096 : 1024) == 0 && kCX >= 1, "activation copies must split evenly");
};

// Per-lane source offsets of the copies of one ring step (bytes from the
// step's uniform bases W + 128 kb, SZ + kb * words, X + kb * kKS; rows past N /
// M clamped to the last one), computed once per workgroup: a step's copies
// then cost no vector arithmetic.  Tile rows 0..31 are weight rows n0 ..,
// tile rows 32..63 are n1 .. (n1 = n0 + 32 except in the SiLU map).
template <int WBITS, int MR>
struct SkCopy {
  using R = SkRing<WBITS, MR>;
  static constexpr int kWpr = R::kSRow / 4;  // scale words per row per step
  uint32_t wo[2], so[R::kCS > 0 ? R::kCS : 1], xo[R::kCX];

  __device__ __forceinline__ void init(int M, int N, int K, int n0, int n1, int wave, int lane) {
    const uint32_t row_bytes = (uint32_t)K * WBITS / 8;
    auto row = [&](int r) { return min(r < 32 ? n0 + r : n1 + (r - 32), N - 1); };
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // weights: copy c covers tile rows 8c .. 8c+7
      const int c = 2 * wave + i, r = 8 * c + (lane >> 3);
      const int piece = (lane & 7) ^ (r & 7);
      wo[i] = (uint32_t)row(r) * row_bytes + 16 * piece;
    }
    if constexpr (WBITS != 16) {
      constexpr int rpc = 64 / kWpr;  // rows per 256-byte copy
#pragma unroll
      for (int i = 0; i < R::kCS; ++i) {
        const int c = R::kCS * wave + i, r = rpc * c + lane / kWpr;
        so[i] = 4u * ((uint32_t)row(r) * (uint32_t)(K / 32) + lane % kWpr);
      }
    }
#pragma unroll
    for (int i = 0; i < R::kCX; ++i) {
      const int c = R::kCX * wave + i;
      if constexpr (R::kX16) {  // 1 KB per copy, 16 bytes per lane
        const int off = 1024 * c + 16 * lane;
        const int r = off / R::kXRow, slot = (off % R::kXRow) / 16;
        xo[i] = 2u * ((uint32_t)min(r, M - 1) * K + 8 * (slot ^ (r & 7)));
      } else {  // 256 B per copy, 4 bytes per lane
        const int off = 256 * c + 4 * lane;
        const int r = off / R::kXRow, slot = (off % R::kXRow) / 16;
        xo[i] = 2u * ((uint32_t)min(r, M - 1) * K + 8 * (slot ^ (r & 7)) + 2 * (lane & 3));
      }
    }
  }

  // step kb of the workgroup's weight rows, scale words and activation rows
  // into ring stage `stage`
  __device__ __forceinline__ void issue(lds8* stage, const uint16_t* __restrict__ X,
                                        const uint8_t* __restrict__ W,
                                        const uint32_t* __restrict__ SZ, int kb,
                                        int wave) const {
    const uint8_t* wb = W + (int64_t)kb * 128;
#pragma unroll
    for (int i = 0; i < 2; ++i) copy16s(wb, wo[i], stage + 1024 * (2 * wave + i));
    if constexpr (WBITS != 16) {
      const uint32_t* sb = SZ + (int64_t)kb * kWpr;
#pragma unroll
      for (int i = 0; i < R::kCS; ++i) copy4s(sb, so[i], stage + R::kW + 256 * (R::kCS * wave + i));
    }
    const uint16_t* xs = X + (int64_t)kb * R::kKS;
#pragma unroll
    for (int i = 0; i < R::kCX; ++i) {
      const int c = R::kCX * wave + i;
      if constexpr (R::kX16) copy16s(xs, xo[i], stage + R::kW + R::kS + 1024 * c);
      else copy4s(xs, xo[i], stage + R::kW + R::kS + 256 * c);
    }
  }
};

// The K loop of one workgroup.  The ring stage of a step is a template
// argument (the loop is unrolled by the ring depth), so that the LDS reads
// address each stage through their immediate offset from per-lane offsets
// computed once.
template <int WBITS, int MR, int D>
struct SkLoop {
  using R = SkRing<WBITS, MR>;
  static_assert(D >= 3 && (D - 2) * R::kPer <= 63, "ring depth: copy waits fit vmcnt");
  lds8* ring;
  const uint16_t* X;
  const uint8_t* W;
  const uint32_t* SZ;
  SkCopy<WBITS, MR> cp;
  int kb0, nk, wave;
  uint32_t ob0, ob1, osw, ox[R::kSteps];  // per-lane LDS offsets within a stage
  f4_t acc;

  template <int ST>
  __device__ __forceinline__ void step(int i) {
    wait_copies<(D - 2) * R::kPer>();  // this wave's copies of step i have landed
    ring_barrier();                    // every wave's; every wave is done with step i-1
    cp.issue(ring + ((ST + D - 1) % D) * R::kStage, X, W, SZ, kb0 + min(i + D - 1, nk - 1),
             wave);
    const lds8* st = ring + ST * R::kStage;
    const u4_t b0 = lds_ld<u4_t>(st + ob0);
    const u4_t b1 = lds_ld<u4_t>(st + ob1);
    uint32_t sw0 = 0u, sw1 = 0u;
    if constexpr (WBITS == 4) {  // blocks 2g, 2g+1 of the step
      const u2_t v = lds_ld<u2_t>(st + osw);
      sw0 = v[0];
      sw1 = v[1];
    } else if constexpr (WBITS == 8) {  // block g
      sw0 = lds_ld<uint32_t>(st + osw);
    }
#pragma unroll
    for (int j = 0; j < R::kSteps; ++j) {
      // activation piece holding k labels k0 + (KS/4) g + 8 j .. +7
      const h8_t a = lds_ld<h8_t>(st + ox[j]);
      h8_t b;
      if constexpr (WBITS == 4) b = skinny_b<4>(j < 4 ? b0 : b1, j < 4 ? sw0 : sw1, j & 3);
      else if constexpr (WBITS == 8) b = skinny_b<8>(j < 2 ? b0 : b1, sw0, j & 1);
      else b = __builtin_bit_cast(h8_t, j == 0 ? b0 : b1);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc, 0, 0, 0);
    }
  }

  // steps i, i+1, ... from ring stage ST to D-1 (one round of the ring)
  template <int ST>
  __device__ __forceinline__ void round_from(int i) {
    step<ST>(i);
    if constexpr (ST + 1 < D) round_from<ST + 1>(i + 1);
  }
  // the last nk - i < D steps, from stage 0
  template <int ST>
  __device__ __forceinline__ void tail_from(int i) {
    if (i < nk) {
      step<ST>(i);
      if constexpr (ST + 2 < D) tail_from<ST + 1>(i + 1);
    }
  }

  __device__ __forceinline__ void run() {
#pragma unroll
    for (int s = 0; s < D - 1; ++s)
      cp.issue(ring + s * R::kStage, X, W, SZ, kb0 + min(s, nk - 1), wave);
    int i = 0;
    for (; i + D <= nk; i += D) round_from<0>(i);
    tail_from<0>(i);
  }
};

// Balanced SiLU tail (SILU, tail.part != NULL): units 0 .. umain-1 (whole
// rounds of 256) run one workgroup each over all of K; each of the other
// units is cut along K into S pieces of kps steps (workgroups umain + u' S +
// s), which leave fp32 partials and count in on the unit's counter; the last
// piece to arrive sums the S partials in piece order and finishes the unit.
// Without it the units past the last whole round (544 = 2 x 256 + 32 at I =
// 17408) ran as a third workgroup on 32 CUs, which then finished a whole
// unit after the rest.
struct SkTail {
  float* part = nullptr;  // [tail units][S][8 rows][64 tile rows] fp32
  int* cnt = nullptr;     // [tail units] arrivals, zero before and after a launch
  int umain = 0, S = 1, kps = 0;
};

// Device-coherent 32-bit load and store (agent scope: past the caches of the
// other XCDs), for partials that workgroups hand to each other in a launch.
__device__ __forceinline__ float ld_agent(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int WBITS, int MR, bool SILU, int D = kSkStages>
__global__ __launch_bounds__(256) void gemm_skinny_kernel(const uint16_t* __restrict__ X,
                                                          const uint8_t* __restrict__ W,
                                                          const uint32_t* __restrict__ SZ,
                                                          uint16_t* __restrict__ Y,
                                                          float* __restrict__ part, int M, int N,
                                                          int K, int ntiles, int kps, int silu_I,
                                                          SkTail tail) {
  static_assert(!SILU || MR == 8, "the SiLU epilogue maps 8 rows x 32 elements to 256 threads");
  using R = SkRing<WBITS, MR>;
  __shared__ __align__(16) uint8_t ring[D * R::kStage];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tile = blockIdx.x % ntiles, sp = blockIdx.x / ntiles;
  // SiLU tail piece: unit tile, piece sp of tail.S (workgroup-uniform)
  const bool piece = SILU && tail.part && (int)blockIdx.x >= tail.umain;
  if (piece) {
    const int j = (int)blockIdx.x - tail.umain;
    tile = tail.umain + j / tail.S;
    sp = j % tail.S;
    kps = tail.kps;
  }
  const int n0 = SILU ? 32 * tile : tile * kSkTile;
  const int n1 = SILU ? silu_I + 32 * tile : n0 + 32;
  const int kt = K / R::kKS;
  const int col = lane & 15, g = lane >> 4;
  const int wrow = 16 * wave + col;                   // this lane's weight row in the tile
  const int xr = col % MR;                            // activation row (rows >= MR: duplicates)

  SkLoop<WBITS, MR, D> lp;
  lp.ring = (lds8*)ring;
  lp.X = X;
  lp.W = W;
  lp.SZ = SZ;
  lp.kb0 = sp * kps;
  lp.nk = min(kt - lp.kb0, kps);  // >= 1 (host)
  lp.wave = wave;
  lp.cp.init(M, N, K, n0, n1, wave, lane);
  // weight bytes [32 g, 32 g + 32) of row wrow: pieces 2g, 2g+1
  lp.ob0 = 128 * wrow + 16 * ((2 * g) ^ (wrow & 7));
  lp.ob1 = 128 * wrow + 16 * ((2 * g + 1) ^ (wrow & 7));
  lp.osw = R::kW + R::kSRow * wrow + (WBITS == 4 ? 8 * g : 4 * g);
#pragma unroll
  for (int j = 0; j < R::kSteps; ++j)
    lp.ox[j] = R::kW + R::kS + R::kXRow * xr + 16 * ((R::kSteps * g + j) ^ (xr & 7));
  lp.acc = f4_t{0.f, 0.f, 0.f, 0.f};
  lp.run();
  const f4_t acc = lp.acc;
  wait_copies<0>();  // no copy into LDS outlives the workgroup
  // C: lane holds activation rows 4g + r (rows >= MR repeat rows < MR), tile
  // row 16 wave + col
  if constexpr (SILU) {
#pragma clang fp contract(off)  // g / (1 + e^-g) * u in separately rounded steps
    __syncthreads();  // every wave is done with the ring, which now holds
    float* us = reinterpret_cast<float*>(ring);  // us[m][tile row], 8 x 64
    const int m = threadIdx.x >> 5, i = threadIdx.x & 31;
    float gv, uv;
    if (piece) {
      // partials out as device-coherent stores, which every wave waits for
      // before thread 0 counts the piece in; the last of the unit's S pieces
      // resets the counter for the next launch and sums the partials
      const int tu = tile - tail.umain;
      float* tp = tail.part + ((int64_t)tu * tail.S + sp) * 512;
      if (g < 2) {
#pragma unroll
        for (int r = 0; r < 4; ++r) st_agent(tp + (4 * g + r) * 64 + 16 * wave + col, acc[r]);
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      int* last = reinterpret_cast<int*>(us + 512);
      if (threadIdx.x == 0) {
        int* c = tail.cnt + tu;
        const int prev = __hip_atomic_fetch_add(c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *last = prev == tail.S - 1;
        if (prev == tail.S - 1) __hip_atomic_store(c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      if (*last == 0) return;
      // the split reduce's arithmetic: fp32 sums in piece order, one fp16 rounding
      const float* tb = tail.part + (int64_t)tu * tail.S * 512 + m * 64 + i;
      float ga = ld_agent(tb), ua = ld_agent(tb + 32);
      for (int z = 1; z < tail.S; ++z) {
        ga += ld_agent(tb + z * 512);
        ua += ld_agent(tb + z * 512 + 32);
      }
      gv = h2f(f2h(ga));
      uv = h2f(f2h(ua));
    } else {
      if (g < 2) {
#pragma unroll
        for (int r = 0; r < 4; ++r) us[(4 * g + r) * 64 + 16 * wave + col] = h2f(f2h(acc[r]));
      }
      __syncthreads();
      gv = us[m * 64 + i];
      uv = us[m * 64 + 32 + i];
    }
    float v = gv / (1.0f + expf(-gv)) * uv;
#pragma unroll
    for (int bit = 1; bit <= 16; bit <<= 1) {
      const float o = __shfl_xor(v, bit);
      v = (i & bit) ? o - v : v + o;
    }
    v *= kInvSqrt32;
    if (m < M) Y[(int64_t)m * silu_I + 32 * tile + i] = f2h(v);
    return;
  }
  const int n = n0 + 16 * wave + col;
  if (n < N) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 4 * g + r;
      if (m < M) {
        if (part) part[((int64_t)sp * M + m) * N + n] = acc[r];
        else Y[(int64_t)m * N + n] = f2h(acc[r]);
      }
    }
  }
}

// Y[m][n] = fp16(sum over s of part[s][m][n]), in split order.
__global__ __launch_bounds__(256) void gemm_skinny_reduce_kernel(const float* __restrict__ part,
                                                                 uint16_t* __restrict__ Y, int M,
                                                                 int N, int S) {
  const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (n >= N) return;
  const int64_t plane = (int64_t)M * N;
  const float* p = part + (int64_t)m * N + n;
  float v = p[0];
  for (int z = 1; z < S; ++z) v += p[z * plane];
  Y[(int64_t)m * N + n] = f2h(v);
}

// Split sum fused with the SiLU gate of a gate/up projection (N = 2I
// columns: gate 0..I-1, up I..2I-1), four lanes per 32-column chunk: lane q
// of chunk c of row m sums gate and up columns 32c + 8q .. + 7 over the
// splits in order and rounds each sum to fp16 (what gemm_skinny_reduce_kernel
// stores), applies silu(g) * u as silu_kernel<true> does, then runs the
// butterfly stages 1, 2, 4 of the FWHT-32 in registers and stages 8 and 16
// with the lanes q ^ 1 and q ^ 2 -- the stage order and (a + b, a - b) pairs
// of fwht32, so the fp16 output is the same bit for bit.  (One thread per
// chunk left 72 waves on the chip for I = 17408 and took 6.2 us.)
__device__ __forceinline__ void skinny_sum8(const float* __restrict__ p, int64_t plane, int S,
                                            float* v) {
  const float4* q = reinterpret_cast<const float4*>(p);
  float4 t0 = q[0], t1 = q[1];
  v[0] = t0.x, v[1] = t0.y, v[2] = t0.z, v[3] = t0.w;
  v[4] = t1.x, v[5] = t1.y, v[6] = t1.z, v[7] = t1.w;
  for (int z = 1; z < S; ++z) {
    q = reinterpret_cast<const float4*>(p + z * plane);
    t0 = q[0];
    t1 = q[1];
    v[0] += t0.x, v[1] += t0.y, v[2] += t0.z, v[3] += t0.w;
    v[4] += t1.x, v[5] += t1.y, v[6] += t1.z, v[7] += t1.w;
  }
}

constexpr int kSiluRedThreads = 256;
__global__ __launch_bounds__(kSiluRedThreads) void gemm_skinny_reduce_silu_kernel(
    const float* __restrict__ part, uint16_t* __restrict__ Y, int M, int I, int S) {
#pragma clang fp contract(off)  // g / (1 + e^-g) * u in separately rounded steps
  const int tid = blockIdx.x * kSiluRedThreads + threadIdx.x, m = blockIdx.y;
  const int c = tid >> 2, q = tid & 3;
  // lanes past the row read chunk 0 and store nothing, but take part in the
  // cross-lane stages of their chunk group
  const bool live = c * 32 < I;
  const int64_t plane = (int64_t)M * 2 * I;
  const float* pg = part + (int64_t)m * 2 * I + (live ? c : 0) * 32 + 8 * q;
  float a[8], b[8];
  skinny_sum8(pg, plane, S, a);
  skinny_sum8(pg + I, plane, S, b);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float g = h2f(f2h(a[i])), u = h2f(f2h(b[i]));
    a[i] = g / (1.0f + expf(-g)) * u;
  }
#pragma unroll
  for (int step = 1; step < 8; step <<= 1) {
#pragma unroll
    for (int i = 0; i < 8; i += 2 * step) {
#pragma unroll
      for (int j = i; j < i + step; ++j) {
        const float x = a[j], y = a[j + step];
        a[j] = x + y;
        a[j + step] = x - y;
      }
    }
  }
#pragma unroll
  for (int lm = 1; lm <= 2; lm <<= 1) {  // stages 8 and 16: partner lane q ^ lm
    const bool upper = (q & lm) != 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float o = __shfl_xor(a[j], lm);
      a[j] = upper ? o - a[j] : a[j] + o;
    }
  }
  if (!live) return;
  u4_t w;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    w[k] = (uint32_t)f2h(a[2 * k] * kInvSqrt32) | ((uint32_t)f2h(a[2 * k + 1] * kInvSqrt32) << 16);
  *reinterpret_cast<u4_t*>(Y + (int64_t)m * I + c * 32 + 8 * q) = w;
}

}  // namespace

bool gemm_skinny_ok(int64_t M, int64_t N, int64_t K, int wbits) {
  const int64_t ks = 1024 / (wbits == 4 ? 4 : wbits == 8 ? 8 : 16);  // k per ring step
  // the copies address the weights with 32-bit byte offsets
  return M >= 2 && M <= 16 && K % ks == 0 && N * K * wbits / 8 < ((int64_t)1 << 32);
}

// Split count of the skinny ring.  A CU streams its workgroups' weight
// tiles at about the same rate whether it holds one or several, so the step
// ends with the most-loaded CU: cost(S) = ceil(ntiles S / CUs) * kps + S,
// the last term charging each split its fp32 partials and share of the
// reduce.  S runs over 1..8 with at most 8 workgroups per CU (past that the
// quantisation the model prices is smoothed out and splitting loses: FP16
// 151936 x 5120 at M = 8, 2 splits 279 us against 268); ties go to more
// splits.  Measured at M = 8 (us, chosen / unsplit / old rule): INT4 o
// 5120 x 5120 3 splits 10.5 / 17.1 / 12.1, qkv 7168 x 5120 2: 12.9 / 17.8,
// gate_up 34816 x 5120 3: 34.8 / 39.4, down 5120 x 17408 3: 23.1 / 51.6 /
// 23.2; INT8 o 3: 11.5 / 18.7 / 13.1, qkv 2: 14.0 / 19.3 / 17.3, down 3:
// 25.7 / 55.1 / 29.9.  S > 1 needs S * M * N fp32 of workspace.
int skinny_splits(int64_t M, int64_t N, int64_t K, int wbits, size_t ws_bytes) {
  constexpr int64_t kCUs = 256;  // MI355X
  const int64_t ntiles = (N + kSkTile - 1) / kSkTile;
  const int64_t kt = K / (1024 / wbits);
  int64_t S = 1, best = INT64_MAX;
  for (int64_t s = 1; s <= std::min<int64_t>(kSkMaxSplits, kt); ++s) {
    const int64_t kps = (kt + s - 1) / s;
    const int64_t se = (kt + kps - 1) / kps;  // splits left non-empty
    if (se > 1 && ntiles * se > 8 * kCUs) break;
    const int64_t c = (ntiles * se + kCUs - 1) / kCUs * kps + se;
    if (c <= best) best = c, S = se;
  }
  if (const int v = tuning().skinny_splits.load()) S = v;  // measurement override (r4q_tune)
  if (S < 2) return 1;
  // every split non-empty
  const int64_t kps = (kt + S - 1) / S;
  S = (kt + kps - 1) / kps;
  if ((size_t)S * M * N * 4 > ws_bytes) return 1;
  return (int)S;
}

size_t skinny_ws_bytes(int64_t M, int64_t N, int64_t K, int wbits) {
  const int S = skinny_splits(M, N, K, wbits, SIZE_MAX);
  return S > 1 ? (size_t)S * M * N * 4 : 0;
}

namespace {
size_t skinny_tail_part_bytes(int64_t T, int64_t S) {
  return ((size_t)T * S * 512 * 4 + 255) & ~(size_t)255;
}
size_t skinny_tail_cnt_bytes(int64_t T) { return ((size_t)T * 4 + 255) & ~(size_t)255; }

// Tail plan of the unsplit SiLU GEMM (see SkTail) for I / 32 units over 256
// CUs: the units past the last whole round of 256, each cut into S pieces
// of kps K steps with S about 128 / tail units (measured at 32 tail units:
// 4 pieces each 3.845 ms per batch-8 step, 2 / 3 / 8 / 16 pieces 3.935 /
// 3.877 / 3.852 / 3.892 ms).  No tail
// (part == NULL) without a workspace, below one round, on whole rounds, or
// when a unit would not be cut.  Workspace: the counters, then the partials.
SkTail skinny_tail_plan(int64_t I, int64_t K, int wbits, void* ws) {
  SkTail t;
  const int64_t units = I / 32, kt = K / (1024 / wbits);
  const int64_t T = units % 256;
  if (!ws || units <= 256 || T == 0) return t;
  const int64_t S0 = std::min<int64_t>(kt, std::max<int64_t>(1, 128 / T));
  const int64_t kps = (kt + S0 - 1) / S0, S = (kt + kps - 1) / kps;  // every piece non-empty
  if (S < 2) return t;
  t.umain = (int)(units - T);
  t.S = (int)S;
  t.kps = (int)kps;
  t.cnt = static_cast<int*>(ws);  // counters first: the same place for every width
  t.part = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + skinny_tail_cnt_bytes(T));
  return t;
}

// silu_I > 0: N = 2 silu_I gate/up columns into y (M x silu_I) gated by
// SiLU + FWHT-32: split (S > 1) and reduced by
// gemm_skinny_reduce_silu_kernel, or unsplit (S == 1, M <= 8: checked by the
// caller) with the gate in the GEMM's epilogue.  keep_part: no reduce, the
// S fp32 partial planes stay in ws (S > 1) for the consumer to sum.
int skinny_run(const void* x, const void* w, const void* sz, void* y, int64_t M, int64_t N,
               int64_t K, int wbits, hipStream_t st, void* ws, size_t ws_bytes, int64_t silu_I,
               bool keep_part = false, void* tail_ws = nullptr) {
  const auto* xp = static_cast<const uint16_t*>(x);
  const auto* wp = static_cast<const uint8_t*>(w);
  const auto* sp = static_cast<const uint32_t*>(sz);
  auto* yp = static_cast<uint16_t*>(y);
  const int S = skinny_splits(M, N, K, wbits, ws ? ws_bytes : 0);
  const int64_t ntiles = (N + kSkTile - 1) / kSkTile;
  const int64_t kt = K / (1024 / wbits);
  const int kps = (int)((kt + S - 1) / S);
  float* part = S > 1 ? static_cast<float*>(ws) : nullptr;
  const dim3 grid((unsigned)(ntiles * S));
  const bool m8 = M <= 8;
  if (silu_I > 0 && S == 1) {  // unsplit: the SiLU gate in the epilogue
    R4Q_REQUIRE(M <= 8 && silu_I % 32 == 0 && N == 2 * silu_I,
                "gate_up_silu: the unsplit epilogue takes at most 8 rows (M=%lld)", (long long)M);
    const SkTail tl = skinny_tail_plan(silu_I, K, wbits, tail_ws);
    const int64_t units = silu_I / 32;
    const int64_t wgs = tl.part ? tl.umain + (units - tl.umain) * tl.S : units;
#define R4Q_SKINNY_SILU(WB)                                                                      \
  hipLaunchKernelGGL((gemm_skinny_kernel<WB, 8, true>), dim3((unsigned)wgs), dim3(256), 0, st,   \
                     xp, wp, sp, yp, nullptr, (int)M, (int)N, (int)K, (int)units, kps,           \
                     (int)silu_I, tl)
    if (wbits == 4) R4Q_SKINNY_SILU(4);
    else if (wbits == 8) R4Q_SKINNY_SILU(8);
    else R4Q_SKINNY_SILU(16);
#undef R4Q_SKINNY_SILU
    return launch_status("gemm_skinny_silu");
  }
  const bool deep = ntiles * S <= 256;  // one workgroup per CU: LDS for a deeper ring
#define R4Q_SKINNY_D(WB, MRR, DD)                                                              \
  hipLaunchKernelGGL((gemm_skinny_kernel<WB, MRR, false, DD>), grid, dim3(256), 0, st, xp, wp, \
                     sp, yp, part, (int)M, (int)N, (int)K, (int)ntiles, kps, 0, SkTail{})
#define R4Q_SKINNY(WB, MRR)                                                                    \
  if (deep) R4Q_SKINNY_D(WB, MRR, kSkDeepStages);                                            \
  else R4Q_SKINNY_D(WB, MRR, kSkStages)
  switch (wbits) {
    case 4:
      if (m8) R4Q_SKINNY(4, 8);
      else R4Q_SKINNY(4, 16);
      break;
    case 8:
      if (m8) R4Q_SKINNY(8, 8);
      else R4Q_SKINNY(8, 16);
      break;
    default:
      if (m8) R4Q_SKINNY(16, 8);
      else R4Q_SKINNY(16, 16);
  }
#undef R4Q_SKINNY
#undef R4Q_SKINNY_D
  R4Q_TRY(launch_status("gemm_skinny"));
  if (keep_part) return R4Q_OK;
  if (silu_I > 0) {
    hipLaunchKernelGGL(gemm_skinny_reduce_silu_kernel,
                       dim3((unsigned)((silu_I / 8 + kSiluRedThreads - 1) / kSiluRedThreads),
                            (unsigned)M),
                       dim3(kSiluRedThreads), 0, st, part, yp, (int)M, (int)silu_I, S);
    R4Q_TRY(launch_status("gemm_skinny_reduce_silu"));
  } else if (S > 1) {
    hipLaunchKernelGGL(gemm_skinny_reduce_kernel, dim3((unsigned)((N + 255) / 256), (unsigned)M),
                       dim3(256), 0, st, part, yp, (int)M, (int)N, S);
    R4Q_TRY(launch_status("gemm_skinny_reduce"));
  }
  return R4Q_OK;
}
}  // namespace

int gemm_skinny_launch(const void* x, const void* w, const void* sz, void* y, int64_t M,
                       int64_t N, int64_t K, int wbits, hipStream_t st, void* ws,
                       size_t ws_bytes) {
  return skinny_run(x, w, sz, y, M, N, K, wbits, st, ws, ws_bytes, 0);
}

int gemm_skinny_part_launch(const void* x, const void* w, const void* sz, void* y, int64_t M,
                            int64_t N, int64_t K, int wbits, hipStream_t st, void* ws,
                            size_t ws_bytes, int* S) {
  R4Q_REQUIRE(gemm_skinny_ok(M, N, K, wbits), "skinny GEMM: unsupported shape");
  *S = skinny_splits(M, N, K, wbits, ws ? ws_bytes : 0);
  return skinny_run(x, w, sz, y, M, N, K, wbits, st, ws, ws_bytes, 0, true);
}

bool gemm_skinny_silu_ok(int64_t M, int64_t I, int64_t K, int wbits, size_t ws_bytes) {
  return gemm_skinny_ok(M, 2 * I, K, wbits) && I > 0 && I % 32 == 0 &&
         (M <= 8 || skinny_splits(M, 2 * I, K, wbits, ws_bytes) > 1);
}

int gemm_skinny_silu_launch(const void* x, const void* w, const void* sz, void* y, int64_t M,
                            int64_t I, int64_t K, int wbits, hipStream_t st, void* ws,
                            size_t ws_bytes) {
  R4Q_REQUIRE(gemm_skinny_silu_ok(M, I, K, wbits, ws ? ws_bytes : 0),
              "gate_up_silu: needs I %% 32 == 0, and above 8 rows a workspace that splits K");
  return skinny_run(x, w, sz, y, M, 2 * I, K, wbits, st, ws, ws_bytes, I);
}

size_t skinny_silu_tail_bytes(int64_t I, int64_t K, int wbits) {
  int dummy = 0;
  const SkTail t = skinny_tail_plan(I, K, wbits, &dummy);
  if (!t.part) return 0;
  const int64_t T = I / 32 - t.umain;
  return skinny_tail_cnt_bytes(T) + skinny_tail_part_bytes(T, t.S);
}

size_t skinny_silu_tail_cnt_bytes(int64_t I) {
  const int64_t units = I / 32;
  return units > 256 && units % 256 ? skinny_tail_cnt_bytes(units % 256) : 0;
}

int gemm_skinny_silu_tail_launch(const void* x, const void* w, const void* sz, void* y, int64_t M,
                                 int64_t I, int64_t K, int wbits, hipStream_t st, void* tail_ws) {
  R4Q_REQUIRE(M <= 8 && gemm_skinny_silu_ok(M, I, K, wbits, 0),
              "gate_up_silu: the unsplit epilogue takes at most 8 rows and I %% 32 == 0");
  return skinny_run(x, w, sz, y, M, 2 * I, K, wbits, st, nullptr, 0, I, false, tail_ws);
}

// Work split of gemm_tile_kernel: dp whole tiles, then sk stream-K workgroups
// over the other tiles.
struct TilePlan {
  int dp = 0, sk = 0, U = 1, maxseg = 1;
  size_t ws = 0;  // partials: (tiles - dp) * maxseg tiles
};

// MI355X compute units.  Their LDS holds one workgroup of a 256 x 256 tile, two of
// the others.
constexpr int kTileCUs = 256;

// Host restatement of sk_lo / sk_owner (the kernel's unit split).
static int64_t host_sk_lo(int64_t w, int64_t TU, int64_t sk) { return w * TU / sk; }
static int64_t host_sk_owner(int64_t u, int64_t TU, int64_t sk) {
  int64_t w = u * sk / TU;
  while (w + 1 < sk && host_sk_lo(w + 1, TU, sk) <= u) ++w;
  while (w > 0 && host_sk_lo(w, TU, sk) > u) --w;
  return w;
}

// dp / sk split of `tiles` tiles of U units each (see tile_plan), with
// partials of tile_bytes per (shared tile, segment).
static TilePlan split_plan(int64_t tiles, int U, int64_t tile_bytes, size_t ws_bytes) {
  // Every CU gets the same number of K units: the tiles of the full rounds
  // of 256 workgroups are computed whole, the remaining tiles' units are
  // shared by 256 stream-K workgroups (each then writes at most two
  // partials).  Whole tiles throughout when their rounds are at least 7/8
  // full: the partials and their reduce then cost what the idle CUs would
  // (the LM head of a 512-token prompt, 1188 tiles in 5 rounds).
  TilePlan pl;
  pl.U = U;
  int64_t dp = tiles, sk = 0;
  const int v = tuning().gemm_splits.load();  // measurement override
  if (v >= 2) {                                // about v segments per tile, all tiles shared
    dp = 0;
    sk = std::min<int64_t>(tiles * v, tiles * pl.U);
  } else if (v == 1 || 8 * tiles >= 7 * kTileCUs * ((tiles + kTileCUs - 1) / kTileCUs)) {
    dp = tiles;
  } else if (tiles > kTileCUs) {
    dp = (tiles / kTileCUs) * kTileCUs;
    // no more stream-K workgroups than shared units: every one owns at
    // least one, so every partial slot the reduce reads is written
    sk = std::min<int64_t>(kTileCUs, (tiles - dp) * pl.U);
  } else if (kTileCUs / tiles >= 2) {
    // at most 128 tiles: each split into floor(256 / tiles) equal pieces, so
    // that every workgroup stays inside one tile and writes one partial
    dp = 0;
    sk = std::min<int64_t>(tiles * (kTileCUs / tiles), tiles * pl.U);
  } else {
    dp = 0;
    sk = std::min<int64_t>(kTileCUs, tiles * pl.U);
  }
  if (sk > 0) {
    const int64_t TU = (tiles - dp) * pl.U;
    int64_t maxseg = 1;
    for (int64_t t = 0; t < tiles - dp; ++t)
      maxseg = std::max(maxseg, host_sk_owner(t * pl.U + pl.U - 1, TU, sk) -
                                    host_sk_owner(t * pl.U, TU, sk) + 1);
    const size_t ws = maxseg > 1 ? (size_t)(tiles - dp) * maxseg * tile_bytes : 0;
    if (ws <= ws_bytes) {
      pl.dp = (int)dp;
      pl.sk = (int)sk;
      pl.maxseg = (int)maxseg;
      pl.ws = ws;
      return pl;
    }
  }
  pl.dp = (int)tiles;  // whole tiles only
  return pl;
}

// Tile shape.  M >= 256: 256 x 256, the K of its tiles split.  Operands of 4 GiB and
// more take the shapes below, in whole tiles, as they did before there were tiles
// of 256 rows: the copies would allow more (their 32-bit offsets count from the
// tile's first row), but fp16 partials would round what is not rounded now.
// M < 256 (and those): whole tiles over all of K, one fp32 chain per output,
// so the tile decides how many CUs work.  The time follows the most loaded
// CU, ceil(tiles / 256) x the time of a tile's K step, which hardly depends on
// how many tiles of a shape share the CU; measured at INT4 per 128 k (us): 32 x 64
// 0.34, 48 x 64 0.40, 64 x 64 0.45, 64 x 128 0.88, 96 x 128 0.98, 128 x 128 1.15.  INT8
// and FP16 steps copy more bytes of weights; no table of their own was measured,
// but on 13 row counts from 17 to 255 and 8 widths the choice was 1.2 to 7 times as
// fast as the 128 x 128 kernel before it in every format.  E.g.
// (us) 96 x 7168 x 5120 INT4 29 / 22 / 24 / 41 / 47 / 52 over those shapes, 96 x 34816 x
// 5120 98 / 83 / 91 / 104 / 84 / 87, 96 x 5120 x 17408 INT8 58 / 73 / 73 / 138 / 174 / 174,
// 200 x 34816 x 5120 195 / 169 / 156 / 166 / 150 / 141.
struct TileShape {
  int mt, nf, mg;
};
TileShape tile_shape(int64_t M, int64_t N, int64_t K, int wbits) {
  const int64_t lim = (int64_t)1 << 32;
  if (M >= 256 && M * K * 2 < lim && N * K * wbits / 8 < lim && N * (K / 32) * 4 < lim)
    return TileShape{8, 4, 2};
  static const struct { int mt, nf, cost; } kShapes[] = {{8, 2, 115}, {6, 2, 98}, {4, 2, 88},
                                                         {4, 1, 45},  {3, 1, 40}, {2, 1, 34}};
  TileShape best{8, 2, 1};
  int64_t least = INT64_MAX;
  for (const auto& c : kShapes) {
    if (c.mt == 3 && wbits == 16) continue;  // 6 KB of X do not split over 4 waves
    const int64_t tiles = ((M + 16 * c.mt - 1) / (16 * c.mt)) * ((N + 64 * c.nf - 1) / (64 * c.nf));
    const int64_t t = (tiles + kTileCUs - 1) / kTileCUs * c.cost;
    if (t < least) least = t, best = TileShape{c.mt, c.nf, 1};
  }
  return best;
}
// f(Tile of the shape, its weight bits)
template <class F>
auto with_tile(int wbits, TileShape s, F f) {
  using W4 = std::integral_constant<int, 4>;
  using W8 = std::integral_constant<int, 8>;
  using W16 = std::integral_constant<int, 16>;
#define R4Q_TILE(MT, NF, MG)                                                               \
  if (s.mt == MT && s.nf == NF)                                                            \
    return wbits == 4 ? f(Tile<4, MT, NF, MG>(), W4())                                     \
           : wbits == 8 ? f(Tile<8, MT, NF, MG>(), W8()) : f(Tile<16, MT, NF, MG>(), W16());
  R4Q_TILE(8, 4, 2)
  R4Q_TILE(2, 1, 1)
  R4Q_TILE(4, 1, 1)
  R4Q_TILE(4, 2, 1)
  R4Q_TILE(6, 2, 1)
  R4Q_TILE(8, 2, 1)
#undef R4Q_TILE
  return wbits == 4 ? f(Tile<4, 3, 1, 1>(), W4()) : f(Tile<8, 3, 1, 1>(), W8());
}
int tile_unit(int wbits) {
  return wbits == 4 ? Tile<4, 8, 4, 2>::kUnit : wbits == 8 ? Tile<8, 8, 4, 2>::kUnit
                                                            : Tile<16, 8, 4, 2>::kUnit;
}
TilePlan tile_plan(int64_t M, int64_t N, int64_t K, int wbits, size_t ws_bytes) {
  const TileShape s = tile_shape(M, N, K, wbits);
  const int64_t bm = 16 * s.mt * s.mg, bn = 64 * s.nf, unit = tile_unit(wbits);
  const int64_t tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  const int U = (int)((K + unit - 1) / unit);
  if (s.mg == 2) return split_plan(tiles, U, bm * bn * 2, ws_bytes);
  TilePlan pl;  // whole tiles
  pl.U = U;
  pl.dp = (int)tiles;
  return pl;
}

void gemm_plan(int64_t M, int64_t N, int64_t K, int wbits, size_t ws_bytes, int32_t* out) {
  const TileShape s = tile_shape(M, N, K, wbits);
  const TilePlan pl = tile_plan(M, N, K, wbits, ws_bytes);
  out[0] = 16 * s.mt * s.mg;
  out[1] = 64 * s.nf;
  out[2] = pl.dp;
  out[3] = pl.sk;
}

size_t gemm_ws_bytes(int64_t M, int64_t N, int64_t K, int wbits) {
  return tile_plan(M, N, K, wbits, (size_t)-1).ws;
}

int gemm_mfma_launch(const void* x, const void* w, const void* sz, void* y, int64_t M, int64_t N,
                     int64_t K, int wbits, hipStream_t st, void* ws, size_t ws_bytes) {
  const auto* xp = static_cast<const uint16_t*>(x);
  const auto* wp = static_cast<const uint8_t*>(w);
  const auto* sp = static_cast<const uint32_t*>(sz);
  auto* yp = static_cast<uint16_t*>(y);
  const TilePlan pl = tile_plan(M, N, K, wbits, ws ? ws_bytes : 0);
  return with_tile(wbits, tile_shape(M, N, K, wbits), [&](auto tl, auto wb) {
    using T = decltype(tl);
    constexpr int WB = decltype(wb)::value, MT = T::BM / 16 / T::kMG, NF = T::BN / 64;
    uint16_t* part = pl.ws ? static_cast<uint16_t*>(ws) : nullptr;
    const int vec = N % T::kOut == 0 && (reinterpret_cast<uintptr_t>(yp) & (2 * T::kOut - 1)) == 0;
    hipLaunchKernelGGL((gemm_tile_kernel<WB, MT, NF, T::kMG>), dim3((unsigned)(pl.dp + pl.sk)),
                       dim3(T::kThreads), 0, st, xp, wp, sp, yp, part, (int)M, (int)N, (int)K,
                       pl.dp, pl.sk, pl.U, tile_unit(wbits), pl.maxseg, vec);
    R4Q_TRY(launch_status("gemm_tile"));
    if constexpr (T::kMG == 2) {
      if (pl.ws) {
        const int64_t tiles = ((M + T::BM - 1) / T::BM) * ((N + T::BN - 1) / T::BN);
        const int64_t threads = (tiles - pl.dp) * (T::BM * T::BN / T::kOut);
        hipLaunchKernelGGL((gemm_tile_reduce_kernel<T>), dim3((unsigned)((threads + 255) / 256)),
                           dim3(256), 0, st, part, yp, (int)M, (int)N, pl.dp, pl.sk, pl.U,
                           pl.maxseg, vec);
        R4Q_TRY(launch_status("gemm_tile_reduce"));
      }
    }
    return R4Q_OK;
  });
}

}  // namespace r4q
