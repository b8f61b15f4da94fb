// Flash-style attention forward for gfx950, bf16 Q/K/V/O, fp32 softmax and
// accumulation:  O = softmax(scale * Q K^T [causal mask]) V  per (batch, head).
//
// Semantics: runtime/cpu/bwpp_cpu_ref.c:92-144 (row max, sum of exp, inv =
// sum > 0 ? 1/sum : 0, weighted sum of V) generalised with a score scale and
// a bottom-right aligned causal mask (keys n > m + N - M excluded); the MSL
// kernel it replaces is codegen_metal.c:435-556.
//
// Layout of the work: a block of 8 waves (two per SIMD) owns a tile of 256
// queries of one (batch, head) (causal: two such tiles, one after the
// other); each wave owns 32 queries of the tile.  Keys stream through LDS in
// tiles of 128 (K and V, 32 KiB each for d = 128) in a 2-stage ring, filled
// by global -> LDS DMA.  Two waves per SIMD let one wave's softmax (VALU)
// run while the other's MFMAs issue; 32 queries per wave keep the
// registers (Q^T operands, S^T tile, O^T accumulators) under 256 per wave.
//
// Why S^T: the wave computes S^T = K Q^T with v_mfma_f32_32x32x16_bf16
// (MFMA "A" = a 32-key block of K, "B" = Q^T held in registers).  The
// accumulator then gives lane l the scores of ONE query (l % 32) for 16 of
// the 32 keys; the other 16 are in lane l ^ 32.  Running max, exp, sum and
// the rescale of the output accumulator are therefore lane-local plus one
// lane exchange.  The P V product is computed as O^T += V^T P^T: the
// probabilities go into the MFMA "B" operand straight from the accumulator
// registers, because the key order implied by the accumulator layout
// (lane half h holds keys 4h..4h+3, 8+4h..8+4h+3 of each 16) is applied to
// V^T as well: V^T is read from the [key][d] LDS tile with
// ds_read_b64_tr_b16 at exactly those key rows.
//
// Softmax runs in base 2: scores are multiplied by scale * log2(e) and
// exponentiated with v_exp_f32.  The exponent offset (running maximum) is
// only raised when a tile's maximum exceeds it by more than kLazy (log2
// units): probabilities then stay below 2^kLazy, the common factor cancels
// in O = (sum p v) / (sum p), and the O rescale is skipped on most tiles.
#include <type_traits>

#include "common.h"
#include "../kargs.h"

using namespace bwpp;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef short v8s_t __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s_t lds_v4s_t;

namespace {

typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

// Eight fp32 probabilities (registers r0 .. r0 + 7 of an accumulator) as two
// bf16 terms: the upper 16 bits, and the rounded rest.  The rest is kept
// above zero wherever p is (by 2^-23 p), so that p * inf stays inf.
__device__ __forceinline__ void split_bf16x8(const f32x16_t *s, int r0, bf16x8_t &hi, bf16x8_t &lo) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float p0 = (*s)[r0 + 2 * i], p1 = (*s)[r0 + 2 * i + 1];
    const uint32_t u0 = __float_as_uint(p0) & 0xffff0000u, u1 = __float_as_uint(p1) & 0xffff0000u;
    h[i] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
    l[i] = pack_bf16x2(__builtin_fmaf(p0, 1.00000012f, -__uint_as_float(u0)),
                       __builtin_fmaf(p1, 1.00000012f, -__uint_as_float(u1)));
  }
  hi = __builtin_bit_cast(bf16x8_t, make_uint4(h[0], h[1], h[2], h[3]));
  lo = __builtin_bit_cast(bf16x8_t, make_uint4(l[0], l[1], l[2], l[3]));
}

// m ln 2 + ln l, rounded once: l = 2^k f with f in [0.71, 1.42), so that logf's
// error is one of a small number, ln 2 in two terms, and every rounding on the
// way carried to the end (B1 H16 S1664 d64, error against 64 bits: 5.4e-8 with
// plain arithmetic, 4.3e-8 in the generic path).
__device__ __forceinline__ float lse_of(float m, float l) {
#pragma clang fp contract(off)
  constexpr float kHi = 0.693147182f, kLo = -1.90465421e-9f;
  if (!(l < INFINITY)) return l;
  const uint32_t u = __float_as_uint(l);
  const int k = (int)(u - 0x3f3504f3u) >> 23;
  const float e = (float)k, lf = logf(__uint_as_float(u - ((uint32_t)k << 23)));
  const float a = m * kHi, b = e * kHi, t = a + b, td = t - a, r = t + lf, rd = r - t;
  const float lo = ((a - (t - td)) + (b - td)) + ((t - (r - rd)) + (lf - rd));  // of the two sums
  return r + (lo + (__builtin_fmaf(m, kHi, -a) + __builtin_fmaf(e, kHi, -b) + (m + e) * kLo));
}

// Running maximum of |v| as bit patterns, two bf16 lanes at a time (0x7f80
// and above: infinity or NaN).
__device__ __forceinline__ u16x2_t max_abs_bf16(u16x2_t m, v8s_t v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const u16x2_t w = {(unsigned short)(v[2 * i] & 0x7fff), (unsigned short)(v[2 * i + 1] & 0x7fff)};
    m = __builtin_elementwise_max(m, w);
  }
  return m;
}

constexpr int kWaves = 4;               // generic path
constexpr int kFW = 8;                  // flash path: waves per block
constexpr int kQW = 32;                 // queries per wave
constexpr int kBQ = kFW * kQW;          // queries per block
constexpr float kLazy = 8.0f;

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// 16 bytes per lane global -> LDS (M0 = destination of lane 0, lane l at
// +16 l), from a wave-uniform 64-bit base in SGPRs plus a 32-bit per-lane
// byte offset; inline asm keeps the compiler from adding vmcnt(0) before every
// LDS read (completion is awaited with wait_vmcnt + a barrier).  M0 cannot
// be declared clobbered (it is reserved); these kernels use M0 for nothing
// else, which the generated code confirms (only these s_mov_b32 m0 write it).
__device__ __forceinline__ void g2lds16_so(const void *sbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(sbase)
               : "memory");
}

// K tile [64 keys][D] (256-byte rows for D = 128): chunk c of row r at
// c ^ (r & 15), so the 16 rows read by a ds_read_b128 quarter-wave hit 16
// distinct bank groups.  V tile [64 keys][D]: chunk c of row r at
// c ^ (4 * (r & 3)), conflict-free for the transposing reads (4 rows x 2
// chunks per 16-lane group, two groups per half-wave).
__device__ __forceinline__ uint32_t k_off(uint32_t r, uint32_t c) { return r * 256u + 16u * (c ^ (r & 15u)); }
__device__ __forceinline__ uint32_t v_off(uint32_t r, uint32_t c) { return r * 256u + 16u * (c ^ (4u * (r & 3u))); }

// One query tile (256 queries) of one (batch, head) slice.
template <bool CAUSAL>
__device__ __forceinline__ void attn_bf16_d128_tile(const BwppAttnArgs &a, const uint32_t bh, const uint32_t qt) {
  // Key tiles: 128 keys in a 2-stage ring (half the barriers and DMA issues
  // per key of 64-key tiles: 4 % faster at C4 unmasked, 5 % causal, where a
  // masked tile skips the 32-key blocks its wave sees none of).
  constexpr int kBKV = 128;
  constexpr int kStages = 2;
  constexpr int D = 128;
  constexpr int KS = D / 16;  // k-steps of S over d
  constexpr int DB = D / 32;  // 32-wide d blocks of O^T
  constexpr int kTile = kBKV * D * 2;
  constexpr int kStage = 2 * kTile;
  constexpr int kRing = kStages * kStage;
  constexpr int kOut = kBQ * D * 2;
  constexpr int kBlkPW = (kBKV / 4) / kFW;  // 1 KiB DMA blocks per wave per K (or V) tile
  constexpr int KB = kBKV / 32;             // 32-key blocks per tile
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kRing > kOut ? kRing : kOut];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t b = bh / a.heads, h = bh % a.heads;
  const uint16_t *Q = static_cast<const uint16_t *>(a.q) + b * a.q_bs + h * a.q_hs;
  const uint16_t *K = static_cast<const uint16_t *>(a.k) + b * a.k_bs + h * a.k_hs;
  const uint16_t *V = static_cast<const uint16_t *>(a.v) + b * a.v_bs + h * a.v_hs;
  uint16_t *O = static_cast<uint16_t *>(a.o) + b * a.o_bs + h * a.o_hs;
  const int64_t diag = (int64_t)a.N - (int64_t)a.M;  // key n visible to query m iff n <= m + diag

  const uint32_t qb0 = qt * kBQ;                    // block's first query
  const uint32_t q0 = qb0 + (uint32_t)wave * kQW;   // wave's first query
  const uint32_t lq = (uint32_t)(lane & 31), lh = (uint32_t)(lane >> 5);
  const uint32_t qi = q0 + lq;                      // this lane's query

  // Key tiles this block needs.
  uint32_t kend = a.N;
  if (CAUSAL) {
    const int64_t last_q = (int64_t)min(qb0 + kBQ, a.M) - 1;
    const int64_t lim = last_q + diag + 1;
    kend = lim <= 0 ? 0u : (uint32_t)min<int64_t>(lim, a.N);
  }
  const uint32_t nkt = (kend + kBKV - 1) / kBKV;

  // Q^T operands: lane holds query qi, d = 16 ks + 8 lh .. +7.
  bf16x8_t qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    uint4 v = make_uint4(0, 0, 0, 0);
    if (qi < a.M) v = *reinterpret_cast<const uint4 *>(Q + (size_t)qi * a.ldq + 16 * ks + 8 * lh);
    qf[ks] = __builtin_bit_cast(bf16x8_t, v);
  }
  // Let the Q loads land before any DMA is issued: the compiler cannot see
  // the DMA, and an outstanding Q load at the loop head would make it wait
  // for vmcnt(0) -- every tile in flight -- on each iteration.
  wait_vmcnt<0>();

  // DMA: each wave loads kBlkPW of the kBKV / 4 1-KiB blocks of the K tile
  // and of the V tile.  Rows past N re-read row N - 1 (finite data; masked to -inf).
  // Lane l of block i fills 16-byte slot l of it: key row r = 4 i' + l / 16
  // of the tile (i' the block index), physical chunk l % 16, which holds the
  // logical chunk given by the K / V swizzles below.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
  uint32_t dma_row[kBlkPW], dma_kcol[kBlkPW], dma_vcol[kBlkPW];
#pragma unroll
  for (int i = 0; i < kBlkPW; ++i) {
    const uint32_t q = (uint32_t)(wave * kBlkPW + i) * 64u + (uint32_t)lane;
    const uint32_t r = q >> 4, pc = q & 15u;
    dma_row[i] = r;
    dma_kcol[i] = 8u * (pc ^ (r & 15u));
    dma_vcol[i] = 8u * (pc ^ (4u * (r & 3u)));
  }
  auto issue = [&](uint32_t t) {
    const uint32_t st = lds0 + (t % kStages) * kStage + (uint32_t)(wave * kBlkPW) * 1024u;
#pragma unroll
    for (int i = 0; i < kBlkPW; ++i) {
      uint32_t key = t * kBKV + dma_row[i];
      key = key < a.N ? key : a.N - 1;
      // Byte offsets inside the (batch, head) slice fit 32 bits (the runtime
      // checks (N - 1) * ld + D < 2^31 before choosing this kernel).
      g2lds16_so(K, 2u * (key * a.ldk + dma_kcol[i]), st + (uint32_t)i * 1024u);
      g2lds16_so(V, 2u * (key * a.ldv + dma_vcol[i]), st + kTile + (uint32_t)i * 1024u);
    }
  };
  constexpr int kDmaPerTile = 2 * kBlkPW;

  f32x16_t o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
  float mrow = -INFINITY, lrow = 0.0f;
  const float c = a.scale_log2;

  // Per-lane LDS read offsets inside a stage.  K operand of k-step ks, key
  // block kb: koff[ks] + kb * 32 rows.  V^T operand of d block d, keys
  // 32 kb + 16 kq (+8 for the upper four): voff[d] + (32 kb + 16 kq (+8))
  // rows; the V swizzle depends on the row only through r & 3, which those
  // row steps keep.
  const uint32_t grp = (uint32_t)((lane >> 4) & 3), L = (uint32_t)(lane & 15);
  uint32_t koff[KS], voff[DB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = k_off(lq, 2u * ks + lh);
  {
    const uint32_t kbase = 4u * (grp >> 1) + (L >> 2);
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      const uint32_t col = 32u * d + 16u * (grp & 1u) + 4u * (L & 3u);
      voff[d] = kTile + v_off(kbase, col >> 3) + (col & 7u) * 2u;
    }
  }

  // One key tile.  MASK: some (key, query) pair of the tile is masked out.
  auto tile = [&](auto mask_tag, const unsigned char *Ks, uint32_t k0) {
    constexpr bool MASK = decltype(mask_tag)::value;
    // Masked tiles: 32-key blocks past every key this wave's queries see
    // are skipped (their scores are masked to -inf below, p = 0).
    int kbmax = KB - 1;
    if constexpr (MASK) {
      int64_t kv = (int64_t)a.N - 1 - (int64_t)k0;
      if (CAUSAL) {
        const int64_t kc = (int64_t)(q0 + kQW - 1) + diag - (int64_t)k0;
        kv = kc < kv ? kc : kv;
      }
      kbmax = kv < 0 ? -1 : (int)(kv / 32 < KB - 1 ? kv / 32 : KB - 1);
      kbmax = __builtin_amdgcn_readfirstlane(kbmax);
    }
    // S^T blocks: s[kb] = K[32 kb .. 32 kb + 31] . Q^T.
    f32x16_t s[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[kb][r] = 0.0f;
      if (MASK && kb > kbmax) continue;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bf16x8_t kf =
            __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(Ks + koff[ks] + 32u * 256u * kb));
        s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[kb], 0, 0, 0);
      }
    }
    // Keep two K reads ahead of the MFMAs instead of hoisting all sixteen
    // (which would not fit the 256 registers of a two-wave-per-SIMD wave).
    if constexpr (!MASK) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
      for (int i = 0; i < KB * KS - 2; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }

    // Online softmax for this lane's query (plus partner lane ^ 32).
    float mx = -INFINITY;
    if constexpr (MASK) {
      // Key of register r in block kb is k0 + 4 lh + (32 kb + 8 (r >> 2) +
      // (r & 3)); visible iff that offset is below `lim` (key < N and, when
      // causal, key <= query + diag).  Wave-uniform per block: blocks past
      // kbmax are all masked (their scores stay out of the max, and their
      // probabilities are 0 below), and a block whose last key every query
      // of the wave sees needs no per-element test.
      int64_t lim64 = (int64_t)a.N - (int64_t)(k0 + 4u * lh);
      if (CAUSAL) {
        const int64_t c64 = (int64_t)qi + diag + 1 - (int64_t)(k0 + 4u * lh);
        lim64 = c64 < lim64 ? c64 : lim64;
      }
      const int lim = (int)(lim64 < -1 ? -1 : (lim64 > kBKV ? kBKV : lim64));
      int64_t vis = (int64_t)a.N - 1 - (int64_t)k0;  // last key offset every query of the wave sees
      if (CAUSAL) {
        const int64_t vc = (int64_t)q0 + diag - (int64_t)k0;
        vis = vc < vis ? vc : vis;
      }
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        if (kb > kbmax) continue;
        if ((int64_t)(32 * kb + 31) <= vis) {
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float x = (32 * kb + 8 * (r >> 2) + (r & 3)) < lim ? s[kb][r] : -INFINITY;
            s[kb][r] = x;
            mx = fmaxf(mx, x);
          }
        }
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
    }
    {
      // Lanes l and l ^ 32 hold the two halves of one query's keys.
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * c;
    }
    // Raise the offset only past the lazy margin (or from -inf).
    float alpha = 1.0f;
    if (mx > mrow + kLazy) {
      alpha = __builtin_amdgcn_exp2f(mrow - mx);  // 0 when mrow is -inf
      mrow = mx;
    }
    const float muse = mrow == -INFINITY ? 0.0f : mrow;
    float sum = 0.0f;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      if (MASK && kb > kbmax) continue;  // p = 0: adds nothing, and its P.V is skipped
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], c, -muse));
        s[kb][r] = p;
        sum += p;
      }
    }
    {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
      sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    lrow = lrow * alpha + sum;
    if (__ballot(alpha != 1.0f)) {
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
    }

    // O^T += V^T P^T over the blocks of 16 keys.
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      if (MASK && kb > kbmax) continue;
#pragma unroll
      for (int kq = 0; kq < 2; ++kq) {
        const int r0 = 8 * kq;
        uint4 w;
        w.x = pack_bf16x2(s[kb][r0 + 0], s[kb][r0 + 1]);
        w.y = pack_bf16x2(s[kb][r0 + 2], s[kb][r0 + 3]);
        w.z = pack_bf16x2(s[kb][r0 + 4], s[kb][r0 + 5]);
        w.w = pack_bf16x2(s[kb][r0 + 6], s[kb][r0 + 7]);
        const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, w);
        // Key rows of this lane's operand: 32 kb + 16 kq + 4 h (+8).
        constexpr uint32_t kRowB = 256u;
        const uint32_t rstep = (32u * kb + 16u * kq) * kRowB;
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(Ks + voff[d] + rstep));
          const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(Ks + voff[d] + rstep + 8u * kRowB));
          const v8s_t vv = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vv), pf, o[d], 0, 0, 0);
        }
      }
    }
    // Two V^T operands (four transposing reads) ahead of the MFMAs.
    if constexpr (!MASK) {
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 0; i < 2 * KB * DB - 2; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
  };

#pragma unroll
  for (int st = 0; st < kStages - 1; ++st)
    if ((uint32_t)st < nkt) issue((uint32_t)st);

  // Tiles before t_mask need no mask for any query of the block; the rest
  // go through the masked variant.  Two loops (not one with a branch, which
  // made the compiler keep a second copy of the O accumulators and spill)
  // with a block-uniform boundary: every wave passes every tile's barrier
  // from the same loop.  Inside the masked loop the waves differ only in
  // wave-uniform branches around MFMA work (the 32-key blocks and tiles
  // their queries see none of).
  uint32_t t_mask = a.N / kBKV;  // first tile with keys past N
  if (CAUSAL) {
    // First tile holding a key past the block's first query's limit.
    const int64_t first_hidden = (int64_t)qb0 + diag + 1;
    const uint32_t tc = first_hidden <= 0 ? 0u : (uint32_t)min<int64_t>(first_hidden / kBKV, (int64_t)nkt);
    t_mask = min(t_mask, tc);
  }
  t_mask = min(t_mask, nkt);

  auto step = [&](uint32_t t) {
    // Tiles t + 1 .. t + kStages - 2 may still be in flight.
    const uint32_t younger = min(nkt - 1 - t, (uint32_t)(kStages - 2));
    if (younger >= 2) wait_vmcnt<2 * kDmaPerTile>();
    else if (younger == 1) wait_vmcnt<kDmaPerTile>();
    else wait_vmcnt<0>();
    __syncthreads();
    if (t + kStages - 1 < nkt) issue(t + kStages - 1);
    // The stage base goes through readfirstlane so that loop strength
    // reduction does not turn every LDS address into its own induction
    // variable (it would need ~50 registers); the per-read offsets are then
    // base + lane offset + an immediate.
    return smem + __builtin_amdgcn_readfirstlane((t % kStages) * kStage);
  };
  for (uint32_t t = 0; t < t_mask; ++t) {
    const unsigned char *Ks = step(t);
    tile(std::integral_constant<bool, false>{}, Ks, t * kBKV);
  }
  for (uint32_t t = t_mask; t < nkt; ++t) {
    const unsigned char *Ks = step(t);
    const uint32_t k0 = t * kBKV;
    // Whole tile masked for this wave's queries: nothing to do.
    if (CAUSAL && (int64_t)k0 > (int64_t)(q0 + kQW - 1) + diag) continue;
    tile(std::integral_constant<bool, true>{}, Ks, k0);
  }
  __syncthreads();

  // O = O^T / l, staged through LDS ([query][d] bf16 per wave, 256-byte
  // rows, 16-byte chunk c of row q at c ^ (q & 15)), then stored with
  // 16-byte row chunks.  Without the swizzle the 32 rows a staging write
  // touches at one column all fall on the same banks.  The row stores are
  // non-temporal: O is not read again by this kernel, and written back
  // from the caches later it took bandwidth from the next launch (C4
  // 542 -> 530 us unmasked, 318 -> 301 causal, back to back).
  uint16_t *os = reinterpret_cast<uint16_t *>(smem) + (size_t)wave * kQW * D;
  // Natural-log log-sum-exp of the scaled scores when asked for: the sum of
  // exp(scale s) is 2^mrow * lrow (mrow in log2 units).
  if (a.lse && lh == 0 && qi < a.M)
    a.lse[(size_t)bh * a.M + qi] =
        lrow > 0.0f ? ((mrow == -INFINITY ? 0.0f : mrow) + log2f(lrow)) * 0.69314718055994531f : -INFINITY;
  {
    const float inv = lrow > 0.0f ? 1.0f / lrow : 0.0f;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const uint32_t chunk = (4u * d + q4) ^ (lq & 15u);
        uint2 w;
        w.x = pack_bf16x2(o[d][4 * q4 + 0] * inv, o[d][4 * q4 + 1] * inv);
        w.y = pack_bf16x2(o[d][4 * q4 + 2] * inv, o[d][4 * q4 + 3] * inv);
        *reinterpret_cast<uint2 *>(os + lq * D + 8u * chunk + 4u * lh) = w;
      }
  }
  __syncthreads();
  constexpr int kRowChunks = D / 8;
#pragma unroll 4
  for (int it = 0; it < kQW * kRowChunks / 64; ++it) {
    const int q = lane + it * 64;
    const uint32_t ql = (uint32_t)(q / kRowChunks), cc = (uint32_t)(q % kRowChunks);
    const uint32_t qo = q0 + ql;
    if (qo < a.M)
      __builtin_nontemporal_store(*reinterpret_cast<const u32x4_t *>(os + ql * D + 8u * (cc ^ (ql & 15u))),
                                  reinterpret_cast<u32x4_t *>(O + (size_t)qo * a.ldo + 8u * cc));
  }
  __syncthreads();  // the block's next tile reuses smem
}

// Persistent form of the kernel: a block (one per CU) works through its
// items -- unmasked: (slice, query tile) items, item k of block b being
// k * G + b' (b' the XCD renumbering of b below, so each XCD's blocks take
// the query tiles of a few slices together in every round); causal: the
// same over pairs of query tiles, as attn_bf16_d128 pairs them.  Per item the
// work is attn_bf16_d128_tile's; what differs is the item boundary: the
// next item's first K / V stage is requested at the start of the current
// item's last key tile (into the stage that tile does not use), its Q rows
// as soon as the last tile's S products have read the current ones, and O
// is staged through the last tile's stage -- so the next item's loads are
// in flight during the last tile and the O epilogue instead of after them
// (with one item per block they cost 2.7 us for Q, 1.3 us for the first
// stage and 1.5 us for O of each 62 us item at C4).
template <bool CAUSAL>
__device__ __forceinline__ void attn_bf16_d128_persist(const BwppAttnArgs &a) {
  constexpr int kBKV = 128;
  constexpr int D = 128;
  constexpr int KS = D / 16;
  constexpr int DB = D / 32;
  constexpr int kTile = kBKV * D * 2;
  constexpr int kStage = 2 * kTile;
  constexpr int kOut = kBQ * D * 2;
  static_assert(kOut <= kStage, "O is staged through one ring stage");
  constexpr int kBlkPW = (kBKV / 4) / kFW;
  constexpr int KB = kBKV / 32;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * kStage];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lq = (uint32_t)(lane & 31), lh = (uint32_t)(lane >> 5);
  const uint32_t G = gridDim.x, QT = a.q_tiles;
  const uint32_t bp = G % 8u == 0 ? (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u : blockIdx.x;
  // Unmasked: a.items (slice, query tile) items.  Causal: a.items pairs of
  // query tiles QT - 1 - p and p of one slice, as attn_bf16_d128 pairs them
  // (one item when they coincide); block b' takes pairs j G + b'.
  const uint32_t P = (QT + 1) / 2;
  const uint32_t nunits = bp < a.items ? (a.items - bp + G - 1) / G : 0u;
  const uint32_t nitems = CAUSAL ? 2u * nunits : nunits;  // slots; a causal pair's second may be empty
  if (nitems == 0) return;
  const int64_t diag = (int64_t)a.N - (int64_t)a.M;  // key n visible to query m iff n <= m + diag

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
  uint32_t dma_row[kBlkPW], dma_kcol[kBlkPW], dma_vcol[kBlkPW];
#pragma unroll
  for (int i = 0; i < kBlkPW; ++i) {
    const uint32_t q = (uint32_t)(wave * kBlkPW + i) * 64u + (uint32_t)lane;
    const uint32_t r = q >> 4, pc = q & 15u;
    dma_row[i] = r;
    dma_kcol[i] = 8u * (pc ^ (r & 15u));
    dma_vcol[i] = 8u * (pc ^ (4u * (r & 3u)));
  }
  struct Item {
    const uint16_t *Q, *K, *V;
    uint16_t *O;
    uint32_t bh, q0, qb0;
  };
  // Slot k: its slice and query tile; valid(k) is false only for the empty
  // second slot of a causal pair whose two tiles coincide.
  auto slot_tile = [&](uint32_t k, uint32_t &bh) {
    if (!CAUSAL) {
      const uint32_t li = k * G + bp;
      bh = li / QT;
      return QT - 1 - li % QT;
    }
    const uint32_t pi = (k >> 1) * G + bp, p = pi % P;
    bh = pi / P;
    return (k & 1u) ? p : QT - 1 - p;
  };
  auto valid = [&](uint32_t k) {
    if (!CAUSAL || !(k & 1u)) return k < nitems;
    const uint32_t p = ((k >> 1) * G + bp) % P;
    return k < nitems && p != QT - 1 - p;
  };
  auto item = [&](uint32_t k) {
    uint32_t bh;
    const uint32_t qt = slot_tile(k, bh);
    const uint32_t b = bh / a.heads, h = bh % a.heads;
    Item it;
    it.Q = static_cast<const uint16_t *>(a.q) + b * a.q_bs + h * a.q_hs;
    it.K = static_cast<const uint16_t *>(a.k) + b * a.k_bs + h * a.k_hs;
    it.V = static_cast<const uint16_t *>(a.v) + b * a.v_bs + h * a.v_hs;
    it.O = static_cast<uint16_t *>(a.o) + b * a.o_bs + h * a.o_hs;
    it.bh = bh;
    it.qb0 = qt * kBQ;
    it.q0 = it.qb0 + (uint32_t)wave * kQW;
    return it;
  };
  // Key tiles an item needs, and its first tile with a masked (key, query).
  auto key_tiles = [&](const Item &it) {
    uint32_t kend = a.N;
    if (CAUSAL) {
      const int64_t lim = (int64_t)min(it.qb0 + kBQ, a.M) - 1 + diag + 1;
      kend = lim <= 0 ? 0u : (uint32_t)min<int64_t>(lim, a.N);
    }
    return (kend + kBKV - 1) / kBKV;
  };
  auto first_masked = [&](const Item &it, uint32_t nkt) {
    uint32_t tm = a.N / kBKV;
    if (CAUSAL) {
      const int64_t first_hidden = (int64_t)it.qb0 + diag + 1;
      tm = min(tm, first_hidden <= 0 ? 0u : (uint32_t)min<int64_t>(first_hidden / kBKV, (int64_t)nkt));
    }
    return min(tm, nkt);
  };
  auto issue = [&](const Item &it, uint32_t t, uint32_t stage) {
    const uint32_t st = lds0 + stage * kStage + (uint32_t)(wave * kBlkPW) * 1024u;
#pragma unroll
    for (int i = 0; i < kBlkPW; ++i) {
      uint32_t key = t * kBKV + dma_row[i];
      key = key < a.N ? key : a.N - 1;
      g2lds16_so(it.K, 2u * (key * a.ldk + dma_kcol[i]), st + (uint32_t)i * 1024u);
      g2lds16_so(it.V, 2u * (key * a.ldv + dma_vcol[i]), st + kTile + (uint32_t)i * 1024u);
    }
  };
  bf16x8_t qf[KS];
  auto load_q = [&](const Item &it) {
    const uint32_t qi = it.q0 + lq;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (qi < a.M) v = *reinterpret_cast<const uint4 *>(it.Q + (size_t)qi * a.ldq + 16 * ks + 8 * lh);
      qf[ks] = __builtin_bit_cast(bf16x8_t, v);
    }
  };

  // Per-lane LDS read offsets of k-step 0 / d block 0 (as in
  // attn_bf16_d128_tile); the others differ in chunk bits the swizzles XOR
  // and never carry into: K operand of k-step ks at koff0 ^ 32 ks, V^T of d
  // block d at voff0 ^ 64 d.  The tile recomputes them (see below).
  const uint32_t grp = (uint32_t)((lane >> 4) & 3), L = (uint32_t)(lane & 15);
  const uint32_t koff0 = k_off(lq, lh);
  const uint32_t voff0 = kTile + v_off(4u * (grp >> 1) + (L >> 2), 2u * (grp & 1u) + ((L & 3u) >> 1)) + (4u * (L & 1u)) * 2u;
  const float c = a.scale_log2;

  // First item: Q, then its first stage (the Q loads land first, as in
  // attn_bf16_d128_tile).
  Item cur = item(0);
  load_q(cur);
  wait_vmcnt<0>();
  issue(cur, 0, 0);
  uint32_t s0 = 0;  // ring stage of the current item's key tile 0

  for (uint32_t k = 0; k < nitems; ++k) {
    if (!valid(k)) continue;
    const uint32_t kn = valid(k + 1) ? k + 1 : k + 2;  // the next item's slot
    const bool has_next = kn < nitems;
    const Item nxt = item(has_next ? kn : k);
    const uint32_t qi = cur.q0 + lq;
    const uint32_t nkt = key_tiles(cur), t_mask = first_masked(cur, nkt);
    f32x16_t o[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
    float mrow = -INFINITY, lrow = 0.0f;

    auto tile = [&](auto mask_tag, const unsigned char *Ks, uint32_t k0, bool last) {
      constexpr bool MASK = decltype(mask_tag)::value;
      // The offsets through an empty asm tied to the tile, so that their
      // XORed forms stay inside the tile instead of occupying twelve
      // registers across the whole item loop (the causal kernel spilled).
      uint32_t ko = koff0, vo = voff0;
      asm("" : "+v"(ko), "+v"(vo) : "s"(k0));
      int kbmax = KB - 1;
      if constexpr (MASK) {
        int64_t kv = (int64_t)a.N - 1 - (int64_t)k0;
        if (CAUSAL) {
          const int64_t kc = (int64_t)(cur.q0 + kQW - 1) + diag - (int64_t)k0;
          kv = kc < kv ? kc : kv;
        }
        kbmax = kv < 0 ? -1 : (int)(kv / 32 < KB - 1 ? kv / 32 : KB - 1);
        kbmax = __builtin_amdgcn_readfirstlane(kbmax);
      }
      f32x16_t s[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = 0.0f;
        if (MASK && kb > kbmax) continue;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const bf16x8_t kf =
              __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(Ks + (ko ^ (32u * ks)) + 32u * 256u * kb));
          s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[kb], 0, 0, 0);
        }
      }
      if constexpr (!MASK) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int i = 0; i < KB * KS - 2; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      }
      // The current Q rows are no longer needed: request the next item's.
      if (last && has_next) load_q(nxt);

      float mx = -INFINITY;
      if constexpr (MASK) {
        // As in attn_bf16_d128_tile: blocks past kbmax are left out, and a
        // block every query of the wave sees whole needs no element test.
        int64_t lim64 = (int64_t)a.N - (int64_t)(k0 + 4u * lh);
        if (CAUSAL) {
          const int64_t c64 = (int64_t)qi + diag + 1 - (int64_t)(k0 + 4u * lh);
          lim64 = c64 < lim64 ? c64 : lim64;
        }
        const int lim = (int)(lim64 < -1 ? -1 : (lim64 > kBKV ? kBKV : lim64));
        int64_t vis = (int64_t)a.N - 1 - (int64_t)k0;
        if (CAUSAL) {
          const int64_t vc = (int64_t)cur.q0 + diag - (int64_t)k0;
          vis = vc < vis ? vc : vis;
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          if (kb > kbmax) continue;
          if ((int64_t)(32 * kb + 31) <= vis) {
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
          } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const float x = (32 * kb + 8 * (r >> 2) + (r & 3)) < lim ? s[kb][r] : -INFINITY;
              s[kb][r] = x;
              mx = fmaxf(mx, x);
            }
          }
        }
      } else {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
      }
      {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * c;
      }
      float alpha = 1.0f;
      if (mx > mrow + kLazy) {
        alpha = __builtin_amdgcn_exp2f(mrow - mx);
        mrow = mx;
      }
      const float muse = mrow == -INFINITY ? 0.0f : mrow;
      float sum = 0.0f;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        if (MASK && kb > kbmax) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], c, -muse));
          s[kb][r] = p;
          sum += p;
        }
      }
      {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
        sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      }
      lrow = lrow * alpha + sum;
      if (__ballot(alpha != 1.0f)) {
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
      }
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        if (MASK && kb > kbmax) continue;
#pragma unroll
        for (int kq = 0; kq < 2; ++kq) {
          const int r0 = 8 * kq;
          uint4 w;
          w.x = pack_bf16x2(s[kb][r0 + 0], s[kb][r0 + 1]);
          w.y = pack_bf16x2(s[kb][r0 + 2], s[kb][r0 + 3]);
          w.z = pack_bf16x2(s[kb][r0 + 4], s[kb][r0 + 5]);
          w.w = pack_bf16x2(s[kb][r0 + 6], s[kb][r0 + 7]);
          const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, w);
          constexpr uint32_t kRowB = 256u;
          const uint32_t rstep = (32u * kb + 16u * kq) * kRowB;
#pragma unroll
          for (int d = 0; d < DB; ++d) {
            const uint32_t vd = vo ^ (64u * d);
            const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(Ks + vd + rstep));
            const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(Ks + vd + rstep + 8u * kRowB));
            const v8s_t vv = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vv), pf, o[d], 0, 0, 0);
          }
        }
      }
      if constexpr (!MASK) {
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < 2 * KB * DB - 2; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      }
    };

    // Tile t lives in stage (s0 + t) % 2.  At tile t's barrier every wave is
    // done with tile t - 1, whose stage then takes tile t + 1 -- or, at the
    // last tile, the next item's tile 0.
    auto step = [&](uint32_t t) {
      wait_vmcnt<0>();
      __syncthreads();
      const uint32_t nst = (s0 + t + 1) & 1u;
      if (t + 1 < nkt) issue(cur, t + 1, nst);
      else if (has_next) issue(nxt, 0, nst);
      return smem + __builtin_amdgcn_readfirstlane(((s0 + t) & 1u) * kStage);
    };
    for (uint32_t t = 0; t < t_mask; ++t) {
      const unsigned char *Ks = step(t);
      tile(std::integral_constant<bool, false>{}, Ks, t * kBKV, t + 1 == nkt);
    }
    // A tile whose keys this wave's queries see none of goes through tile()
    // too: no MFMA runs (kbmax = -1), the all -inf scores leave the running
    // max, the sum and O exactly as they were, and the next item's Q rows
    // are requested at one place (a second one, in a skip branch, made the
    // compiler keep two versions of them and spill).
    for (uint32_t t = t_mask; t < nkt; ++t) {
      const unsigned char *Ks = step(t);
      tile(std::integral_constant<bool, true>{}, Ks, t * kBKV, t + 1 == nkt);
    }
    __syncthreads();
    if (nkt == 0 && has_next) {
      // No key tile: the next item's loads start here (after this item's
      // own, unused, first-stage DMA into the same stage has landed).
      wait_vmcnt<0>();
      load_q(nxt);
      issue(nxt, 0, s0);
    }

    // O through the last tile's stage (the other one holds the next item's
    // tile 0); the next item's tile 1 goes into this stage after its first
    // barrier, which comes after these reads.
    uint16_t *os = reinterpret_cast<uint16_t *>(smem + ((s0 + nkt + 1) & 1u) * kStage) + (size_t)wave * kQW * D;
    if (a.lse && lh == 0 && qi < a.M)
      a.lse[(size_t)cur.bh * a.M + qi] =
          lrow > 0.0f ? ((mrow == -INFINITY ? 0.0f : mrow) + log2f(lrow)) * 0.69314718055994531f : -INFINITY;
    {
      const float inv = lrow > 0.0f ? 1.0f / lrow : 0.0f;
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const uint32_t chunk = (4u * d + q4) ^ (lq & 15u);
          uint2 w;
          w.x = pack_bf16x2(o[d][4 * q4 + 0] * inv, o[d][4 * q4 + 1] * inv);
          w.y = pack_bf16x2(o[d][4 * q4 + 2] * inv, o[d][4 * q4 + 3] * inv);
          *reinterpret_cast<uint2 *>(os + lq * D + 8u * chunk + 4u * lh) = w;
        }
    }
    __syncthreads();
    constexpr int kRowChunks = D / 8;
#pragma unroll 4
    for (int it = 0; it < kQW * kRowChunks / 64; ++it) {
      const int q = lane + it * 64;
      const uint32_t ql = (uint32_t)(q / kRowChunks), cc = (uint32_t)(q % kRowChunks);
      const uint32_t qo = cur.q0 + ql;
      if (qo < a.M)
        __builtin_nontemporal_store(*reinterpret_cast<const u32x4_t *>(os + ql * D + 8u * (cc ^ (ql & 15u))),
                                    reinterpret_cast<u32x4_t *>(cur.O + (size_t)qo * a.ldo + 8u * cc));
    }
    s0 = (s0 + nkt) & 1u;
    cur = nxt;
  }
}

// Work per block.  Blocks are dispatched round-robin over the 8 XCDs; the
// renumbering below gives each XCD a contiguous run of (batch, head) slices
// with all of their query tiles, so the blocks that stream the same K / V
// run together on one L2.  Unmasked: one query tile per block.  Causal: a
// block takes query tiles QT - 1 - p and p of one slice, whose visible key
// counts add up to the same total for every p (up to the clamping at 0 and
// N when M != N), so the blocks carry equal work (the runtime launches
// slices * ceil(QT / 2) blocks).
template <bool CAUSAL>
__device__ __forceinline__ void attn_bf16_d128(const BwppAttnArgs &a) {
  const uint32_t G = gridDim.x, QT = a.q_tiles;
  const uint32_t lb = G % 8u == 0 ? (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u : blockIdx.x;
  if (!CAUSAL) {
    attn_bf16_d128_tile<CAUSAL>(a, lb / QT, QT - 1 - lb % QT);
    return;
  }
  const uint32_t P = (QT + 1) / 2, bh = lb / P, pi = lb % P;
  for (uint32_t i = 0; i < 2; ++i) {
    if (i == 1 && QT - 1 - pi == pi) break;
    attn_bf16_d128_tile<CAUSAL>(a, bh, i == 0 ? QT - 1 - pi : pi);
  }
}

// ------------------------------------------------------------- generic path
// Any head dims K, D <= 512, fp32 or bf16 storage, fp32 arithmetic with
// expf: the reference's accumulation conventions (dot products in k order,
// bwpp_cpu_ref.c:110-113) with an online max/sum over chunks of 64 keys.
// A wave processes one query at a time: lanes split the keys for the
// scores (one key per lane per chunk), the probabilities go through LDS,
// and lanes split d for the weighted sum of V.  4 waves per block, a.items
// rows (queries, or keys in the dK / dV pass) per block: 16, or one per wave
// where 16 would leave CUs idle.
constexpr int kGenMaxDim = 512;

template <class T>
__device__ __forceinline__ float ld_elem(const T *p) {
  if constexpr (sizeof(T) == 2)
    return bf16_bits_to_f32(*reinterpret_cast<const uint16_t *>(p));
  else
    return *p;
}
template <class T>
__device__ __forceinline__ void st_elem(T *p, float v) {
  if constexpr (sizeof(T) == 2)
    *reinterpret_cast<uint16_t *>(p) = f32_to_bf16_bits(v);
  else
    *p = v;
}

// acc + sum over k of q[k] * row[k], in k order.  The row comes in 16-byte
// loads (at any address), several in flight: element loads, one row per lane,
// were what bound these kernels (forward and backward of B2 H16 S58 d96
// bf16 271 -> 29 us, of fp32 B3 H4 S127 d96 963 -> 91, of bf16 B1 H4 S800 d96
// 5616 -> 235; the same bits).
template <class T>
__device__ __forceinline__ float dot_row(const float *q, const T *row, uint32_t n, float acc) {
  constexpr uint32_t W = 16 / sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(W), aligned(sizeof(T))));
  uint32_t k = 0;
#pragma unroll 4
  for (; k + W <= n; k += W) {
    const vec_t v = *reinterpret_cast<const vec_t *>(row + k);
#pragma unroll
    for (uint32_t e = 0; e < W; ++e) {
      const T x = v[e];
      acc += q[k + e] * ld_elem(&x);
    }
  }
  for (; k < n; ++k) acc += q[k] * ld_elem(row + k);
  return acc;
}

// acc[j] += w[t] * row t's element 64 j + lane, rows in order t = 0 .. cnt -
// 1, eight rows' loads in flight.
template <class T, int DPL>
__device__ __forceinline__ void axpy_rows(float (&acc)[DPL], const float *w, const T *rows, uint32_t ld, uint32_t cnt,
                                          uint32_t n, int lane) {
#pragma unroll
  for (int j = 0; j < DPL; ++j) {
    const uint32_t d = (uint32_t)lane + 64u * j;
    if (64u * j >= n) break;  // uniform
    if (d >= n) continue;
    uint32_t t = 0;
    for (; t + 8 <= cnt; t += 8) {
      T x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = rows[(size_t)(t + i) * ld + d];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[j] += w[t + i] * ld_elem(&x[i]);
    }
    for (; t < cnt; ++t) acc[j] += w[t] * ld_elem(rows + (size_t)t * ld + d);
  }
}

// One query by one wave.  qs: [>= kdim] floats, ps: [64] floats of LDS of
// the wave's own; DPL: ceil(vdim / 64) at most.
template <class T, bool CAUSAL, int DPL>
__device__ __forceinline__ void attn_generic_query(const BwppAttnArgs &a, uint32_t bh, uint32_t qi, float scale,
                                                   float *qs, float *ps) {
  const uint32_t Kd = a.kdim, Dv = a.vdim;
  const int lane = threadIdx.x & 63;
  const uint32_t b = bh / a.heads, h = bh % a.heads;
  const T *Q = static_cast<const T *>(a.q) + b * a.q_bs + h * a.q_hs;
  const T *K = static_cast<const T *>(a.k) + b * a.k_bs + h * a.k_hs;
  const T *V = static_cast<const T *>(a.v) + b * a.v_bs + h * a.v_hs;
  T *O = static_cast<T *>(a.o) + b * a.o_bs + h * a.o_hs;
  const int64_t diag = (int64_t)a.N - (int64_t)a.M;

  for (uint32_t k = (uint32_t)lane; k < Kd; k += 64) qs[k] = ld_elem(Q + (size_t)qi * a.ldq + k);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  int64_t lim = CAUSAL ? (int64_t)qi + diag + 1 : (int64_t)a.N;
  lim = lim < 0 ? 0 : (lim > (int64_t)a.N ? (int64_t)a.N : lim);
  const uint32_t kend = (uint32_t)lim;
  float m = -INFINITY, l = 0.0f;
  float o[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) o[j] = 0.0f;
  for (uint32_t n0 = 0; n0 < kend; n0 += 64) {
    const uint32_t n = n0 + (uint32_t)lane;
    float s = -INFINITY;
    if (n < kend) {
      s = dot_row(qs, K + (size_t)n * a.ldk, Kd, 0.0f) * scale;
    }
    const float cm = wave_max(s);
    const float mnew = fmaxf(m, cm);
    const float muse = mnew == -INFINITY ? 0.0f : mnew;
    const float alpha = expf(m - muse);
    const float p = n < kend ? expf(s - muse) : 0.0f;
    l = l * alpha + wave_sum(p);
    m = mnew;
    __builtin_amdgcn_wave_barrier();
    ps[lane] = p;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t cnt = min(64u, kend - n0);
#pragma unroll
    for (int j = 0; j < DPL; ++j) o[j] *= alpha;
    axpy_rows<T, DPL>(o, ps, V + (size_t)n0 * a.ldv, a.ldv, cnt, Dv, lane);
    __builtin_amdgcn_wave_barrier();
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
  for (int j = 0; j < DPL; ++j) {
    const uint32_t d = (uint32_t)lane + 64u * j;
    if (d < Dv) st_elem(O + (size_t)qi * a.ldo + d, o[j] * inv);
  }
  if (a.lse && lane == 0) a.lse[(size_t)bh * a.M + qi] = l > 0.0f ? m + logf(l) : -INFINITY;
  __builtin_amdgcn_wave_barrier();
}

template <class T, bool CAUSAL>
__device__ __forceinline__ void attn_generic(const BwppAttnArgs &a) {
  __shared__ float qs[kWaves][kGenMaxDim];
  __shared__ float ps[kWaves][64];
  const int wave = threadIdx.x >> 6;
  const uint32_t nbh = gridDim.x / a.q_tiles;
  const uint32_t qt = a.q_tiles - 1 - blockIdx.x / nbh;
  const uint32_t bh = blockIdx.x % nbh;
  for (uint32_t qq = (uint32_t)wave; qq < a.items; qq += kWaves) {
    const uint32_t qi = qt * a.items + qq;
    if (qi >= a.M) break;  // wave-uniform
    attn_generic_query<T, CAUSAL, kGenMaxDim / 64>(a, bh, qi, a.scale_log2 /* the plain scale on this path */, qs[wave],
                                                  ps[wave]);
  }
}

// --------------------------------------- bf16 forward, head dims 32, 64, 96
// The flash scheme above (S^T = K Q^T on the matrix cores, softmax on the
// accumulator registers, O^T += V^T P^T) for the smaller head dims, with the
// probabilities at fp32 precision: P enters the second product as two bf16
// terms, its upper 16 bits and the rounded rest (2^-16 of p together), so O
// is as the fp32 arithmetic of the generic path gives it (error against 64
// bits at B4 H16 S1000 d64: the rounding of the bf16 result, 1.6e-3, both
// ways).  The second MFMA per V^T operand is cheap here: at d = 64 the
// softmax (exp, max, sum, split: ~14 VALU slots per score) bounds the loop,
// not the matrix pipe.
//
// A block of 4 waves owns 128 queries, each wave 32; keys stream in tiles of
// 64 through a two-stage LDS ring filled by DMA.  Smaller tiles than d =
// 128's: 16 KiB per stage and 126 registers leave room for four blocks per
// CU, whose waves cover each other's barriers, and 128-query blocks fill the
// chip at training's usual batch x heads (B4 H16 S1000: 512 blocks).
// Measured there, causal: generic path 3784 us, this 32 us.
//
// Values that no query sees stay out: a masked key has p = 0, but 0 * v is
// NaN for an infinite or NaN v.  Tiles with masked keys therefore look for
// non-finite V elements, and a wave that finds one takes its queries through
// the generic path's loop instead, which reads visible keys only.
template <int D>
struct AttnTile {
  static constexpr int kSlots = D <= 64 ? 8 : 16;  // 16-byte chunks per LDS row (D / 8 of them in use)
  static constexpr int kRowB = 16 * kSlots;
  // Chunk c of K row r: the 16 rows of a quarter-wave's ds_read_b128 fall
  // on 16 distinct 16-byte slots of the 64 banks.
  static __device__ __forceinline__ uint32_t k_swz(uint32_t r) { return kSlots == 8 ? (r >> 1) & 7u : r & 15u; }
  // Chunk c of V row r: the 4 rows x 4 chunks of a half-wave's transposing
  // reads likewise; unchanged by steps of 8 rows.
  static __device__ __forceinline__ uint32_t v_swz(uint32_t r) {
    return kSlots == 8 ? 4u * ((r >> 1) & 1u) : 4u * (r & 3u);
  }
};

template <int D, bool CAUSAL>
__device__ __forceinline__ void attn_bf16_small(const BwppAttnArgs &a) {
  using T = AttnTile<D>;
  constexpr int NW = 4, kBKV = 64, KS = D / 16, DB = D / 32, KB = kBKV / 32;
  constexpr int kTile = kBKV * T::kRowB, kStage = 2 * kTile;
  constexpr int kBlkPW = kTile / 1024 / NW;  // 1 KiB DMA blocks per wave per K (or V) tile
  constexpr int kOut = NW * kQW * T::kRowB;
  static_assert(2 * kStage >= kOut && 2 * kStage >= NW * 4 * (D + 64), "epilogues reuse the ring");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * kStage];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // Contiguous runs of slices per XCD, as in attn_bf16_d128; the longest
  // (last) query tile of a slice first.
  const uint32_t G = gridDim.x, QT = a.q_tiles;
  const uint32_t lb = G % 8u == 0 ? (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u : blockIdx.x;
  const uint32_t bh = lb / QT, qt = QT - 1 - lb % QT;
  const uint32_t b = bh / a.heads, h = bh % a.heads;
  const uint16_t *Q = static_cast<const uint16_t *>(a.q) + b * a.q_bs + h * a.q_hs;
  const uint16_t *K = static_cast<const uint16_t *>(a.k) + b * a.k_bs + h * a.k_hs;
  const uint16_t *V = static_cast<const uint16_t *>(a.v) + b * a.v_bs + h * a.v_hs;
  uint16_t *O = static_cast<uint16_t *>(a.o) + b * a.o_bs + h * a.o_hs;
  const int64_t diag = (int64_t)a.N - (int64_t)a.M;  // key n visible to query m iff n <= m + diag

  const uint32_t qb0 = qt * (NW * kQW), q0 = qb0 + (uint32_t)wave * kQW;
  const uint32_t lq = (uint32_t)(lane & 31), lh = (uint32_t)(lane >> 5);
  const uint32_t qi = q0 + lq;

  uint32_t kend = a.N;
  if (CAUSAL) {
    const int64_t lim = (int64_t)min(qb0 + NW * kQW, a.M) + diag;
    kend = lim <= 0 ? 0u : (uint32_t)min<int64_t>(lim, a.N);
  }
  const uint32_t nkt = (kend + kBKV - 1) / kBKV;

  bf16x8_t qf[KS];  // query qi, d = 16 ks + 8 lh .. + 7
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    uint4 v = make_uint4(0, 0, 0, 0);
    if (qi < a.M) v = *reinterpret_cast<const uint4 *>(Q + (size_t)qi * a.ldq + 16 * ks + 8 * lh);
    qf[ks] = __builtin_bit_cast(bf16x8_t, v);
  }
  wait_vmcnt<0>();  // no load of the compiler's outstanding beside the DMA

  // DMA: lane l of block i fills 16-byte slot l of it.  Rows past N re-read
  // row N - 1 (masked below), slots past D / 8 a chunk of their row (unread).
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
  uint32_t dma_row[kBlkPW], dma_kcol[kBlkPW], dma_vcol[kBlkPW];
#pragma unroll
  for (int i = 0; i < kBlkPW; ++i) {
    const uint32_t q = (uint32_t)(wave * kBlkPW + i) * 64u + (uint32_t)lane;
    const uint32_t r = q / T::kSlots, pc = q % T::kSlots;
    const uint32_t kc = pc ^ T::k_swz(r), vc = pc ^ T::v_swz(r);
    dma_row[i] = r;
    dma_kcol[i] = 8u * (kc < D / 8 ? kc : kc % (D / 8));
    dma_vcol[i] = 8u * (vc < D / 8 ? vc : vc % (D / 8));
  }
  auto issue = [&](uint32_t t) {
    const uint32_t st = lds0 + (t & 1u) * kStage + (uint32_t)(wave * kBlkPW) * 1024u;
#pragma unroll
    for (int i = 0; i < kBlkPW; ++i) {
      uint32_t key = t * kBKV + dma_row[i];
      key = key < a.N ? key : a.N - 1;
      g2lds16_so(K, 2u * (key * a.ldk + dma_kcol[i]), st + (uint32_t)i * 1024u);
      g2lds16_so(V, 2u * (key * a.ldv + dma_vcol[i]), st + kTile + (uint32_t)i * 1024u);
    }
  };

  f32x16_t o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
  float mrow = -INFINITY, lrow = 0.0f;
  bool redo = false;  // wave-uniform
  const float c = a.scale_log2;

  const uint32_t grp = (uint32_t)((lane >> 4) & 3), L = (uint32_t)(lane & 15);
  uint32_t koff[KS], voff[DB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = lq * T::kRowB + 16u * ((2u * ks + lh) ^ T::k_swz(lq));
  {
    const uint32_t kbase = 4u * (grp >> 1) + (L >> 2);
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      const uint32_t col = 32u * d + 16u * (grp & 1u) + 4u * (L & 3u);
      voff[d] = kTile + kbase * T::kRowB + 16u * ((col >> 3) ^ T::v_swz(kbase)) + (col & 7u) * 2u;
    }
  }

  auto tile = [&](auto mask_tag, const unsigned char *Ks, uint32_t k0) {
    constexpr bool MASK = decltype(mask_tag)::value;
    int kbmax = KB - 1;  // last 32-key block that a query of this wave sees
    if constexpr (MASK) {
      int64_t kv = (int64_t)a.N - 1 - (int64_t)k0;
      if (CAUSAL) kv = min(kv, (int64_t)(q0 + kQW - 1) + diag - (int64_t)k0);
      kbmax = __builtin_amdgcn_readfirstlane(kv < 0 ? -1 : (int)min<int64_t>(kv / 32, KB - 1));
    }
    f32x16_t s[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[kb][r] = 0.0f;
      if (MASK && kb > kbmax) continue;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bf16x8_t kf =
            __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(Ks + koff[ks] + 32u * T::kRowB * kb));
        s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[kb], 0, 0, 0);
      }
    }
    float mx = -INFINITY;
    if constexpr (MASK) {
      // Key of register r in block kb: k0 + 4 lh + 32 kb + 8 (r >> 2) + (r & 3).
      int64_t lim64 = (int64_t)a.N - (int64_t)(k0 + 4u * lh);
      if (CAUSAL) lim64 = min(lim64, (int64_t)qi + diag + 1 - (int64_t)(k0 + 4u * lh));
      const int lim = (int)(lim64 < -1 ? -1 : (lim64 > kBKV ? kBKV : lim64));
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        if (kb > kbmax) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float x = (32 * kb + 8 * (r >> 2) + (r & 3)) < lim ? s[kb][r] : -INFINITY;
          s[kb][r] = x;
          mx = fmaxf(mx, x);
        }
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
    }
    {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * c;
    }
    float alpha = 1.0f;
    if (mx > mrow + kLazy) {
      alpha = __builtin_amdgcn_exp2f(mrow - mx);  // 0 when mrow is -inf
      mrow = mx;
    }
    const float muse = mrow == -INFINITY ? 0.0f : mrow;
    float sum = 0.0f;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      if (MASK && kb > kbmax) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], c, -muse));
        s[kb][r] = p;
        sum += p;
      }
    }
    {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
      sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    lrow = lrow * alpha + sum;
    if (__ballot(alpha != 1.0f)) {
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
    }
    u16x2_t big = {0, 0};  // largest |V| bit patterns of a masked tile
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      if (MASK && kb > kbmax) continue;
#pragma unroll
      for (int kq = 0; kq < 2; ++kq) {
        bf16x8_t ph, pl;
        split_bf16x8(&s[kb], 8 * kq, ph, pl);
        const uint32_t rstep = (32u * kb + 16u * kq) * T::kRowB;
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(Ks + voff[d] + rstep));
          const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(Ks + voff[d] + rstep + 8u * T::kRowB));
          const v8s_t vv = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          if constexpr (MASK) big = max_abs_bf16(big, vv);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vv), ph, o[d], 0, 0, 0);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vv), pl, o[d], 0, 0, 0);
        }
      }
    }
    if constexpr (MASK) redo = redo || __ballot(big[0] >= 0x7f80u || big[1] >= 0x7f80u) != 0;
  };

  if (nkt > 0) issue(0);
  // Tiles before t_mask need no mask for any query of the block.
  uint32_t t_mask = a.N / kBKV;
  if (CAUSAL) {
    const int64_t first_hidden = (int64_t)qb0 + diag + 1;
    t_mask = min(t_mask, first_hidden <= 0 ? 0u : (uint32_t)min<int64_t>(first_hidden / kBKV, (int64_t)nkt));
  }
  t_mask = min(t_mask, nkt);
  auto step = [&](uint32_t t) {
    wait_vmcnt<0>();
    __syncthreads();
    if (t + 1 < nkt) issue(t + 1);
    return smem + __builtin_amdgcn_readfirstlane((t & 1u) * kStage);
  };
  for (uint32_t t = 0; t < t_mask; ++t) {
    const unsigned char *Ks = step(t);
    tile(std::integral_constant<bool, false>{}, Ks, t * kBKV);
  }
  for (uint32_t t = t_mask; t < nkt; ++t) {
    const unsigned char *Ks = step(t);
    const uint32_t k0 = t * kBKV;
    if (CAUSAL && (int64_t)k0 > (int64_t)(q0 + kQW - 1) + diag) continue;  // no query of the wave sees it
    tile(std::integral_constant<bool, true>{}, Ks, k0);
  }
  __syncthreads();

  if (redo) {
    float *qs = reinterpret_cast<float *>(smem) + wave * (D + 64);
    for (uint32_t q = q0; q < min(q0 + kQW, a.M); ++q)
      attn_generic_query<uint16_t, CAUSAL, (D + 63) / 64>(a, bh, q, a.scale, qs, qs + D);
  }
  __syncthreads();  // a wave's staging below may lie in another's qs
  if (redo) return;
  if (a.lse && lh == 0 && qi < a.M)
    a.lse[(size_t)bh * a.M + qi] =
        lrow > 0.0f ? lse_of(mrow == -INFINITY ? 0.0f : mrow, lrow) : -INFINITY;
  uint16_t *os = reinterpret_cast<uint16_t *>(smem) + (size_t)wave * kQW * (T::kRowB / 2);
  const float inv = lrow > 0.0f ? 1.0f / lrow : 0.0f;
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      uint2 w;
      w.x = pack_bf16x2(o[d][4 * q4 + 0] * inv, o[d][4 * q4 + 1] * inv);
      w.y = pack_bf16x2(o[d][4 * q4 + 2] * inv, o[d][4 * q4 + 3] * inv);
      *reinterpret_cast<uint2 *>(os + lq * (T::kRowB / 2) + 8u * ((4u * d + q4) ^ T::k_swz(lq)) + 4u * lh) = w;
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  constexpr int kRowChunks = D / 8;
#pragma unroll
  for (int it = 0; it < kQW * kRowChunks / 64; ++it) {
    const uint32_t q = (uint32_t)(lane + it * 64), ql = q / kRowChunks, cc = q % kRowChunks;
    if (q0 + ql < a.M)
      __builtin_nontemporal_store(
          *reinterpret_cast<const u32x4_t *>(os + ql * (T::kRowB / 2) + 8u * (cc ^ T::k_swz(ql))),
          reinterpret_cast<u32x4_t *>(O + (size_t)(q0 + ql) * a.ldo + 8u * cc));
  }
}

// -------------------------------------------------- bf16, at most 32 queries
// Decoding: a few queries against a long cache, bound by reading K and V
// once (4 flop per byte and query).  A block of 4 waves owns one slice and a
// range of its keys; every wave holds all the queries as the MFMA "B" operand
// and streams key tiles of 32 of its own (every fourth of the block's)
// through a DMA ring of its own, so the waves never wait for one another:
// 16 KiB of K and V per wave in flight while the previous tile is multiplied.
// The waves' (offset, sum, O) triples meet in LDS at the end, and those of a
// split slice in bwpp_attn_dec_combine.  P enters the second product as two
// bf16 terms (see above).  B8 H32 M1 N4095 d128: 256-query tiles, one block
// per slice 116-144 us, this 94 us (537 MB at 5.7 TB/s); B1 H32 M1 N8192 172
// -> 27 (split 8 ways).
//
// Tiles with masked keys look for non-finite V elements; where one is found
// the tile's sums are formed element by element over visible keys only.
template <int D, bool CAUSAL>
__device__ __forceinline__ void attn_bf16_dec(const BwppAttnArgs &a) {
  using T = AttnTile<D>;
  constexpr int NW = 4, kKeys = 32, KS = D / 16, DB = D / 32;
  constexpr int kTile = kKeys * T::kRowB, kStage = 2 * kTile;
  constexpr int kStages = 32768 / kStage;      // 32 KiB per wave
  constexpr int kDma = kTile / 1024;           // DMA instructions per K (or V) tile
  constexpr int kCld = D + 4;                  // merge: [wave][32 queries][D + 4] floats
  static_assert(kStages >= 2 && NW * 32 * kCld * 4 <= NW * kStages * kStage, "merge reuses the rings");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[NW * kStages * kStage];
  __shared__ float ps[NW][kKeys][33];          // a tile's probabilities (non-finite V only)
  __shared__ float mls[NW][32][2];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const uint32_t bh = blockIdx.x / a.ksplit, sp = blockIdx.x % a.ksplit;
  const uint32_t b = bh / a.heads, h = bh % a.heads;
  const uint16_t *Q = static_cast<const uint16_t *>(a.q) + b * a.q_bs + h * a.q_hs;
  const uint16_t *K = static_cast<const uint16_t *>(a.k) + b * a.k_bs + h * a.k_hs;
  const uint16_t *V = static_cast<const uint16_t *>(a.v) + b * a.v_bs + h * a.v_hs;
  const int64_t diag = (int64_t)a.N - (int64_t)a.M;  // key n visible to query m iff n <= m + diag
  const uint32_t lq = (uint32_t)(lane & 31), lh = (uint32_t)(lane >> 5);

  // Keys of this block: [kbeg, kend), kbeg a multiple of 32.
  const uint32_t kbeg = sp * a.kchunk, kend = min(a.N, kbeg + a.kchunk);
  const uint32_t ntile = kbeg < kend ? (kend - kbeg + kKeys - 1) / kKeys : 0u;
  const uint32_t nmine = ntile > (uint32_t)wave ? (ntile - (uint32_t)wave + NW - 1) / NW : 0u;

  bf16x8_t qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    uint4 v = make_uint4(0, 0, 0, 0);
    if (lq < a.M) v = *reinterpret_cast<const uint4 *>(Q + (size_t)lq * a.ldq + 16 * ks + 8 * lh);
    qf[ks] = __builtin_bit_cast(bf16x8_t, v);
  }
  wait_vmcnt<0>();  // no load of the compiler's outstanding beside the DMA

  unsigned char *ring = smem + wave * (kStages * kStage);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)ring;
  uint32_t dma_row[kDma], dma_kcol[kDma], dma_vcol[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const uint32_t q = (uint32_t)i * 64u + (uint32_t)lane, r = q / T::kSlots, pc = q % T::kSlots;
    dma_row[i] = r;
    dma_kcol[i] = 8u * (pc ^ T::k_swz(r));
    dma_vcol[i] = 8u * (pc ^ T::v_swz(r));
  }
  static_assert(D / 8 == T::kSlots, "every slot of a row is in use");
  // Tile j of this wave: keys from kbeg + 32 (4 j + wave); rows past N
  // re-read row N - 1 (masked below).
  auto issue = [&](uint32_t j) {
    const uint32_t k0 = kbeg + kKeys * (NW * j + (uint32_t)wave), st = lds0 + (j % kStages) * kStage;
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
      const uint32_t key = min(k0 + dma_row[i], a.N - 1);
      g2lds16_so(K, 2u * (key * a.ldk + dma_kcol[i]), st + (uint32_t)i * 1024u);
      g2lds16_so(V, 2u * (key * a.ldv + dma_vcol[i]), st + kTile + (uint32_t)i * 1024u);
    }
  };

  f32x16_t o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
  float mrow = -INFINITY, lrow = 0.0f;
  const float c = a.scale_log2;
  const uint32_t grp = (uint32_t)((lane >> 4) & 3), L = (uint32_t)(lane & 15);
  uint32_t koff[KS], voff[DB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = lq * T::kRowB + 16u * ((2u * ks + lh) ^ T::k_swz(lq));
  {
    const uint32_t kbase = 4u * (grp >> 1) + (L >> 2);
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      const uint32_t col = 32u * d + 16u * (grp & 1u) + 4u * (L & 3u);
      voff[d] = kTile + kbase * T::kRowB + 16u * ((col >> 3) ^ T::v_swz(kbase)) + (col & 7u) * 2u;
    }
  }

#pragma unroll
  for (int j = 0; j < kStages - 1; ++j)
    if ((uint32_t)j < nmine) issue((uint32_t)j);
  for (uint32_t j = 0; j < nmine; ++j) {
    const uint32_t k0 = kbeg + kKeys * (NW * j + (uint32_t)wave);
    const uint32_t younger = min(nmine - 1 - j, (uint32_t)(kStages - 2));
    if (kStages >= 4 && younger >= 2) wait_vmcnt<(kStages >= 4 ? 4 * kDma : 0)>();
    else if (kStages >= 3 && younger >= 1) wait_vmcnt<(kStages >= 3 ? 2 * kDma : 0)>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): done reading the stage that is refilled now
    if (j + kStages - 1 < nmine) issue(j + kStages - 1);
    const unsigned char *st = ring + __builtin_amdgcn_readfirstlane((j % kStages) * kStage);
    f32x16_t s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(st + koff[ks])), qf[ks], s, 0, 0, 0);
    // Key of register r: k0 + 4 lh + 8 (r >> 2) + (r & 3); visible below lim.
    const bool masked = k0 + kKeys > kend || (CAUSAL && (int64_t)k0 + kKeys - 1 > diag);  // wave-uniform
    int64_t lim64 = (int64_t)kend - (int64_t)(k0 + 4u * lh);
    if (CAUSAL) lim64 = min(lim64, (int64_t)lq + diag + 1 - (int64_t)(k0 + 4u * lh));
    const int lim = (int)(lim64 < -1 ? -1 : (lim64 > kKeys ? kKeys : lim64));
    if (masked) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 8 * (r >> 2) + (r & 3) < lim ? s[r] : -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * c;
    }
    float alpha = 1.0f;
    if (mx > mrow + kLazy) {
      alpha = __builtin_amdgcn_exp2f(mrow - mx);  // 0 when mrow is -inf
      mrow = mx;
    }
    const float muse = mrow == -INFINITY ? 0.0f : mrow;
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c, -muse));
      s[r] = p;
      sum += p;
    }
    {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
      sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    lrow = lrow * alpha + sum;
    if (__ballot(alpha != 1.0f)) {
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
    }
    v8s_t vv[2][DB];
#pragma unroll
    for (int kq = 0; kq < 2; ++kq)
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const unsigned char *p = st + voff[d] + 16u * kq * T::kRowB;
        const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)p);
        const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(p + 8u * T::kRowB));
        vv[kq][d] = v8s_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    bool plain = true;
    if (masked) {
      u16x2_t big = {0, 0};
#pragma unroll
      for (int kq = 0; kq < 2; ++kq)
#pragma unroll
        for (int d = 0; d < DB; ++d) big = max_abs_bf16(big, vv[kq][d]);
      plain = __ballot(big[0] >= 0x7f80u || big[1] >= 0x7f80u) == 0;
    }
    if (plain) {
#pragma unroll
      for (int kq = 0; kq < 2; ++kq) {
        bf16x8_t ph, pl;
        split_bf16x8(&s, 8 * kq, ph, pl);
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vv[kq][d]), ph, o[d], 0, 0, 0);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vv[kq][d]), pl, o[d], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) ps[wave][8 * (r >> 2) + 4 * lh + (r & 3)][lq] = s[r];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int64_t vis = lim64 + 4 * (int64_t)lh;  // keys of the tile that this lane's query sees
      for (int key = 0; key < kKeys; ++key) {
        const float p = ps[wave][key][lq];
        const unsigned char *vr = st + kTile + (uint32_t)key * T::kRowB;
        if (key < vis) {
#pragma unroll
          for (int d = 0; d < DB; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const uint32_t col = 32u * d + 8u * (r >> 2) + 4u * lh + (r & 3);
              const uint16_t *e = reinterpret_cast<const uint16_t *>(
                  vr + 16u * ((col >> 3) ^ T::v_swz((uint32_t)key)) + 2u * (col & 7u));
              o[d][r] += p * bf16_bits_to_f32(*e);
            }
        }
      }
    }
  }

  // The four waves' triples: O (this lane's query, d = 32 db + 8 (r >> 2) +
  // 4 lh + (r & 3)) and (offset, sum).
  __syncthreads();
  float *os = reinterpret_cast<float *>(smem) + wave * (32 * kCld);
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4)
      *reinterpret_cast<float4 *>(os + lq * kCld + 32 * d + 8 * q4 + 4 * (int)lh) =
          make_float4(o[d][4 * q4], o[d][4 * q4 + 1], o[d][4 * q4 + 2], o[d][4 * q4 + 3]);
  if (lh == 0) {
    mls[wave][lq][0] = mrow;
    mls[wave][lq][1] = lrow;
  }
  __syncthreads();
  uint16_t *O = static_cast<uint16_t *>(a.o) + b * a.o_bs + h * a.o_hs;
  for (uint32_t i = threadIdx.x; i < a.M * (D / 4); i += 64 * NW) {
    const uint32_t q = i / (D / 4), d4 = 4u * (i % (D / 4));
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) m = fmaxf(m, mls[w][q][0]);
    float l = 0.0f;
    float4 t = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = mls[w][q][0];
      // No key seen (offset -inf): sums of 0 (or NaN, kept).
      const float f = mw == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(mw - m);
      const float4 u = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(smem) + (w * 32 + q) * kCld + d4);
      l += mls[w][q][1] * f;
      t.x += u.x * f, t.y += u.y * f, t.z += u.z * f, t.w += u.w * f;
    }
    if (a.ksplit > 1) {
      const size_t row = (size_t)blockIdx.x * a.M + q;
      *reinterpret_cast<float4 *>(a.part_o + row * D + d4) = t;
      if (d4 == 0) {
        a.part_ml[2 * row] = m;
        a.part_ml[2 * row + 1] = l;
      }
      continue;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    *reinterpret_cast<uint2 *>(O + (size_t)q * a.ldo + d4) =
        make_uint2(pack_bf16x2(t.x * inv, t.y * inv), pack_bf16x2(t.z * inv, t.w * inv));
    if (a.lse && d4 == 0)
      a.lse[(size_t)bh * a.M + q] =
          l > 0.0f ? lse_of(m == -INFINITY ? 0.0f : m, l) : -INFINITY;
  }
}

// Merges the ksplit partial triples of a slice's queries: a thread per four
// d of one query.
template <class T>
__device__ __forceinline__ void attn_dec_combine(const BwppAttnArgs &a, uint32_t slices) {
  const uint32_t D = a.vdim, n4 = D / 4;
  const uint64_t total = (uint64_t)slices * a.M * n4;
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < total; i += (uint64_t)gridDim.x * 256u) {
    const uint32_t d4 = 4u * (uint32_t)(i % n4), q = (uint32_t)(i / n4 % a.M), bh = (uint32_t)(i / n4 / a.M);
    const size_t row0 = (size_t)bh * a.ksplit * a.M + q;
    float m = -INFINITY;
    for (uint32_t s = 0; s < a.ksplit; ++s) m = fmaxf(m, a.part_ml[2 * (row0 + (size_t)s * a.M)]);
    float l = 0.0f;
    float4 t = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 4
    for (uint32_t s = 0; s < a.ksplit; ++s) {
      const size_t row = row0 + (size_t)s * a.M;
      const float mw = a.part_ml[2 * row];
      const float f = mw == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(mw - m);
      const float4 u = *reinterpret_cast<const float4 *>(a.part_o + row * D + d4);
      l += a.part_ml[2 * row + 1] * f;
      t.x += u.x * f, t.y += u.y * f, t.z += u.z * f, t.w += u.w * f;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    T *O = static_cast<T *>(a.o) + bh / a.heads * a.o_bs + bh % a.heads * a.o_hs + (size_t)q * a.ldo + d4;
    st_elem(O, t.x * inv), st_elem(O + 1, t.y * inv), st_elem(O + 2, t.z * inv), st_elem(O + 3, t.w * inv);
    if (a.lse && d4 == 0)
      a.lse[(size_t)bh * a.M + q] =
          l > 0.0f ? lse_of(m == -INFINITY ? 0.0f : m, l) : -INFINITY;
  }
}

// ------------------------------------------------------- backward (generic)
// O = softmax(scale Q K^T [mask]) V.  With the saved lse (natural-log
// log-sum-exp per query) the probabilities are recomputed as
// p = exp(scale q.k - lse) and, with D_m = rowsum(dO * O)[m],
//   dS = p (dO.v - D_m),  dQ = scale dS K,  dK = scale dS^T Q,  dV = P^T dO.
// Two passes, both one wave per row with fp32 arithmetic and any head dims
// up to 512: attn_bwd_dq (one query per wave; also writes D_m) and then
// attn_bwd_dkdv (one key per wave, looping over the queries that see it).

template <class T, bool CAUSAL>
__device__ __forceinline__ void attn_bwd_dq(const BwppAttnArgs &a) {
  const uint32_t Kd = a.kdim, Dv = a.vdim;
  __shared__ float qs[kWaves][kGenMaxDim];
  __shared__ float gs[kWaves][kGenMaxDim];
  __shared__ float ps[kWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t nbh = gridDim.x / a.q_tiles;
  const uint32_t qt = a.q_tiles - 1 - blockIdx.x / nbh;
  const uint32_t bh = blockIdx.x % nbh;
  const uint32_t b = bh / a.heads, h = bh % a.heads;
  const T *Q = static_cast<const T *>(a.q) + b * a.q_bs + h * a.q_hs;
  const T *K = static_cast<const T *>(a.k) + b * a.k_bs + h * a.k_hs;
  const T *V = static_cast<const T *>(a.v) + b * a.v_bs + h * a.v_hs;
  const T *O = static_cast<const T *>(a.o) + b * a.o_bs + h * a.o_hs;
  const T *dO = static_cast<const T *>(a.dout) + b * a.o_bs + h * a.o_hs;
  T *dQ = static_cast<T *>(a.dq) + b * a.q_bs + h * a.q_hs;
  const int64_t diag = (int64_t)a.N - (int64_t)a.M;
  const float scale = a.scale_log2;  // the plain scale on this path
  constexpr int DPL = kGenMaxDim / 64;

  for (uint32_t qq = (uint32_t)wave; qq < a.items; qq += kWaves) {
    const uint32_t qi = qt * a.items + qq;
    if (qi >= a.M) break;  // wave-uniform
    for (uint32_t k = (uint32_t)lane; k < Kd; k += 64) qs[wave][k] = ld_elem(Q + (size_t)qi * a.ldq + k);
    float dsum = 0.0f;
    for (uint32_t d = (uint32_t)lane; d < Dv; d += 64) {
      const float g = ld_elem(dO + (size_t)qi * a.ldo + d);
      gs[wave][d] = g;
      dsum += g * ld_elem(O + (size_t)qi * a.ldo + d);
    }
    dsum = wave_sum(dsum);
    if (lane == 0) a.dsum[(size_t)bh * a.M + qi] = dsum;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float lse = a.lse[(size_t)bh * a.M + qi];
    int64_t lim = CAUSAL ? (int64_t)qi + diag + 1 : (int64_t)a.N;
    lim = lim < 0 ? 0 : (lim > (int64_t)a.N ? (int64_t)a.N : lim);
    const uint32_t kend = (uint32_t)lim;
    float acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0.0f;
    for (uint32_t n0 = 0; n0 < kend; n0 += 64) {
      const uint32_t n = n0 + (uint32_t)lane;
      float ds = 0.0f;
      if (n < kend) {
        const float s = dot_row(qs[wave], K + (size_t)n * a.ldk, Kd, 0.0f);
        const float dp = dot_row(gs[wave], V + (size_t)n * a.ldv, Dv, 0.0f);
        const float p = expf(s * scale - lse);
        ds = p * (dp - dsum);
      }
      __builtin_amdgcn_wave_barrier();
      ps[wave][lane] = ds;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const uint32_t cnt = min(64u, kend - n0);
      axpy_rows<T, DPL>(acc, ps[wave], K + (size_t)n0 * a.ldk, a.ldk, cnt, Kd, lane);
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
      const uint32_t k = (uint32_t)lane + 64u * j;
      if (k < Kd) st_elem(dQ + (size_t)qi * a.ldq + k, acc[j] * scale);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <class T, bool CAUSAL>
__device__ __forceinline__ void attn_bwd_dkdv(const BwppAttnArgs &a) {
  const uint32_t Kd = a.kdim, Dv = a.vdim;
  __shared__ float ks[kWaves][kGenMaxDim];
  __shared__ float vs[kWaves][kGenMaxDim];
  __shared__ float pp[kWaves][64];
  __shared__ float dd[kWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t nbh = gridDim.x / a.q_tiles;  // q_tiles holds the key tiles here
  const uint32_t kt = a.q_tiles - 1 - blockIdx.x / nbh;
  const uint32_t bh = blockIdx.x % nbh;
  const uint32_t b = bh / a.heads, h = bh % a.heads;
  const T *Q = static_cast<const T *>(a.q) + b * a.q_bs + h * a.q_hs;
  const T *K = static_cast<const T *>(a.k) + b * a.k_bs + h * a.k_hs;
  const T *V = static_cast<const T *>(a.v) + b * a.v_bs + h * a.v_hs;
  const T *dO = static_cast<const T *>(a.dout) + b * a.o_bs + h * a.o_hs;
  T *dK = static_cast<T *>(a.dk) + b * a.k_bs + h * a.k_hs;
  T *dV = static_cast<T *>(a.dv) + b * a.v_bs + h * a.v_hs;
  const float *lse = a.lse + (size_t)bh * a.M;
  const float *dsum = a.dsum + (size_t)bh * a.M;
  const int64_t diag = (int64_t)a.N - (int64_t)a.M;
  const float scale = a.scale_log2;
  constexpr int DPL = kGenMaxDim / 64;

  for (uint32_t kk = (uint32_t)wave; kk < a.items; kk += kWaves) {
    const uint32_t n = kt * a.items + kk;
    if (n >= a.N) break;  // wave-uniform
    for (uint32_t k = (uint32_t)lane; k < Kd; k += 64) ks[wave][k] = ld_elem(K + (size_t)n * a.ldk + k);
    for (uint32_t d = (uint32_t)lane; d < Dv; d += 64) vs[wave][d] = ld_elem(V + (size_t)n * a.ldv + d);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // Queries that see key n: m >= n - diag (causal), all otherwise.
    int64_t first = CAUSAL ? (int64_t)n - diag : 0;
    first = first < 0 ? 0 : first;
    const uint32_t mbeg = first > (int64_t)a.M ? a.M : (uint32_t)first;
    float gk[DPL], gv[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) gk[j] = gv[j] = 0.0f;
    for (uint32_t m0 = mbeg; m0 < a.M; m0 += 64) {
      const uint32_t m = m0 + (uint32_t)lane;
      float p = 0.0f, ds = 0.0f;
      if (m < a.M) {
        const float s = dot_row(ks[wave], Q + (size_t)m * a.ldq, Kd, 0.0f);
        const float dp = dot_row(vs[wave], dO + (size_t)m * a.ldo, Dv, 0.0f);
        p = expf(s * scale - lse[m]);
        ds = p * (dp - dsum[m]);
      }
      __builtin_amdgcn_wave_barrier();
      pp[wave][lane] = p;
      dd[wave][lane] = ds;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const uint32_t cnt = min(64u, a.M - m0);
      axpy_rows<T, DPL>(gk, dd[wave], Q + (size_t)m0 * a.ldq, a.ldq, cnt, Kd, lane);
      axpy_rows<T, DPL>(gv, pp[wave], dO + (size_t)m0 * a.ldo, a.ldo, cnt, Dv, lane);
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
      const uint32_t c = (uint32_t)lane + 64u * j;
      if (c < Kd) st_elem(dK + (size_t)n * a.ldk + c, gk[j] * scale);
      if (c < Dv) st_elem(dV + (size_t)n * a.ldv + c, gv[j]);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace

#define BWPP_ATTN_BWD(NAME, T, CAUSAL)                                                      \
  extern "C" __global__ __launch_bounds__(256) void NAME##_dq(const BwppAttnArgs a) {       \
    attn_bwd_dq<T, CAUSAL>(a);                                                             \
  }                                                                                        \
  extern "C" __global__ __launch_bounds__(256) void NAME##_dkdv(const BwppAttnArgs a) {     \
    attn_bwd_dkdv<T, CAUSAL>(a);                                                           \
  }
BWPP_ATTN_BWD(bwpp_attn_bwd_f32, float, false)
BWPP_ATTN_BWD(bwpp_attn_bwd_f32_causal, float, true)
BWPP_ATTN_BWD(bwpp_attn_bwd_bf16, uint16_t, false)
BWPP_ATTN_BWD(bwpp_attn_bwd_bf16_causal, uint16_t, true)

// WPE: waves per SIMD the registers are cut to (the accumulators then stay
// in VGPRs: with the compiler's own choice they moved to AGPRs and every
// score was copied back for the softmax).
#define BWPP_ATTN_SMALL(D, WPE)                                                                \
  extern "C" __global__ __attribute__((amdgpu_flat_work_group_size(256, 256),                  \
                                       amdgpu_waves_per_eu(WPE, WPE))) void                    \
      bwpp_attn_bf16_d##D(const BwppAttnArgs a) {                                              \
    attn_bf16_small<D, false>(a);                                                              \
  }                                                                                            \
  extern "C" __global__ __attribute__((amdgpu_flat_work_group_size(256, 256),                  \
                                       amdgpu_waves_per_eu(WPE, WPE))) void                    \
      bwpp_attn_bf16_d##D##_causal(const BwppAttnArgs a) {                                     \
    attn_bf16_small<D, true>(a);                                                               \
  }
BWPP_ATTN_SMALL(32, 4)
BWPP_ATTN_SMALL(64, 3)
BWPP_ATTN_SMALL(96, 2)

#define BWPP_ATTN_DEC(D)                                                                       \
  extern "C" __global__ __launch_bounds__(256) void bwpp_attn_bf16_dec_d##D(const BwppAttnArgs a) { \
    attn_bf16_dec<D, false>(a);                                                                \
  }                                                                                            \
  extern "C" __global__ __launch_bounds__(256) void bwpp_attn_bf16_dec_d##D##_causal(          \
      const BwppAttnArgs a) {                                                                  \
    attn_bf16_dec<D, true>(a);                                                                 \
  }
BWPP_ATTN_DEC(64)
BWPP_ATTN_DEC(128)
extern "C" __global__ __launch_bounds__(256) void bwpp_attn_dec_combine_bf16(const BwppAttnArgs a) {
  attn_dec_combine<uint16_t>(a, a.items);
}
extern "C" __global__ __launch_bounds__(256) void bwpp_attn_dec_combine_f32(const BwppAttnArgs a) {
  attn_dec_combine<float>(a, a.items);
}

// Generic path entry points, one per storage type x mask.
#define BWPP_ATTN_GENERIC(NAME, T, CAUSAL)                                                  \
  extern "C" __global__ __launch_bounds__(256) void NAME(const BwppAttnArgs a) {            \
    attn_generic<T, CAUSAL>(a);                                                            \
  }
BWPP_ATTN_GENERIC(bwpp_attn_generic_f32, float, false)
BWPP_ATTN_GENERIC(bwpp_attn_generic_f32_causal, float, true)
BWPP_ATTN_GENERIC(bwpp_attn_generic_bf16, uint16_t, false)
BWPP_ATTN_GENERIC(bwpp_attn_generic_bf16_causal, uint16_t, true)

extern "C" __global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void
bwpp_attn_bf16_d128(const BwppAttnArgs a) {
  attn_bf16_d128<false>(a);
}
// Persistent unmasked form (a.items (slice, query tile) items over one
// block per CU).
extern "C" __global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void
bwpp_attn_bf16_d128_p(const BwppAttnArgs a) {
  attn_bf16_d128_persist<false>(a);
}
extern "C" __global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void
bwpp_attn_bf16_d128_causal_p(const BwppAttnArgs a) {
  attn_bf16_d128_persist<true>(a);
}
extern "C" __global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void
bwpp_attn_bf16_d128_causal(const BwppAttnArgs a) {
  attn_bf16_d128<true>(a);
}
