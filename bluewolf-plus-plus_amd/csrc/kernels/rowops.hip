// Bandwidth-bound row operators for gfx950: softmax, RMSNorm, LayerNorm,
// reduce_max (value + argmax), reduce_max mask, and the reduce_max grads.
//
// Semantics follow runtime/cpu/bwpp_cpu_ref.c (softmax :37-61, rmsnorm
// :63-90, reduce_max mask :146-190, grad :192-219); LayerNorm and the
// argmax forms are the closed forms documented in include/bwpp_hip.h.
//
// Main path ("reg"): the row is read from HBM once with 128-bit
// non-temporal loads into registers, reduced with DPP + lane exchanges,
// transformed and written once with 128-bit non-temporal stores (the data is
// streamed exactly once, so it is kept out of the caches' way).  WPR waves
// share a row: WPR < 4 packs 4/WPR rows into a 256-thread block; WPR >= 4
// gives each row a block of 64*WPR threads with a cross-wave step through
// LDS.  Thread g of the row group owns float4 chunks g, g + 64*WPR, ...,
// so each load instruction of the group covers 1 KiB * WPR of contiguous
// memory.  VPT chunks per thread (<= 16) keep the row in registers.
// Blocks loop over row groups with stride gridDim.x (the host may cap the
// grid); the next group's loads are issued before the current group's
// reductions, and gamma/beta chunks are loaded once per block.
//
// Rows start at any 4-byte address (an odd row length): the 128-bit accesses
// need no more, and a misaligned 1 KiB wave access touches nine 128-byte
// lines instead of eight (2047 x 5003: softmax 30.6 -> 17.0 us, LayerNorm 40 ->
// 17.1, RMSNorm 24.4 -> 15.7, reduce_max 11.0 -> 8.8 against the multi-pass
// fallback, 4.8 TB/s; 1 to 3 columns take a thread per row).
//
// Fallback path ("gen"): one 256-thread block per row, scalar loads, several
// passes; rows longer than 32768.
#include "common.h"
#include "../kargs.h"

using namespace bwpp;

namespace {

enum RowOp : int {
  OP_SOFTMAX = 0,
  OP_RMSNORM = 1,
  OP_LAYERNORM = 2,
  OP_MAX = 3,      // maxv + argmax
  OP_MAX_GRAD = 4, // dx one-hot from x
  OP_MASK = 5,     // reference mask (all ties)
};

constexpr uint32_t kNoIndex = 0xFFFFFFFFu;

// Cross-wave steps of the row reductions.  A block holds 4/WPR rows
// (WPR < 4) or one row of WPR waves; waves w0 .. w0+WPR-1 share a row.
// PAIRS: the waves' sums are added in pairs, as the multi-pass fallback adds
// them: rows of any length are as exact as there (softmax's scale at 5003
// columns 0.79 x 2^-24 rms, 0.96 with the eight added one after another).
template <int WPR, bool PAIRS = false>
__device__ __forceinline__ float row_sum(float v, float *red) {
  v = wave_sum(v);
  if constexpr (WPR > 1) {
    const int w = threadIdx.x >> 6, w0 = (w / WPR) * WPR;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    if constexpr (PAIRS) {
      float p[WPR];
#pragma unroll
      for (int i = 0; i < WPR; ++i) p[i] = red[w0 + i];
#pragma unroll
      for (int n = WPR / 2; n > 0; n /= 2)
#pragma unroll
        for (int i = 0; i < n; ++i) p[i] = p[2 * i] + p[2 * i + 1];
      v = p[0];
    } else {
      v = red[w0];
#pragma unroll
      for (int i = 1; i < WPR; ++i) v += red[w0 + i];
    }
  }
  return v;
}

template <int WPR>
__device__ __forceinline__ float row_max(float v, float *red) {
  v = wave_max(v);
  if constexpr (WPR > 1) {
    const int w = threadIdx.x >> 6, w0 = (w / WPR) * WPR;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    v = red[w0];
#pragma unroll
    for (int i = 1; i < WPR; ++i) v = fmaxf(v, red[w0 + i]);
  }
  return v;
}

template <int WPR>
__device__ __forceinline__ void row_argmax(float &v, uint32_t &i, float *redf,
                                           uint32_t *redu) {
  wave_argmax(v, i);
  if constexpr (WPR > 1) {
    const int w = threadIdx.x >> 6, w0 = (w / WPR) * WPR;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
      redf[w] = v;
      redu[w] = i;
    }
    __syncthreads();
    v = redf[w0];
    i = redu[w0];
#pragma unroll
    for (int k = 1; k < WPR; ++k) argmax_merge(v, i, redf[w0 + k], redu[w0 + k]);
  }
}

// Row mean and M2 = sum (x - mean)^2 from per-thread statistics over equal
// counts n (full rows): the equal-weight form of Chan, Golub & LeVeque's
// pairwise update, one exchange per step; WPR waves' (mean, M2) combine as
// mean = average of the means, M2 = sum of M2 + n_wave * sum (mean_i - mean)^2.
template <int WPR>
__device__ __forceinline__ void row_chan_equal(float &n, float &mu, float &m2, float *red) {
  auto merge = [&](float mu2, float m22) {
    const float d = mu2 - mu;
    mu = mu + 0.5f * d;
    m2 = m2 + m22 + d * d * (0.5f * n);
    n = 2.0f * n;
  };
  merge(dpp_f32<kDppQuadXor1>(mu), dpp_f32<kDppQuadXor1>(m2));
  merge(dpp_f32<kDppQuadXor2>(mu), dpp_f32<kDppQuadXor2>(m2));
  merge(dpp_f32<kDppRowHalfMirror>(mu), dpp_f32<kDppRowHalfMirror>(m2));
  merge(dpp_f32<kDppRowMirror>(mu), dpp_f32<kDppRowMirror>(m2));
  merge(xor_f32(mu, 16), xor_f32(m2, 16));
  merge(xor_f32(mu, 32), xor_f32(m2, 32));
  if constexpr (WPR > 1) {
    const int w = threadIdx.x >> 6, w0 = (w / WPR) * WPR;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
      red[2 * w] = mu;
      red[2 * w + 1] = m2;
    }
    __syncthreads();
    float smu = 0.0f;
#pragma unroll
    for (int i = 0; i < WPR; ++i) smu += red[2 * (w0 + i)];
    const float gmu = smu * (1.0f / (float)WPR);
    float sm2 = 0.0f;
#pragma unroll
    for (int i = 0; i < WPR; ++i) {
      const float d = red[2 * (w0 + i)] - gmu;
      sm2 += red[2 * (w0 + i) + 1] + d * d * n;
    }
    mu = gmu;
    m2 = sm2;
    n = n * (float)WPR;
  }
}

template <int WPR>
struct RowGeom {
  static constexpr int kBlock = WPR >= 4 ? 64 * WPR : 256;  // threads per block
  static constexpr int kGroup = 64 * WPR;                    // threads per row
  static constexpr int kRows = kBlock / kGroup;              // rows per block
};

__device__ __forceinline__ float get(const float4 &v, int e) {
  return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w;
}
__device__ __forceinline__ void set(float4 &v, int e, float t) {
  if (e == 0) v.x = t;
  else if (e == 1) v.y = t;
  else if (e == 2) v.z = t;
  else v.w = t;
}

template <int OP, int VPT, int WPR, bool FULL>
__device__ __forceinline__ void row_reg(const BwppRowArgs &a) {
  using G = RowGeom<WPR>;
  constexpr int GT = G::kGroup;
  constexpr bool kNorm = (OP == OP_RMSNORM || OP == OP_LAYERNORM);
  // 16 chunks per thread already fill half the register file: no prefetch
  // buffer and no hoisted gamma/beta there (they would spill).
  constexpr bool kPrefetch = VPT <= 8;
  constexpr bool kHoist = kNorm && VPT <= 8;
  __shared__ float redf[3 * 16];
  __shared__ uint32_t redu[16];
  const int tid = threadIdx.x;
  const int g = tid % GT;
  const uint32_t sub = (uint32_t)(tid / GT);  // row slot in the block
  const uint32_t cols = a.cols;
  const uint32_t ngroups = (a.rows + G::kRows - 1) / G::kRows;

  auto chunk_col = [&](int j) { return (uint32_t)(j * GT + g) * 4u; };
  // A chunk that would pass the row's end starts at the row's last four
  // columns instead (also one wholly past it), so that loads need neither
  // tests nor branches (with them the compiler waited for one chunk before
  // it issued the next).  Such a chunk repeats columns of other threads:
  // harmless for maxima, left out of sums, and stored again with the same
  // values.  Needs 4 columns.
  auto chunk_at = [&](int j) { return FULL ? chunk_col(j) : min(chunk_col(j), cols - 4u); };
  auto own = [&](int j, int e) { return FULL || chunk_at(j) + (uint32_t)e >= chunk_col(j); };

  // Loads the row of group `grp` (rows past the end re-read the last row;
  // their results are never stored), and for the max grad its dy with it.
  auto load_row = [&](uint32_t grp, float4 *v, float &dyv) {
    // The row is wave-uniform (a row is owned by whole waves): through
    // readfirstlane its base stays in SGPRs and the loads take the
    // SGPR-base + 32-bit lane offset form, with no 64-bit address VGPRs
    // (which the compiler otherwise recycled into the prefetch buffer,
    // waiting for all memory operations at the loop head).
    const uint32_t row = __builtin_amdgcn_readfirstlane(grp * G::kRows + sub);
    const uint32_t rr = row < a.rows ? row : a.rows - 1;
    const float *xr = a.x + (size_t)rr * a.ld;
    if constexpr (OP == OP_MAX_GRAD) dyv = a.dy[rr];
#pragma unroll
    for (int j = 0; j < VPT; ++j) v[j] = load_nt4(xr + chunk_at(j));
  };

  // gamma / beta chunk j (1 / 0 where absent).
  auto affine_chunk = [&](int j, float4 &gj, float4 &bj) {
    gj = a.gamma ? load4(a.gamma + chunk_at(j)) : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    bj = a.beta ? load4(a.beta + chunk_at(j)) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  };
  // Hoisted copies, reused for every row the block normalises.
  float4 gm[kHoist ? VPT : 1], bt[kHoist ? VPT : 1];
  if constexpr (kHoist) {
#pragma unroll
    for (int j = 0; j < VPT; ++j) affine_chunk(j, gm[j], bt[j]);
  }

  // Processes the row group `grp` held in v[] (reductions + stores).
  auto process = [&](float4(&v)[VPT], uint32_t grp, float dyv) {
    const uint32_t row = __builtin_amdgcn_readfirstlane(grp * G::kRows + sub);  // wave-uniform
    const bool valid = row < a.rows;
    float *yr = a.y ? a.y + (size_t)(valid ? row : 0) * a.ld : nullptr;
    auto store = [&](int j, const float4 &o) {
      if (valid && (FULL || chunk_col(j) < cols)) store_nt4(yr + chunk_at(j), o);
    };

    if constexpr (OP == OP_SOFTMAX) {
      float m = -INFINITY;
#pragma unroll
      for (int j = 0; j < VPT; ++j)
        m = fmaxf(fmaxf(m, fmaxf(v[j].x, v[j].y)), fmaxf(v[j].z, v[j].w));
      m = row_max<WPR>(m, redf);
      float s = 0.0f;
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        v[j].x = __expf(v[j].x - m);
        v[j].y = __expf(v[j].y - m);
        v[j].z = __expf(v[j].z - m);
        v[j].w = __expf(v[j].w - m);
        if constexpr (FULL) {
          s += (v[j].x + v[j].y) + (v[j].z + v[j].w);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) s += own(j, e) ? get(v[j], e) : 0.0f;
        }
      }
      s = row_sum<WPR, !FULL>(s, redf);
      const float inv = s > 0.0f ? 1.0f / s : 0.0f;
#pragma unroll
      for (int j = 0; j < VPT; ++j)
        store(j, make_float4(v[j].x * inv, v[j].y * inv, v[j].z * inv, v[j].w * inv));
    } else if constexpr (kNorm) {
      // v past the row is not 0 (it repeats the row): sums take own columns.
      auto mine = [&](int j, int e, float t) { return own(j, e) ? t : 0.0f; };
      float mean = 0.0f, ss = 0.0f;
      if constexpr (OP == OP_LAYERNORM) {
        float n = 4.0f * VPT, s = 0.0f;
#pragma unroll
        for (int j = 0; j < VPT; ++j)
          s += (mine(j, 0, v[j].x) + mine(j, 1, v[j].y)) + (mine(j, 2, v[j].z) + mine(j, 3, v[j].w));
        float mu, m2 = 0.0f;
        if constexpr (FULL) {
          // Thread-local mean and M2 from registers (two passes, exact),
          // then one merged reduction of (count, mean, M2) across the row.
          // Every thread holds 4 VPT values, so every merge step joins equal
          // counts n and Chan's update needs no division:
          // mu = (mu_a + mu_b) / 2, M2 = M2_a + M2_b + (mu_b - mu_a)^2 n / 2.
          mu = s / n;
        } else {
          // Other rows: the row's mean first (a second reduction costs less
          // than merging unequal counts, which divides at every step).
          mu = row_sum<WPR, true>(s, redf) / (float)cols;
        }
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float d = mine(j, e, get(v[j], e) - mu);
            m2 += d * d;
          }
        }
        if constexpr (FULL) row_chan_equal<WPR>(n, mu, m2, redf);
        else m2 = row_sum<WPR, true>(m2, redf);
        mean = mu;
        ss = m2;
      } else {
#pragma unroll
        for (int j = 0; j < VPT; ++j)
          ss += (mine(j, 0, v[j].x * v[j].x) + mine(j, 1, v[j].y * v[j].y)) +
                (mine(j, 2, v[j].z * v[j].z) + mine(j, 3, v[j].w * v[j].w));
        ss = row_sum<WPR, !FULL>(ss, redf);
      }
      const float inv = 1.0f / sqrtf(ss / (float)cols + a.eps);
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        float4 o, gj, bj;
        if constexpr (kHoist) {
          gj = gm[j];
          bj = bt[j];
        } else {
          affine_chunk(j, gj, bj);
        }
        o.x = (v[j].x - mean) * inv * gj.x + bj.x;
        o.y = (v[j].y - mean) * inv * gj.y + bj.y;
        o.z = (v[j].z - mean) * inv * gj.z + bj.z;
        o.w = (v[j].w - mean) * inv * gj.w + bj.w;
        store(j, o);
      }
    } else if constexpr (OP == OP_MAX || OP == OP_MAX_GRAD) {
      // Two passes over the registers: the lane's max (fmaxf skips NaN,
      // -inf when the lane holds no number), then its first column
      // holding that value and the element there (a backward scan, the
      // last hit wins), which is the first strict-or-equal maximum of the
      // fold in column order (the element, not fmaxf's result, carries the
      // sign of a zero maximum).  Repeated chunks are scanned first and
      // name columns of the row, so an earlier hit replaces theirs.
      float m = -INFINITY;
      uint32_t mi = kNoIndex;
#pragma unroll
      for (int j = 0; j < VPT; ++j) m = fmaxf(fmaxf(m, fmaxf(v[j].x, v[j].y)), fmaxf(v[j].z, v[j].w));
      float mv = m;
#pragma unroll
      for (int j = VPT - 1; j >= 0; --j) {
        const uint32_t c = chunk_at(j);
#pragma unroll
        for (int e = 3; e >= 0; --e) {
          const float t = get(v[j], e);
          const bool hit = t == m;
          mi = hit ? c + e : mi;
          mv = hit ? t : mv;
        }
      }
      m = mv;
      row_argmax<WPR>(m, mi, redf, redu);
      if constexpr (OP == OP_MAX) {
        if (g == 0 && valid) {
          if (a.maxv) a.maxv[row] = m;
          if (a.argmax) a.argmax[row] = (mi == kNoIndex) ? -1 : (int32_t)mi;
        }
      } else {
        const float gv = valid ? dyv : 0.0f;
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
          const uint32_t c = chunk_at(j);
          float4 o;
          o.x = (c + 0 == mi) ? gv : 0.0f;
          o.y = (c + 1 == mi) ? gv : 0.0f;
          o.z = (c + 2 == mi) ? gv : 0.0f;
          o.w = (c + 3 == mi) ? gv : 0.0f;
          store(j, o);
        }
      }
    } else if constexpr (OP == OP_MASK) {
      float m = -INFINITY;
#pragma unroll
      for (int j = 0; j < VPT; ++j)
        m = fmaxf(fmaxf(m, fmaxf(v[j].x, v[j].y)), fmaxf(v[j].z, v[j].w));
      m = row_max<WPR>(m, redf);
#pragma unroll
      for (int j = 0; j < VPT; ++j)
        store(j, make_float4(v[j].x == m ? 1.0f : 0.0f, v[j].y == m ? 1.0f : 0.0f,
                             v[j].z == m ? 1.0f : 0.0f, v[j].w == m ? 1.0f : 0.0f));
    }

  };

  // Group loop, two groups per trip so the prefetch buffers alternate
  // without copies; every trip count is block-uniform.  The last group of a
  // block is processed on a path of its own, so inside the loop the
  // next-group loads are issued unconditionally: the compiler's vmcnt
  // waits then count them as younger than the current group's loads (with
  // a conditional prefetch it merges both paths and waits for the prefetch
  // too, which serialises the rows).
  uint32_t grp = blockIdx.x;
  if (grp >= ngroups) return;  // block-uniform
  float4 va[VPT], vb[VPT];
  float da = 0.0f, db = 0.0f;
  load_row(grp, va, da);
  for (;;) {
    uint32_t next = grp + gridDim.x;
    if (next >= ngroups) {
      process(va, grp, da);
      break;
    }
    if (kPrefetch) load_row(next, vb, db);
    process(va, grp, da);
    if (!kPrefetch) load_row(next, vb, db);
    grp = next;
    next = grp + gridDim.x;
    if (next >= ngroups) {
      process(vb, grp, db);
      break;
    }
    if (kPrefetch) load_row(next, va, da);
    process(vb, grp, db);
    if (!kPrefetch) load_row(next, va, da);
    grp = next;
  }
}

// Rows of 1 to 3 columns: a thread per row.
template <int OP>
__device__ __forceinline__ void row_tiny(const BwppRowArgs &a) {
  const uint64_t row = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (row >= a.rows) return;
  const uint32_t cols = a.cols;
  float v[3], m = -INFINITY;
  uint32_t mi = kNoIndex;
#pragma unroll
  for (uint32_t c = 0; c < 3; ++c) {
    v[c] = c < cols ? a.x[row * a.ld + c] : 0.0f;
    if (c < cols && (v[c] > m || (mi == kNoIndex && v[c] == m))) {
      m = v[c];
      mi = c;
    }
  }
  auto put = [&](auto f) {
#pragma unroll
    for (uint32_t c = 0; c < 3; ++c)
      if (c < cols) a.y[row * a.ld + c] = f(c);
  };
  if constexpr (OP == OP_SOFTMAX) {
    float s = 0.0f;
#pragma unroll
    for (uint32_t c = 0; c < 3; ++c) {
      v[c] = __expf(v[c] - m);
      s += c < cols ? v[c] : 0.0f;
    }
    const float inv = s > 0.0f ? 1.0f / s : 0.0f;
    put([&](uint32_t c) { return v[c] * inv; });
  } else if constexpr (OP == OP_RMSNORM || OP == OP_LAYERNORM) {
    const float mean = OP == OP_LAYERNORM ? (v[0] + v[1] + v[2]) / (float)cols : 0.0f;
    float ss = 0.0f;
#pragma unroll
    for (uint32_t c = 0; c < 3; ++c) {
      const float d = c < cols ? v[c] - mean : 0.0f;
      ss += d * d;
    }
    const float inv = 1.0f / sqrtf(ss / (float)cols + a.eps);
    put([&](uint32_t c) {
      return (v[c] - mean) * inv * (a.gamma ? a.gamma[c] : 1.0f) + (a.beta ? a.beta[c] : 0.0f);
    });
  } else if constexpr (OP == OP_MAX) {
    if (a.maxv) a.maxv[row] = m;
    if (a.argmax) a.argmax[row] = (mi == kNoIndex) ? -1 : (int32_t)mi;
  } else if constexpr (OP == OP_MAX_GRAD) {
    const float gv = a.dy[row];
    put([&](uint32_t c) { return c == mi ? gv : 0.0f; });
  } else {
    put([&](uint32_t c) { return v[c] == m ? 1.0f : 0.0f; });
  }
}

// ---------------------------------------------------------------- fallback

__device__ __forceinline__ float block_sum(float v, float *red) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}
__device__ __forceinline__ float block_max(float v, float *red) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

template <int OP>
__device__ __forceinline__ void row_gen(const BwppRowArgs &a) {
  __shared__ float redf[4];
  __shared__ uint32_t redu[4];
  const uint32_t row = blockIdx.x;
  if (row >= a.rows) return;  // block-uniform
  const uint32_t cols = a.cols;
  const uint32_t t = threadIdx.x;
  const float *xr = a.x + (size_t)row * a.ld;
  float *yr = a.y ? a.y + (size_t)row * a.ld : nullptr;

  if constexpr (OP == OP_SOFTMAX) {
    float m = -INFINITY;
    for (uint32_t c = t; c < cols; c += 256) m = fmaxf(m, xr[c]);
    m = block_max(m, redf);
    float s = 0.0f;
    for (uint32_t c = t; c < cols; c += 256) s += __expf(xr[c] - m);
    s = block_sum(s, redf);
    const float inv = s > 0.0f ? 1.0f / s : 0.0f;
    for (uint32_t c = t; c < cols; c += 256) yr[c] = __expf(xr[c] - m) * inv;
  } else if constexpr (OP == OP_RMSNORM || OP == OP_LAYERNORM) {
    float mean = 0.0f;
    if constexpr (OP == OP_LAYERNORM) {
      float s = 0.0f;
      for (uint32_t c = t; c < cols; c += 256) s += xr[c];
      mean = block_sum(s, redf) / (float)cols;
    }
    float ss = 0.0f;
    for (uint32_t c = t; c < cols; c += 256) {
      const float d = xr[c] - mean;
      ss += d * d;
    }
    ss = block_sum(ss, redf);
    const float inv = 1.0f / sqrtf(ss / (float)cols + a.eps);
    for (uint32_t c = t; c < cols; c += 256) {
      float o = (xr[c] - mean) * inv;
      if (a.gamma) o *= a.gamma[c];
      if (a.beta) o += a.beta[c];
      yr[c] = o;
    }
  } else if constexpr (OP == OP_MAX || OP == OP_MAX_GRAD) {
    float m = -INFINITY;
    uint32_t mi = kNoIndex;
    for (uint32_t c = t; c < cols; c += 256) {
      const float v = xr[c];
      if (v > m || (mi == kNoIndex && v == m)) {
        m = v;
        mi = c;
      }
    }
    row_argmax<4>(m, mi, redf, redu);
    if constexpr (OP == OP_MAX) {
      if (t == 0) {
        if (a.maxv) a.maxv[row] = m;
        if (a.argmax) a.argmax[row] = (mi == kNoIndex) ? -1 : (int32_t)mi;
      }
    } else {
      const float gv = a.dy[row];
      for (uint32_t c = t; c < cols; c += 256) yr[c] = (c == mi) ? gv : 0.0f;
    }
  } else if constexpr (OP == OP_MASK) {
    float m = -INFINITY;
    for (uint32_t c = t; c < cols; c += 256) m = fmaxf(m, xr[c]);
    m = block_max(m, redf);
    for (uint32_t c = t; c < cols; c += 256) yr[c] = (xr[c] == m) ? 1.0f : 0.0f;
  }
}

}  // namespace

// ------------------------------------------------------------ entry points
// Register path: bwpp_row_<op>_v<VPT>_w<WPR>_<f|p>  (f: cols == 256*WPR*VPT)
#define BWPP_ROW_REG(NAME, OP, VPT, WPR)                                      \
  extern "C" __global__ __launch_bounds__(RowGeom<WPR>::kBlock) void          \
      bwpp_row_##NAME##_v##VPT##_w##WPR##_f(const BwppRowArgs a) {            \
    row_reg<OP, VPT, WPR, true>(a);                                           \
  }                                                                           \
  extern "C" __global__ __launch_bounds__(RowGeom<WPR>::kBlock) void          \
      bwpp_row_##NAME##_v##VPT##_w##WPR##_p(const BwppRowArgs a) {            \
    row_reg<OP, VPT, WPR, false>(a);                                          \
  }

// Keep this list in sync with kRowCfgs in runtime/bwpp_hip.cpp.
#define BWPP_ROW_ALL_CFG(NAME, OP)                                            \
  BWPP_ROW_REG(NAME, OP, 1, 1)                                                \
  BWPP_ROW_REG(NAME, OP, 2, 1)                                                \
  BWPP_ROW_REG(NAME, OP, 4, 1)                                                \
  BWPP_ROW_REG(NAME, OP, 8, 1)                                                \
  BWPP_ROW_REG(NAME, OP, 16, 1)                                               \
  BWPP_ROW_REG(NAME, OP, 2, 2)                                                \
  BWPP_ROW_REG(NAME, OP, 4, 2)                                                \
  BWPP_ROW_REG(NAME, OP, 8, 2)                                                \
  BWPP_ROW_REG(NAME, OP, 1, 4)                                                \
  BWPP_ROW_REG(NAME, OP, 2, 4)                                                \
  BWPP_ROW_REG(NAME, OP, 4, 4)                                                \
  BWPP_ROW_REG(NAME, OP, 8, 4)                                                \
  BWPP_ROW_REG(NAME, OP, 16, 4)                                               \
  BWPP_ROW_REG(NAME, OP, 2, 8)                                                \
  BWPP_ROW_REG(NAME, OP, 4, 8)                                                \
  BWPP_ROW_REG(NAME, OP, 8, 8)                                                \
  BWPP_ROW_REG(NAME, OP, 16, 8)                                               \
  extern "C" __global__ __launch_bounds__(256) void bwpp_row_##NAME##_tiny(const BwppRowArgs a) { \
    row_tiny<OP>(a);                                                          \
  }                                                                           \
  extern "C" __global__ __launch_bounds__(256) void bwpp_row_##NAME##_gen(const BwppRowArgs a) { \
    row_gen<OP>(a);                                                           \
  }

BWPP_ROW_ALL_CFG(softmax, OP_SOFTMAX)
BWPP_ROW_ALL_CFG(rmsnorm, OP_RMSNORM)
BWPP_ROW_ALL_CFG(layernorm, OP_LAYERNORM)
BWPP_ROW_ALL_CFG(max, OP_MAX)
BWPP_ROW_ALL_CFG(maxgrad, OP_MAX_GRAD)
BWPP_ROW_ALL_CFG(mask, OP_MASK)

// ------------------------------------------------------- streaming kernels

// reduce_max grad from saved indices, axis 1: dx[r, c] = (c == idx[r]) ? dy[r] : 0.
// Block per row (grid-stride), each thread writes columns t, t+256, ...
extern "C" __global__ __launch_bounds__(256) void bwpp_row_maxgrad_idx(const BwppRowArgs a) {
  for (uint32_t r = blockIdx.x; r < a.rows; r += gridDim.x) {
    const int32_t idx = a.idx_in[r];
    const float gv = a.dy[r];
    float *yr = a.y + (size_t)r * a.ld;
    for (uint32_t c = threadIdx.x; c < a.cols; c += 256)
      yr[c] = ((int32_t)c == idx) ? gv : 0.0f;
  }
}

// Same, 128-bit stores (host checks dx alignment and ld % 4 == 0).
extern "C" __global__ __launch_bounds__(256) void bwpp_row_maxgrad_idx_v4(const BwppRowArgs a) {
  for (uint32_t r = blockIdx.x; r < a.rows; r += gridDim.x) {
    const int32_t idx = a.idx_in[r];
    const float gv = a.dy[r];
    float *yr = a.y + (size_t)r * a.ld;
    const uint32_t c4 = a.cols & ~3u;
    for (uint32_t c = threadIdx.x * 4u; c < c4; c += 1024u) {
      float4 o;
      o.x = ((int32_t)c == idx) ? gv : 0.0f;
      o.y = ((int32_t)c + 1 == idx) ? gv : 0.0f;
      o.z = ((int32_t)c + 2 == idx) ? gv : 0.0f;
      o.w = ((int32_t)c + 3 == idx) ? gv : 0.0f;
      *reinterpret_cast<float4 *>(yr + c) = o;
    }
    for (uint32_t c = c4 + threadIdx.x; c < a.cols; c += 256)
      yr[c] = ((int32_t)c == idx) ? gv : 0.0f;
  }
}

// Reference grad (bwpp_cpu_ref.c:192-219): dx = mask * dy[line].
// axis 1: dy per row; axis 0 variant below: dy per column.
extern "C" __global__ __launch_bounds__(256) void bwpp_row_maskgrad(const BwppRowArgs a) {
  for (uint32_t r = blockIdx.x; r < a.rows; r += gridDim.x) {
    const float gv = a.dy[r];
    const float *mr = a.x + (size_t)r * a.ld;
    float *yr = a.y + (size_t)r * a.ld;
    for (uint32_t c = threadIdx.x; c < a.cols; c += 256) yr[c] = mr[c] * gv;
  }
}
extern "C" __global__ __launch_bounds__(256) void bwpp_col_maskgrad(const BwppRowArgs a) {
  for (uint32_t r = blockIdx.x; r < a.rows; r += gridDim.x) {
    const float *mr = a.x + (size_t)r * a.ld;
    float *yr = a.y + (size_t)r * a.ld;
    for (uint32_t c = threadIdx.x; c < a.cols; c += 256) yr[c] = mr[c] * a.dy[c];
  }
}

// ---------------------------------------------------------- axis 0 (columns)
// Reductions over rows.  HBM-bound: x is read once, coalesced, by enough
// blocks to fill the chip, in two launches: bwpp_col_max_band reduces bands
// of rows (a block owns 64 columns x one band; its 4 waves take every fourth
// row, 8 rows' loads in flight per wave) to (value, first row) pairs, and
// bwpp_col_max_final merges the bands.  The pair rule is the strict fold in
// row order (bwpp_cpu_ref.c:156-171): a larger value wins, an equal one
// keeps the lower row, so any split gives the fold's bits.  Mask and
// gradient then stream their output in a further kernel whose blocks tile
// rows as well as columns.  4096 x 4096: maximum and index 2450 us with one
// thread per column walking all rows (16 blocks, one load in flight per
// lane), 13.3 + 4.6 us so (5.0 TB/s in the first pass); the gradient from
// saved indices 128 -> 12.9 us.

extern "C" __global__ __launch_bounds__(256) void bwpp_col_max_band(const BwppRowArgs a) {
  __shared__ float sv[4][64];
  __shared__ uint32_t si[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t c = blockIdx.x * 64u + (uint32_t)lane;
  const uint64_t band = ((uint64_t)a.rows + gridDim.y - 1) / gridDim.y;
  const uint64_t r0 = band * blockIdx.y, r1 = min((uint64_t)a.rows, r0 + band);
  float m = -INFINITY;
  uint32_t mi = kNoIndex;
  auto take = [&](float v, uint64_t r) {
    if (v > m || (mi == kNoIndex && v == m)) {
      m = v;
      mi = (uint32_t)r;
    }
  };
  if (c < a.cols) {
    const float *x = a.x + c;
    uint64_t r = r0 + (uint64_t)wave;
    for (; r + 28 < r1; r += 32) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = x[(r + 4 * i) * a.ld];
#pragma unroll
      for (int i = 0; i < 8; ++i) take(v[i], r + 4 * i);
    }
    for (; r < r1; r += 4) take(x[r * a.ld], r);
  }
  sv[wave][lane] = m;
  si[wave][lane] = mi;
  __syncthreads();
  if (wave != 0 || c >= a.cols) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) argmax_merge(m, mi, sv[w][lane], si[w][lane]);
  if (gridDim.y > 1) {
    a.part_v[(size_t)blockIdx.y * a.cols + c] = m;
    a.part_i[(size_t)blockIdx.y * a.cols + c] = mi;
    return;
  }
  if (a.maxv) a.maxv[c] = m;
  if (a.argmax) a.argmax[c] = (mi == kNoIndex) ? -1 : (int32_t)mi;
}

// Merges a.bands partials per column: 64 columns x 4 band groups per block.
extern "C" __global__ __launch_bounds__(256) void bwpp_col_max_final(const BwppRowArgs a) {
  __shared__ float sv[4][64];
  __shared__ uint32_t si[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t c = blockIdx.x * 64u + (uint32_t)lane;
  float m = -INFINITY;
  uint32_t mi = kNoIndex;
  if (c < a.cols) {
    uint32_t b = (uint32_t)wave;
    for (; b + 28 < a.bands; b += 32) {  // 8 bands' loads in flight
      float v[8];
      uint32_t i8[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = a.part_v[(size_t)(b + 4 * i) * a.cols + c];
        i8[i] = a.part_i[(size_t)(b + 4 * i) * a.cols + c];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) argmax_merge(m, mi, v[i], i8[i]);
    }
    for (; b < a.bands; b += 4)
      argmax_merge(m, mi, a.part_v[(size_t)b * a.cols + c], a.part_i[(size_t)b * a.cols + c]);
  }
  sv[wave][lane] = m;
  si[wave][lane] = mi;
  __syncthreads();
  if (wave != 0 || c >= a.cols) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) argmax_merge(m, mi, sv[w][lane], si[w][lane]);
  if (a.maxv) a.maxv[c] = m;
  if (a.argmax) a.argmax[c] = (mi == kNoIndex) ? -1 : (int32_t)mi;
}

namespace {

// The second pass of the axis-0 mask (y = x == max[c]) and gradient
// (y = row == idx[c] ? dy[c] : 0): a wave owns 64 column chunks (4 columns
// with VEC, else 1), whose per-column values stay in registers, and every
// (4 * gridDim.y)-th row, four rows per trip.  y may be x: each element is
// read and written by one thread.
template <bool MASK, bool VEC>
__device__ __forceinline__ void col_apply(const BwppRowArgs &a) {
  constexpr int W = VEC ? 4 : 1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t c = (blockIdx.x * 64u + (uint32_t)lane) * W;
  if (c >= a.cols) return;
  float g[W];      // MASK: the column's maximum, else dy
  int32_t idx[W];  // row that takes dy
#pragma unroll
  for (int e = 0; e < W; ++e) {
    g[e] = MASK ? a.part_v[c + e] : a.dy[c + e];
    idx[e] = MASK ? 0 : a.idx_in[c + e];
  }
  auto apply = [&](uint64_t r) {
    float x[W], o[W];
    if constexpr (MASK) {
      if constexpr (VEC) {
        const float4 t = load_nt4(a.x + r * a.ld + c);
        x[0] = t.x, x[1] = t.y, x[2] = t.z, x[3] = t.w;
      } else {
        x[0] = a.x[r * a.ld + c];
      }
    }
#pragma unroll
    for (int e = 0; e < W; ++e) {
      if constexpr (MASK) o[e] = x[e] == g[e] ? 1.0f : 0.0f;
      else o[e] = (int32_t)r == idx[e] ? g[e] : 0.0f;
    }
    if constexpr (VEC) store_nt4(a.y + r * a.ld + c, make_float4(o[0], o[1], o[2], o[3]));
    else a.y[r * a.ld + c] = o[0];
  };
  const uint64_t step = 4ull * gridDim.y;
  uint64_t r = 4ull * blockIdx.y + (uint64_t)wave;
  for (; r + 3 * step < a.rows; r += 4 * step) {
#pragma unroll
    for (int i = 0; i < 4; ++i) apply(r + i * step);
  }
  for (; r < a.rows; r += step) apply(r);
}

// One thread per column, rows walked in order: mask and gradient without a
// workspace for the column maxima.
__device__ __forceinline__ void col_argmax(const BwppRowArgs &a, uint32_t c,
                                           float &m, int32_t &mi) {
  m = -INFINITY;
  for (uint32_t r = 0; r < a.rows; ++r) {
    const float v = a.x[(size_t)r * a.ld + c];
    if (v > m) m = v;
  }
  mi = -1;
  for (uint32_t r = 0; r < a.rows; ++r) {
    if (a.x[(size_t)r * a.ld + c] == m) {
      mi = (int32_t)r;
      break;
    }
  }
}

}  // namespace

#define BWPP_COL_APPLY(NAME, MASK, VEC)                                                       \
  extern "C" __global__ __launch_bounds__(256) void NAME(const BwppRowArgs a) {                \
    col_apply<MASK, VEC>(a);                                                                  \
  }
BWPP_COL_APPLY(bwpp_col_mask_apply, true, false)
BWPP_COL_APPLY(bwpp_col_mask_apply_v4, true, true)
BWPP_COL_APPLY(bwpp_col_maxgrad_apply, false, false)
BWPP_COL_APPLY(bwpp_col_maxgrad_apply_v4, false, true)

extern "C" __global__ __launch_bounds__(256) void bwpp_col_maxgrad(const BwppRowArgs a) {
  const uint32_t c = blockIdx.x * 256 + threadIdx.x;
  if (c >= a.cols) return;
  int32_t mi;
  float m;
  col_argmax(a, c, m, mi);
  const float gv = a.dy[c];
  for (uint32_t r = 0; r < a.rows; ++r) a.y[(size_t)r * a.ld + c] = ((int32_t)r == mi) ? gv : 0.0f;
}

extern "C" __global__ __launch_bounds__(256) void bwpp_col_mask(const BwppRowArgs a) {
  const uint32_t c = blockIdx.x * 256 + threadIdx.x;
  if (c >= a.cols) return;
  float m = -INFINITY;
  for (uint32_t r = 0; r < a.rows; ++r) m = fmaxf(m, a.x[(size_t)r * a.ld + c]);
  for (uint32_t r = 0; r < a.rows; ++r) {
    const size_t o = (size_t)r * a.ld + c;
    a.y[o] = (a.x[o] == m) ? 1.0f : 0.0f;
  }
}
