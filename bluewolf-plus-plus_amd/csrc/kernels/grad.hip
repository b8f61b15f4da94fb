// Autodiff grad ops and elementwise glue for gfx950 (fp32).
//
// The reference's autodiff (compiler/graph_ir.c:1485-1839) emits these
// internal ops; the reference has no numeric kernels for them, so the
// semantics are the closed forms restated in oracle/bwpp_oracle.c:
//   silu_grad      (graph_ir.c:1709-1720)  dx = dy * s * (1 + x (1 - s))
//   softmax_grad   (graph_ir.c:1722-1733)  dx = y * (dy - sum(dy * y))
//   rmsnorm_grad   (graph_ir.c:1735-1789)  dx, dgamma = sum_r dy * xhat,
//                                          dbeta = sum_r dy
//   reduce_sum     (graph_ir.c:1410-1455)  along rows or over rows
//   add/sub/mul/div with broadcasting, broadcast (graph_ir.c:697-770,
//   1457-1470, 1585-1654)
// All are HBM-bound: one read of each input, one write of each output,
// 128-bit accesses where rows are 16-byte aligned.
#include "common.h"
#include "../kargs.h"

using namespace bwpp;

namespace {

__device__ __forceinline__ float block_sum256(float v, float *red) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

__device__ __forceinline__ float silu_grad1(float x, float dy) {
  const float s = 1.0f / (1.0f + __expf(-x));
  return dy * (s * (1.0f + x * (1.0f - s)));
}

}  // namespace

// Flat elementwise silu_grad over n elements; vec: 16-byte aligned buffers.
extern "C" __global__ __launch_bounds__(256) void bwpp_silu_grad(const BwppGradArgs g) {
  const uint64_t stride = (uint64_t)gridDim.x * 256u;
  const uint64_t n4 = g.vec ? g.n / 4 : 0;
  const float4 *x4 = reinterpret_cast<const float4 *>(g.a);
  const float4 *d4 = reinterpret_cast<const float4 *>(g.b);
  float4 *o4 = reinterpret_cast<float4 *>(g.out);
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n4; i += stride) {
    const float4 x = load_nt4(reinterpret_cast<const float *>(x4 + i));
    const float4 d = load_nt4(reinterpret_cast<const float *>(d4 + i));
    store_nt4(reinterpret_cast<float *>(o4 + i),
              make_float4(silu_grad1(x.x, d.x), silu_grad1(x.y, d.y), silu_grad1(x.z, d.z), silu_grad1(x.w, d.w)));
  }
  for (uint64_t i = n4 * 4 + (uint64_t)blockIdx.x * 256u + threadIdx.x; i < g.n; i += stride)
    g.out[i] = silu_grad1(g.a[i], g.b[i]);
}

// Columns of a row that thread g of its group of GT threads holds in chunk
// j, element e: runs of four (VEC: 128-bit accesses), or every GT-th column
// (rows at any 4-byte address: 4-byte accesses, still 256 contiguous bytes
// per wave and instruction).
template <int GT, bool VEC>
__device__ __forceinline__ uint32_t elem_col(int g, int j, int e) {
  return VEC ? 4u * (uint32_t)(j * GT + g) + (uint32_t)e : (uint32_t)((4 * j + e) * GT + g);
}

// One thread's share of a row, v[4 j + e] = p[elem_col(j, e)]; columns past
// the end re-read the last ones (callers zero or skip them), so the loads
// issue without branches.
template <int VPT, int GT, bool VEC, bool NT = true>
__device__ __forceinline__ void load_share(float (&v)[4 * VPT], const float *p, int g, uint32_t cols) {
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if constexpr (VEC) {
      const uint32_t c = elem_col<GT, VEC>(g, j, 0);
      const float *q = p + (c < cols ? c : cols - 4u);
      const float4 t = NT ? load_nt4(q) : *reinterpret_cast<const float4 *>(q);
      v[4 * j] = t.x, v[4 * j + 1] = t.y, v[4 * j + 2] = t.z, v[4 * j + 3] = t.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t c = elem_col<GT, VEC>(g, j, e);
        v[4 * j + e] = p[c < cols ? c : cols - 1u];
      }
    }
  }
}
template <int VPT, int GT, bool VEC, bool NT = true>
__device__ __forceinline__ void store_share(float *p, const float (&v)[4 * VPT], int g, uint32_t cols) {
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if constexpr (VEC) {
      const uint32_t c = elem_col<GT, VEC>(g, j, 0);
      const float4 t = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
      if (c < cols) {
        if constexpr (NT) store_nt4(p + c, t);
        else *reinterpret_cast<float4 *>(p + c) = t;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t c = elem_col<GT, VEC>(g, j, e);
        if (c < cols) p[c] = v[4 * j + e];
      }
    }
  }
}

// Row-wise softmax_grad with the row in registers: y and dy are read once.
// WPR waves share a row (WPR = 1: four rows per block, no barrier); the
// block holds one group of rows, so blocks overlap each other's loads and
// reductions.  4096 x 4096: re-reading the row for the second pass with
// 4-byte loads took 50.5 us, this 32.0 us (201 MB at 6.3 TB/s).
template <int VPT, int WPR, bool VEC>
__device__ __forceinline__ void softmax_grad_reg(const BwppGradArgs &g) {
  constexpr int GT = 64 * WPR, kBlock = WPR >= 4 ? GT : 256;
  __shared__ float red[kBlock / 64];
  const int tid = (int)threadIdx.x, gi = tid % GT, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t row = blockIdx.x * (uint32_t)(kBlock / GT) + (uint32_t)(wave / WPR);
  const uint32_t r = row < g.rows ? row : g.rows - 1u;
  float y[4 * VPT], d[4 * VPT];
  load_share<VPT, GT, VEC>(y, g.a + (size_t)r * g.ld, gi, g.cols);
  load_share<VPT, GT, VEC>(d, g.b + (size_t)r * g.ld, gi, g.cols);
  float dot = 0.0f;
#pragma unroll
  for (int i = 0; i < 4 * VPT; ++i)
    if (elem_col<GT, VEC>(gi, i / 4, i % 4) < g.cols) dot += d[i] * y[i];
  dot = wave_sum(dot);
  if constexpr (WPR > 1) {
    if ((tid & 63) == 0) red[wave] = dot;
    __syncthreads();
    dot = red[wave / WPR * WPR];
#pragma unroll
    for (int w = 1; w < WPR; ++w) dot += red[wave / WPR * WPR + w];
  }
  if (row >= g.rows) return;
#pragma unroll
  for (int i = 0; i < 4 * VPT; ++i) y[i] = y[i] * (d[i] - dot);
  store_share<VPT, GT, VEC>(g.out + (size_t)row * g.ld, y, gi, g.cols);
}

#define BWPP_SOFTMAX_GRAD(VPT, WPR)                                                                \
  extern "C" __global__ __launch_bounds__(WPR >= 4 ? 64 * WPR : 256) void                           \
      bwpp_softmax_grad_v##VPT##_w##WPR(const BwppGradArgs g) {                                     \
    softmax_grad_reg<VPT, WPR, true>(g);                                                           \
  }                                                                                                \
  extern "C" __global__ __launch_bounds__(WPR >= 4 ? 64 * WPR : 256) void                           \
      bwpp_softmax_grad_v##VPT##_w##WPR##_u(const BwppGradArgs g) {                                 \
    softmax_grad_reg<VPT, WPR, false>(g);                                                          \
  }
// Keep this list in sync with kGradCfgs in runtime/bwpp_hip.cpp.
#define BWPP_GRAD_ALL_CFG(MAC) MAC(1, 1) MAC(2, 1) MAC(4, 1) MAC(2, 4) MAC(2, 8) MAC(4, 8)
BWPP_GRAD_ALL_CFG(BWPP_SOFTMAX_GRAD)
BWPP_SOFTMAX_GRAD(8, 8)

// Longer rows: one block per row (grid-stride); the second pass re-reads
// the row (L2).
extern "C" __global__ __launch_bounds__(256) void bwpp_softmax_grad(const BwppGradArgs g) {
  __shared__ float red[4];
  for (uint32_t r = blockIdx.x; r < g.rows; r += gridDim.x) {
    const float *y = g.a + (size_t)r * g.ld;
    const float *dy = g.b + (size_t)r * g.ld;
    float *dx = g.out + (size_t)r * g.ld;
    float dot = 0.0f;
    for (uint32_t c = threadIdx.x; c < g.cols; c += 256) dot += dy[c] * y[c];
    dot = block_sum256(dot, red);
    for (uint32_t c = threadIdx.x; c < g.cols; c += 256) dx[c] = y[c] * (dy[c] - dot);
  }
}

// Mean-square loss and its gradient in one pass over x: block b adds x^2
// over its rows (rows b, b + grid, ...; thread order fixed) into partial
// part_g[b] and, with out, writes dx = x * s_grad; bwpp_mean_square_final
// then sums the partials in index order.  Deterministic for a given grid.
extern "C" __global__ __launch_bounds__(256) void bwpp_mean_square_part(const BwppGradArgs g) {
  __shared__ float red[4];
  const float gs = g.s_grad ? *g.s_grad : 1.0f;
  float acc = 0.0f;
  for (uint32_t r = blockIdx.x; r < g.rows; r += gridDim.x) {
    const float *x = g.a + (size_t)r * g.ld;
    float *dx = g.out ? g.out + (size_t)r * g.ld : nullptr;
    if (g.vec) {  // 16-byte rows
      for (uint32_t c = 4u * threadIdx.x; c < g.cols; c += 1024u) {
        const float4 v = *reinterpret_cast<const float4 *>(x + c);
        acc += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
        if (dx) *reinterpret_cast<float4 *>(dx + c) = make_float4(v.x * gs, v.y * gs, v.z * gs, v.w * gs);
      }
    } else {
      for (uint32_t c = threadIdx.x; c < g.cols; c += 256u) {
        const float v = x[c];
        acc += v * v;
        if (dx) dx[c] = v * gs;
      }
    }
  }
  acc = block_sum256(acc, red);
  if (threadIdx.x == 0) g.part_g[blockIdx.x] = acc;
}

// out2[0] = s_loss * (sum of the nparts partials), one block.
extern "C" __global__ __launch_bounds__(256) void bwpp_mean_square_final(const BwppGradArgs g) {
  __shared__ float red[4];
  float acc = 0.0f;
  for (uint32_t i = threadIdx.x; i < g.nparts; i += 256u) acc += g.part_g[i];
  acc = block_sum256(acc, red);
  if (threadIdx.x == 0) g.out2[0] = acc * (g.s_loss ? *g.s_loss : 1.0f);
}

// rmsnorm_grad with the row in registers: x, dy (and acc) are read once,
// WPR waves share a row, and a block strides over rows with the next row's
// loads in flight while it reduces the current one; the dgamma / dbeta
// column sums stay in registers and leave once per block as a partial row
// (summed by bwpp_col_partials_sum; rows that share a block with WPR = 1
// first meet in LDS).  The two row sums take one barrier: the LDS slots
// alternate between rows.  gamma NULL means 1; with g.acc, dx = acc + the
// gradient (acc may be dx itself: a thread has read its acc elements before
// it writes them).  4096 x 4096 with dgamma and dbeta: two passes over the
// row and per-element LDS accumulators took 148 us, this 31.4 us (201 MB
// and 8 MB of partials).
//
// No contraction anywhere in the row's arithmetic: with plain roundings
// every copy of the code gives the same bits, and dx = acc + gradient is
// exactly the two ops.
template <int VPT, int WPR, bool VEC>
__device__ __forceinline__ void rmsnorm_grad_reg(const BwppGradArgs &g) {
#pragma clang fp contract(off)
  constexpr int GT = 64 * WPR, kBlock = WPR >= 4 ? GT : 256, kRows = kBlock / GT, E = 4 * VPT;
  // One wave per row (rows of at most 1024 columns): no prefetch, the block's
  // other rows cover the latency, and cached accesses, such rows mostly being
  // a layer's own, just written (4096 x 1024: 14.5 us; with prefetch and
  // non-temporal accesses 15.3).
  constexpr bool kPrefetch = WPR > 1 && (VEC || VPT < 4), kNT = WPR > 1;
  __shared__ float red[2][2][kBlock / 64];
  extern __shared__ float colacc[];  // [kRows][2][cols] when partials are requested and kRows > 1
  const int tid = (int)threadIdx.x, gi = tid % GT, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t sub = (uint32_t)(wave / WPR), cols = g.cols;
  const bool parts = g.part_g != nullptr, has_acc = g.acc != nullptr;
  float gm[E], ag[E], ab[E];
#pragma unroll
  for (int i = 0; i < E; ++i) {
    gm[i] = 1.0f;
    ag[i] = ab[i] = 0.0f;
  }
  if (g.gamma) load_share<VPT, GT, VEC, false>(gm, g.gamma, gi, cols);
  struct Row {
    float x[E], d[E], a[E];
  };
  auto load = [&](uint32_t row, Row &v) {
    const size_t at = (size_t)(row < g.rows ? row : g.rows - 1u) * g.ld;
    load_share<VPT, GT, VEC, kNT>(v.x, g.a + at, gi, cols);
    load_share<VPT, GT, VEC, kNT>(v.d, g.b + at, gi, cols);
    if (has_acc) load_share<VPT, GT, VEC, kNT>(v.a, g.acc + at, gi, cols);
  };
  auto process = [&](uint32_t row, Row &v, int slot) {
    const bool valid = row < g.rows;
    float ss = 0.0f, t = 0.0f;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      if (!valid || elem_col<GT, VEC>(gi, i / 4, i % 4) >= cols) v.x[i] = v.d[i] = 0.0f;
      ss += v.x[i] * v.x[i];
      t += v.x[i] * gm[i] * v.d[i];
    }
    ss = wave_sum(ss);
    t = wave_sum(t);
    if constexpr (WPR > 1) {
      if ((tid & 63) == 0) {
        red[slot][0][wave] = ss;
        red[slot][1][wave] = t;
      }
      __syncthreads();
      const int w0 = wave / WPR * WPR;
      ss = red[slot][0][w0];
      t = red[slot][1][w0];
#pragma unroll
      for (int w = 1; w < WPR; ++w) {
        ss += red[slot][0][w0 + w];
        t += red[slot][1][w0 + w];
      }
    }
    const float inv = 1.0f / sqrtf(ss / (float)cols + g.eps);
    const float mdot = inv * t / (float)cols;  // mean(xhat * gamma * dy)
    float o[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const float h = v.x[i] * inv;
      o[i] = inv * (gm[i] * v.d[i] - h * mdot);
      o[i] = has_acc ? v.a[i] + o[i] : o[i];  // acc: a separate rounded add
      ag[i] += v.d[i] * h;
      ab[i] += v.d[i];
    }
    if (valid) store_share<VPT, GT, VEC, kNT>(g.out + (size_t)row * g.ld, o, gi, cols);
  };
  const uint32_t ngroups = (g.rows + kRows - 1) / kRows;
  uint32_t grp = blockIdx.x;
  if constexpr (!kPrefetch) {
    for (int slot = 0; grp < ngroups; grp += gridDim.x, slot ^= 1) {
      Row v;
      load(grp * kRows + sub, v);
      process(grp * kRows + sub, v, slot);
    }
  } else if (grp < ngroups) {
    // Two rows per trip so that the buffers alternate without copies; the
    // last row of a block is processed on a path of its own, so that inside
    // the loop the next row's loads are issued unconditionally.
    Row ra, rb;
    load(grp * kRows + sub, ra);
    for (;;) {
      uint32_t next = grp + gridDim.x;
      if (next >= ngroups) {
        process(grp * kRows + sub, ra, 0);
        break;
      }
      load(next * kRows + sub, rb);
      process(grp * kRows + sub, ra, 0);
      grp = next;
      next = grp + gridDim.x;
      if (next >= ngroups) {
        process(grp * kRows + sub, rb, 1);
        break;
      }
      load(next * kRows + sub, ra);
      process(grp * kRows + sub, rb, 1);
      grp = next;
    }
  }
  if (!parts) return;  // block-uniform
  if constexpr (kRows == 1) {
    store_share<VPT, GT, VEC>(g.part_g + (size_t)blockIdx.x * cols, ag, gi, cols);
    store_share<VPT, GT, VEC>(g.part_b + (size_t)blockIdx.x * cols, ab, gi, cols);
  } else {
    float *mine = colacc + (size_t)sub * 2 * cols;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const uint32_t c = elem_col<GT, VEC>(gi, i / 4, i % 4);
      if (c < cols) {
        mine[c] = ag[i];
        mine[cols + c] = ab[i];
      }
    }
    __syncthreads();
    for (uint32_t c = threadIdx.x; c < cols; c += kBlock) {
      float sg = 0.0f, sb = 0.0f;
#pragma unroll
      for (int w = 0; w < kRows; ++w) {
        sg += colacc[(size_t)w * 2 * cols + c];
        sb += colacc[(size_t)w * 2 * cols + cols + c];
      }
      g.part_g[(size_t)blockIdx.x * cols + c] = sg;
      g.part_b[(size_t)blockIdx.x * cols + c] = sb;
    }
  }
}

#define BWPP_RMSNORM_GRAD(VPT, WPR)                                                                \
  extern "C" __global__ __launch_bounds__(WPR >= 4 ? 64 * WPR : 256) void                           \
      bwpp_rmsnorm_grad_v##VPT##_w##WPR(const BwppGradArgs g) {                                     \
    rmsnorm_grad_reg<VPT, WPR, true>(g);                                                           \
  }                                                                                                \
  extern "C" __global__ __launch_bounds__(WPR >= 4 ? 64 * WPR : 256) void                           \
      bwpp_rmsnorm_grad_v##VPT##_w##WPR##_u(const BwppGradArgs g) {                                 \
    rmsnorm_grad_reg<VPT, WPR, false>(g);                                                          \
  }
BWPP_GRAD_ALL_CFG(BWPP_RMSNORM_GRAD)

// Rows of more than 8192 columns (no partials there): one block per row,
// the row read twice.
extern "C" __global__ __launch_bounds__(256) void bwpp_rmsnorm_grad(const BwppGradArgs g) {
  __shared__ float red[4];
  for (uint32_t r = blockIdx.x; r < g.rows; r += gridDim.x) {
    const float *x = g.a + (size_t)r * g.ld;
    const float *dy = g.b + (size_t)r * g.ld;
    float *dx = g.out + (size_t)r * g.ld;
    const float *ac = g.acc ? g.acc + (size_t)r * g.ld : nullptr;
    float ss = 0.0f, t = 0.0f;
    for (uint32_t c = threadIdx.x; c < g.cols; c += 256) {
      const float xv = x[c];
      const float gd = g.gamma ? g.gamma[c] * dy[c] : dy[c];
      ss += xv * xv;
      t += xv * gd;
    }
    ss = block_sum256(ss, red);
    t = block_sum256(t, red);
    const float inv = 1.0f / sqrtf(ss / (float)g.cols + g.eps);
    const float mdot = inv * t / (float)g.cols;  // mean(xhat * gamma * dy)
    for (uint32_t c = threadIdx.x; c < g.cols; c += 256) {
      const float xh = x[c] * inv;
      const float d = dy[c];
      const float gd = g.gamma ? g.gamma[c] * d : d;
      const float v = inv * (gd - xh * mdot);
      if (ac) {
#pragma clang fp contract(off)
        dx[c] = ac[c] + v;  // never contracted into the product
      } else {
        dx[c] = v;
      }
    }
  }
}

// out[c] = sum_p part[p][c] for the two partial arrays (dgamma, dbeta); the
// outputs may be NULL.  A block owns 16 columns: thread (g, c) of 16 x 16
// sums parts g, g + 16, ... of column c (16 consecutive columns = 64-byte
// rows per part), then the 16 partial sums of each column are added in LDS
// in a fixed order.
extern "C" __global__ __launch_bounds__(256) void bwpp_col_partials_sum(const BwppGradArgs g) {
  __shared__ float red[2][16][17];
  const uint32_t cl = threadIdx.x & 15u, grp = threadIdx.x >> 4;
  const uint32_t c = blockIdx.x * 16u + cl;
  float sg = 0.0f, sb = 0.0f;
  if (c < g.cols) {
    // Eight parts' loads issued before their adds (same order of addition
    // as one at a time): the loop is bound by the L2 round trip, not by
    // bandwidth, and a load-add-wait per part took 32 round trips at 512
    // parts.
    uint32_t p = grp;
    for (; p + 16u * 7u < g.nparts; p += 16u * 8u) {
      float a[8], b[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        a[i] = g.part_g[(size_t)(p + 16u * i) * g.cols + c];
        b[i] = g.part_b[(size_t)(p + 16u * i) * g.cols + c];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sg += a[i];
        sb += b[i];
      }
    }
    for (; p < g.nparts; p += 16u) {
      sg += g.part_g[(size_t)p * g.cols + c];
      sb += g.part_b[(size_t)p * g.cols + c];
    }
  }
  red[0][grp][cl] = sg;
  red[1][grp][cl] = sb;
  __syncthreads();
  if (threadIdx.x < 32) {
    const uint32_t which = threadIdx.x >> 4, col = blockIdx.x * 16u + cl;
    float t = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += red[which][i][cl];
    float *out = which ? g.out2 : g.out;
    if (col < g.cols && out) out[col] = t;
  }
}

// reduce_sum along each row (axis 1): one block per row.
extern "C" __global__ __launch_bounds__(256) void bwpp_reduce_sum_rows(const BwppGradArgs g) {
  __shared__ float red[4];
  for (uint32_t r = blockIdx.x; r < g.rows; r += gridDim.x) {
    const float *x = g.a + (size_t)r * g.ld;
    float s = 0.0f;
    for (uint32_t c = threadIdx.x; c < g.cols; c += 256) s += x[c];
    s = block_sum256(s, red);
    if (threadIdx.x == 0) g.out[r] = s;
  }
}

// reduce_sum over rows (axis 0): a block owns 64 columns x one band of rows
// (blockIdx.y), its 4 waves every fourth row with 8 rows' loads in flight;
// the band sums go to part_g for bwpp_col_partials_sum, or with one band to
// out.  4096 x 4096: 36.4 us with a serial walk of 64-row bands, 13.2 us
// so.
extern "C" __global__ __launch_bounds__(256) void bwpp_reduce_sum_cols(const BwppGradArgs g) {
  __shared__ float red[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t c = blockIdx.x * 64u + (uint32_t)lane;
  const uint64_t band = ((uint64_t)g.rows + gridDim.y - 1) / gridDim.y;
  const uint64_t r0 = band * blockIdx.y, r1 = min((uint64_t)g.rows, r0 + band);
  float s = 0.0f;
  if (c < g.cols) {
    const float *x = g.a + c;
    uint64_t r = r0 + (uint64_t)wave;
    for (; r + 28 < r1; r += 32) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = x[(r + 4 * i) * g.ld];
      s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    for (; r < r1; r += 4) s += x[r * g.ld];
  }
  red[wave][lane] = s;
  __syncthreads();
  if (wave != 0 || c >= g.cols) return;
  s = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
  if (gridDim.y > 1) g.part_g[(size_t)blockIdx.y * g.cols + c] = s;
  else g.out[c] = s;
}

// Binary elementwise with broadcasting of b, and broadcast itself (op 4:
// out = b broadcast).  rows x cols, leading dimension ld for a / out, ldb
// for b when full.  vec (cols, ld, ldb multiples of 4, 16-byte aligned
// pointers): one float4 per thread per step, 128-bit loads and stores.
namespace {
__device__ __forceinline__ float ew1(uint32_t op, float a, float b) {
  switch (op) {
    case 0: return a + b;
    case 1: return a - b;
    case 2: return a * b;
    case 3: return a / b;
    case 5: return b / (1.0f + expf(-b));  // SiLU of b (bwpp_cpu_ref.c:4-6)
    default: return b;
  }
}
}  // namespace

extern "C" __global__ __launch_bounds__(256) void bwpp_elementwise(const BwppGradArgs g) {
  if (g.vec) {
    const uint32_t c4n = g.cols / 4;
    for (uint32_t r = blockIdx.x; r < g.rows; r += gridDim.x) {
      const float4 *ar = g.a ? reinterpret_cast<const float4 *>(g.a + (size_t)r * g.ld) : nullptr;
      float4 *orow = reinterpret_cast<float4 *>(g.out + (size_t)r * g.ld);
      const float4 *brow = g.bmode == 0 ? reinterpret_cast<const float4 *>(g.b + (size_t)r * g.ldb)
                                        : reinterpret_cast<const float4 *>(g.b);
      const float bs = g.bmode == 2 ? g.b[r] : g.b[0];
      for (uint32_t c = threadIdx.x; c < c4n; c += 256) {
        const float4 bv = g.bmode <= 1 ? brow[c] : make_float4(bs, bs, bs, bs);
        const float4 av = ar ? ar[c] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        orow[c] = make_float4(ew1(g.op, av.x, bv.x), ew1(g.op, av.y, bv.y), ew1(g.op, av.z, bv.z),
                              ew1(g.op, av.w, bv.w));
      }
    }
    return;
  }
  for (uint32_t r = blockIdx.x; r < g.rows; r += gridDim.x) {
    const float *ar = g.a ? g.a + (size_t)r * g.ld : nullptr;
    float *orow = g.out + (size_t)r * g.ld;
    for (uint32_t c = threadIdx.x; c < g.cols; c += 256) {
      float bv;
      switch (g.bmode) {
        case 0: bv = g.b[(size_t)r * g.ldb + c]; break;
        case 1: bv = g.b[c]; break;
        case 2: bv = g.b[r]; break;
        default: bv = g.b[0]; break;
      }
      orow[c] = ew1(g.op, ar ? ar[c] : 0.0f, bv);
    }
  }
}

// Several row-strided copies in one launch (the plan's multi-pair copy:
// weights into their column blocks of a concatenation, or the blocks of a
// concatenated gradient out to the separate outputs).  Block rows stride
// over the segments' rows laid end to end.
extern "C" __global__ __launch_bounds__(256) void bwpp_copy_multi(const BwppCopyArgs a) {
  const uint32_t total = a.row0[a.n];
  for (uint32_t r = blockIdx.x; r < total; r += gridDim.x) {
    uint32_t sg = 0;
    while (sg + 1 < a.n && r >= a.row0[sg + 1]) ++sg;
    const uint32_t rr = r - a.row0[sg], cols = a.cols[sg];
    const float *src = a.src[sg] + (size_t)rr * a.ld_src[sg];
    float *dst = a.dst[sg] + (size_t)rr * a.ld_dst[sg];
    if (a.vec) {
      for (uint32_t c = threadIdx.x; c < cols / 4; c += 256)
        reinterpret_cast<float4 *>(dst)[c] = reinterpret_cast<const float4 *>(src)[c];
    } else {
      for (uint32_t c = threadIdx.x; c < cols; c += 256) dst[c] = src[c];
    }
  }
}
