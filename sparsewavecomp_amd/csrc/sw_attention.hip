// sparsewave.sddmm, csr_row_reduce, csr_rowwise_map and the six-kernel
// sparse-attention chain on gfx950.
//
// Reference kernels (generated IR):
//   sddmm            ThreadPerRowSDDMMPattern, SparseWaveToGPU.cpp:667-750
//   csr_row_reduce   ThreadPerRowCSRRowReducePattern, SparseWaveToGPU.cpp:752-818
//   csr_rowwise_map  ThreadPerRowCSRRowwiseMapPattern, SparseWaveToGPU.cpp:820-878
//   attention chain  examples/pytorch/integration/SparseAttentionToSparseWave.cpp:230-315
//
// SDDMM: 64- and 16-row matrix-core tiles for block masks, runs of positions
// over a transposed right-hand side where scratch memory was given, one wave
// per row for small calls, and one thread per row for the rest.  Row
// reductions: groups of 2 to 64 lanes per row.  Row-wise maps: cut by
// positions.  Attention: one kernel for the whole chain where its shapes fit.
#include "sw_device.h"
#include "sw_internal.h"
#include "sw_sddmm_tile64.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

using namespace swd;

namespace sw {
int launch_spmm(const int32_t *ro, const int32_t *col, const float *val,
                const float *rhs, float *out, int64_t rows, int64_t rhs_rows,
                int64_t nnz, int64_t k, const sw_options &o, const char *what,
                hipStream_t st);
int launch_spmm(const int32_t *ro, const int32_t *col, const uint16_t *val,
                const uint16_t *rhs, uint16_t *out, int64_t rows,
                int64_t rhs_rows, int64_t nnz, int64_t k, const sw_options &o,
                const char *what, hipStream_t st);
}

namespace {

// waves per 16-row SDDMM tile (4: 20.9 us on configuration 5; 8: 24.6 us)
constexpr int kSddmmTileWaves = 4;

__device__ __forceinline__ float combine_sddmm(int kind, float sample,
                                               float dot, float alpha,
                                               float beta) {
  if (kind == SW_SDDMM_MUL)
    return sample * dot;
  if (kind == SW_SDDMM_AFFINE)
    return sample * beta + dot * alpha;
  return dot;
}

// arith.maximumf: NaN propagates, +0 is above -0 -- the IEEE 754-2019
// maximum, which gfx950 computes in one v_maximum3_f32 (llvm.maximum)
__device__ __forceinline__ float maximumf(float a, float b) {
  return __builtin_elementwise_maximum(a, b);
}

// A result as its op stores it: unchanged in fp32, rounded to bf16 (and
// widened back) for bf16 buffers.  The fused bf16 kernels round each
// intermediate where the separate ops would store it, so every bf16 schedule
// computes the six ops on bf16 buffers.
template <typename T>
__device__ __forceinline__ float as_stored(float v) {
  if constexpr (sizeof(T) == 4)
    return v;
  else
    return bf16_to_f32(f32_to_bf16(v));
}

__device__ __forceinline__ float map_value(int kind, float v, float rv) {
  switch (kind) {
  case SW_MAP_EXP_SUB:
    return expf(v - rv);
  case SW_MAP_DIV:
    return v / rv;
  case SW_MAP_SUB:
    return v - rv;
  default:
    return v * rv;
  }
}

// ---- SDDMM -----------------------------------------------------------------
// Thread-per-row (the reference's mapping and launch).  TKB > 0 (kdim = 64
// TKB, a block size that is a multiple of 64, for bf16 a 16-byte aligned
// lhs, which the host checks): each wave first tries its 64 consecutive
// rows as one matrix-core tile (sw_sddmm_tile64.h); rows of a tile without
// the shared column prefix are then computed by their own threads as below.
template <typename T, int RP, int LB, int TKB = 0>
__global__ __launch_bounds__(LB) void sddmm_thread_per_row(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const T *__restrict__ val, const T *__restrict__ lhs,
    const T *__restrict__ rhs, T *__restrict__ out, int32_t rows,
    int64_t cols, int32_t kdim, int kind, float alpha, float beta) {
  if constexpr (TKB > 0) {
    __shared__ int32_t lcol[LB / kWave][sw_tile64::kTileCols];
    const int64_t r0 = block_id() * blockDim.x +
                       (int64_t)wave_in_group() * kWave;
    if (r0 >= rows)
      return; // wave-uniform
    auto combine = [&](float sample, float dot) {
      return combine_sddmm(kind, sample, dot, alpha, beta);
    };
    if (val != nullptr ? sw_tile64::sddmm_tile64<T, TKB, true, true>(
                             ro, col, val, lhs, rhs, out, rows, cols, r0,
                             lcol[wave_in_group()], combine)
                       : sw_tile64::sddmm_tile64<T, TKB, false, false>(
                             ro, col, val, lhs, rhs, out, rows, cols, r0,
                             lcol[wave_in_group()], combine))
      return;
  }
  int64_t r = block_id() * blockDim.x + threadIdx.x;
  if (r >= rows)
    return;
  const T *a = lhs + r * kdim;
  // RP positions at a time, sixteen terms of each in flight: the
  // launch has one thread per row (8192 rows are 128 waves), so a row is a
  // chain of memory trips and registers are plentiful (LB, the launch
  // bound, sets how many).  Each position's dot is still added term by term
  // in order.
  const int32_t e = ro[r + 1];
  for (int32_t p = ro[r]; p < e; p += RP) {
    int64_t c[RP];
    float dot[RP];
#pragma unroll
    for (int j = 0; j < RP; ++j) {
      c[j] = col[std::min(p + j, e - 1)];
      dot[j] = 0.0f;
    }
    // the dot products of the step's positions, whose columns are cc
    auto dots = [&](const auto &cc) __attribute__((always_inline)) {
      int32_t i = 0;
      for (; i + 15 < kdim; i += 16) {
        float av[16], bv[RP][16];
#pragma unroll
        for (int u = 0; u < 16; ++u)
          av[u] = ldv(a + i + u);
#pragma unroll
        for (int j = 0; j < RP; ++j)
#pragma unroll
          for (int u = 0; u < 16; ++u)
            bv[j][u] = ldv(rhs + (int64_t)(i + u) * cols + cc[j]);
#pragma unroll
        for (int j = 0; j < RP; ++j)
#pragma unroll
          for (int u = 0; u < 16; ++u)
            dot[j] = __builtin_fmaf(av[u], bv[j][u], dot[j]);
      }
      for (; i < kdim; ++i) {
        const float av = ldv(a + i);
#pragma unroll
        for (int j = 0; j < RP; ++j)
          dot[j] = __builtin_fmaf(av, ldv(rhs + (int64_t)i * cols + cc[j]),
                                  dot[j]);
      }
    };
    // fp32: rows of a block-structured mask share their columns position
    // by position (83% of configuration 5's steps).  When every active
    // lane's step has the first active lane's columns, the rhs addresses are
    // wave-uniform and the rhs values scalar loads (configuration 5: 479 ->
    // 416 us).  The products and their order are the same either way.  (bf16
    // elements at odd columns cannot be scalar loads; the test alone made
    // it slower, 423 -> 475 us.)
    bool uniform = false;
    if constexpr (sizeof(T) == 4) {
      bool same = true;
#pragma unroll
      for (int j = 0; j < RP; ++j)
        same &= (int32_t)c[j] ==
                __builtin_amdgcn_readfirstlane((int32_t)c[j]);
      uniform = __builtin_amdgcn_ballot_w64(!same) == 0;
    }
    if (uniform) {
      int32_t cu[RP];
#pragma unroll
      for (int j = 0; j < RP; ++j)
        cu[j] = __builtin_amdgcn_readfirstlane((int32_t)c[j]);
      dots(cu);
    } else {
      dots(c);
    }
#pragma unroll
    for (int j = 0; j < RP; ++j)
      if (p + j < e)
        stv(out + p + j,
            combine_sddmm(kind, val != nullptr ? ldv(val + p + j) : 0.0f,
                          dot[j], alpha, beta));
  }
}

// One wave computes the SDDMM entries of row r: lane l takes positions
// start+l, start+l+64, ...; the row of lhs is held 64 values at a time, one
// per lane, and broadcast with v_readlane.
template <typename T>
__device__ __forceinline__ void sddmm_row_wave(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const T *__restrict__ val, const T *__restrict__ lhs,
    const T *__restrict__ rhs, T *__restrict__ out, int64_t r,
    int64_t cols, int32_t kdim, int kind, float alpha, float beta) {
  const int l = lane_id();
  const int32_t s = ro[r], e = ro[r + 1];
  const T *a = lhs + r * kdim;
  for (int32_t p0 = s; p0 < e; p0 += 4 * kWave) {
    float dot[4] = {0.f, 0.f, 0.f, 0.f};
    int64_t c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      int32_t p = p0 + j * kWave + l;
      c[j] = p < e ? (int64_t)col[p] : 0;
    }
    for (int32_t i0 = 0; i0 < kdim; i0 += kWave) {
      const float mine = (i0 + l < kdim) ? ldv(a + i0 + l) : 0.0f;
      const int n = std::min<int32_t>(kWave, kdim - i0);
      for (int t = 0; t < n; ++t) {
        const float av =
            __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine), t));
        const T *rrow = rhs + (int64_t)(i0 + t) * cols;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          dot[j] = __builtin_fmaf(av, ldv(rrow + c[j]), dot[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      int32_t p = p0 + j * kWave + l;
      if (p < e)
        stv(out + p, combine_sddmm(kind, val != nullptr ? ldv(val + p) : 0.0f,
                                   dot[j], alpha, beta));
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void sddmm_wave_per_row(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const T *__restrict__ val, const T *__restrict__ lhs,
    const T *__restrict__ rhs, T *__restrict__ out, int32_t rows,
    int64_t cols, int32_t kdim, int kind, float alpha, float beta) {
  const int64_t r = block_id() * (blockDim.x / kWave) +
                    wave_in_group();
  if (r >= rows)
    return; // wave-uniform
  sddmm_row_wave(ro, col, val, lhs, rhs, out, r, cols, kdim, kind, alpha,
                 beta);
}

// SDDMM over 16-row tiles on the matrix cores (kdim = 64 * KB).
//
// A workgroup of W waves owns rows r0 .. r0+15.  When every row's columns
// are a prefix of the last row's (tile_prefix_ok_block), the tile's dot products
// for 16 of the last row's columns at a time are one 16 x 16 x kdim product
//   D = lhs[r0 .. r0+15][:] * rhs[:][c_t0 .. c_t0+15]
// computed with v_mfma_f32_16x16x4_f32 (lane (i, g) supplies
// lhs[r0+i][16g+s] at step s, lane (j, g) supplies rhs[16g+s][c_j]); wave w
// takes the column chunks w, w+W, ...  Each result lands at its CSR position
// ro[row] + t when t is inside that row.  Tiles without the shared structure
// are computed row by row on the vector ALUs.
//
// Latency: the row bounds and lhs rows are requested before the structure
// check waits, and a chunk pair's sampled values before its rhs loads wait
// (checking the structure inside the chunk loop instead measured slower).
template <int KB, int W>
__global__ __launch_bounds__(64 * W) void sddmm_tile_mfma(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const float *__restrict__ val, const float *__restrict__ lhs,
    const float *__restrict__ rhs, float *__restrict__ out, int32_t rows,
    int64_t cols, int32_t kdim, int kind, float alpha, float beta) {
  if (block_id() * 16 >= rows)
    return; // a folded grid's surplus workgroup (workgroup-uniform)
  const int r0 = (int)block_id() * 16;
  const int nt = std::min(16, rows - r0);
  const int wave = wave_in_group();
  const int l = lane_id(), i = l & 15, g = l >> 4;
  // loads are unconditional from clamped, valid addresses, their values
  // selected afterwards (a guarded load becomes a branch that waits for it
  // on the spot)
  int32_t rb[4], rl[4];
  {
    int32_t b[5];
#pragma unroll
    for (int v = 0; v < 5; ++v)
      b[v] = ro[std::min(r0 + 4 * g + v, rows)];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      rb[v] = b[v];
      rl[v] = 4 * g + v < nt ? b[v + 1] - b[v] : 0;
    }
  }
  float qa[16 * KB];
  const int64_t qrow = (int64_t)std::min(r0 + i, rows - 1) * kdim;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int st = 0; st < 16; ++st) {
      const float x = lhs[qrow + kb * 64 + 16 * g + st];
      qa[kb * 16 + st] = i < nt ? x : 0.0f;
    }
  __shared__ int verdict;
  if (!tile_prefix_ok_block(ro, col, r0, nt, &verdict)) {
    for (int r = r0 + wave; r < r0 + nt; r += W)
      sddmm_row_wave(ro, col, val, lhs, rhs, out, r, cols, kdim, kind, alpha,
                     beta);
    return;
  }
  const int last = r0 + nt - 1;
  const int32_t bl = ro[last];
  const int32_t len_last = ro[last + 1] - bl;
  // two column chunks per iteration (W chunks apart): two independent
  // accumulators and 32 outstanding rhs loads per lane
  for (int32_t t0 = wave * 16; t0 < len_last; t0 += 32 * W) {
    const int32_t t1 = t0 + 16 * W;
    const bool two = t1 < len_last; // wave-uniform
    const int32_t ta = t0 + i, tb = t1 + i;
    const int64_t cj0 = ta < len_last ? (int64_t)col[bl + ta] : 0;
    const int64_t cj1 = two && tb < len_last ? (int64_t)col[bl + tb] : 0;
    float s0[4], s1[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      // position bl is inside the last row, always a valid index
      const bool in0 = val != nullptr && ta < rl[v];
      const bool in1 = val != nullptr && two && tb < rl[v];
      const float x0 = val != nullptr ? val[in0 ? rb[v] + ta : bl] : 0.0f;
      const float x1 = val != nullptr ? val[in1 ? rb[v] + tb : bl] : 0.0f;
      s0[v] = in0 ? x0 : 0.0f;
      s1[v] = in1 ? x1 : 0.0f;
    }
    v4f acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      float bv0[16], bv1[16];
#pragma unroll
      for (int st = 0; st < 16; ++st) {
        const float *rrow = rhs + (int64_t)(kb * 64 + 16 * g + st) * cols;
        bv0[st] = rrow[cj0];
        bv1[st] = two ? rrow[cj1] : 0.0f;
      }
#pragma unroll
      for (int st = 0; st < 16; ++st) {
        acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[kb * 16 + st], bv0[st],
                                                    acc0, 0, 0, 0);
        if (two)
          acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[kb * 16 + st],
                                                      bv1[st], acc1, 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (ta < rl[v])
        out[rb[v] + ta] = combine_sddmm(kind, s0[v], acc0[v], alpha, beta);
      if (two && tb < rl[v])
        out[rb[v] + tb] = combine_sddmm(kind, s1[v], acc1[v], alpha, beta);
    }
  }
}

// ---- SDDMM over a transposed rhs --------------------------------------------
// A stored entry's dot product reads a column of rhs, kdim elements a row of
// rhs apart: where neighbouring entries do not share the cache lines (a
// graph's columns) every element is a line of its own.  With scratch memory
// for the transposed rhs (the _ws entry points) it is transposed once, and
// an entry reads kdim consecutive elements.

// rhs[kdim][cols] as rhst[cols][kp], columns of kp >= kdim elements (a
// multiple of 16 bytes), zero past kdim.  64 x 64 tiles through LDS, both
// sides in whole lines.
template <typename T>
__global__ __launch_bounds__(256) void transpose_rhs(
    const T *__restrict__ rhs, T *__restrict__ rhst, int64_t cols,
    int32_t kdim, int32_t kp, int64_t col_tiles) {
  __shared__ T tile[64][64 + 4 / sizeof(T)];
  const int64_t id = block_id();
  const int64_t kt = id / col_tiles;
  const int64_t c0 = (id - kt * col_tiles) * 64;
  const int32_t k0 = (int32_t)kt * 64;
  if (k0 >= kp)
    return; // a folded grid's surplus workgroup (workgroup-uniform)
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  // unconditional loads from clamped addresses, all sixteen in flight, and
  // 16-byte stores (guarded loads and one element a store: 2.6 us longer for
  // 50,021 x 64 in fp32)
  const int64_t cc = std::min<int64_t>(c0 + x, cols - 1);
  T in[16];
#pragma unroll
  for (int u = 0; u < 16; ++u)
    in[u] = rhs[(int64_t)std::min(k0 + 4 * u + y, kdim - 1) * cols + cc];
#pragma unroll
  for (int u = 0; u < 16; ++u)
    tile[4 * u + y][x] = k0 + 4 * u + y < kdim ? in[u] : T(0);
  __syncthreads();
  // 16 bytes of a column of rhs a lane (kp is a multiple of V)
  constexpr int V = 16 / (int)sizeof(T), L = 64 / V;
  const int kx = V * (int)(threadIdx.x & (L - 1)), cy = threadIdx.x / L;
#pragma unroll
  for (int u = 0; u < 64 * L / 256; ++u) {
    const int ct = cy + 256 / L * u;
    if (c0 + ct < cols && k0 + kx < kp) {
      T o[V];
#pragma unroll
      for (int v = 0; v < V; ++v)
        o[v] = tile[kx + v][ct];
      v4u w;
      __builtin_memcpy(&w, o, sizeof w);
      *reinterpret_cast<v4u *>(rhst + (c0 + ct) * kp + k0 + kx) = w;
    }
  }
}

// A wave takes 64 consecutive positions, lane l holding position l's row
// (wave-uniform searches for the first and last, then its own between them),
// column and sample.  G lanes compute an entry's dot product, V = 16 bytes'
// worth of elements a lane and step from the lhs row and the transposed
// column, 64 / G entries at a time and U such steps' loads in flight; the
// sums return to the entries' lanes, whose stores are consecutive.  The work
// is cut by entries, so rows of any length cost the same.
// It is bound by the gathered columns' trips from L2 and the MALL (246 MB).
// 60,013 x 50,021, 960,000 entries, kdim = 64, fp32: 1904 us one thread per
// row, 643 one wave per row, 44.5 here.
template <typename T, int G>
__global__ __launch_bounds__(256) void sddmm_positions(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const T *val, const T *__restrict__ lhs, const T *__restrict__ rhst,
    T *out, int32_t rows, int32_t nnz, int32_t kdim, int32_t kp, int kind,
    float alpha, float beta) {
  constexpr int V = 16 / (int)sizeof(T);
  constexpr int E = kWave / G; // entries a step
  constexpr int U = G < 4 ? G : 4;
  using Vec = std::conditional_t<sizeof(T) == 4, v4f, v4u>;
  const int64_t first =
      (block_id() * (blockDim.x / kWave) + wave_in_group()) * kWave;
  if (first >= nnz)
    return; // wave-uniform
  const int l = lane_id(), gl = l & (G - 1), q = l / G;
  const int32_t n = (int32_t)std::min<int64_t>(kWave, nnz - first);
  // (lanes past the end repeat the last position)
  const int32_t p = (int32_t)first + std::min(l, n - 1);
  // positions outside the rows (ro may be a slice of a matrix's offsets, the
  // arrays longer than the rows): their columns are not used, their row is
  // the first or last one, and nothing is stored; a wave that holds no other
  // ends here, so that a slice costs its own entries
  const int32_t base = ro[0], top = ro[rows];
  if (first >= top || first + n <= base)
    return; // wave-uniform
  const bool stored = p >= base && p < top;
  const int32_t cp = col[p];
  const int32_t c = stored ? cp : 0;
  const float sample = val != nullptr ? ldv(val + p) : 0.0f;
  const int fr = row_search_uniform(ro, 1u, (uint32_t)rows, (int32_t)first);
  const int lr = row_search_gallop(ro, (uint32_t)fr + 1u, (uint32_t)rows,
                                   (int32_t)first + n - 1);
  const int32_t r = row_search_lane(ro, (uint32_t)fr + 1u, (uint32_t)lr + 1u,
                                    p);
  float mine = 0.0f;
  for (int e0 = 0; e0 < n; e0 += E * U) { // wave-uniform
    float dot[U];
    int32_t rr[U], cc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int src = (e0 + E * u + q) << 2; // < 64: E U divides 64
      rr[u] = __builtin_amdgcn_ds_bpermute(src, r);
      cc[u] = __builtin_amdgcn_ds_bpermute(src, c);
      dot[u] = 0.0f;
    }
    for (int32_t k0 = 0; k0 < kdim; k0 += G * V) {
      const int32_t k = k0 + gl * V;
      Vec a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        a[u] = b[u] = Vec{};
      if (k < kdim) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          b[u] = *reinterpret_cast<const Vec *>(rhst + (int64_t)cc[u] * kp +
                                                k);
        // (a lhs row ends at kdim, the next one's elements must not be read
        // past the last row's end)
        if (k + V <= kdim) {
#pragma unroll
          for (int u = 0; u < U; ++u)
            __builtin_memcpy(&a[u], lhs + (int64_t)rr[u] * kdim + k,
                             sizeof(Vec));
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            T x[V];
#pragma unroll
            for (int v = 0; v < V; ++v)
              x[v] = k + v < kdim ? lhs[(int64_t)rr[u] * kdim + k + v] : T(0);
            __builtin_memcpy(&a[u], x, sizeof x);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        T x[V], y[V];
        __builtin_memcpy(x, &a[u], sizeof x);
        __builtin_memcpy(y, &b[u], sizeof y);
#pragma unroll
        for (int v = 0; v < V; ++v)
          dot[u] = __builtin_fmaf(tof(x[v]), tof(y[v]), dot[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float sum = group_sum<G>(dot[u]);
      // entry e0 + E u + j was computed by the lanes G j .. G j + G - 1
      const float s = __int_as_float(__builtin_amdgcn_ds_bpermute(
          (G * (l & (E - 1))) << 2, __float_as_int(sum)));
      mine = l / E == (e0 / E) + u ? s : mine;
    }
  }
  if (l < n && stored)
    stv(out + p, combine_sddmm(kind, sample, mine, alpha, beta));
}

__device__ __forceinline__ float wave_max(float v) {
  v = maximumf(v, dpp_f<kQuadXor1>(-INFINITY, v));
  v = maximumf(v, dpp_f<kQuadXor2>(-INFINITY, v));
  v = maximumf(v, dpp_f<kRowHalfMirror>(-INFINITY, v));
  v = maximumf(v, dpp_f<kRowMirror>(-INFINITY, v));
  v = maximumf(v, swizzle_xor16(v));
  v = maximumf(v, shfl_xor32(v));
  return v;
}

// ---- row reductions ---------------------------------------------------------
// A group of G lanes takes a row (64 / G consecutive rows a wave), each lane
// eight of its entries a step in 16-byte windows, so that neighbouring groups
// stream neighbouring memory; rows of more than kGroupSteps steps are taken
// by the whole wave, one after another.  The sums' order is fixed by the
// row's length and G.  300,007 rows of 24 entries on average (lognormal, up
// to 4,096), fp32: maximum 40 us one thread per row (each lane walking its
// own lines), 12 us here, 29 MB.
constexpr int kRowEntries = 8; // entries a lane holds
constexpr int kGroupSteps = 4;

// The W = 16 bytes' worth of entries from position p on, those below `end`
// valid (others undefined); nothing is read past nnz.
template <typename T>
__device__ __forceinline__ void load_window(const T *val, int64_t p,
                                            int32_t end, int32_t nnz,
                                            T (&x)[16 / sizeof(T)]) {
  constexpr int W = 16 / (int)sizeof(T);
#pragma unroll
  for (int u = 0; u < W; ++u)
    x[u] = T(0);
  if (p < end) {
    if (p + W <= nnz) {
      __builtin_memcpy(x, val + p, sizeof x);
    } else {
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (p + u < end)
          x[u] = val[p + u];
    }
  }
}

template <bool MAX, typename T>
__device__ __forceinline__ float fold(float acc, const T *x, int64_t p,
                                      int32_t end) {
  constexpr int W = 16 / (int)sizeof(T);
#pragma unroll
  for (int u = 0; u < W; ++u) {
    const float v = tof(x[u]);
    acc = p + u < end ? (MAX ? maximumf(acc, v) : acc + v) : acc;
  }
  return acc;
}

template <int G>
__device__ __forceinline__ float group_max(float v) {
  if constexpr (G >= 2) v = maximumf(v, dpp_f<kQuadXor1>(-INFINITY, v));
  if constexpr (G >= 4) v = maximumf(v, dpp_f<kQuadXor2>(-INFINITY, v));
  if constexpr (G >= 8) v = maximumf(v, dpp_f<kRowHalfMirror>(-INFINITY, v));
  if constexpr (G >= 16) v = maximumf(v, dpp_f<kRowMirror>(-INFINITY, v));
  if constexpr (G >= 32) v = maximumf(v, swizzle_xor16(v));
  if constexpr (G >= 64) v = maximumf(v, shfl_xor32(v));
  return v;
}

template <bool MAX, typename T, int G>
__global__ __launch_bounds__(1024) void row_reduce_group(
    const int32_t *__restrict__ ro, const T *__restrict__ val,
    T *__restrict__ out, int32_t rows, int32_t nnz) {
  constexpr int W = 16 / (int)sizeof(T), N = kRowEntries / W;
  const int64_t r = (block_id() * blockDim.x + threadIdx.x) / G;
  const int gl = threadIdx.x & (G - 1);
  const bool in = r < rows;
  const int32_t s = in ? ro[r] : 0, e = in ? ro[r + 1] : 0;
  bool wide = e - s > kGroupSteps * kRowEntries * G;
  uint64_t m = ballot(wide && gl == 0);
  if (m != 0) {
    // the wave's long rows one after another, a trip and more each, unless the
    // groups' steps over the longest are fewer (neighbours as long, as where
    // rows are sorted by length: 445,278 rows of 19, bf16, 22.5 us otherwise,
    // one thread per row 11.9)
    int32_t longest = 0, trips = 0;
    for (uint64_t left = m; left != 0; left &= left - 1) { // wave-uniform
      const int src = __builtin_ctzll(left);
      const int32_t len = __builtin_amdgcn_readlane(e, src) -
                          __builtin_amdgcn_readlane(s, src);
      longest = len > longest ? len : longest;
      trips += 1 + len / (4 * W * kWave);
    }
    if (trips >= longest / (kRowEntries * G)) {
      wide = false;
      m = 0;
    }
  }
  const int32_t end = wide ? s : e;
  float acc = MAX ? -INFINITY : 0.0f;
  for (int32_t at = s; ballot(at < end) != 0; at += kRowEntries * G) {
    T x[N][W];
#pragma unroll
    for (int n = 0; n < N; ++n)
      load_window(val, (int64_t)at + W * (gl + G * n), end, nnz, x[n]);
#pragma unroll
    for (int n = 0; n < N; ++n)
      acc = fold<MAX>(acc, x[n], (int64_t)at + W * (gl + G * n), end);
  }
  acc = MAX ? group_max<G>(acc) : group_sum<G>(acc);
  if (in && !wide && gl == 0)
    stv(out + r, acc);
  // the wave's long rows
  while (m != 0) { // wave-uniform
    const int src = __builtin_ctzll(m);
    m &= m - 1;
    const int32_t ls = __builtin_amdgcn_readlane(s, src);
    const int32_t le = __builtin_amdgcn_readlane(e, src);
    float a = MAX ? -INFINITY : 0.0f;
    for (int64_t p = ls + (int64_t)W * lane_id(); p - W * lane_id() < le;
         p += 4 * W * kWave) {
      T y[4][W];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        load_window(val, p + W * kWave * u, le, nnz, y[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        a = fold<MAX>(a, y[u], p + W * kWave * u, le);
    }
    a = MAX ? wave_max(a) : group_sum<kWave>(a);
    if (lane_id() == src)
      stv(out + r, a);
  }
}

// ---- row-wise map ----------------------------------------------------------
// Cut by entries: a wave takes N windows of 64 W consecutive positions, W =
// 16 bytes' worth a lane, so that every load and store is a whole coalesced
// window whatever the rows' lengths.  The wave finds the rows of its first
// and last position by 64 probes a trip under the loads, stages the rows'
// ends and values between them in LDS, and each lane searches the row of its
// first position there and steps on from it; over wider spans each entry
// searches ro itself.  out may be val (in place): a
// lane reads its entries before it writes them.  KIND is a template argument:
// no switch per entry.  300,007 rows of 24 entries on average (lognormal), fp32:
// exp(v - max) 147 us one thread per row, 21 us here, 58 MB.
constexpr int kMapRows = 512; // rows staged per wave

template <typename T, int KIND, int N>
__global__ __launch_bounds__(256) void rowwise_map_positions(
    const int32_t *__restrict__ ro, const T *val, const T *__restrict__ rowv,
    T *out, int32_t rows, int32_t nnz) {
  constexpr int W = 16 / (int)sizeof(T);
  __shared__ int32_t ends[256 / kWave][kMapRows];
  __shared__ float values[256 / kWave][kMapRows];
  const int wave = wave_in_group(), l = lane_id();
  const int64_t first =
      (block_id() * (blockDim.x / kWave) + wave) * (int64_t)(kWave * W * N);
  if (first >= nnz)
    return; // wave-uniform; the kernel has no workgroup barrier
  const int64_t last = std::min<int64_t>(first + kWave * W * N, nnz) - 1;
  // positions outside the rows (ro may be a slice of a matrix's offsets, the
  // arrays longer than the rows) find the first or last row and are not
  // stored; a wave that holds no other ends here, so that a slice costs its
  // own entries (2,000 of 2,000,000 rows of 20, fp32: 31 us otherwise, 9 so)
  const int32_t base = ro[0], top = ro[rows];
  if (first >= top || last < base)
    return; // wave-uniform
  T x[N][W];
#pragma unroll
  for (int n = 0; n < N; ++n)
    load_window(val, first + W * (l + kWave * n), nnz, nnz, x[n]);
  int fr, lr;
  row_search_wave(ro, 1, rows, (int32_t)first, (int32_t)last, &fr, &lr);
  const int span = lr - fr; // wave-uniform
  const bool staged = span < kMapRows;
  int32_t *win = ends[wave];
  float *rvs = values[wave];
  if (staged) {
    for (int j = l; j <= span; j += kWave) {
      win[j] = ro[fr + 1 + j];
      rvs[j] = ldv(rowv + fr + j);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int64_t p0 = first + W * (l + kWave * n);
    if (p0 >= top)
      break;
    T y[W];
    if (staged) {
      int row = 0, hi = span; // the first row that ends past p0
      auto search = [&](int64_t p) __attribute__((always_inline)) {
        while (row < hi) {
          const int mid = (row + hi) >> 1;
          if (win[mid] <= p)
            row = mid + 1;
          else
            hi = mid;
        }
      };
      search(p0);
      int32_t next = win[row];
      float rv = rvs[row];
#pragma unroll
      for (int u = 0; u < W; ++u) {
        // (row < span also ends the walk past the last row)
        if (p0 + u >= next && row < span) {
          // mostly the next row; past empty ones by bisection
          ++row;
          hi = win[row] > p0 + u ? row : span;
          search(p0 + u);
          next = win[row];
          rv = rvs[row];
        }
        stv(&y[u], map_value(KIND, tof(x[n][u]), rv));
      }
    } else {
      // each entry's own bisection, W probes in flight: a run of empty rows
      // between two entries may be of any length (100,000 of them: 10,963 us
      // row by row, 9.2 so)
      uint32_t lo[W], hi[W];
#pragma unroll
      for (int u = 0; u < W; ++u) {
        lo[u] = (uint32_t)fr + 1u;
        hi[u] = (uint32_t)lr + 1u;
      }
      for (int left = span; left > 0; left >>= 1) // wave-uniform
#pragma unroll
        for (int u = 0; u < W; ++u) {
          const uint32_t mid = lo[u] + ((hi[u] - lo[u]) >> 1);
          const bool up = ro[std::min(mid, (uint32_t)lr)] <= p0 + u;
          const bool open = lo[u] < hi[u];
          lo[u] = open && up ? mid + 1 : lo[u];
          hi[u] = open && !up ? mid : hi[u];
        }
#pragma unroll
      for (int u = 0; u < W; ++u)
        stv(&y[u], map_value(KIND, tof(x[n][u]), ldv(rowv + lo[u] - 1)));
    }
    if (p0 >= base && p0 + W <= top) {
      __builtin_memcpy(out + p0, y, sizeof y);
    } else {
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (p0 + u >= base && p0 + u < top)
          out[p0 + u] = y[u];
    }
  }
}

// The four row ops of the attention chain fused (row max, exp(s - max), row
// sum, s / sum): one wave per row.  Rows of up to 64 * kSoftmaxRegs entries
// stay in registers between the ops (one read and one write of the scores);
// longer rows take a max pass and two read/write passes.  rowMaximum and
// rowSum are written as the separate ops would write them.
constexpr int kSoftmaxRegs = 8;

template <typename T>
__global__ __launch_bounds__(256) void row_softmax_wave(
    const int32_t *__restrict__ ro, T *scores, T *__restrict__ rmax,
    T *__restrict__ rsum, int32_t rows) {
  const int64_t r = block_id() * (blockDim.x / kWave) +
                    wave_in_group();
  if (r >= rows)
    return;
  const int l = lane_id();
  const int32_t s = ro[r], e = ro[r + 1];
  float m = -INFINITY;
  float sum = 0.0f;
  if (e > s && e - s <= kWave * kSoftmaxRegs) { // wave-uniform
    float v[kSoftmaxRegs];
#pragma unroll
    for (int j = 0; j < kSoftmaxRegs; ++j) {
      // unconditional load from a clamped index, then select (a guarded
      // load would wait on the spot)
      const int32_t p = s + l + j * kWave;
      const float x = ldv(scores + (p < e ? p : e - 1));
      v[j] = p < e ? x : -INFINITY;
      m = maximumf(m, v[j]);
    }
    m = wave_max(m);
#pragma unroll
    for (int j = 0; j < kSoftmaxRegs; ++j)
      if (s + l + j * kWave < e) {
        v[j] = as_stored<T>(expf(v[j] - m));
        sum += v[j];
      }
    sum = as_stored<T>(group_sum<kWave>(sum));
#pragma unroll
    for (int j = 0; j < kSoftmaxRegs; ++j) {
      const int32_t p = s + l + j * kWave;
      if (p < e)
        stv(scores + p, v[j] / sum);
    }
  } else {
    for (int32_t p = s + l; p < e; p += kWave)
      m = maximumf(m, ldv(scores + p));
    m = wave_max(m);
    for (int32_t p = s + l; p < e; p += kWave) {
      const float v = as_stored<T>(expf(ldv(scores + p) - m));
      stv(scores + p, v);
      sum += v;
    }
    sum = as_stored<T>(group_sum<kWave>(sum));
    for (int32_t p = s + l; p < e; p += kWave)
      stv(scores + p, ldv(scores + p) / sum);
  }
  if (l == 0) {
    stv(rmax + r, m);
    stv(rsum + r, sum);
  }
}

// Row r of the attention output computed by one wave from the row's
// normalised scores (the fused kernel's per-row path): lanes over the output
// columns, sequential over the row's positions.
template <typename T>
__device__ __forceinline__ void attention_row_output(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const T *scores, const T *__restrict__ value, T *__restrict__ out,
    int64_t r, int64_t dv) {
  const int32_t s = ro[r], e = ro[r + 1];
  for (int64_t c = lane_id(); c < dv; c += kWave) {
    float acc = 0.0f;
    for (int32_t p = s; p < e; ++p)
      acc = __builtin_fmaf(ldv(scores + p),
                           ldv(value + (int64_t)col[p] * dv + c), acc);
    stv(out + r * dv + c, acc);
  }
}

// One row's softmax in global memory by one wave (the fused kernel's
// per-row path): the long-row branch of row_softmax_wave.
template <typename T>
__device__ __forceinline__ void attention_row_softmax(
    const int32_t *__restrict__ ro, T *scores, T *__restrict__ rmax,
    T *__restrict__ rsum, int64_t r) {
  const int l = lane_id();
  const int32_t s = ro[r], e = ro[r + 1];
  float m = -INFINITY, sum = 0.0f;
  for (int32_t p = s + l; p < e; p += kWave)
    m = maximumf(m, ldv(scores + p));
  m = wave_max(m);
  for (int32_t p = s + l; p < e; p += kWave) {
    const float v = as_stored<T>(expf(ldv(scores + p) - m));
    stv(scores + p, v);
    sum += v;
  }
  sum = as_stored<T>(group_sum<kWave>(sum));
  for (int32_t p = s + l; p < e; p += kWave)
    stv(scores + p, ldv(scores + p) / sum);
  if (l == 0) {
    stv(rmax + r, m);
    stv(rsum + r, sum);
  }
}

// the eight K^T values K^T[32 s + 8 g + e][c] (e = 0..7) as four bf16 pairs;
// base is K^T row 32 s, lane_off the byte offset of column c plus 8 g rows
__device__ __forceinline__ v4u gather_kt8(const uint16_t *base,
                                          uint32_t row_bytes,
                                          uint32_t lane_off) {
  uint32_t x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    x[e] = *at_bytes(at_bytes(base, e * row_bytes), lane_off);
  return v4u{x[0] | (x[1] << 16), x[2] | (x[3] << 16), x[4] | (x[5] << 16),
             x[6] | (x[7] << 16)};
}

// exp and division of the fused tiles.  LIBM: the library's expf and the
// IEEE division, as the six separate ops compute them; otherwise the hardware
// base-2 exponential (exp_by_exp2) and a multiply by the row's reciprocal.
template <bool LIBM>
__device__ __forceinline__ float tile_exp(float x) {
  if constexpr (LIBM)
    return expf(x);
  else
    return exp_by_exp2(x);
}
template <bool LIBM>
__device__ __forceinline__ float tile_div(float v, float sum, float rsum) {
  if constexpr (LIBM)
    return v / sum;
  else
    return v * rsum;
}

// the fused tiles' waves, and the entries of a row that they hold in
// registers (each wave kFusedChunks chunks of 16)
constexpr int kFusedCols = 512;
constexpr int kFusedWaves = 8;
constexpr int kFusedChunks = kFusedCols / (16 * kFusedWaves);

// The structure check of a tile whose last row holds more than kFusedCols
// entries: row after row against the last row's columns, wave w rows w and
// w + W (nt <= 16 = 2 W), 512 entries a trip as 16-byte windows.  A window
// of a row before the last that holds a compared entry starts below bl <=
// nnz - kFusedCols and is never moved; the last row's are read from
// min(e, amax) and shifted.  Every thread of the workgroup calls it.
template <int W>
__device__ __forceinline__ bool long_tile_prefix_ok(
    const int32_t *__restrict__ col, int32_t my_ro, int nt, int32_t bl,
    int32_t len_last, uint32_t amax, int *verdict /* __shared__ int[W] */) {
  const int wave = wave_in_group();
  const int l = lane_id();
  int32_t b[2], len[2];
  bool ok = true;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int rr = wave + h * W;
    const int rc = rr < nt - 1 ? rr : nt - 1; // the last row against itself
    b[h] = __builtin_amdgcn_readlane(my_ro, rc);
    len[h] = __builtin_amdgcn_readlane(my_ro, rc + 1) - b[h];
    ok &= len[h] <= len_last;
    if (rr >= nt - 1)
      len[h] = 0; // nothing to compare
  }
  const int32_t most = std::min(std::max(len[0], len[1]), len_last);
  for (int32_t t0 = 0; t0 < most; t0 += 8 * kWave) { // wave-uniform
    v4i x[2][2], y[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int32_t t = t0 + 4 * (l + u * kWave);
      auto at = [&](int32_t row) __attribute__((always_inline)) {
        v4i z;
        __builtin_memcpy(
            &z, at_bytes(col, 4u * std::min((uint32_t)(row + t), amax)),
            sizeof z);
        return z;
      };
      y[u] = at(bl);
      x[0][u] = at(b[0]);
      x[1][u] = at(b[1]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int32_t t = t0 + 4 * (l + u * kWave);
      const uint32_t e = (uint32_t)(bl + t);
      const uint32_t d = e - std::min(e, amax);
      const v4i z = {d == 0 ? y[u].x : d == 1 ? y[u].y : d == 2 ? y[u].z
                                                                : y[u].w,
                     d == 0 ? y[u].y : d == 1 ? y[u].z : y[u].w,
                     d == 0 ? y[u].z : y[u].w, y[u].w};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < 4; ++m)
          ok &= (t + m >= len[h]) | (x[h][u][m] == z[m]);
    }
  }
  const bool mine = __builtin_amdgcn_ballot_w64(!ok) == 0;
  if (l == 0)
    verdict[wave] = mine;
  __syncthreads();
  ok = true;
#pragma unroll
  for (int w = 0; w < W; ++w)
    ok &= verdict[w] != 0;
  return ok;
}

// A 16-row tile with the shared column structure whose last row holds more
// entries than the fused kernels keep in registers (kFusedCols): the same
// chunks, products and roundings in three passes over the tile's chunks,
// wave w taking the 16-entry chunks w, w + W, ...
//   A. S^T = K_chunk Q^T; the scores, as their op stores them, go to the
//      score buffer (each lane re-reads only what it wrote itself) and into
//      the running row maxima;
//   B. (after the maxima met in LDS) the exponentials' row sums;
//   C. P = exp / sum, stored over the scores, and output = P V, 64 columns
//      at a time, the waves' partial tiles summed through LDS.
// The extra passes re-read 2 or 4 bytes per entry from L2, against a K^T
// column and a V row per entry and 16 rows.  SO: pass A alone.  Every wave
// of the workgroup calls it; returns with every output stored.
// 16,384 positions of up to 768 entries, d = dv = 128, bf16: 2002 us row by
// row, 80 us here; fp32 2039 and 126 us.  Without the K^T or the V gathers
// it would take 71 or 68 us: two rounds of a chain of about twenty dependent
// trips, two workgroups a CU.
template <typename T, int KB, int W, bool IL, bool SO, bool NS, bool LIBM>
__device__ __forceinline__ void attention_long_tile(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const T *__restrict__ mask, const T *__restrict__ q,
    const T *__restrict__ kt, const T *__restrict__ value, T *scores,
    T *__restrict__ rmax, T *__restrict__ rsum, T *__restrict__ out,
    int64_t cols, int32_t kdim, int64_t dv, float alpha, float beta,
    uint32_t amax, int region, int r0, int nt, int32_t rbase, int32_t la,
    int32_t bl, int32_t len_last,
    const std::conditional_t<std::is_same_v<T, float>, float, v4u> (
        &qb)[std::is_same_v<T, float> ? 16 * KB : 2 * KB],
    float (&part)[W][4][4][kWave], float (&wred)[2][W][16],
    int &v_nonfinite) {
  constexpr bool kF32 = std::is_same_v<T, float>;
  constexpr int S = kF32 ? 16 * KB : 2 * KB;
  using Op = std::conditional_t<kF32, float, v4u>;
  using Win = std::conditional_t<kF32, v4f, v2u>; // four entries
  const int wave = wave_in_group();
  const int l = lane_id(), i = l & 15, g = l >> 4;
  // (its own copies of the strides: shared with the register path, their
  // multiples stayed live through both and spilled)
  asm volatile("" : "+s"(cols), "+s"(dv));
  // the column of entry t0 + i of the last row (its final column past it)
  auto column = [&](int32_t t0) __attribute__((always_inline)) {
    return (uint32_t)*at_bytes(
        col, 4u * (uint32_t)(bl + std::min(t0 + i, len_last - 1)));
  };
  // entries t0 + 4g .. + 3 of row i: a window read from min(e, amax)
  auto window = [&](const T *p, int32_t t0) __attribute__((always_inline)) {
    const uint32_t e = (uint32_t)(rbase + t0 + 4 * g);
    const uint32_t w = std::min(e, amax);
    Win y;
    __builtin_memcpy(&y, at_bytes(p, (uint32_t)sizeof(T) * w), sizeof y);
    return y;
  };
  auto entries = [&](const Win &y, int32_t t0, float (&x)[4])
      __attribute__((always_inline)) {
    const uint32_t e = (uint32_t)(rbase + t0 + 4 * g);
    const uint32_t d = e - std::min(e, amax);
    if constexpr (kF32) {
      x[0] = d == 0 ? y.x : d == 1 ? y.y : d == 2 ? y.z : y.w;
      x[1] = d == 0 ? y.y : d == 1 ? y.z : y.w;
      x[2] = d == 0 ? y.z : y.w;
      x[3] = y.w;
    } else {
      const uint64_t w = ((uint64_t)y.y << 32) | y.x;
      const uint64_t z = d < 4 ? w >> (16 * d) : 0ull;
#pragma unroll
      for (int v = 0; v < 4; ++v)
        x[v] = bf16_to_f32((uint16_t)(z >> (16 * v)));
    }
  };
  auto valid = [&](int32_t t0, int v) __attribute__((always_inline)) {
    return t0 + 4 * g + v < la;
  };
  auto store = [&](int32_t t0, const float (&x)[4])
      __attribute__((always_inline)) {
    T *dst = scores + rbase + t0 + 4 * g;
    Win y;
    if constexpr (kF32)
      y = v4f{x[0], x[1], x[2], x[3]};
    else
      y = v2u{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
    if (valid(t0, 3)) {
      __builtin_memcpy(dst, &y, sizeof y);
    } else {
#pragma unroll
      for (int v = 0; v < 3; ++v)
        if (valid(t0, v))
          stv(dst + v, x[v]);
    }
  };
  const uint32_t row_bytes = (uint32_t)sizeof(T) * (uint32_t)cols;
  const __amdgpu_buffer_rsrc_t kt_rsrc =
      buffer_rsrc(kt, (uint32_t)kdim * row_bytes);
  auto gather_k = [&](uint32_t c, Op (&a)[S]) __attribute__((always_inline)) {
    if constexpr (kF32) {
      const uint32_t ko = 16u * g * row_bytes + 4u * c;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int st = 0; st < 16; ++st)
          a[kb * 16 + st] = buffer_load_f32(kt_rsrc, ko,
                                            (uint32_t)(kb * 64 + st) *
                                                row_bytes);
    } else {
      const uint32_t ko = 2u * c + 8u * g * row_bytes;
#pragma unroll
      for (int s = 0; s < S; ++s)
        a[s] = gather_kt8(kt + (int64_t)(32 * s) * cols, row_bytes, ko);
    }
  };
  // A.  The next columns a step ahead (two chunks' gathers in flight
  // measured no faster).
  float m = -INFINITY;
  uint32_t cn = column(16 * wave);
  for (int32_t t0 = 16 * wave; t0 < len_last; t0 += 16 * W) {
    Op a[S];
    gather_k(cn, a);
    Win mw = Win{};
    if constexpr (!NS)
      mw = window(mask, t0);
    cn = column(t0 + 16 * W);
    __builtin_amdgcn_sched_barrier(0);
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    if constexpr (kF32) {
      v4f acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < S; st += 2) {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[st], qb[st], acc, 0, 0,
                                                   0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[st + 1], qb[st + 1],
                                                    acc1, 0, 0, 0);
      }
      acc += acc1;
    } else {
#pragma unroll
      for (int s = 0; s < S; ++s)
        acc = mfma_16x16x32_bf16(a[s], qb[s], acc);
    }
    float x[4], sv[4];
    entries(mw, t0, x);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      sv[v] = as_stored<T>(combine_sddmm(
          region, valid(t0, v) ? x[v] : 0.0f, acc[v], alpha, beta));
      if constexpr (!SO)
        m = valid(t0, v) ? maximumf(m, sv[v]) : m;
    }
    store(t0, sv);
  }
  if constexpr (SO)
    return;
  m = maximumf(m, swizzle_xor16(m));
  m = maximumf(m, shfl_xor32(m));
  if (g == 0)
    wred[0][wave][i] = m;
  if (threadIdx.x == 0)
    v_nonfinite = 0;
  __syncthreads();
  m = wred[0][0][i];
#pragma unroll
  for (int w = 1; w < W; ++w)
    m = maximumf(m, wred[0][w][i]);
  // B.
  auto exps = [&](const Win &y, int32_t t0, float (&x)[4])
      __attribute__((always_inline)) {
    entries(y, t0, x);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float e = as_stored<T>(tile_exp<LIBM>(x[v] - m));
      x[v] = valid(t0, v) ? e : 0.0f;
    }
  };
  float sum = 0.0f;
  for (int32_t t0 = 16 * wave; t0 < len_last; t0 += 64 * W) {
    Win y[4]; // chunks past the row hold nothing valid
#pragma unroll
    for (int h = 0; h < 4; ++h)
      y[h] = window(scores, t0 + 16 * W * h);
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float x[4];
      exps(y[h], t0 + 16 * W * h, x);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        sum += x[v];
    }
  }
  sum += swizzle_xor16(sum);
  sum += shfl_xor32(sum);
  if (g == 0)
    wred[1][wave][i] = sum;
  __syncthreads();
  sum = wred[1][0][i];
#pragma unroll
  for (int w = 1; w < W; ++w)
    sum += wred[1][w][i];
  sum = as_stored<T>(sum);
  const float rsum_i = 1.0f / sum;
  if (wave == 0 && g == 0 && i < nt) {
    stv(rmax + r0 + i, m);
    stv(rsum + r0 + i, sum);
  }
  // C.  The next columns a step ahead; bf16 takes two 64-column blocks of
  // the output in one pass over the entries.
  constexpr int NB = kF32 ? 1 : 2;
  bool nonfinite = false;
  for (int64_t nb0 = 0; nb0 < dv; nb0 += 64 * NB) {
    const int ntiles0 = (int)std::min<int64_t>(4, (dv - nb0) / 16);
    const bool both = NB == 2 && nb0 + 64 < dv; // wave-uniform
    v4f acc[NB][4];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int n = 0; n < 4; ++n)
        acc[j][n] = v4f{0.f, 0.f, 0.f, 0.f};
    uint32_t cc = column(16 * wave);
    for (int32_t t0 = 16 * wave; t0 < len_last; t0 += 16 * W) {
      Win bq[NB][4];
      const Win y = window(scores, t0);
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const uint32_t cs = (uint32_t)__builtin_amdgcn_ds_bpermute(
            (4 * g + st) << 2, (int)cc);
        if constexpr (IL || !kF32) {
          const uint32_t vo =
              (uint32_t)sizeof(T) * (cs * (uint32_t)dv + 4u * (uint32_t)i);
          bq[0][st] =
              *reinterpret_cast<const Win *>(at_bytes(value + nb0, vo));
          if constexpr (NB == 2) {
            bq[1][st] = Win{};
            if (both)
              bq[1][st] = *reinterpret_cast<const Win *>(
                  at_bytes(value + nb0 + 64, vo));
          }
        } else {
          const uint32_t vo = 4u * (cs * (uint32_t)dv + (uint32_t)i);
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            const int nn = n < ntiles0 ? n : 0; // wave-uniform
            bq[0][st][n] = *at_bytes(value + nb0 + 16 * nn, vo);
          }
        }
      }
      cc = column(t0 + 16 * W);
      __builtin_amdgcn_sched_barrier(0);
      float p[4];
      if (nb0 == 0) { // P from the scores, stored over them
        exps(y, t0, p);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          p[v] = as_stored<T>(tile_div<LIBM>(p[v], sum, rsum_i));
          p[v] = valid(t0, v) ? p[v] : 0.0f;
        }
        store(t0, p);
      } else { // P as the first pass stored it
        entries(y, t0, p);
#pragma unroll
        for (int v = 0; v < 4; ++v)
          p[v] = valid(t0, v) ? p[v] : 0.0f;
      }
      if constexpr (kF32) {
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int st = 0; st < 4; ++st)
            acc[0][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                p[st], bq[0][st][n], acc[0][n], 0, 0, 0);
      } else {
        const v2u pk = v2u{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3])};
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            const v2u bn = v2u{bf16_pair(bq[j][0], bq[j][1], n),
                               bf16_pair(bq[j][2], bq[j][3], n)};
            acc[j][n] = mfma_16x16x16_bf16(pk, bn, acc[j][n]);
          }
      }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int64_t nb = nb0 + 64 * j;
      if (nb >= dv)
        break; // wave-uniform
      const int ntiles = (int)std::min<int64_t>(4, (dv - nb) / 16);
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          part[wave][n][v][l] = acc[j][n][v];
      __syncthreads();
      if (wave < (IL || !kF32 ? 4 : ntiles)) {
        // IL: wave w finishes rows 4g + w, columns nb + 4i .. nb + 4i + 3;
        // else wave n the tile of columns nb + 16n + i, rows 4g + v
        float o[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          o[x] = 0.0f;
#pragma unroll
          for (int w = 0; w < W; ++w)
            o[x] += IL || !kF32 ? part[w][x][wave][l] : part[w][wave][x][l];
        }
        if constexpr (IL || !kF32) {
          const int rr = 4 * g + wave;
          if (rr < nt) {
            T *dst = out + (int64_t)(r0 + rr) * dv + nb + 4 * i;
            if constexpr (kF32)
              *reinterpret_cast<v4f *>(dst) = v4f{o[0], o[1], o[2], o[3]};
            else
              *reinterpret_cast<v2u *>(dst) =
                  v2u{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
#pragma unroll
            for (int x = 0; x < 4; ++x)
              nonfinite |= !__builtin_isfinite(o[x]);
          }
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (4 * g + v < nt) {
              stv(out + (int64_t)(r0 + 4 * g + v) * dv + nb + 16 * wave + i,
                  o[v]);
              nonfinite |= !__builtin_isfinite(o[v]);
            }
        }
        if (__builtin_amdgcn_ballot_w64(nonfinite) != 0 && l == 0)
          v_nonfinite = 1;
      }
      __syncthreads();
    }
  }
  // (the barrier above also made every wave's stored P visible)
  if (v_nonfinite != 0) // workgroup-uniform
    for (int r = r0 + wave; r < r0 + nt; r += W)
      attention_row_output(ro, col, scores, value, out, r, dv);
}

// The attention chain fused over 16-row tiles (d = 64 * KB, dv % 16 == 0):
// scores = alpha * Q K^T + beta * mask on the mask's positions, the row
// softmax (rowMaximum, rowSum and the normalised scores written as the
// separate ops write them), and output = P V, in one kernel.  A tile whose
// rows share the last row's column structure (tile_prefix_ok_block) and
// whose last row holds at most kFusedCols entries keeps its scores in
// registers.  Wave w takes the 16-entry chunks k = 0..3 at entries
// t0(k) = 16 (w + W k) of the last row:
//   A. S^T = K_chunk Q^T with 16 x 16 x 4 MFMAs (the gathered K rows as the
//      A operand, Q as the B operand), so that lane (i, g) holds the scores
//      of row i at entries t0 + 4g .. t0 + 4g + 3, which is the A operand
//      the P V product takes;
//   B. the row maxima, then the row sums, are reduced over the four lanes of
//      a row in each wave and over the waves through LDS (two barriers);
//      every final score, row maximum and row sum is written once;
//   C. output = P V from those registers against the gathered V rows, the
//      waves' partial output tiles summed through LDS.
// The scores thus cross HBM once (written) instead of five times, and the
// chain is one launch.  Other tiles run row by row: each wave computes a row's
// scores, softmax and output in global memory.
//
// The loads are batched so that the chain of dependent memory trips is
// short: (1) the tile's row offsets (one load, spread to the lanes by
// permutes) and its Q rows; (2) the rows' column indices for the structure
// check; (3) the K^T gathers and mask windows of chunks 0-1, then of chunks
// 2-3; the V rows of chunks 0-1 fly over the softmax.  Entries past the last row read the last row's
// final column, so no load is guarded; their scores are never used and
// their P is zero.  A V row that is inf or NaN makes the tile's output
// non-finite wherever it is read (0 * inf); such tiles are recomputed row by
// row from the stored scores, adding exactly each row's own entries.
// Scheduling barriers keep each batch of loads together and in order, so
// that waiting for one batch leaves the later ones in flight.
// The host guarantees that the byte offsets into mask / scores (positions),
// K^T (kdim * cols) and V (cols * dv) fit 32 bits and that nnz >= 4
// (amax = nnz - 4, the last 4-entry window of the mask).
//
// IL (dv % 64 == 0, V and the output 16-byte aligned): the four 16-column
// output tiles of a 64-column block interleave -- tile n's column j is
// output column 4j + n of the block -- so that one 128-bit load of a V row
// gives a lane its values for all four tiles, and one 128-bit store writes
// four outputs of a row.
// SO (SDDMM only): the kernel serves the sddmm op on its own -- mask is the
// op's sample values, q its lhs, kt its rhs, scores its output, and `kind`
// its region; the tile stores its scores and ends (value, rmax, rsum, out
// and dv are unused).  The attention chain takes the affine region.
// NS (with SO; no sample values, mask is null): every sample reads as zero
// and no sample window is loaded.
// FLOOR (the chain only; the tile-floor diagnostic sw_attention_tile_floor):
// the same loads, structure check, barrier, stores and output reduction,
// with every product, exponential and division replaced by an XOR of the
// words the lane loaded and without the softmax's two barriers.  Its time is
// the floor of the tile's chain of memory trips.
// (at most 128 VGPRs: the two workgroups of a CU need four waves per SIMD)
// LIBM: see tile_exp (calls without mapping options).
// LONG: tiles with the shared structure and rows past kFusedCols entries
// take attention_long_tile instead of running row by row.  Its code beside
// the register path makes the allocator spill there (configuration 5 19.2
// -> 20.3 us, d = 128 31.0 -> 33.5 us; the bf16 kernel, which always has it,
// 14.4 -> 14.6 us), so the host takes it for long rows only.
template <int KB, int W, bool IL, bool SO, bool NS = false, bool FLOOR = false,
          bool LIBM = false, bool LONG = false>
__global__ __launch_bounds__(64 * W, 4) void attention_tile_fused(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const float *__restrict__ mask, const float *__restrict__ q,
    const float *__restrict__ kt, const float *__restrict__ value,
    float *scores, float *__restrict__ rmax, float *__restrict__ rsum,
    float *__restrict__ out, int32_t rows, int64_t cols, int32_t kdim,
    int64_t dv, float alpha, float beta, uint32_t amax, int kind) {
  const int region = SO ? kind : SW_SDDMM_AFFINE;
  static_assert(W == 8 && kFusedCols == 8 * kWave && kFusedChunks == 4,
                "check layout");
  static_assert(SO || !NS, "the attention chain reads its mask");
  static_assert(!(SO && FLOOR), "the floor runs the chain");
  __shared__ float part[W][4][4][kWave]; // [wave][n tile][v][lane]
  __shared__ float wred[2][W][16];       // [max, sum][wave][row]
  __shared__ int32_t lcol[kFusedCols];   // the last row's columns
  __shared__ int wshared[W]; // each wave's rows share the last row's columns
  __shared__ int v_nonfinite; // an output of the tile is inf or NaN
  if (block_id() * 16 >= rows)
    return; // a folded grid's surplus workgroup (workgroup-uniform)
  const int r0 = (int)block_id() * 16;
  const int nt = std::min(16, rows - r0);
  const int wave = wave_in_group();
  const int l = lane_id(), i = l & 15, g = l >> 4;
  // 1. lanes 0..nt hold ro[r0 .. r0 + nt]; Q row r0 + i, elements
  //    kb 64 + 16 g + st (the B operand of step st)
  const int32_t my_ro = ro[r0 + (l < nt ? l : nt)];
  float qa[16 * KB];
  const int64_t qrow = (int64_t)std::min(r0 + i, rows - 1) * kdim;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      v4f x;
      __builtin_memcpy(&x, q + qrow + kb * 64 + 16 * g + 4 * u, sizeof x);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        qa[kb * 16 + 4 * u + e] = i < nt ? x[e] : 0.0f;
    }
  __builtin_amdgcn_sched_barrier(0);
  // row i's first position and length (0 past nt); the permutes run on
  // every lane, as a permute reads zero from a lane that is switched off
  const int ic = i < nt ? i : nt - 1;
  const int32_t rbase = __builtin_amdgcn_ds_bpermute(ic << 2, my_ro);
  const int32_t rnext = __builtin_amdgcn_ds_bpermute((ic + 1) << 2, my_ro);
  const int32_t la = i < nt ? rnext - rbase : 0;
  const int32_t bl = __builtin_amdgcn_readlane(my_ro, nt - 1);
  const int32_t len_last = __builtin_amdgcn_readlane(my_ro, nt) - bl;
  // first entry of this wave's chunk k (entries past len_last: no chunk)
  auto chunk_t0 = [&](int k) __attribute__((always_inline)) {
    return 16 * (wave + W * k);
  };
  // entry (k, v) of lane (i, g): row i, entry chunk_t0(k) + 4g + v
  auto valid = [&](int k, int v) __attribute__((always_inline)) {
    return chunk_t0(k) + 4 * g + v < la;
  };
  // row i's mask values at entries t0(k) + 4g .. + 3: the raw window, read
  // from position min(e, amax) for the window's first position e and
  // shifted by e - min(e, amax) where the values are used
  auto window_at = [&](int k) __attribute__((always_inline)) {
    const uint32_t e = rbase + chunk_t0(k) + 4 * g;
    return e < amax ? e : amax;
  };
  if constexpr (LONG) {
    if (len_last > kFusedCols && // workgroup-uniform
        long_tile_prefix_ok<W>(col, my_ro, nt, bl, len_last, amax, wshared)) {
      attention_long_tile<float, KB, W, IL, SO, NS, LIBM>(
          ro, col, mask, q, kt, value, scores, rmax, rsum, out, cols, kdim,
          dv, alpha, beta, amax, region, r0, nt, rbase, la, bl, len_last, qa,
          part, wred, v_nonfinite);
      return;
    }
  }
  // The structure check and the LDS copy of the last row's column indices
  // share one batch of loads: wave w compares rows w and w + W (at most two,
  // nt <= 16 = 2W) against the last row, a row of at most kFusedCols entries
  // being 8 loads per lane, and stores entries [64w, 64w + 64) of the last
  // row to LDS, where both products read their K / V row indices.
  bool ok = len_last <= kFusedCols; // workgroup-uniform
  if (ok) {
    if (threadIdx.x == 0)
      v_nonfinite = 0;
    int32_t x[2][8], yl[8];
    // unconditional loads from clamped, valid positions (nnz > 0): a row's
    // first position as the wave-uniform base (scalar registers) and the
    // clamped entry index as a 32-bit lane offset (4 nnz fits 32 bits)
    auto row_entry = [&](int32_t b, int32_t len, int32_t t)
        __attribute__((always_inline)) {
      const int32_t *rb = col + (len > 0 ? b : 0);
      return *at_bytes(rb, 4u * (uint32_t)std::min(t, std::max(len - 1, 0)));
    };
#pragma unroll
    for (int u = 0; u < 8; ++u)
      yl[u] = row_entry(bl, len_last, l + u * kWave);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int rr = wave + h * W;
      const int rc = rr < nt - 1 ? rr : 0; // rows past nt-2 are not checked
      const int32_t b = __builtin_amdgcn_readlane(my_ro, rc);
      const int32_t len = __builtin_amdgcn_readlane(my_ro, rc + 1) - b;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        x[h][u] = row_entry(b, len, l + u * kWave);
    }
    // without branches: a compare inside a branch would pull its loads
    // into the branch
    bool mine = true;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int rr = wave + h * W;
      const int rc = rr < nt - 1 ? rr : 0;
      const int32_t b = __builtin_amdgcn_readlane(my_ro, rc);
      const int32_t len = __builtin_amdgcn_readlane(my_ro, rc + 1) - b;
      bool same = len <= len_last;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        same &= (l + u * kWave >= len) | (x[h][u] == yl[u]);
      mine &= (rr >= nt - 1) | same;
    }
    // wave w stores the last row's entries 64w .. 64w + 63; those past the
    // row hold its final column (the clamped loads above), so that the
    // gathers read lcol without clamping an index
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (u == wave)
        lcol[l + u * kWave] = yl[u];
    const bool shared_cols = __builtin_amdgcn_ballot_w64(!mine) == 0;
    if (l == 0)
      wshared[wave] = shared_cols;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W; ++w)
      ok &= wshared[w] != 0;
  }
  if (!ok) { // workgroup-uniform
    for (int r = r0 + wave; r < r0 + nt; r += W) {
      sddmm_row_wave(ro, col, mask, q, kt, scores, r, cols, kdim, region,
                     alpha, beta);
      if constexpr (!SO) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        attention_row_softmax(ro, scores, rmax, rsum, r);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        attention_row_output(ro, col, scores, value, out, r, dv);
      }
    }
    return;
  }
  // 3. the gathers; entries past the last row read its final column
  // K_chunk rows (A operand of step kb 16 + st): K^T[kb 64 + 16 g + st][c]
  // for the column c of entry t0 + i -- the lane's byte offset (16 g rows
  // and c columns on) plus the wave-uniform offset of row kb 64 + st, as
  // buffer loads, whose wave-uniform offset costs no vector instruction
  // (configuration 5: 21.2 -> 20.3 us; d = 128: 31.2 -> 28.5 us)
  const __amdgpu_buffer_rsrc_t kt_rsrc =
      buffer_rsrc(kt, 4u * (uint32_t)kdim * (uint32_t)cols);
  auto gather_k = [&](int k, float (&a)[16 * KB])
      __attribute__((always_inline)) {
    const uint32_t cj = lcol[chunk_t0(k) + i];
    const uint32_t ko = 4u * (16u * g * (uint32_t)cols + cj);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int st = 0; st < 16; ++st)
        a[kb * 16 + st] = buffer_load_f32(
            kt_rsrc, ko, 4u * (uint32_t)(kb * 64 + st) * (uint32_t)cols);
  };
  // V rows (B operand of P V, [n tile][st]): for t = t0(k) + 4g + st, lane
  // (j, g) takes V[c_t][nb + 4j + n] (IL) or V[c_t][nb + 16n + j]; tiles
  // n >= ntiles read tile 0 again -- their outputs are never stored, so
  // their values need no select (a select on the wave-uniform n < ntiles
  // would become a branch around each load)
  auto load_v = [&](int k, int64_t nb, float (&bv)[4][4])
      __attribute__((always_inline)) {
    const int ntiles = (int)std::min<int64_t>(4, (dv - nb) / 16);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int32_t t = chunk_t0(k) + 4 * g + st;
      const uint32_t c = lcol[t];
      if constexpr (IL) {
        const uint32_t vo = 4u * (c * (uint32_t)dv + 4u * (uint32_t)i);
        const v4f x = *reinterpret_cast<const v4f *>(at_bytes(value + nb, vo));
#pragma unroll
        for (int n = 0; n < 4; ++n)
          bv[n][st] = x[n];
      } else {
        const uint32_t vo = 4u * (c * (uint32_t)dv + (uint32_t)i);
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const int nn = n < ntiles ? n : 0; // wave-uniform
          bv[n][st] = *at_bytes(value + nb + 16 * nn, vo);
        }
      }
    }
  };
  auto load_window = [&](int k, v4f &w) __attribute__((always_inline)) {
    if constexpr (NS)
      w = v4f{0.f, 0.f, 0.f, 0.f};
    else
      __builtin_memcpy(&w, mask + window_at(k), sizeof(v4f));
  };
  // A. S^T per chunk: sv[k][v] = score (i, t0(k) + 4g + v)
  float sv[kFusedChunks][4];
  auto sddmm_chunk = [&](int k, const float (&a)[16 * KB], const v4f &w)
      __attribute__((always_inline)) {
    if constexpr (FLOOR) {
      uint32_t x = 0;
#pragma unroll
      for (int st = 0; st < 16 * KB; ++st)
        x ^= __float_as_uint(a[st]);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        sv[k][v] = __uint_as_float(x ^ __float_as_uint(w[v]));
      return;
    }
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    if (chunk_t0(k) < len_last) { // wave-uniform
      // two independent chains of products (even and odd K steps): one
      // chain of 16 dependent MFMAs held the wave (18.0 -> 17.6 us; four
      // chains: no faster at d = 64, slower at d = 128)
      v4f acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < 16 * KB; st += 2) {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[st], qa[st], acc, 0, 0,
                                                   0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[st + 1], qa[st + 1],
                                                    acc1, 0, 0, 0);
      }
      acc += acc1;
    }
    const uint32_t d = rbase + chunk_t0(k) + 4 * g - window_at(k);
    const v4f x = {d == 0 ? w.x : d == 1 ? w.y : d == 2 ? w.z : w.w,
                   d == 0 ? w.y : d == 1 ? w.z : w.w, d == 0 ? w.z : w.w, w.w};
#pragma unroll
    for (int v = 0; v < 4; ++v)
      sv[k][v] = combine_sddmm(region, valid(k, v) ? x[v] : 0.0f, acc[v],
                               alpha, beta);
  };
  float bv[kFusedChunks][4][4];
  // two chunks' K^T gathers and mask windows per batch; a chunk past the
  // last row's entries loads nothing (each branch holds its loads and the
  // products that take them, so no branch waits for a load it does not use)
#pragma unroll
  for (int k0 = 0; k0 < kFusedChunks; k0 += 2) {
    if (chunk_t0(k0 + 1) < len_last) { // wave-uniform
      float a[2][16 * KB];
      v4f w[2];
      gather_k(k0, a[0]);
      gather_k(k0 + 1, a[1]);
      load_window(k0, w[0]);
      load_window(k0 + 1, w[1]);
      __builtin_amdgcn_sched_barrier(0);
      sddmm_chunk(k0, a[0], w[0]);
      sddmm_chunk(k0 + 1, a[1], w[1]);
    } else {
      if (chunk_t0(k0) < len_last) {
        float a[16 * KB];
        v4f w;
        gather_k(k0, a);
        load_window(k0, w);
        __builtin_amdgcn_sched_barrier(0);
        sddmm_chunk(k0, a, w);
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          sv[k0][v] = 0.0f;
      }
#pragma unroll
      for (int v = 0; v < 4; ++v)
        sv[k0 + 1][v] = 0.0f;
    }
  }
  if constexpr (SO) {
    // the scores of entries t0(k) + 4g .. + 3 of row i: one (unaligned)
    // vector store when all four are the row's, else the row's ones one by
    // one
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      if (chunk_t0(k) >= len_last) // wave-uniform
        continue;
      float *dst = scores + rbase + chunk_t0(k) + 4 * g;
      if (valid(k, 3)) {
        const v4f x = v4f{sv[k][0], sv[k][1], sv[k][2], sv[k][3]};
        __builtin_memcpy(dst, &x, sizeof x);
      } else {
#pragma unroll
        for (int v = 0; v < 3; ++v)
          if (valid(k, v))
            dst[v] = sv[k][v];
      }
    }
    return;
  }
  // in flight over the softmax (the V rows of chunks 2-3 are loaded after
  // it: holding all four chunks' rows over it would take more registers
  // than four waves per SIMD leave)
  load_v(0, 0, bv[0]);
  load_v(1, 0, bv[1]);
  if constexpr (FLOOR) {
    // the scores' stores and the row outputs' stores, no softmax
    uint32_t x = 0;
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      if (chunk_t0(k) >= len_last) // wave-uniform
        continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        sv[k][v] = valid(k, v) ? sv[k][v] : 0.0f;
        x ^= __float_as_uint(sv[k][v]);
      }
      float *dst = scores + rbase + chunk_t0(k) + 4 * g;
      if (valid(k, 3)) {
        const v4f y = v4f{sv[k][0], sv[k][1], sv[k][2], sv[k][3]};
        __builtin_memcpy(dst, &y, sizeof y);
      } else {
#pragma unroll
        for (int v = 0; v < 3; ++v)
          if (valid(k, v))
            dst[v] = sv[k][v];
      }
    }
    if (wave == 0 && g == 0 && i < nt) {
      rmax[r0 + i] = __uint_as_float(x);
      rsum[r0 + i] = __uint_as_float(x);
    }
  } else {
  // B. row softmax: lanes (i, 0..3) of every wave hold row i's entries
  {
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (valid(k, v))
          m = maximumf(m, sv[k][v]);
    m = maximumf(m, swizzle_xor16(m));
    m = maximumf(m, shfl_xor32(m));
    if (g == 0)
      wred[0][wave][i] = m;
    __syncthreads();
    m = wred[0][0][i];
#pragma unroll
    for (int w = 1; w < W; ++w)
      m = maximumf(m, wred[0][w][i]);
    // per chunk of entries (a chunk past the last row is skipped whole),
    // each entry's value computed unconditionally and selected afterwards:
    // no branch per entry
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      if (chunk_t0(k) < len_last) { // wave-uniform
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float e = tile_exp<LIBM>(sv[k][v] - m);
          sv[k][v] = valid(k, v) ? e : 0.0f;
          sum += sv[k][v];
        }
      }
    }
    sum += swizzle_xor16(sum);
    sum += shfl_xor32(sum);
    if (g == 0)
      wred[1][wave][i] = sum;
    __syncthreads();
    sum = wred[1][0][i];
#pragma unroll
    for (int w = 1; w < W; ++w)
      sum += wred[1][w][i];
    // one correctly rounded reciprocal per row, one multiply per entry
    // (within 1.5 ulp of the quotient)
    const float rsum_i = 1.0f / sum;
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      if (chunk_t0(k) >= len_last) { // wave-uniform
#pragma unroll
        for (int v = 0; v < 4; ++v)
          sv[k][v] = 0.0f;
        continue;
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) { // zero past the row: P V adds nothing
        const float p = tile_div<LIBM>(sv[k][v], sum, rsum_i);
        sv[k][v] = valid(k, v) ? p : 0.0f;
      }
      // entries t0(k) + 4g .. + 3 of row i: one (unaligned) vector store
      // when all four are the row's, else the row's ones one by one
      float *dst = scores + rbase + chunk_t0(k) + 4 * g;
      if (valid(k, 3)) {
        const v4f x = v4f{sv[k][0], sv[k][1], sv[k][2], sv[k][3]};
        __builtin_memcpy(dst, &x, sizeof x);
      } else {
#pragma unroll
        for (int v = 0; v < 3; ++v)
          if (valid(k, v))
            dst[v] = sv[k][v];
      }
    }
    if (wave == 0 && g == 0 && i < nt) {
      rmax[r0 + i] = m;
      rsum[r0 + i] = sum;
    }
  }
  } // FLOOR
  // C. output = P V with P from sv (lane (i, g) holds P[i][t0(k)+4g+st],
  // the A operand of step st); the waves' partial tiles are summed in LDS
  auto mfma_chunk = [&](int k, const float (&b)[4][4], v4f (&acc)[4])
      __attribute__((always_inline)) {
    if constexpr (FLOOR) {
      if (chunk_t0(k) < len_last) // wave-uniform
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int st = 0; st < 4; ++st)
            acc[n][st] = __uint_as_float(__float_as_uint(acc[n][st]) ^
                                         __float_as_uint(sv[k][st]) ^
                                         __float_as_uint(b[n][st]));
      return;
    }
    if (chunk_t0(k) < len_last) // wave-uniform
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int st = 0; st < 4; ++st)
          acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[k][st], b[n][st],
                                                        acc[n], 0, 0, 0);
  };
  // the waves' partial tiles combine by sum (by XOR in the floor)
  auto combine = [&](float a, float b) __attribute__((always_inline)) {
    if constexpr (FLOOR)
      return __uint_as_float(__float_as_uint(a) ^ __float_as_uint(b));
    else
      return a + b;
  };
  bool nonfinite = false;
  for (int64_t nb = 0; nb < dv; nb += 64) {
    const int ntiles = (int)std::min<int64_t>(4, (dv - nb) / 16);
    v4f acc[4];
#pragma unroll
    for (int n = 0; n < 4; ++n)
      acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
    if (nb > 0) {
#pragma unroll
      for (int k = 0; k < kFusedChunks; ++k)
        load_v(k, nb, bv[k]);
    } else {
      load_v(2, 0, bv[2]);
      load_v(3, 0, bv[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k)
      mfma_chunk(k, bv[k], acc);
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        part[wave][n][v][l] = acc[n][v];
    __syncthreads();
    if constexpr (IL) {
      if (wave < 4) {
        // wave w finishes rows 4g + w, columns nb + 4i .. nb + 4i + 3
        v4f o;
        bool nf = false;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          float sum = 0.0f;
#pragma unroll
          for (int w = 0; w < W; ++w)
            sum = combine(sum, part[w][n][wave][l]);
          o[n] = sum;
          nf |= !FLOOR && !__builtin_isfinite(sum);
        }
        const int rr = 4 * g + wave;
        if (rr < nt) {
          *reinterpret_cast<v4f *>(out + (int64_t)(r0 + rr) * dv + nb +
                                   4 * i) = o;
          nonfinite |= nf;
        }
        if (__builtin_amdgcn_ballot_w64(nonfinite) != 0 && l == 0)
          v_nonfinite = 1;
      }
    } else if (wave < ntiles) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w)
          sum = combine(sum, part[w][wave][v][l]);
        const int rr = 4 * g + v;
        if (rr < nt) {
          out[(int64_t)(r0 + rr) * dv + nb + 16 * wave + i] = sum;
          nonfinite |= !FLOOR && !__builtin_isfinite(sum);
        }
      }
      if (__builtin_amdgcn_ballot_w64(nonfinite) != 0 && l == 0)
        v_nonfinite = 1;
    }
    __syncthreads();
  }
  // workgroup-uniform; the barrier above also made every wave's stored
  // scores visible to the others
  if (v_nonfinite != 0)
    for (int r = r0 + wave; r < r0 + nt; r += W)
      attention_row_output(ro, col, scores, value, out, r, dv);
}

// ---- bf16 matrix-core kernels ----------------------------------------------
// The bf16 forms of the SDDMM tile and the fused attention tile: the same
// 16-row tiles, row structure check, fallbacks and outputs as the fp32
// kernels above, with bf16 operands on the matrix cores (fp32 accumulation):
//   Q K^T: v_mfma_f32_16x16x32_bf16, lane group g supplying K elements
//     32 s + 8 g .. 32 s + 8 g + 7 at step s -- one 128-bit load of a Q row
//     and eight 16-bit K^T gathers per lane and step;
//   P V:   v_mfma_f32_16x16x16_bf16 per 16-entry chunk, lane group g
//     supplying entries 4 g .. 4 g + 3 of the chunk, with four output tiles
//     whose columns interleave (tile n's column j is output column
//     4 j + n of the 64-column block), so that one 64-bit load of a V row
//     gives a lane its values for all four tiles.
// Every result is rounded to bf16 where the separate op would store it.

// SDDMM over 16-row tiles, bf16 (kdim = 64 * KB; the host guarantees that
// 2 * kdim * cols and 2 * nnz fit 32 bits and that lhs is 16-byte aligned).
template <int KB, int W>
__global__ __launch_bounds__(64 * W) void sddmm_tile_mfma_bf16(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const uint16_t *__restrict__ val, const uint16_t *__restrict__ lhs,
    const uint16_t *__restrict__ rhs, uint16_t *__restrict__ out,
    int32_t rows, int64_t cols, int32_t kdim, int kind, float alpha,
    float beta) {
  constexpr int S = 2 * KB; // 32-deep K steps
  if (block_id() * 16 >= rows)
    return; // a folded grid's surplus workgroup (workgroup-uniform)
  const int r0 = (int)block_id() * 16;
  const int nt = std::min(16, rows - r0);
  const int wave = wave_in_group();
  const int l = lane_id(), i = l & 15, g = l >> 4;
  int32_t rb[4], rl[4];
  {
    int32_t b[5];
#pragma unroll
    for (int v = 0; v < 5; ++v)
      b[v] = ro[std::min(r0 + 4 * g + v, rows)];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      rb[v] = b[v];
      rl[v] = 4 * g + v < nt ? b[v + 1] - b[v] : 0;
    }
  }
  // A operand: lhs row r0 + i, elements 32 s + 8 g .. + 7
  v4u qa[S];
  const int64_t qrow = (int64_t)std::min(r0 + i, rows - 1) * kdim;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const v4u x = *reinterpret_cast<const v4u *>(lhs + qrow + 32 * s + 8 * g);
    qa[s] = i < nt ? x : v4u{0u, 0u, 0u, 0u};
  }
  __shared__ int verdict;
  if (!tile_prefix_ok_block(ro, col, r0, nt, &verdict)) {
    for (int r = r0 + wave; r < r0 + nt; r += W)
      sddmm_row_wave(ro, col, val, lhs, rhs, out, r, cols, kdim, kind, alpha,
                     beta);
    return;
  }
  const int last = r0 + nt - 1;
  const int32_t bl = ro[last];
  const int32_t len_last = ro[last + 1] - bl;
  const uint32_t row_bytes = 2u * (uint32_t)cols;
  for (int32_t t0 = wave * 16; t0 < len_last; t0 += 32 * W) {
    const int32_t t1 = t0 + 16 * W;
    const bool two = t1 < len_last; // wave-uniform
    const int32_t ta = t0 + i, tb = t1 + i;
    const uint32_t cj0 = ta < len_last ? (uint32_t)col[bl + ta] : 0u;
    const uint32_t cj1 = two && tb < len_last ? (uint32_t)col[bl + tb] : 0u;
    float s0[4], s1[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const bool in0 = val != nullptr && ta < rl[v];
      const bool in1 = val != nullptr && two && tb < rl[v];
      const float x0 = val != nullptr ? ldv(val + (in0 ? rb[v] + ta : bl)) : 0.f;
      const float x1 = val != nullptr ? ldv(val + (in1 ? rb[v] + tb : bl)) : 0.f;
      s0[v] = in0 ? x0 : 0.0f;
      s1[v] = in1 ? x1 : 0.0f;
    }
    const uint32_t lo0 = 2u * cj0 + 8u * g * row_bytes;
    const uint32_t lo1 = 2u * cj1 + 8u * g * row_bytes;
    v4f acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    v4u b0[S], b1[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const uint16_t *base = rhs + (int64_t)(32 * s) * cols;
      b0[s] = gather_kt8(base, row_bytes, lo0);
      b1[s] = gather_kt8(base, row_bytes, lo1); // column 0 when !two
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      acc0 = mfma_16x16x32_bf16(qa[s], b0[s], acc0);
      if (two)
        acc1 = mfma_16x16x32_bf16(qa[s], b1[s], acc1);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (ta < rl[v])
        stv(out + rb[v] + ta,
            combine_sddmm(kind, s0[v], acc0[v], alpha, beta));
      if (two && tb < rl[v])
        stv(out + rb[v] + tb,
            combine_sddmm(kind, s1[v], acc1[v], alpha, beta));
    }
  }
}

// The attention chain fused over 16-row tiles, bf16 (d = 64 * KB,
// dv % 64 == 0): the fp32 attention_tile_fused's tiles, waves, chunks,
// structure check and fallbacks, with the products on bf16 matrix cores.
// Its loads are batched so that the chain of dependent memory trips is short:
//   1. the tile's row offsets (one load, spread to the lanes by permutes) and
//      its Q rows;
//   2. the rows' column indices for the structure check, with every chunk's
//      mask window in flight over the check;
//   3. the K^T gathers of chunks 0-1, then of chunks 2-3 (none for chunks
//      past the last row); the V rows of chunks 0-1 fly over the second
//      batch (d = 64) or the softmax, those of chunks 2-3 over the softmax
//      (d = 64) or are loaded after it.
// The products do not wait for the structure check: its verdict is read at
// the softmax's first barrier, before anything is stored.  Entries past the
// last row read the last row's final column, so no load is guarded; their
// scores are never used and their P is zero.  A V row that is inf or NaN
// makes the tile's output non-finite wherever it is read (0 * inf), and such
// tiles are recomputed row by row, as in the fp32 kernel.
// The host guarantees that the byte offsets into mask / scores (2 * nnz),
// K^T (2 * d * cols) and V (2 * cols * dv) fit 32 bits, that nnz >= 4
// (amax = nnz - 4) and that Q is 16-byte and V 8-byte aligned.
// (at most 128 VGPRs: the two workgroups of a CU need four waves per SIMD)
// FLOOR: the tile-floor diagnostic, as for the fp32 kernel above.
// LIBM: see tile_exp (calls without mapping options).
template <int KB, int W, bool SO, bool NS = false, bool FLOOR = false,
          bool LIBM = false>
__global__ __launch_bounds__(64 * W, 4) void attention_tile_fused_bf16(
    const int32_t *__restrict__ ro, const int32_t *__restrict__ col,
    const uint16_t *__restrict__ mask, const uint16_t *__restrict__ q,
    const uint16_t *__restrict__ kt, const uint16_t *__restrict__ value,
    uint16_t *scores, uint16_t *__restrict__ rmax, uint16_t *__restrict__ rsum,
    uint16_t *__restrict__ out, int32_t rows, int64_t cols, int32_t kdim,
    int64_t dv, float alpha, float beta, uint32_t amax, int kind) {
  static_assert(W == 8 && kFusedCols == 8 * kWave && kFusedChunks == 4,
                "check layout");
  constexpr int S = 2 * KB;
  // SO: the SDDMM alone (combine kind `kind`), its scores stored from
  // registers; no softmax and no P V.  NS (with SO): no sample values (mask
  // is null), every sample reads as zero
  const int region = SO ? kind : SW_SDDMM_AFFINE;
  static_assert(SO || !NS, "the attention chain reads its mask");
  static_assert(!(SO && FLOOR), "the floor runs the chain");
  __shared__ float part[W][4][4][kWave]; // [wave][n tile][v][lane]
  __shared__ float wred[2][W][16];       // [max, sum][wave][row]
  __shared__ int wshared[W]; // each wave's rows share the last row's columns
  __shared__ int v_nonfinite;
  if (block_id() * 16 >= rows)
    return; // a folded grid's surplus workgroup (workgroup-uniform)
  const int r0 = (int)block_id() * 16;
  const int nt = std::min(16, rows - r0);
  const int wave = wave_in_group();
  const int l = lane_id(), i = l & 15, g = l >> 4;
  // 1. lanes 0..nt hold ro[r0 .. r0 + nt]; Q row r0 + i, elements
  //    32 s + 8 g .. + 7 (the B operand of S^T = K_chunk Q^T)
  const int32_t my_ro = ro[r0 + (l < nt ? l : nt)];
  v4u qb[S];
  const int64_t qrow = (int64_t)std::min(r0 + i, rows - 1) * kdim;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const v4u x = *reinterpret_cast<const v4u *>(q + qrow + 32 * s + 8 * g);
    qb[s] = i < nt ? x : v4u{0u, 0u, 0u, 0u};
  }
  // (scheduling barriers keep each batch of loads together and in order,
  // so that waiting for one batch leaves the later ones in flight)
  __builtin_amdgcn_sched_barrier(0);
  // row i's first position and length (0 past nt); the permutes run on
  // every lane, as a permute reads zero from a lane that is switched off
  const int ic = i < nt ? i : nt - 1;
  const int32_t rbase = __builtin_amdgcn_ds_bpermute(ic << 2, my_ro);
  const int32_t rnext = __builtin_amdgcn_ds_bpermute((ic + 1) << 2, my_ro);
  const int32_t la = i < nt ? rnext - rbase : 0;
  const int32_t bl = __builtin_amdgcn_readlane(my_ro, nt - 1);
  const int32_t len_last = __builtin_amdgcn_readlane(my_ro, nt) - bl;
  auto chunk_t0 = [&](int k) __attribute__((always_inline)) {
    return 16 * (wave + W * k);
  };
  auto valid = [&](int k, int v) __attribute__((always_inline)) {
    return chunk_t0(k) + 4 * g + v < la;
  };
  // 2. row i's mask values at entries t0(k) + 4g .. + 3: the raw 8-byte
  //    window, read from position min(e, amax) for the window's first
  //    position e and shifted by e - min(e, amax) where the values are used
  auto window_at = [&](int k) __attribute__((always_inline)) {
    const uint32_t e = rbase + chunk_t0(k) + 4 * g;
    return e < amax ? e : amax;
  };
  uint64_t mw[kFusedChunks];
  if constexpr (!FLOOR) {
    if (len_last > kFusedCols && // workgroup-uniform
        long_tile_prefix_ok<W>(col, my_ro, nt, bl, len_last, amax, wshared)) {
      attention_long_tile<uint16_t, KB, W, true, SO, NS, LIBM>(
          ro, col, mask, q, kt, value, scores, rmax, rsum, out, cols, kdim,
          dv, alpha, beta, amax, region, r0, nt, rbase, la, bl, len_last, qb,
          part, wred, v_nonfinite);
      return;
    }
  }
  // The structure check and the products run together: each wave checks its
  // rows against the last row and computes its chunks with the last row's
  // columns right away; the verdict is read at the softmax's first barrier,
  // before anything is stored, and a tile that fails it is redone row by
  // row.  The last row's column indices stay in registers: lane j of yl[u]
  // holds entry 64u + j (clamped to the last entry), and a lane takes the
  // column of an entry from there with a permute.
  bool ok = len_last <= kFusedCols; // workgroup-uniform
  if (threadIdx.x == 0)
    v_nonfinite = 0;
  // yk[k]: the yl register holding chunk k's entries 16 (w + 8k) .. + 15,
  // in lanes 16 (w & 3) .. + 15
  int32_t yk[kFusedChunks];
  auto col_of = [&](int k, int off) __attribute__((always_inline)) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute(
        (16 * (wave & 3) + off) << 2, yk[k]);
  };
  // K_chunk rows (A operand): K^T[32 s + 8 g .. + 7][column of entry t0 + i]
  const uint32_t row_bytes = 2u * (uint32_t)cols;
  auto gather_k = [&](int k, v4u (&a)[S]) __attribute__((always_inline)) {
    const uint32_t ko = 2u * col_of(k, i) + 8u * g * row_bytes;
#pragma unroll
    for (int s = 0; s < S; ++s)
      a[s] = gather_kt8(kt + (int64_t)(32 * s) * cols, row_bytes, ko);
  };
  // V rows (B operand of P V): lane (j, g) takes V[c_t][nb + 4j .. + 3] for
  // t = t0(k) + 4g + st, tile n taking element n
  auto load_v = [&](int k, int64_t nb, v2u (&bv)[4])
      __attribute__((always_inline)) {
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const uint32_t c = col_of(k, 4 * g + st);
      const uint32_t vo = 2u * (c * (uint32_t)dv + 4u * (uint32_t)i);
      bv[st] = *reinterpret_cast<const v2u *>(at_bytes(value + nb, vo));
    }
  };
  // A. S^T per chunk: sv[k][v] = score (i, t0(k) + 4g + v), rounded to bf16
  float sv[kFusedChunks][4];
  auto sddmm_chunk = [&](int k, const v4u (&a)[S])
      __attribute__((always_inline)) {
    if constexpr (FLOOR) {
      uint32_t x = (uint32_t)mw[k] ^ (uint32_t)(mw[k] >> 32);
#pragma unroll
      for (int s2 = 0; s2 < S; ++s2)
        x ^= a[s2].x ^ a[s2].y ^ a[s2].z ^ a[s2].w;
#pragma unroll
      for (int v = 0; v < 4; ++v)
        sv[k][v] = __uint_as_float(x ^ (uint32_t)v);
      return;
    }
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    if (chunk_t0(k) < len_last) { // wave-uniform
#pragma unroll
      for (int s = 0; s < S; ++s)
        acc = mfma_16x16x32_bf16(a[s], qb[s], acc);
    }
    const uint32_t d = rbase + chunk_t0(k) + 4 * g - window_at(k);
    const uint64_t w = d < 4 ? mw[k] >> (16 * d) : 0ull;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float x = valid(k, v) ? bf16_to_f32((uint16_t)(w >> (16 * v)))
                                  : 0.0f;
      sv[k][v] = as_stored<uint16_t>(
          combine_sddmm(region, x, acc[v], alpha, beta));
    }
  };
  // two chunks' K^T gathers per batch; a chunk past the last row's entries
  // loads nothing (each branch holds its loads and the products that take
  // them, so no branch waits for a load it does not use)
  auto batch = [&](int k0) __attribute__((always_inline)) {
    if (chunk_t0(k0 + 1) < len_last) { // wave-uniform
      v4u a[2][S];
      gather_k(k0, a[0]);
      gather_k(k0 + 1, a[1]);
      __builtin_amdgcn_sched_barrier(0);
      sddmm_chunk(k0, a[0]);
      sddmm_chunk(k0 + 1, a[1]);
    } else {
      if (chunk_t0(k0) < len_last) {
        v4u a[S];
        gather_k(k0, a);
        __builtin_amdgcn_sched_barrier(0);
        sddmm_chunk(k0, a);
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          sv[k0][v] = 0.0f;
      }
#pragma unroll
      for (int v = 0; v < 4; ++v)
        sv[k0 + 1][v] = 0.0f;
    }
  };
  v2u bv[kFusedChunks][4];
  v2u pk[kFusedChunks]; // P as bf16 pairs: entries 4g, 4g + 1 | 4g + 2, 4g + 3
  if (ok) {
    int32_t x[2][8], yl[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int32_t t = l + u * kWave;
      yl[u] = col[len_last > 0 ? bl + std::min(t, len_last - 1) : 0];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int rr = wave + h * W;
      const int rc = rr < nt - 1 ? rr : 0;
      const int32_t b = __builtin_amdgcn_readlane(my_ro, rc);
      const int32_t len = __builtin_amdgcn_readlane(my_ro, rc + 1) - b;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int32_t t = l + u * kWave;
        x[h][u] = col[len > 0 ? b + std::min(t, len - 1) : 0];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      if constexpr (NS)
        mw[k] = 0;
      else
        __builtin_memcpy(&mw[k], mask + window_at(k), sizeof(uint64_t));
    }
    __builtin_amdgcn_sched_barrier(0);
    // without branches: a compare inside a branch would pull its loads
    // into the branch, behind the mask windows
    bool mine = true;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int rr = wave + h * W;
      const int rc = rr < nt - 1 ? rr : 0;
      const int32_t b = __builtin_amdgcn_readlane(my_ro, rc);
      const int32_t len = __builtin_amdgcn_readlane(my_ro, rc + 1) - b;
      bool same = len <= len_last;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        same &= (l + u * kWave >= len) | (x[h][u] == yl[u]);
      mine &= (rr >= nt - 1) | same;
    }
    const bool shared_cols = __builtin_amdgcn_ballot_w64(!mine) == 0;
    if (l == 0)
      wshared[wave] = shared_cols;
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k)
      yk[k] = wave >= 4 ? yl[2 * k + 1] : yl[2 * k];
    batch(0);
    if constexpr (KB == 1 && !SO) { // in flight over the second batch and softmax
      load_v(0, 0, bv[0]);
      load_v(1, 0, bv[1]);
    }
    batch(2);
    if constexpr (SO) {
    } else if constexpr (KB == 1) { // in flight over the softmax
      load_v(2, 0, bv[2]);
      load_v(3, 0, bv[3]);
    } else {
      load_v(0, 0, bv[0]);
      load_v(1, 0, bv[1]);
    }
    if constexpr (!SO && !FLOOR) {
      // B. row softmax on the stored (bf16) scores, each op's result
      // rounded: this wave's row maxima
      float m = -INFINITY;
#pragma unroll
      for (int k = 0; k < kFusedChunks; ++k)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (valid(k, v))
            m = maximumf(m, sv[k][v]);
      m = maximumf(m, swizzle_xor16(m));
      m = maximumf(m, shfl_xor32(m));
      if (g == 0)
        wred[0][wave][i] = m;
    }
  }
  __syncthreads();
  if (ok) {
#pragma unroll
    for (int w = 0; w < W; ++w)
      ok &= wshared[w] != 0;
  }
  if (!ok) { // workgroup-uniform; nothing has been stored yet
    for (int r = r0 + wave; r < r0 + nt; r += W) {
      sddmm_row_wave(ro, col, mask, q, kt, scores, r, cols, kdim, region,
                     alpha, beta);
      if constexpr (!SO) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        attention_row_softmax(ro, scores, rmax, rsum, r);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        attention_row_output(ro, col, scores, value, out, r, dv);
      }
    }
    return;
  }
  if constexpr (SO) {
    // the scores, already rounded to bf16, as pairs
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      if (chunk_t0(k) < len_last) { // wave-uniform
        const v2u pr = v2u{pack_bf16x2(sv[k][0], sv[k][1]),
                           pack_bf16x2(sv[k][2], sv[k][3])};
        uint16_t *dst = scores + rbase + chunk_t0(k) + 4 * g;
        if (valid(k, 3)) {
          __builtin_memcpy(dst, &pr, sizeof pr);
        } else {
#pragma unroll
          for (int v = 0; v < 3; ++v)
            if (valid(k, v))
              dst[v] = (uint16_t)(pr[v >> 1] >> (16 * (v & 1)));
        }
      }
    }
    return;
  }
  if constexpr (FLOOR) {
    // the scores' stores and the row outputs' stores, no softmax
    uint32_t x = 0;
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      pk[k] = v2u{valid(k, 0) ? __float_as_uint(sv[k][0]) : 0u,
                  valid(k, 2) ? __float_as_uint(sv[k][2]) : 0u};
      x ^= pk[k].x ^ pk[k].y;
      uint16_t *dst = scores + rbase + chunk_t0(k) + 4 * g;
      if (valid(k, 3)) {
        __builtin_memcpy(dst, &pk[k], sizeof pk[k]);
      } else {
#pragma unroll
        for (int v = 0; v < 3; ++v)
          if (valid(k, v))
            dst[v] = (uint16_t)(pk[k][v >> 1] >> (16 * (v & 1)));
      }
    }
    if (wave == 0 && g == 0 && i < nt) {
      rmax[r0 + i] = (uint16_t)x;
      rsum[r0 + i] = (uint16_t)(x >> 16);
    }
  } else {
    float m = wred[0][0][i];
#pragma unroll
    for (int w = 1; w < W; ++w)
      m = maximumf(m, wred[0][w][i]);
    // per chunk of entries (a chunk past the last row is skipped whole),
    // each entry's value computed unconditionally and selected afterwards:
    // no branch per entry (adding the zeros leaves the sum's bits as they are)
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      if (chunk_t0(k) < len_last) { // wave-uniform
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float e = as_stored<uint16_t>(tile_exp<LIBM>(sv[k][v] - m));
          sv[k][v] = valid(k, v) ? e : 0.0f;
          sum += sv[k][v];
        }
      }
    }
    sum += swizzle_xor16(sum);
    sum += shfl_xor32(sum);
    if (g == 0)
      wred[1][wave][i] = sum;
    __syncthreads();
    sum = wred[1][0][i];
#pragma unroll
    for (int w = 1; w < W; ++w)
      sum += wred[1][w][i];
    sum = as_stored<uint16_t>(sum);
    // one correctly rounded reciprocal per row, one multiply per entry
    // (within 1.5 ulp of the quotient before the bf16 rounding)
    const float rsum_i = 1.0f / sum;
    // P rounded to bf16 once, as pairs: the stored scores and the A operand
    // of P V are the same bits
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k) {
      float p[4];
#pragma unroll
      for (int v = 0; v < 4; ++v)
        p[v] = valid(k, v) ? tile_div<LIBM>(sv[k][v], sum, rsum_i) : 0.0f;
      pk[k] = v2u{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3])};
      uint16_t *dst = scores + rbase + chunk_t0(k) + 4 * g;
      if (valid(k, 3)) {
        __builtin_memcpy(dst, &pk[k], sizeof pk[k]);
      } else {
#pragma unroll
        for (int v = 0; v < 3; ++v)
          if (valid(k, v))
            dst[v] = (uint16_t)(pk[k][v >> 1] >> (16 * (v & 1)));
      }
    }
    if (wave == 0 && g == 0 && i < nt) {
      stv(rmax + r0 + i, m);
      stv(rsum + r0 + i, sum);
    }
  }
  // C. output = P V: P from pk (lane (i, g) holds P[i][t0(k) + 4g + st])
  auto mfma_chunk = [&](int k, const v2u (&b)[4], v4f (&acc)[4])
      __attribute__((always_inline)) {
    if constexpr (FLOOR) {
      if (chunk_t0(k) < len_last) // wave-uniform
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int st = 0; st < 4; ++st)
            acc[n][st] = __uint_as_float(__float_as_uint(acc[n][st]) ^
                                         pk[k][st >> 1] ^ b[n][st & 1]);
      return;
    }
    if (chunk_t0(k) < len_last) { // wave-uniform
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const v2u bn = v2u{bf16_pair(b[0], b[1], n), bf16_pair(b[2], b[3], n)};
        acc[n] = mfma_16x16x16_bf16(pk[k], bn, acc[n]);
      }
    }
  };
  bool nonfinite = false;
  for (int64_t nb = 0; nb < dv; nb += 64) {
    v4f acc[4];
#pragma unroll
    for (int n = 0; n < 4; ++n)
      acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
    if (nb > 0) {
#pragma unroll
      for (int k = 0; k < kFusedChunks; ++k)
        load_v(k, nb, bv[k]);
    } else if constexpr (KB != 1) {
      load_v(2, 0, bv[2]);
      load_v(3, 0, bv[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kFusedChunks; ++k)
      mfma_chunk(k, bv[k], acc);
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        part[wave][n][v][l] = acc[n][v];
    __syncthreads();
    if (wave < 4) {
      // wave w finishes rows 4g + w, columns nb + 4i .. nb + 4i + 3
      float o[4];
      bool nf = false;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
          if constexpr (FLOOR) // the waves' partial words combine by XOR
            sum = __uint_as_float(__float_as_uint(sum) ^
                                  __float_as_uint(part[w][n][wave][l]));
          else
            sum += part[w][n][wave][l];
        }
        o[n] = sum;
        nf |= !FLOOR && !__builtin_isfinite(sum);
      }
      const int rr = 4 * g + wave;
      if (rr < nt) {
        *reinterpret_cast<v2u *>(out + (int64_t)(r0 + rr) * dv + nb + 4 * i) =
            FLOOR ? v2u{__float_as_uint(o[0]) ^ __float_as_uint(o[1]),
                        __float_as_uint(o[2]) ^ __float_as_uint(o[3])}
                  : v2u{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
        nonfinite |= nf;
      }
      if (__builtin_amdgcn_ballot_w64(nonfinite) != 0 && l == 0)
        v_nonfinite = 1;
    }
    __syncthreads();
  }
  if (v_nonfinite != 0)
    for (int r = r0 + wave; r < r0 + nt; r += W)
      attention_row_output(ro, col, scores, value, out, r, dv);
}

int grid_for(int64_t work, int64_t per_block, const char *what,
             int64_t *grid) {
  *grid = std::max<int64_t>(sw::ceil_div(work, per_block), 1);
  // (every kernel launched with it has at most 1024 work-items a workgroup)
  return sw::check_grid(*grid, 1024, what);
}

} // namespace

namespace sw {

// Whether rows past kFusedCols entries are to be expected: more than 400
// entries in the mean row.  Block masks whose rows hold up to 512 stay below
// it (configuration 5: rows of up to 384, 345 in the mean), a causal mask of
// 850 positions is past it.
bool long_rows(int64_t rows, int64_t nnz) { return nnz / 400 > rows; }

// Rows of more than 96 entries in the mean are taken for a block mask's,
// which the 16-row matrix-core tiles share their columns on; those of a
// graph are shorter.  (Tiles without shared columns run row by row, one wave
// each: 4,096 rows of 100 random columns, kdim = 64, 46 us, one thread per
// row 645.)
bool block_rows(int64_t rows, int64_t nnz) { return nnz / 96 >= rows; }

// One wave per row was asked for.  (With scratch memory the rhs is transposed
// all the same: 44.5 us against 643 for the graph below.)
bool asks_wave(const sw_options &o) {
  return streq(o.sddmm_mapping, "wave-per-row") ||
         (o.sddmm_lanes_per_row == 64 &&
          !streq(o.sddmm_mapping, "row-tile-mfma"));
}

// The 16-row tiles of the fused attention kernel's product phase serve this
// call: asked for, or rows long enough and no wave per row asked for (rows
// that share no columns gain nothing from a tile: 100 rows of 1,000 random
// columns of 2,000, kdim = 64, 41 us one wave per row, 124 in tiles).  (kdim 256 and bf16's or fp32's other
// tile kernels are chosen in launch_sddmm.)
bool sddmm_tiles(int64_t rows, int64_t nnz, int64_t kdim,
                 const sw_options &o) {
  return streq(o.sddmm_mapping, "row-tile-mfma") ||
         ((kdim == 64 || kdim == 128) && block_rows(rows, nnz) &&
          !asks_wave(o));
}

// Below this many multiply-adds a call is bound by its launches.
bool few_products(int64_t nnz, int64_t kdim) { return nnz < 8000000 / kdim; }

// Few products in few rows: one wave per row without preparation (us, fp32;
// thread per row / wave / transposed: 10,000 rows of 8, kdim = 16 29.7 / 10.5 /
// 14.1; 30,000 of 8, kdim = 4 11.1 / 9.1 / 14.1; 60,000 of 8, kdim = 16 56 /
// 48 / 19.5).  A wave per row costs with the rows, whatever they hold, a
// thread per row with the longest row, and from kdim = 16 on with the lines
// of rhs that its lanes gather at once: 1,000,000 rows of one, kdim = 4 88 /
// 302 / 28; 60,000 of 3, kdim = 8 13 / 23 / 14; 100,000 of one, kdim = 16 86 /
// 78, bf16 92 / 59; 400,000 of 0.2, kdim = 16 55 / 102, of 0.01, kdim = 64 (in
// 1,000,000 rows) 210 / 111.
bool small_sddmm(int64_t rows, int64_t nnz, int64_t kdim) {
  return few_products(nnz, kdim) &&
         (rows <= 16384 || (rows <= 32768 && nnz / 8 >= rows) ||
          (kdim >= 16 &&
           (rows <= 65536 || nnz >= rows || nnz < rows / 64)));
}

// Bytes of scratch memory with which launch_sddmm transposes rhs first (0:
// it would not).  A transposition reads and writes rhs once, a gathered
// column costs a line per element: worth it from one entry per four columns
// on, and not for block masks, whose gathers share their lines (8,192 rows of
// 345 entries, kdim = 96: 71 us one wave per row, 94 transposed).  Few
// products are worth it from 500,000 elements of lhs on (30,000 rows of 3,
// kdim = 32 52 us one wave per row, 15.3 transposed; 30,000 of 8, kdim = 4 9.1
// and 14.1), except the single product of kdim = 1 (1,000,000 rows of 3 41 us
// one thread per row, 53 transposed) and below 200,000 products (100,000 rows
// of 0.2, kdim = 8 9 and 15, kdim = 16 20 and 15; the allocation and the second
// launch alone take the host 5).  At most 1 GiB.
int64_t sddmm_workspace(int64_t rows, int64_t cols, int64_t nnz, int64_t kdim,
                        int64_t elem, const sw_options &o) {
  if (rows <= 0 || cols <= 0 || kdim <= 0 || kdim > INT32_MAX / 2 ||
      (few_products(nnz, kdim) &&
       (kdim == 1 || rows < 500000 / kdim || nnz < 200000 / kdim)) ||
      nnz < cols / 4 || block_rows(rows, nnz) ||
      (streq(o.sddmm_mapping, "row-tile-mfma") &&
       (kdim == 64 || kdim == 128 || kdim == 256)))
    return 0;
  const int64_t kp = ceil_div(kdim, 16 / elem) * (16 / elem);
  if (cols > ((int64_t)1 << 30) / (kp * elem))
    return 0;
  return cols * kp * elem;
}

template <typename T>
int launch_sddmm_transposed(const int32_t *ro, const int32_t *col,
                            const T *val, const T *lhs, const T *rhs, T *out,
                            int64_t rows, int64_t cols, int64_t nnz,
                            int64_t kdim, int kind, float alpha, float beta,
                            T *rhst, hipStream_t st) {
  constexpr int64_t V = 16 / sizeof(T);
  const int64_t kp = ceil_div(kdim, V) * V;
  const int64_t col_tiles = ceil_div(cols, 64);
  const int64_t tiles = col_tiles * ceil_div(kp, 64);
  int rc = check_grid(tiles, 256, "SDDMM rhs transposition");
  if (rc)
    return rc;
  hipLaunchKernelGGL(transpose_rhs<T>, grid_dim(tiles, 256), dim3(256), 0, st,
                     rhs, rhst, cols, (int32_t)kdim, (int32_t)kp, col_tiles);
  rc = launch_check("SDDMM rhs transposition kernel");
  if (rc)
    return rc;
  const int64_t grid = ceil_div(nnz, 256);
  rc = check_grid(grid, 256, "SDDMM");
  if (rc)
    return rc;
  // lanes per entry: one 16-byte step of the dot product, at most 16 lanes
  const int64_t steps = kp / V;
#define SW_POS(G)                                                             \
  hipLaunchKernelGGL((sddmm_positions<T, G>), grid_dim(grid, 256), dim3(256), \
                     0, st, ro, col, val, lhs, rhst, out, (int32_t)rows,      \
                     (int32_t)nnz, (int32_t)kdim, (int32_t)kp, kind, alpha,   \
                     beta)
  if (steps <= 2)
    SW_POS(2);
  else if (steps <= 4)
    SW_POS(4);
  else if (steps <= 8)
    SW_POS(8);
  else
    SW_POS(16);
#undef SW_POS
  return launch_check("SDDMM kernel");
}

// (ws: at least sddmm_workspace bytes, 16-byte aligned, or null)
template <typename T>
int launch_sddmm(const int32_t *ro, const int32_t *col, const T *val,
                 const T *lhs, const T *rhs, T *out, int64_t rows,
                 int64_t cols, int64_t nnz, int64_t kdim, int kind,
                 float alpha, float beta, const sw_options &o,
                 hipStream_t st, T *ws = nullptr) {
  int64_t grid;
  if (ws != nullptr)
    return launch_sddmm_transposed<T>(ro, col, val, lhs, rhs, out, rows, cols,
                                      nnz, kdim, kind, alpha, beta, ws, st);
  const bool apart = val == nullptr || out + nnz <= val || val + nnz <= out;
  if (streq(o.sddmm_mapping, "row-tile-mfma")
          ? kdim == 64 || kdim == 128 || kdim == 256
          : sddmm_tiles(rows, nnz, kdim, o) && apart && nnz >= 4 &&
                narrow_offsets(nnz, 1) && narrow_offsets(cols, kdim) &&
                (sizeof(T) == 4 || aligned16(lhs))) {
    const int kb = (int)(kdim / 64);
    if constexpr (sizeof(T) == 4) {
      int rc = grid_for(rows, 16, "SDDMM", &grid);
      if (rc)
        return rc;
      // d of 64 or 128 with 32-bit offsets, and no sample values or an
      // output apart from them: the fused attention kernel's product phase
      // (its 4-entry sample windows may reach a neighbouring tile's entries)
      if ((kdim == 64 || kdim == 128) && nnz >= 4 &&
          narrow_offsets(nnz, 1) && narrow_offsets(cols, kdim) && apart) {
        const bool lng = long_rows(rows, nnz);
#define SW_SDDMM_FUSED(KB, NS)                                                \
  do {                                                                        \
    if (lng)                                                                  \
      SW_SDDMM_FUSED_AS(KB, NS, true);                                        \
    else                                                                      \
      SW_SDDMM_FUSED_AS(KB, NS, false);                                       \
  } while (0)
#define SW_SDDMM_FUSED_AS(KB, NS, LONG)                                       \
  hipLaunchKernelGGL((attention_tile_fused<KB, kFusedWaves, false, true, NS,  \
                                           false, false, LONG>),              \
                     sw::grid_dim(grid, 64 * kFusedWaves), dim3(64 * kFusedWaves), 0, st, ro, \
                     col, val, lhs, rhs, nullptr, out, nullptr, nullptr,      \
                     nullptr, (int32_t)rows, cols, (int32_t)kdim, (int64_t)0, \
                     alpha, beta, (uint32_t)(nnz - 4), kind)
        if (kb == 1 && val != nullptr)
          SW_SDDMM_FUSED(1, false);
        else if (kb == 1)
          SW_SDDMM_FUSED(1, true);
        else if (val != nullptr)
          SW_SDDMM_FUSED(2, false);
        else
          SW_SDDMM_FUSED(2, true);
#undef SW_SDDMM_FUSED_AS
#undef SW_SDDMM_FUSED
        return launch_check("SDDMM tile MFMA kernel");
      }
#define SW_SDDMM_TILE(KB)                                                     \
  hipLaunchKernelGGL((sddmm_tile_mfma<KB, kSddmmTileWaves>),                  \
                     sw::grid_dim(grid, 64 * kSddmmTileWaves), dim3(64 * kSddmmTileWaves), 0, st, \
                     ro, col, val, lhs, rhs, out, (int32_t)rows, cols,        \
                     (int32_t)kdim, kind, alpha, beta)
      if (kb == 1)
        SW_SDDMM_TILE(1);
      else if (kb == 2)
        SW_SDDMM_TILE(2);
      else
        SW_SDDMM_TILE(4);
#undef SW_SDDMM_TILE
      return launch_check("SDDMM tile MFMA kernel");
    } else if (aligned16(lhs) && narrow_offsets(kdim, cols) &&
               narrow_offsets(nnz, 1)) {
      // bf16 tiles: a 128-bit lhs load per K step, K^T gathered with 32-bit
      // lane byte offsets
      int rc = grid_for(rows, 16, "SDDMM", &grid);
      if (rc)
        return rc;
      // d of 64 or 128, and no sample values or an output apart from them:
      // the fused attention kernel's product phase, as for fp32
      if ((kdim == 64 || kdim == 128) && nnz >= 4 && apart) {
#define SW_SDDMM_FUSED(KB, NS)                                                \
  hipLaunchKernelGGL((attention_tile_fused_bf16<KB, kFusedWaves, true, NS>),  \
                     sw::grid_dim(grid, 64 * kFusedWaves), dim3(64 * kFusedWaves), 0, st, ro, \
                     col, val, lhs, rhs, nullptr, out, nullptr, nullptr,      \
                     nullptr, (int32_t)rows, cols, (int32_t)kdim, (int64_t)0, \
                     alpha, beta, (uint32_t)(nnz - 4), kind)
        if (kb == 1 && val != nullptr)
          SW_SDDMM_FUSED(1, false);
        else if (kb == 1)
          SW_SDDMM_FUSED(1, true);
        else if (val != nullptr)
          SW_SDDMM_FUSED(2, false);
        else
          SW_SDDMM_FUSED(2, true);
#undef SW_SDDMM_FUSED
        return launch_check("SDDMM tile MFMA kernel");
      }
#define SW_SDDMM_TILE(KB)                                                     \
  hipLaunchKernelGGL((sddmm_tile_mfma_bf16<KB, kSddmmTileWaves>),             \
                     sw::grid_dim(grid, 64 * kSddmmTileWaves), dim3(64 * kSddmmTileWaves), 0, st, \
                     ro, col, val, lhs, rhs, out, (int32_t)rows, cols,        \
                     (int32_t)kdim, kind, alpha, beta)
      if (kb == 1)
        SW_SDDMM_TILE(1);
      else if (kb == 2)
        SW_SDDMM_TILE(2);
      else
        SW_SDDMM_TILE(4);
#undef SW_SDDMM_TILE
      return launch_check("SDDMM tile MFMA kernel");
    }
  }
  // (thread-per-row: many short rows without scratch memory; rows of a
  // block mask past its kernels' kdim, 8,192 of 345 entries, kdim = 96, take
  // 562 us one thread per row, 71 one wave)
  if (asks_wave(o) || streq(o.sddmm_mapping, "row-tile-mfma") ||
      small_sddmm(rows, nnz, std::max<int64_t>(kdim, 1)) ||
      block_rows(rows, nnz)) {
    int rc = grid_for(rows, 4, "SDDMM", &grid);
    if (rc)
      return rc;
    hipLaunchKernelGGL(sddmm_wave_per_row<T>, sw::grid_dim(grid, 256), dim3(256),
                       0, st, ro, col, val, lhs, rhs, out, (int32_t)rows, cols,
                       (int32_t)kdim, kind, alpha, beta);
  } else {
    const int64_t B = o.sddmm_block_size;
    int rc = grid_for(rows, B, "SDDMM", &grid);
    if (rc)
      return rc;
    // 16 positions per step where a workgroup of at most 512 threads lets a
    // lane hold 256 registers (configuration 5, fp32: 602 -> 478 us with 256
    // threads); four under the 1024-thread bound.  kdim 64 or 128 and whole
    // waves of at most 256-thread workgroups (one wave per SIMD, so the tile
    // and the per-row steps have 512 registers without spills; bf16 also a
    // 16-byte aligned lhs), with the rhs's bytes within 32 bits (the
    // tile's lane offsets): 64-row matrix-core tiles first
    const bool tiles = (kdim == 64 || kdim == 128) && B % kWave == 0 &&
                       B <= 256 && (sizeof(T) == 4 || aligned16(lhs)) &&
                       (int64_t)sizeof(T) * kdim * cols <= (int64_t)UINT32_MAX;
    if (tiles && kdim == 64)
      hipLaunchKernelGGL((sddmm_thread_per_row<T, 16, 256, 1>),
                         sw::grid_dim(grid, (unsigned)B), dim3((unsigned)B), 0, st, ro,
                         col, val, lhs, rhs, out, (int32_t)rows, cols,
                         (int32_t)kdim, kind, alpha, beta);
    else if (tiles)
      hipLaunchKernelGGL((sddmm_thread_per_row<T, 16, 256, 2>),
                         sw::grid_dim(grid, (unsigned)B), dim3((unsigned)B), 0, st, ro,
                         col, val, lhs, rhs, out, (int32_t)rows, cols,
                         (int32_t)kdim, kind, alpha, beta);
    else if (B <= 512)
      hipLaunchKernelGGL((sddmm_thread_per_row<T, 16, 512>),
                         sw::grid_dim(grid, (unsigned)B), dim3((unsigned)B), 0, st, ro,
                         col, val, lhs, rhs, out, (int32_t)rows, cols,
                         (int32_t)kdim, kind, alpha, beta);
    else
      hipLaunchKernelGGL((sddmm_thread_per_row<T, 4, 1024>),
                         sw::grid_dim(grid, (unsigned)B), dim3((unsigned)B), 0, st, ro,
                         col, val, lhs, rhs, out, (int32_t)rows, cols,
                         (int32_t)kdim, kind, alpha, beta);
  }
  return launch_check("SDDMM kernel");
}

// Lanes per row of the row reductions: a mean row in one step, and more of
// them while the rows are fewer than 2,048 waves (8,548 rows of 11, lognormal
// with sigma 1.5 and sorted by length, bf16: 2 lanes 31 us, 16 lanes 8).
int row_lanes(int64_t rows, int64_t nnz) {
  const int64_t mean = nnz / std::max<int64_t>(rows, 1);
  int g = 2;
  while (g < 64 && (kRowEntries * g < mean || rows * g / kWave < 2048))
    g *= 2;
  return g;
}

template <typename T>
int launch_row_reduce(const int32_t *ro, const T *val, T *out, int64_t rows,
                      int64_t nnz, bool is_max, const sw_options &o,
                      hipStream_t st) {
  const int g = row_lanes(rows, nnz);
  // whole waves (row-reduction-block-size may be any size)
  const int64_t B = ceil_div(o.row_reduction_block_size, kWave) * kWave;
  const int64_t grid = std::max<int64_t>(ceil_div(rows, B / g), 1);
  int rc = check_grid(grid, B, "CSR row reduction");
  if (rc)
    return rc;
#define SW_REDUCE(G)                                                          \
  case G:                                                                     \
    if (is_max)                                                               \
      hipLaunchKernelGGL((row_reduce_group<true, T, G>), grid_dim(grid, B),   \
                         dim3((unsigned)B), 0, st, ro, val, out,              \
                         (int32_t)rows, (int32_t)nnz);                        \
    else                                                                      \
      hipLaunchKernelGGL((row_reduce_group<false, T, G>), grid_dim(grid, B),  \
                         dim3((unsigned)B), 0, st, ro, val, out,              \
                         (int32_t)rows, (int32_t)nnz);                        \
    break;
  switch (g) {
    SW_REDUCE(2) SW_REDUCE(4) SW_REDUCE(8) SW_REDUCE(16) SW_REDUCE(32)
    SW_REDUCE(64)
  }
#undef SW_REDUCE
  return launch_check("CSR row reduction kernel");
}

template <typename T>
int launch_rowwise_map(const int32_t *ro, const T *val, const T *rowv, T *out,
                       int64_t rows, int64_t nnz, int kind, hipStream_t st) {
  // 16 entries a lane share a wave's row searches; few entries are spread
  // over more waves instead (exp, fp32, 16 / 4 entries a lane: 4 M entries in
  // 1 M rows 17.0 / 22.1 us, 400,000 in 100,000 rows 11.1 / 7.8)
  constexpr int W = 16 / (int)sizeof(T);
  const int n = nnz >= 2000000 ? 16 / W : 1;
  const int64_t grid =
      std::max<int64_t>(ceil_div(nnz, (int64_t)256 * W * n), 1);
  int rc = check_grid(grid, 256, "CSR row-wise map");
  if (rc)
    return rc;
#define SW_MAP_N(KIND, N)                                                     \
  hipLaunchKernelGGL((rowwise_map_positions<T, KIND, N>),                     \
                     grid_dim(grid, 256), dim3(256), 0, st, ro, val, rowv,    \
                     out, (int32_t)rows, (int32_t)nnz)
#define SW_MAP(KIND)                                                          \
  case KIND:                                                                  \
    if (n > 1)                                                                \
      SW_MAP_N(KIND, 16 / W);                                                 \
    else                                                                      \
      SW_MAP_N(KIND, 1);                                                      \
    break;
  switch (kind) {
    SW_MAP(SW_MAP_EXP_SUB)
    SW_MAP(SW_MAP_DIV)
    SW_MAP(SW_MAP_SUB)
    SW_MAP(SW_MAP_MUL)
  }
#undef SW_MAP
#undef SW_MAP_N
  return launch_check("CSR row-wise map kernel");
}

// ---- entry points (fp32 and bf16 share them) --------------------------------

template <typename T>
int sddmm_entry(const int32_t *row_offsets, const int32_t *column_indices,
                const T *values, const T *lhs, const T *rhs, T *output_values,
                int64_t rows, int64_t cols, int64_t nnz, int64_t kdim,
                int combine, float alpha, float beta, const sw_options *opts,
                void *workspace, int64_t workspace_bytes, void *stream) {
  clear_error();
  sw_options o;
  int rc = resolve_options(opts, &o);
  if (rc)
    return rc;
  if (combine != SW_SDDMM_MUL && combine != SW_SDDMM_AFFINE &&
      combine != SW_SDDMM_DOT)
    return fail(SW_ERR_INVALID_ARGUMENT, "unknown SDDMM combine kind %d",
                combine);
  rc = check_csr(row_offsets, column_indices,
                 combine == SW_SDDMM_DOT ? (const void *)output_values
                                         : (const void *)values,
                 rows, nnz, true);
  if (!rc)
    rc = check_value_alignment(sizeof(T), {values, lhs, rhs, output_values});
  if (rc)
    return rc;
  if (cols < 0 || kdim < 0 || kdim > INT32_MAX)
    return fail(SW_ERR_INVALID_SHAPE, "invalid SDDMM dense shapes");
  if (rows == 0 || nnz == 0)
    return SW_OK;
  if (!output_values || (kdim > 0 && (!lhs || !rhs)))
    return fail(SW_ERR_INVALID_ARGUMENT, "SDDMM operand pointer is null");
  const int64_t need =
      workspace ? sddmm_workspace(rows, cols, nnz, kdim, sizeof(T), o) : 0;
  const bool use = need > 0 && workspace_bytes >= need && aligned16(workspace);
  return launch_sddmm<T>(row_offsets, column_indices,
                         combine == SW_SDDMM_DOT ? nullptr : values, lhs, rhs,
                         output_values, rows, cols, nnz, kdim, combine, alpha,
                         beta, o, as_stream(stream),
                         use ? static_cast<T *>(workspace) : nullptr);
}

template <typename T>
int row_reduce_entry(const int32_t *row_offsets, const int32_t *column_indices,
                     const T *values, T *output, int64_t rows, int64_t nnz,
                     const char *kind, const sw_options *opts, void *stream) {
  clear_error();
  sw_options o;
  int rc = resolve_options(opts, &o);
  if (rc)
    return rc;
  if (!kind || (!streq(kind, "sum") && !streq(kind, "max")))
    return fail(SW_ERR_INVALID_ARGUMENT,
                "expected CSR row reduction kind 'sum' or 'max', but got '%s'",
                kind ? kind : "(null)");
  rc = check_csr(row_offsets, column_indices, values, rows, nnz, false);
  if (!rc)
    rc = check_value_alignment(sizeof(T), {values, output});
  if (rc)
    return rc;
  if (rows == 0)
    return SW_OK;
  if (!output)
    return fail(SW_ERR_INVALID_ARGUMENT, "output pointer is null");
  return launch_row_reduce<T>(row_offsets, values, output, rows, nnz,
                              streq(kind, "max"), o, as_stream(stream));
}

template <typename T>
int rowwise_map_entry(const int32_t *row_offsets,
                      const int32_t *column_indices, const T *values,
                      const T *row_values, T *output_values, int64_t rows,
                      int64_t nnz, int map, const sw_options *opts,
                      void *stream) {
  clear_error();
  sw_options o;
  int rc = resolve_options(opts, &o);
  if (rc)
    return rc;
  if (map < SW_MAP_EXP_SUB || map > SW_MAP_MUL)
    return fail(SW_ERR_INVALID_ARGUMENT, "unknown row-wise map kind %d", map);
  rc = check_csr(row_offsets, column_indices, values, rows, nnz, false);
  if (!rc)
    rc = check_value_alignment(sizeof(T), {values, row_values, output_values});
  if (rc)
    return rc;
  if (rows == 0 || nnz == 0)
    return SW_OK;
  if (!output_values || !row_values)
    return fail(SW_ERR_INVALID_ARGUMENT, "row-wise map pointer is null");
  return launch_rowwise_map<T>(row_offsets, values, row_values, output_values,
                               rows, nnz, map, as_stream(stream));
}

// No output range shares a byte with an input or with another output.
struct Range {
  const void *p;
  int64_t bytes;
};
bool outputs_apart(std::initializer_list<Range> outs,
                   std::initializer_list<Range> ins) {
  auto apart = [](const Range &a, const Range &b) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a.p),
                    y = reinterpret_cast<uintptr_t>(b.p);
    return a.bytes <= 0 || b.bytes <= 0 || x + (uintptr_t)a.bytes <= y ||
           y + (uintptr_t)b.bytes <= x;
  };
  for (const Range &o : outs) {
    for (const Range &i : ins)
      if (!apart(o, i))
        return false;
    for (const Range &p : outs)
      if (&p != &o && !apart(o, p))
        return false;
  }
  return true;
}

// The whole chain in one kernel per 16-row tile when the options ask for
// matrix-core tiles and the shapes fit the fused kernel; returns true when it
// was launched (rc holds the launch status).
bool launch_fused_attention(const int32_t *ro, const int32_t *col,
                            const float *mask, const float *q,
                            const float *kt, const float *v, float *scores,
                            float *rmax, float *rsum, float *out,
                            int64_t rows, int64_t cols, int64_t nnz,
                            int64_t d, int64_t dv, float alpha, float beta,
                            bool libm, hipStream_t st, int *rc) {
  if (!((d == 64 || d == 128) && dv > 0 && dv % 16 == 0 && nnz >= 4 &&
        narrow_offsets(nnz, 1) && narrow_offsets(cols, d) &&
        narrow_offsets(cols, dv)))
    return false;
  int64_t grid;
  *rc = grid_for(rows, 16, "fused attention", &grid);
  if (*rc)
    return true;
  // interleaved output tiles (configuration 5: 25.2 -> 24.0 us)
  const bool il = dv % 64 == 0 && aligned16(v) && aligned16(out);
  const bool lng = long_rows(rows, nnz);
#define SW_FUSED_AS(KB, IL, LIBM, LONG)                                       \
  hipLaunchKernelGGL(                                                         \
      (attention_tile_fused<KB, kFusedWaves, IL, false, false, false, LIBM,   \
                            LONG>),                                           \
      sw::grid_dim(grid, 64 * kFusedWaves), dim3(64 * kFusedWaves), 0, st,    \
      ro, col, mask, q, kt, v, scores, rmax, rsum, out, (int32_t)rows, cols,  \
      (int32_t)d, dv, alpha, beta, (uint32_t)(nnz - 4),                       \
      (int)SW_SDDMM_AFFINE)
#define SW_FUSED(KB, IL)                                                      \
  do {                                                                        \
    if (libm && lng)                                                          \
      SW_FUSED_AS(KB, IL, true, true);                                        \
    else if (libm)                                                            \
      SW_FUSED_AS(KB, IL, true, false);                                       \
    else if (lng)                                                             \
      SW_FUSED_AS(KB, IL, false, true);                                       \
    else                                                                      \
      SW_FUSED_AS(KB, IL, false, false);                                      \
  } while (0)
  if (d == 64 && il)
    SW_FUSED(1, true);
  else if (d == 64)
    SW_FUSED(1, false);
  else if (il)
    SW_FUSED(2, true);
  else
    SW_FUSED(2, false);
#undef SW_FUSED
#undef SW_FUSED_AS
  *rc = launch_check("fused attention kernel");
  return true;
}

bool launch_fused_attention(const int32_t *ro, const int32_t *col,
                            const uint16_t *mask, const uint16_t *q,
                            const uint16_t *kt, const uint16_t *v,
                            uint16_t *scores, uint16_t *rmax, uint16_t *rsum,
                            uint16_t *out, int64_t rows, int64_t cols,
                            int64_t nnz, int64_t d, int64_t dv, float alpha,
                            float beta, bool libm, hipStream_t st, int *rc) {
  if (!((d == 64 || d == 128) && dv > 0 && dv % 64 == 0 && nnz >= 4 &&
        aligned16(q) &&
        (reinterpret_cast<uintptr_t>(v) & 7u) == 0 &&
        (reinterpret_cast<uintptr_t>(out) & 7u) == 0 &&
        narrow_offsets(nnz, 1) && narrow_offsets(cols, d) &&
        narrow_offsets(cols, dv)))
    return false;
  int64_t grid;
  *rc = grid_for(rows, 16, "fused attention", &grid);
  if (*rc)
    return true;
#define SW_FUSED_AS(KB, LIBM)                                                 \
  hipLaunchKernelGGL(                                                         \
      (attention_tile_fused_bf16<KB, kFusedWaves, false, false, false, LIBM>),\
      sw::grid_dim(grid, 64 * kFusedWaves), dim3(64 * kFusedWaves), 0, st,    \
      ro, col, mask, q, kt, v, scores, rmax, rsum, out, (int32_t)rows, cols,  \
      (int32_t)d, dv, alpha, beta, (uint32_t)(nnz - 4),                       \
      (int)SW_SDDMM_AFFINE)
#define SW_FUSED(KB)                                                          \
  do {                                                                        \
    if (libm)                                                                 \
      SW_FUSED_AS(KB, true);                                                  \
    else                                                                      \
      SW_FUSED_AS(KB, false);                                                 \
  } while (0)
  if (d == 64)
    SW_FUSED(1);
  else
    SW_FUSED(2);
#undef SW_FUSED
#undef SW_FUSED_AS
  *rc = launch_check("fused attention kernel");
  return true;
}

// The tile floor: the fused kernel launch_fused_attention would run for
// these operands, in its FLOOR form; false when the shapes do not take the
// fused kernel.
bool launch_attention_floor(const int32_t *ro, const int32_t *col,
                            const float *mask, const float *q,
                            const float *kt, const float *v, float *scores,
                            float *rmax, float *rsum, float *out,
                            int64_t rows, int64_t cols, int64_t nnz,
                            int64_t d, int64_t dv, hipStream_t st, int *rc) {
  if (!((d == 64 || d == 128) && dv > 0 && dv % 16 == 0 && nnz >= 4 &&
        narrow_offsets(nnz, 1) && narrow_offsets(cols, d) &&
        narrow_offsets(cols, dv)))
    return false;
  int64_t grid;
  *rc = grid_for(rows, 16, "attention tile floor", &grid);
  if (*rc)
    return true;
  const bool il = dv % 64 == 0 && aligned16(v) && aligned16(out);
#define SW_FLOOR(KB, IL)                                                      \
  hipLaunchKernelGGL(                                                         \
      (attention_tile_fused<KB, kFusedWaves, IL, false, false, true>),        \
      sw::grid_dim(grid, 64 * kFusedWaves), dim3(64 * kFusedWaves), 0, st, ro, col, mask, q,  \
      kt, v, scores, rmax, rsum, out, (int32_t)rows, cols, (int32_t)d, dv,    \
      1.0f, 0.0f, (uint32_t)(nnz - 4), (int)SW_SDDMM_AFFINE)
  if (d == 64 && il)
    SW_FLOOR(1, true);
  else if (d == 64)
    SW_FLOOR(1, false);
  else if (il)
    SW_FLOOR(2, true);
  else
    SW_FLOOR(2, false);
#undef SW_FLOOR
  *rc = launch_check("attention tile floor kernel");
  return true;
}

bool launch_attention_floor(const int32_t *ro, const int32_t *col,
                            const uint16_t *mask, const uint16_t *q,
                            const uint16_t *kt, const uint16_t *v,
                            uint16_t *scores, uint16_t *rmax, uint16_t *rsum,
                            uint16_t *out, int64_t rows, int64_t cols,
                            int64_t nnz, int64_t d, int64_t dv,
                            hipStream_t st, int *rc) {
  if (!((d == 64 || d == 128) && dv > 0 && dv % 64 == 0 && nnz >= 4 &&
        aligned16(q) &&
        (reinterpret_cast<uintptr_t>(v) & 7u) == 0 &&
        (reinterpret_cast<uintptr_t>(out) & 7u) == 0 &&
        narrow_offsets(nnz, 1) && narrow_offsets(cols, d) &&
        narrow_offsets(cols, dv)))
    return false;
  int64_t grid;
  *rc = grid_for(rows, 16, "attention tile floor", &grid);
  if (*rc)
    return true;
#define SW_FLOOR(KB)                                                          \
  hipLaunchKernelGGL(                                                         \
      (attention_tile_fused_bf16<KB, kFusedWaves, false, false, true>),       \
      sw::grid_dim(grid, 64 * kFusedWaves), dim3(64 * kFusedWaves), 0, st, ro, col, mask, q,  \
      kt, v, scores, rmax, rsum, out, (int32_t)rows, cols, (int32_t)d, dv,    \
      1.0f, 0.0f, (uint32_t)(nnz - 4), (int)SW_SDDMM_AFFINE)
  if (d == 64)
    SW_FLOOR(1);
  else
    SW_FLOOR(2);
#undef SW_FLOOR
  *rc = launch_check("attention tile floor kernel");
  return true;
}

template <typename T>
int attention_floor_entry(const int32_t *row_offsets,
                          const int32_t *column_indices, const T *mask_values,
                          const T *query, const T *transposed_key,
                          const T *value, T *scores, T *row_maximum,
                          T *row_sum, T *output, int64_t rows, int64_t cols,
                          int64_t nnz, int64_t d, int64_t dv, void *stream) {
  int rc = check_csr(row_offsets, column_indices, mask_values, rows, nnz,
                     true);
  if (!rc)
    rc = check_value_alignment(sizeof(T), {mask_values, query, transposed_key,
                                           value, scores, row_maximum,
                                           row_sum, output});
  if (rc)
    return rc;
  if (cols < 0 || d < 0 || dv < 0 || d > INT32_MAX)
    return fail(SW_ERR_INVALID_SHAPE, "invalid attention shapes");
  if (rows == 0)
    return SW_OK;
  if (!row_maximum || !row_sum || !output || !scores || !query ||
      !transposed_key || !value)
    return fail(SW_ERR_INVALID_ARGUMENT, "attention buffer pointer is null");
  if (!launch_attention_floor(row_offsets, column_indices, mask_values, query,
                              transposed_key, value, scores, row_maximum,
                              row_sum, output, rows, cols, nnz, d, dv,
                              as_stream(stream), &rc))
    return fail(SW_ERR_INVALID_ARGUMENT,
                "the tile floor needs the fused kernel's shapes: d of 64 or "
                "128, dv a multiple of %d, at least 4 entries%s",
                sizeof(T) == 4 ? 16 : 64,
                sizeof(T) == 4 ? "" : ", aligned query, value and output");
  return rc;
}

template <typename T>
int attention_entry(const int32_t *row_offsets, const int32_t *column_indices,
                    const T *mask_values, const T *query,
                    const T *transposed_key, const T *value, T *scores,
                    T *row_maximum, T *row_sum, T *output, int64_t rows,
                    int64_t cols, int64_t nnz, int64_t d, int64_t dv,
                    float alpha, float beta, const sw_options *opts,
                    void *stream) {
  clear_error();
  sw_options o;
  int rc = resolve_options(opts, &o);
  if (rc)
    return rc;
  rc = check_csr(row_offsets, column_indices, mask_values, rows, nnz, true);
  if (!rc)
    rc = check_value_alignment(sizeof(T), {mask_values, query, transposed_key,
                                           value, scores, row_maximum,
                                           row_sum, output});
  if (rc)
    return rc;
  if (cols < 0 || d < 0 || dv < 0 || d > INT32_MAX)
    return fail(SW_ERR_INVALID_SHAPE, "invalid attention shapes");
  if constexpr (std::is_same_v<T, uint16_t>) {
    rc = check_bf16_spmm_mapping(o); // before any launch
    if (rc)
      return rc;
  }
  if (rows == 0)
    return SW_OK;
  if (!row_maximum || !row_sum || (dv > 0 && !output) ||
      (nnz > 0 && (!scores || !query || !transposed_key || (dv > 0 && !value))))
    return fail(SW_ERR_INVALID_ARGUMENT, "attention buffer pointer is null");
  hipStream_t st = as_stream(stream);
  const bool fused = o.sddmm_lanes_per_row == 64 &&
                     streq(o.sddmm_mapping, "row-tile-mfma") &&
                     streq(o.spmm_mapping, "row-tile-mfma");
  // A call that leaves every mapping and block size at its default asks for
  // the chain and not for a schedule: it takes the one-kernel form too, with
  // the separate ops' expf and division (LIBM), when no output buffer shares
  // memory with another operand (the six kernels finish reading an operand
  // before a later one writes).  3,001 positions of up to 384 entries,
  // d = dv = 64, fp32: 536 us in six kernels, 12.4 us in one.  Not many rows
  // of fewer than five entries: tiles of them seldom share columns, and row
  // by row a wave's chain of trips costs the same however short the row is
  // (d = 64, fp32, one kernel / six: 100,000 rows of 0.1 entries 251 / 85 us, of
  // 4 691 / 474, 32,000 in 8 x 8 blocks 156 / 56; 8,000 rows of 4 30 / 46,
  // 32,000 of 8 223 / 196, in 16 x 16 blocks, 8.5 entries a row, 31 / 61; bf16
  // 23,585 rows of 7.6, unequal and sorted by length, 147 / 336).
  const bool defaults =
      (rows <= 16384 || nnz / 5 >= rows) &&
      streq(o.sddmm_mapping, "thread-per-row") &&
      streq(o.spmm_mapping, "thread-per-output") &&
      o.sddmm_lanes_per_row == 1 && o.sddmm_block_size == 256 &&
      o.row_reduction_block_size == 256 && o.rowwise_map_block_size == 256 &&
      o.spmm_block_size == 256 &&
      outputs_apart({{scores, nnz * (int64_t)sizeof(T)},
                     {row_maximum, rows * (int64_t)sizeof(T)},
                     {row_sum, rows * (int64_t)sizeof(T)},
                     {output, rows * dv * (int64_t)sizeof(T)}},
                    {{row_offsets, (rows + 1) * 4},
                     {column_indices, nnz * 4},
                     {mask_values, nnz * (int64_t)sizeof(T)},
                     {query, rows * d * (int64_t)sizeof(T)},
                     {transposed_key, d * cols * (int64_t)sizeof(T)},
                     {value, cols * dv * (int64_t)sizeof(T)}});
  if (nnz > 0 && (fused || defaults) &&
      launch_fused_attention(row_offsets, column_indices, mask_values, query,
                             transposed_key, value, scores, row_maximum,
                             row_sum, output, rows, cols, nnz, d, dv, alpha,
                             beta, !fused, st, &rc))
    return rc;
  if (nnz > 0) {
    rc = launch_sddmm<T>(row_offsets, column_indices, mask_values, query,
                         transposed_key, scores, rows, cols, nnz, d,
                         SW_SDDMM_AFFINE, alpha, beta, o, st);
    if (rc)
      return rc;
  }
  if (o.sddmm_lanes_per_row == 64) {
    // wave row ops: the four softmax ops run as one kernel
    int64_t grid = std::max<int64_t>(ceil_div(rows, 4), 1);
    rc = check_grid(grid, 256, "attention softmax");
    if (rc)
      return rc;
    hipLaunchKernelGGL(row_softmax_wave<T>, sw::grid_dim(grid, 256), dim3(256), 0,
                       st, row_offsets, scores, row_maximum, row_sum,
                       (int32_t)rows);
    rc = launch_check("attention softmax kernel");
    if (rc)
      return rc;
    if (dv == 0)
      return SW_OK;
    return launch_spmm(row_offsets, column_indices, scores, value, output,
                       rows, cols, nnz, dv, o, "attention output SpMM", st);
  }
  rc = launch_row_reduce<T>(row_offsets, scores, row_maximum, rows, nnz, true,
                            o, st);
  if (rc)
    return rc;
  if (nnz > 0) {
    rc = launch_rowwise_map<T>(row_offsets, scores, row_maximum, scores, rows,
                               nnz, SW_MAP_EXP_SUB, st);
    if (rc)
      return rc;
  }
  rc = launch_row_reduce<T>(row_offsets, scores, row_sum, rows, nnz, false, o,
                            st);
  if (rc)
    return rc;
  if (nnz > 0) {
    rc = launch_rowwise_map<T>(row_offsets, scores, row_sum, scores, rows, nnz,
                               SW_MAP_DIV, st);
    if (rc)
      return rc;
  }
  if (dv == 0)
    return SW_OK;
  return launch_spmm(row_offsets, column_indices, scores, value, output, rows,
                     cols, nnz, dv, o, "attention output SpMM", st);
}

} // namespace sw

extern "C" int sw_sddmm_csr_f32(const int32_t *row_offsets,
                                const int32_t *column_indices,
                                const float *values, const float *lhs,
                                const float *rhs, float *output_values,
                                int64_t rows, int64_t cols, int64_t nnz,
                                int64_t kdim, int combine, float alpha,
                                float beta, const sw_options *opts,
                                void *stream) {
  return sw::sddmm_entry<float>(row_offsets, column_indices, values, lhs, rhs,
                                output_values, rows, cols, nnz, kdim, combine,
                                alpha, beta, opts, nullptr, 0, stream);
}

extern "C" int sw_sddmm_csr_f32_ws(
    const int32_t *row_offsets, const int32_t *column_indices,
    const float *values, const float *lhs, const float *rhs,
    float *output_values, int64_t rows, int64_t cols, int64_t nnz,
    int64_t kdim, int combine, float alpha, float beta, const sw_options *opts,
    void *workspace, int64_t workspace_bytes, void *stream) {
  return sw::sddmm_entry<float>(row_offsets, column_indices, values, lhs, rhs,
                                output_values, rows, cols, nnz, kdim, combine,
                                alpha, beta, opts, workspace, workspace_bytes,
                                stream);
}

extern "C" int sw_sddmm_csr_bf16_ws(
    const int32_t *row_offsets, const int32_t *column_indices,
    const uint16_t *values, const uint16_t *lhs, const uint16_t *rhs,
    uint16_t *output_values, int64_t rows, int64_t cols, int64_t nnz,
    int64_t kdim, int combine, float alpha, float beta, const sw_options *opts,
    void *workspace, int64_t workspace_bytes, void *stream) {
  return sw::sddmm_entry<uint16_t>(
      row_offsets, column_indices, values, lhs, rhs, output_values, rows, cols,
      nnz, kdim, combine, alpha, beta, opts, workspace, workspace_bytes,
      stream);
}

extern "C" int64_t sw_sddmm_workspace_bytes(int64_t rows, int64_t cols,
                                            int64_t nnz, int64_t kdim,
                                            int value_bytes,
                                            const sw_options *opts) {
  if (value_bytes != 4 && value_bytes != 2)
    return 0;
  if (opts)
    return sw::sddmm_workspace(rows, cols, nnz, kdim, value_bytes, *opts);
  sw_options o;
  sw_options_init(&o);
  return sw::sddmm_workspace(rows, cols, nnz, kdim, value_bytes, o);
}

extern "C" int sw_sddmm_csr_bf16(const int32_t *row_offsets,
                                 const int32_t *column_indices,
                                 const uint16_t *values, const uint16_t *lhs,
                                 const uint16_t *rhs, uint16_t *output_values,
                                 int64_t rows, int64_t cols, int64_t nnz,
                                 int64_t kdim, int combine, float alpha,
                                 float beta, const sw_options *opts,
                                 void *stream) {
  return sw::sddmm_entry<uint16_t>(row_offsets, column_indices, values, lhs,
                                   rhs, output_values, rows, cols, nnz, kdim,
                                   combine, alpha, beta, opts, nullptr, 0,
                                   stream);
}

extern "C" int sw_csr_row_reduce_f32(const int32_t *row_offsets,
                                     const int32_t *column_indices,
                                     const float *values, float *output,
                                     int64_t rows, int64_t nnz,
                                     const char *kind, const sw_options *opts,
                                     void *stream) {
  return sw::row_reduce_entry<float>(row_offsets, column_indices, values,
                                     output, rows, nnz, kind, opts, stream);
}

extern "C" int sw_csr_row_reduce_bf16(const int32_t *row_offsets,
                                      const int32_t *column_indices,
                                      const uint16_t *values, uint16_t *output,
                                      int64_t rows, int64_t nnz,
                                      const char *kind, const sw_options *opts,
                                      void *stream) {
  return sw::row_reduce_entry<uint16_t>(row_offsets, column_indices, values,
                                        output, rows, nnz, kind, opts, stream);
}

extern "C" int sw_csr_rowwise_map_f32(const int32_t *row_offsets,
                                      const int32_t *column_indices,
                                      const float *values,
                                      const float *row_values,
                                      float *output_values, int64_t rows,
                                      int64_t nnz, int map,
                                      const sw_options *opts, void *stream) {
  return sw::rowwise_map_entry<float>(row_offsets, column_indices, values,
                                      row_values, output_values, rows, nnz,
                                      map, opts, stream);
}

extern "C" int sw_csr_rowwise_map_bf16(const int32_t *row_offsets,
                                       const int32_t *column_indices,
                                       const uint16_t *values,
                                       const uint16_t *row_values,
                                       uint16_t *output_values, int64_t rows,
                                       int64_t nnz, int map,
                                       const sw_options *opts, void *stream) {
  return sw::rowwise_map_entry<uint16_t>(row_offsets, column_indices, values,
                                         row_values, output_values, rows, nnz,
                                         map, opts, stream);
}

extern "C" int sw_sparse_attention_f32(
    const int32_t *row_offsets, const int32_t *column_indices,
    const float *mask_values, const float *query, const float *transposed_key,
    const float *value, float *scores, float *row_maximum, float *row_sum,
    float *output, int64_t rows, int64_t cols, int64_t nnz, int64_t d,
    int64_t dv, float alpha, float beta, const sw_options *opts,
    void *stream) {
  return sw::attention_entry<float>(
      row_offsets, column_indices, mask_values, query, transposed_key, value,
      scores, row_maximum, row_sum, output, rows, cols, nnz, d, dv, alpha,
      beta, opts, stream);
}

extern "C" int sw_attention_tile_floor(
    const int32_t *row_offsets, const int32_t *column_indices,
    const void *mask_values, const void *query, const void *transposed_key,
    const void *value, void *scores, void *row_maximum, void *row_sum,
    void *output, int64_t rows, int64_t cols, int64_t nnz, int64_t d,
    int64_t dv, int value_bytes, void *stream) {
  sw::clear_error();
  if (value_bytes == 4)
    return sw::attention_floor_entry<float>(
        row_offsets, column_indices, static_cast<const float *>(mask_values),
        static_cast<const float *>(query),
        static_cast<const float *>(transposed_key),
        static_cast<const float *>(value), static_cast<float *>(scores),
        static_cast<float *>(row_maximum), static_cast<float *>(row_sum),
        static_cast<float *>(output), rows, cols, nnz, d, dv, stream);
  if (value_bytes == 2)
    return sw::attention_floor_entry<uint16_t>(
        row_offsets, column_indices,
        static_cast<const uint16_t *>(mask_values),
        static_cast<const uint16_t *>(query),
        static_cast<const uint16_t *>(transposed_key),
        static_cast<const uint16_t *>(value), static_cast<uint16_t *>(scores),
        static_cast<uint16_t *>(row_maximum),
        static_cast<uint16_t *>(row_sum), static_cast<uint16_t *>(output),
        rows, cols, nnz, d, dv, stream);
  return sw::fail(SW_ERR_INVALID_ARGUMENT,
                  "tile floor value bytes must be 4 or 2, but got %d",
                  value_bytes);
}

extern "C" int sw_sparse_attention_bf16(
    const int32_t *row_offsets, const int32_t *column_indices,
    const uint16_t *mask_values, const uint16_t *query,
    const uint16_t *transposed_key, const uint16_t *value, uint16_t *scores,
    uint16_t *row_maximum, uint16_t *row_sum, uint16_t *output, int64_t rows,
    int64_t cols, int64_t nnz, int64_t d, int64_t dv, float alpha, float beta,
    const sw_options *opts, void *stream) {
  return sw::attention_entry<uint16_t>(
      row_offsets, column_indices, mask_values, query, transposed_key, value,
      scores, row_maximum, row_sum, output, rows, cols, nnz, d, dv, alpha,
      beta, opts, stream);
}
