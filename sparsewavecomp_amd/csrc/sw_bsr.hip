// sparsewave.bsr_spmm on gfx950 behind sw_bsr_spmm_f32 / sw_bsr_spmm_bf16.
//
// Reference kernel: ThreadPerOutputBSRSpMMPattern
// (lib/Dialect/SparseWave/Transforms/SparseWaveToGPU.cpp:560-665), blocks
// row-major [nnzb][b][b] (SparseWaveOps.td:133-137), shape rules of the
// verifier (lib/Dialect/SparseWave/IR/SparseWaveOps.cpp:144-207, 340-372).
//
// The MI355X path runs each block product on the matrix cores, accumulating
// in fp32 registers across the block row's blocks; for 16 x 16 blocks:
//   fp32, k % 4 == 0: a wave owns a 16 x 64 output strip (four tiles with
//     interleaved columns, 128-bit RHS loads and output stores) and issues
//     v_mfma_f32_16x16x4_f32 four times per block and tile;
//   bf16 with a bf16 output, k % 8 == 0: a wave owns a 16 x 128 output strip
//     (eight tiles with interleaved columns, 128-bit RHS loads) and issues
//     v_mfma_f32_16x16x16_bf16 once per block and tile;
//   other block sizes that are a multiple of 4, other k and unaligned
//     operands take bsr_mfma, the same tiles over 16-row strips.
#include "sw_device.h"
#include "sw_internal.h"

#include <algorithm>
#include <type_traits>

using namespace swd;

namespace {

// thread-per-output for any block size: one thread per output element,
// the products added in block and column order.  BS = 16: the block size
// known, a block's 16 values and rhs rows requested together.  ROW (k and
// the workgroup size multiples of 64): a wave's outputs lie in one row, whose
// index is put in a scalar register, so that the block values and column
// indices are scalar loads shared by the wave.
template <typename T, typename TO, int BS, bool ROW>
__global__ __launch_bounds__(1024) void bsr_thread_per_output(
    const int32_t *__restrict__ bro, const int32_t *__restrict__ bcol,
    const T *__restrict__ bval, const T *__restrict__ rhs,
    TO *__restrict__ out, int64_t rows, int64_t k, int32_t b_any) {
  const int32_t b = BS > 0 ? BS : b_any;
  int64_t e = block_id() * blockDim.x + threadIdx.x;
  if (e >= rows * k)
    return;
  int64_t r = e / k, c = e - r * k;
  if constexpr (ROW) // rows < 2^31
    r = __builtin_amdgcn_readfirstlane((int32_t)r);
  int64_t br = r / b, lr = r - br * b;
  float acc = 0.0f;
  for (int32_t bp = bro[br]; bp < bro[br + 1]; ++bp) {
    const T *blk = bval + (int64_t)bp * b * b + lr * b;
    int64_t rb = (int64_t)bcol[bp] * b;
    if constexpr (BS > 0) {
      float a[BS], x[BS];
#pragma unroll
      for (int lc = 0; lc < BS; ++lc) {
        a[lc] = tof(blk[lc]);
        x[lc] = tof(rhs[(rb + lc) * k + c]);
      }
#pragma unroll
      for (int lc = 0; lc < BS; ++lc)
        acc = __builtin_fmaf(a[lc], x[lc], acc);
    } else {
      for (int32_t lc = 0; lc < b; ++lc)
        acc = __builtin_fmaf(tof(blk[lc]), tof(rhs[(rb + lc) * k + c]), acc);
    }
  }
  stv(out + e, acc);
}

// MFMA operand layouts (one 16 x 16 x K step, wave64, lane l):
//   A[i][k] with i = l % 16, k from the lane group g = l / 16,
//   B[k][j] with j = l % 16, same k,
//   D[4*g + v][l % 16] in accumulator register v.
// The k order inside a block is a free choice as long as A and B agree;
// fp32 uses k = 4*g + s at step s so that one 128-bit load gives a lane its
// four A values.
// Block rows are visited XCD-aware: workgroups are dispatched to the eight
// XCDs round-robin, so workgroup w runs block row
// (w % 8) * (nbr / 8) + w / 8 and each XCD walks a contiguous range of block
// rows, keeping the RHS tiles of a banded matrix in its own L2.
__device__ __forceinline__ int xcd_block_row(int w, int nbr) {
  constexpr int kXcds = 8;
  if (nbr % kXcds != 0)
    return w;
  return (w % kXcds) * (nbr / kXcds) + w / kXcds;
}

// Column-interleaved bf16 kernel (k % 8 == 0, rhs and output 16-byte
// aligned).  A workgroup owns one block row and a 128-column strip as eight
// 16 x 16 tiles whose columns interleave -- tile t's MFMA column j is strip
// column 8j + t -- so one 128-bit load of an RHS row gives a lane its eight
// columns' values, one per tile: per block a lane issues one 64-bit A load
// and four 128-bit B loads (the block's 16 x 128 RHS slab in four wave
// instructions), then eight v_mfma_f32_16x16x16_bf16.  The B operand of tile
// t is element t of the four loaded rows (lane group g: rows 4g .. 4g+3).
// The block row's blocks are split over the SPL waves of the workgroup
// (wave w takes blocks w NB .. w NB + NB - 1, then every NB SPL-th batch),
// which shortens each wave's chain of memory trips; the waves' partial
// tiles are summed in LDS by wave 0.  Each lane ends with eight consecutive
// columns of four output rows: one 128-bit (bf16) or two 128-bit (fp32)
// stores per row.  Workgroups run in XCD-contiguous block-row order.
//
// FLOOR (the slab-floor diagnostic, sw_bsr_slab_floor): the same grid, block
// order, loads, LDS reduction and stores, with the matrix-core products
// replaced by an XOR of every 32-bit word the lane loads; every output
// element of the lane's region then holds that XOR (truncated to 16 bits for
// a bf16 output).  Its time is the floor of the kernel's memory trips.
template <int NB, int SPL, typename TO, bool FLOOR = false>
__global__ __launch_bounds__(64 * SPL) void bsr16_mfma_bf16_x8(
    const int32_t *__restrict__ bro, const int32_t *__restrict__ bcol,
    const uint16_t *__restrict__ bval, const uint16_t *__restrict__ rhs,
    TO *__restrict__ out, int64_t k, int nbr) {
  __shared__ float red[SPL > 1 ? SPL - 1 : 1][8][4][kWave];
  const int64_t br = xcd_contiguous(blockIdx.x, gridDim.x);
  const int sp = wave_in_group();
  const int l = lane_id();
  const int j = l & 15, g = l >> 4;
  const int64_t cb = (int64_t)blockIdx.y * 128 + 8 * j;
  const bool ok = cb < k; // k % 8 == 0: all eight columns or none
  v4f acc[8];
#pragma unroll
  for (int t = 0; t < 8; ++t)
    acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  const int32_t s = bro[br], e = bro[br + 1];
  for (int32_t b0 = s + sp * NB; b0 < e; b0 += NB * SPL) {
    const int nb = e - b0 < NB ? e - b0 : NB; // wave-uniform
    const int bcl = l < nb ? bcol[b0 + l] : 0;
    v2u a[NB];
    v4u q[NB][4];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if (u < nb) {
        const int64_t bc = __builtin_amdgcn_readlane(bcl, u);
        // A[j][4g .. 4g+3] of block b0 + u: 8 contiguous bytes
        a[u] = ld_stream(reinterpret_cast<const v2u *>(
            bval + (int64_t)(b0 + u) * 256 + j * 16 + g * 4));
        const uint16_t *brow = rhs + (bc * 16 + g * 4) * k + cb;
#pragma unroll
        for (int st = 0; st < 4; ++st)
          q[u][st] = ok ? *reinterpret_cast<const v4u *>(brow + st * k)
                        : v4u{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if (u < nb) {
        if constexpr (FLOOR) {
          uint32_t x = a[u].x ^ a[u].y;
#pragma unroll
          for (int st = 0; st < 4; ++st)
            x ^= q[u][st].x ^ q[u][st].y ^ q[u][st].z ^ q[u][st].w;
          acc[0].x = __uint_as_float(__float_as_uint(acc[0].x) ^ x);
          continue;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          // element t of the four rows (dword t / 2, half t % 2), paired by
          // byte permutes
          const int d = t >> 1;
          const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
          const v2u bt = v2u{
              __builtin_amdgcn_perm(q[u][1][d], q[u][0][d], sel),
              __builtin_amdgcn_perm(q[u][3][d], q[u][2][d], sel)};
          acc[t] = mfma_16x16x16_bf16(a[u], bt, acc[t]);
        }
      }
    }
  }
  if constexpr (FLOOR) {
    // the XOR of the waves' words, in every element the lane stores
    if constexpr (SPL > 1) {
      if (sp > 0)
        red[sp - 1][0][0][l] = acc[0].x;
      __syncthreads();
      if (sp > 0)
        return; // after the only barrier
      uint32_t x = __float_as_uint(acc[0].x);
#pragma unroll
      for (int w = 0; w < SPL - 1; ++w)
        x ^= __float_as_uint(red[w][0][0][l]);
      acc[0].x = __uint_as_float(x);
    }
    const uint32_t x = __float_as_uint(acc[0].x);
    if (ok) {
      TO *o = out + (br * 16 + g * 4) * k + cb;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if constexpr (sizeof(TO) == 2) {
          const uint32_t h = (x & 0xFFFFu) | (x << 16);
          __builtin_nontemporal_store(v4u{h, h, h, h},
                                      reinterpret_cast<v4u *>(o + v * k));
        } else {
          const float f = __uint_as_float(x);
          st4_nt(o + v * k, v4f{f, f, f, f});
          st4_nt(o + v * k + 4, v4f{f, f, f, f});
        }
      }
    }
    return;
  }
  if constexpr (SPL > 1) {
    if (sp > 0)
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          red[sp - 1][t][v][l] = acc[t][v];
    __syncthreads();
    if (sp > 0)
      return; // after the only barrier
#pragma unroll
    for (int w = 0; w < SPL - 1; ++w)
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc[t][v] += red[w][t][v][l];
  }
  if (ok) {
    TO *o = out + (br * 16 + g * 4) * k + cb;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if constexpr (sizeof(TO) == 2) {
        __builtin_nontemporal_store(
            v4u{pack_bf16x2(acc[0][v], acc[1][v]),
                pack_bf16x2(acc[2][v], acc[3][v]),
                pack_bf16x2(acc[4][v], acc[5][v]),
                pack_bf16x2(acc[6][v], acc[7][v])},
            reinterpret_cast<v4u *>(o + v * k));
      } else {
        st4_nt(o + v * k, v4f{acc[0][v], acc[1][v], acc[2][v], acc[3][v]});
        st4_nt(o + v * k + 4, v4f{acc[4][v], acc[5][v], acc[6][v], acc[7][v]});
      }
    }
  }
}

// Column-interleaved fp32 variant (k % 4 == 0, 16-byte aligned operands): a
// wave owns a 16 x 64 output strip as four 16 x 16 MFMA tiles whose columns
// interleave -- tile t's MFMA column j is output column 4j + t of the strip --
// so one 128-bit load of an RHS row gives a lane its B values for all four
// tiles, and one 128-bit store writes its four results of an output row.
// Per block and strip a lane issues one A load and four B loads instead of
// one A load and sixteen scalar B loads.
//
// A workgroup covers one block row and up to kF32Strips strips; SPL waves per
// strip split the block row's blocks (wave sp takes batches sp, sp + SPL, ...)
// so that more loads are in flight per block row, and the SPL partial tiles
// are summed through LDS by wave 0 of each strip.
constexpr int kF32Strips = 2;

// FLOOR: the slab-floor diagnostic, as for the bf16 kernel above.
template <int NB, int SPL, bool FLOOR = false>
__global__ __launch_bounds__(64 * kF32Strips * SPL) void bsr16_mfma_f32_x4(
    const int32_t *__restrict__ bro, const int32_t *__restrict__ bcol,
    const float *__restrict__ bval, const float *__restrict__ rhs,
    float *__restrict__ out, int64_t k, int nbr) {
  __shared__ float red[kF32Strips][SPL > 1 ? SPL - 1 : 1][4][4][kWave];
  const int br = xcd_block_row(blockIdx.x, nbr);
  const int strips = blockDim.x / (kWave * SPL);
  const int wv = wave_in_group();
  const int strip = wv % strips, sp = wv / strips;
  const int l = lane_id();
  const int i = l & 15, g = l >> 4;
  const int64_t cb = ((int64_t)blockIdx.y * strips + strip) * 64 + 4 * i;
  const bool ok = cb < k; // k % 4 == 0: all four columns or none
  v4f acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
    acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  const int32_t s = bro[br], e = bro[br + 1];
  for (int32_t b0 = s + sp * NB; b0 < e; b0 += NB * SPL) {
    const int nb = e - b0 < NB ? e - b0 : NB; // wave-uniform
    const int bcl = l < nb ? bcol[b0 + l] : 0;
    v4f a[NB], bv[NB][4];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (j < nb) {
        const int64_t bc = __builtin_amdgcn_readlane(bcl, j);
        a[j] = ld_stream(reinterpret_cast<const v4f *>(
            bval + (int64_t)(b0 + j) * 256 + i * 16 + g * 4));
        const float *brow = rhs + (bc * 16 + g * 4) * k + cb;
#pragma unroll
        for (int st = 0; st < 4; ++st)
          bv[j][st] = ok ? *reinterpret_cast<const v4f *>(brow + st * k)
                         : v4f{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (j < nb) {
        if constexpr (FLOOR) {
          uint32_t x = 0;
#pragma unroll
          for (int st = 0; st < 4; ++st)
            x ^= __float_as_uint(a[j][st]) ^ __float_as_uint(bv[j][st].x) ^
                 __float_as_uint(bv[j][st].y) ^ __float_as_uint(bv[j][st].z) ^
                 __float_as_uint(bv[j][st].w);
          acc[0].x = __uint_as_float(__float_as_uint(acc[0].x) ^ x);
          continue;
        }
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][st], bv[j][st].x,
                                                        acc[0], 0, 0, 0);
          acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][st], bv[j][st].y,
                                                        acc[1], 0, 0, 0);
          acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][st], bv[j][st].z,
                                                        acc[2], 0, 0, 0);
          acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][st], bv[j][st].w,
                                                        acc[3], 0, 0, 0);
        }
      }
    }
  }
  if constexpr (FLOOR) {
    if constexpr (SPL > 1) {
      if (sp > 0)
        red[strip][sp - 1][0][0][l] = acc[0].x;
      __syncthreads();
      if (sp > 0)
        return;
      uint32_t x = __float_as_uint(acc[0].x);
#pragma unroll
      for (int w = 0; w < SPL - 1; ++w)
        x ^= __float_as_uint(red[strip][w][0][0][l]);
      acc[0].x = __uint_as_float(x);
    }
    if (ok) {
      float *o = out + ((int64_t)br * 16 + g * 4) * k + cb;
      const float f = acc[0].x;
#pragma unroll
      for (int v = 0; v < 4; ++v)
        __builtin_nontemporal_store(v4f{f, f, f, f},
                                    reinterpret_cast<v4f *>(o + v * k));
    }
    return;
  }
  if constexpr (SPL > 1) {
    if (sp > 0) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          red[strip][sp - 1][t][v][l] = acc[t][v];
    }
    __syncthreads();
    if (sp > 0)
      return;
#pragma unroll
    for (int w = 0; w < SPL - 1; ++w)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc[t][v] += red[strip][w][t][v][l];
  }
  if (ok) {
    float *o = out + ((int64_t)br * 16 + g * 4) * k + cb;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      __builtin_nontemporal_store(v4f{acc[0][v], acc[1][v], acc[2][v],
                                      acc[3][v]},
                                  reinterpret_cast<v4f *>(o + v * k));
  }
}

// Matrix-core kernel for any block size that is a multiple of 4 and any k,
// fp32 and bf16 (16 x 16 blocks with aligned operands take the two kernels
// above, whose blocks are wave-uniform).
//
// A block row's blocks side by side are a b x (blocks b) matrix, whose
// columns ("virtual k") are taken 16 at a time: lane group g of a wave holds
// virtual k 16 v + 4 g .. + 3 of step v, four columns of one block since b
// is a multiple of 4 -- so 4 x 4 blocks go four to a step, 8 x 8 two, and a
// 32 x 32 block takes two steps.  Each lane tracks its own (block, column)
// and loads that block's rhs rows itself, N = 16 bytes' worth of consecutive
// output columns each: one 128-bit load of an rhs row gives a lane its
// values for N interleaved 16-column tiles, as in the kernels above.  Output
// rows are taken MS 16-row strips at a time, which share those rhs loads; a
// workgroup owns one group of MS strips of one block row and 16 N columns,
// and its SPL waves split the steps (wave w takes w, w + SPL, ...), the
// partial tiles summed through LDS.  Steps past the block row's end load
// nothing and multiply zeros; D rows past b are not stored.
//
// It is bound by the rhs slabs' trips from L2 and the MALL.  2,048 block
// rows of 32 x 32 blocks (9.25 on average), bf16, 200 columns: 1966 us for
// the thread-per-output loop, 34.5 us here (242 MB of slabs, 7 TB/s).
//
// VEC: block values aligned to four elements, rhs and output to 16 bytes
// and k a multiple of N, so that every access is aligned and no lane's
// columns pass k.  Otherwise the same accesses are element-aligned, and a
// lane whose columns pass k reads on into the next row (columns of B are
// independent, and those past k are not stored); a step that could so read
// past the end of rhs (total elements) loads element by element.
template <typename T, typename TO, int MS, int N, int SPL, bool VEC>
__global__ __launch_bounds__(64 * SPL, 4) void bsr_mfma(
    const int32_t *__restrict__ bro, const int32_t *__restrict__ bcol,
    const T *__restrict__ bval, const T *__restrict__ rhs,
    TO *__restrict__ out, int64_t k, int32_t b, int32_t groups,
    int32_t strips, int64_t total) {
  constexpr bool kF32 = sizeof(T) == 4;
  using AV = std::conditional_t<kF32, v4f, v2u>; // four A values
  // N rhs values: a lane's columns, one per tile
  using BV = std::conditional_t<kF32, v4f, std::conditional_t<N == 8, v4u, v2u>>;
  __shared__ v4f red[SPL > 1 ? SPL - 1 : 1][MS][N][kWave];
  // (gridDim.x < 2^32 / 256)
  const uint32_t id = (uint32_t)xcd_contiguous(blockIdx.x, gridDim.x);
  const uint32_t vb = id / (uint32_t)strips;
  const int32_t br = (int32_t)(vb / (uint32_t)groups);
  const int32_t s0 = 16 * MS * (int32_t)(vb - (uint32_t)br * groups);
  const int sp = wave_in_group();
  const int l = lane_id(), i = l & 15, g = l >> 4;
  // column strips in x, fastest, so that a block row's strips share its blocks
  // and the rhs lines between them in one XCD's L2 (strips = 1: in y)
  const int64_t cb =
      ((int64_t)blockIdx.y + (id - vb * (uint32_t)strips)) * (16 * N) + N * i;
  const bool ok = cb < k;
  v4f acc[MS][N];
#pragma unroll
  for (int m = 0; m < MS; ++m)
#pragma unroll
    for (int t = 0; t < N; ++t)
      acc[m][t] = v4f{0.f, 0.f, 0.f, 0.f};
  const int32_t s = bro[br], n = bro[br + 1] - s;
  // the lane's first virtual k and the advance of SPL steps
  int32_t blk = (16 * sp + 4 * g) / b;
  int32_t r = 16 * sp + 4 * g - blk * b;
  const int32_t dblk = 16 * SPL / b, dr = 16 * SPL - dblk * b;
  // a step's operands: its A rows and the rhs rows of block column c
  // (zeros past the block row's end); moves the lane to the next step
  auto load = [&](int32_t c, AV (&a)[MS], BV (&q)[4])
      __attribute__((always_inline)) {
    const bool in = blk < n, live = ok && in;
#pragma unroll
    for (int m = 0; m < MS; ++m)
      a[m] = AV{};
#pragma unroll
    for (int st = 0; st < 4; ++st)
      q[st] = BV{};
    const int64_t at = ((int64_t)c * b + r) * k + cb;
    bool whole = true; // no lane's rhs loads pass the end of rhs
    if constexpr (!VEC)
      whole = __builtin_amdgcn_ballot_w64(live && at + 3 * k + N > total) == 0;
    if (in) {
      const T *ap = bval + (int64_t)(s + blk) * b * b + r;
#pragma unroll
      for (int m = 0; m < MS; ++m) {
        const T *av = ap + (int64_t)std::min(s0 + 16 * m + i, b - 1) * b;
        if constexpr (VEC)
          a[m] = ld_stream(reinterpret_cast<const AV *>(av));
        else
          __builtin_memcpy(&a[m], av, sizeof(AV));
      }
    }
    if (whole) { // wave-uniform
      if (live) {
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          if constexpr (VEC)
            q[st] = *reinterpret_cast<const BV *>(rhs + at + st * k);
          else
            __builtin_memcpy(&q[st], rhs + at + st * k, sizeof(BV));
        }
      }
    } else if (live) {
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        T x[N];
#pragma unroll
        for (int t = 0; t < N; ++t)
          x[t] = cb + t < k ? rhs[at + st * k + t] : T(0);
        __builtin_memcpy(&q[st], x, sizeof(BV));
      }
    }
    r += dr;
    blk += dblk;
    if (r >= b) {
      r -= b;
      ++blk;
    }
  };
  // a step's block column, loaded a step ahead
  auto column = [&](int32_t at) __attribute__((always_inline)) {
    return bcol[s + std::min(at, n - 1)];
  };
  auto products = [&](const AV (&a)[MS], const BV (&q)[4])
      __attribute__((always_inline)) {
    if constexpr (kF32) {
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int t = 0; t < N; ++t)
#pragma unroll
          for (int m = 0; m < MS; ++m)
            acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                a[m][st], q[st][t], acc[m][t], 0, 0, 0);
    } else {
#pragma unroll
      for (int t = 0; t < N; ++t) {
        // element t of the four rows, paired by byte permutes
        const int d = t >> 1;
        const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
        const v2u bt = v2u{__builtin_amdgcn_perm(q[1][d], q[0][d], sel),
                           __builtin_amdgcn_perm(q[3][d], q[2][d], sel)};
#pragma unroll
        for (int m = 0; m < MS; ++m)
          acc[m][t] = mfma_16x16x16_bf16(a[m], bt, acc[m][t]);
      }
    }
  };
  // this wave's steps (a loop that tested lane 0's block instead copied
  // every accumulator in each step; a step's operands requested a whole
  // step ahead, two buffers, measured no faster)
  const int64_t steps = ((int64_t)n * b + 15) / 16;
  const int32_t mine = (int32_t)((steps - sp + SPL - 1) / SPL);
  int32_t c = mine > 0 ? column(blk) : 0;
  for (int32_t t = 0; t < mine; ++t) {
    const int32_t next = column(blk + dblk + (r + dr >= b ? 1 : 0));
    AV a[MS];
    BV q[4];
    load(c, a, q);
    products(a, q);
    c = next;
  }
  // wave m % SPL sums and stores strip m
#pragma unroll
  for (int m = 0; m < MS; ++m)
    if (sp != m % SPL)
#pragma unroll
      for (int t = 0; t < N; ++t)
        red[sp < m % SPL ? sp : sp - 1][m][t][l] = acc[m][t];
  __syncthreads();
  if (!ok)
    return; // after the only barrier
#pragma unroll
  for (int m = 0; m < MS; ++m) {
    if (sp != m % SPL) // wave-uniform
      continue;
#pragma unroll
    for (int w = 0; w < SPL - 1; ++w)
#pragma unroll
      for (int t = 0; t < N; ++t)
        acc[m][t] += red[w][m][t][l];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int32_t row = s0 + 16 * m + 4 * g + v;
      if (row >= b)
        continue;
      TO *o = out + ((int64_t)br * b + row) * k + cb;
      if (VEC || cb + N <= k) {
        if constexpr (sizeof(TO) == 2) {
          uint32_t y[N / 2];
#pragma unroll
          for (int t = 0; t < N; t += 2)
            y[t / 2] = pack_bf16x2(acc[m][t][v], acc[m][t + 1][v]);
          BV z;
          __builtin_memcpy(&z, y, sizeof z);
          if constexpr (VEC)
            __builtin_nontemporal_store(z, reinterpret_cast<BV *>(o));
          else
            __builtin_memcpy(o, &z, sizeof z);
        } else {
#pragma unroll
          for (int t = 0; t < N; t += 4) {
            const v4f y = v4f{acc[m][t][v], acc[m][t + 1][v],
                              acc[m][t + 2][v], acc[m][t + 3][v]};
            if constexpr (VEC)
              st4_nt(o + t, y);
            else
              __builtin_memcpy(o + t, &y, sizeof y);
          }
        }
      } else {
#pragma unroll
        for (int t = 0; t < N; ++t)
          if (cb + t < k)
            stv(o + t, acc[m][t][v]);
      }
    }
  }
}

// fp32 x4 kernel shape: blocks per batch and waves per strip. Configuration
// 4, two strips per workgroup: 1 wave x 4-block batches 134.0 us, 2 x 2
// 127.5 us, 2 x 1 128.3 us, 2 x 4 144.2 us, 4 x 2 130.3 us, 4 x 1 124.0 us.
constexpr int kF32Batch = 1;
constexpr int kF32Split = 4;

int check_bsr(const int32_t *bro, const int32_t *bcol, const void *bval,
              const void *rhs, const void *out, int64_t rows, int64_t cols,
              int64_t nnzb, int64_t k, int64_t b) {
  if (b < 1)
    return sw::fail(SW_ERR_INVALID_SHAPE,
                    "BSR block size must be positive, but got %lld",
                    (long long)b);
  if (rows < 0 || cols < 0 || nnzb < 0 || k < 0)
    return sw::fail(SW_ERR_INVALID_SHAPE, "negative BSR shape");
  if (rows % b != 0 || cols % b != 0)
    return sw::fail(SW_ERR_INVALID_SHAPE,
                    "BSR matrix dimensions %lld x %lld must be divisible by "
                    "block size %lld",
                    (long long)rows, (long long)cols, (long long)b);
  if (nnzb * b * b > (int64_t)INT32_MAX * 16)
    return sw::fail(SW_ERR_INVALID_SHAPE, "too many BSR blocks");
  if (rows / b > INT32_MAX - 1)
    return sw::fail(SW_ERR_INVALID_SHAPE, "too many BSR block rows");
  if (!bro)
    return sw::fail(SW_ERR_INVALID_ARGUMENT, "block row offsets pointer is null");
  if (rows > 0 && k > 0 && !out)
    return sw::fail(SW_ERR_INVALID_ARGUMENT, "output pointer is null");
  if (nnzb > 0 && (!bcol || !bval || (k > 0 && !rhs)))
    return sw::fail(SW_ERR_INVALID_ARGUMENT, "BSR operand pointer is null");
  return SW_OK;
}

// bf16 x8 kernel shape: blocks per batch and waves per block row.
// Configuration 4 (bf16 output), one wave per block row: batches of
// 1 / 2 / 4 / 8 blocks 63.2 / 62.1 / 69.9 / 113.6 us (94 VGPRs at 2, 142 at
// 4); the block row split over waves: 2 waves x 2-block batches 60.8 us,
// 2 x 1 58.3 us, 4 x 1 56.6 us, 4 x 2 62.8 us, 8 x 1 98.2 us.
constexpr int kBf16Batch = 1;
constexpr int kBf16Split = 4;

// Few products per block row: thread-per-output is faster than a 16-row tile
// per block row, whose waves cost the same however little of it b and k fill.
// In products (b rows of k outputs of `entries` terms each, and about four
// terms' worth of addressing).  Sweeps over 131,072 and 524,288 rows, thread
// per output / bsr_mfma, us: fp32 4 x 4 blocks, one a block row, k = 1 9 / 101,
// k = 16 42 / 89, k = 32 84 / 88; six 31 / 143, 152 / 126 (k = 16); 8 x 8, one,
// k = 8 30 / 46, k = 16 57 / 47; 12 x 12, one, k = 4 20 / 32, k = 8 38 / 32;
// 20 x 20, one, k = 8 54 / 64, k = 16 104 / 65, three, k = 1 25 / 27.  bf16
// 4 x 4, one, k = 24 61 / 66, k = 32 78 / 66; 8 x 8, six, k = 2 36 / 55, k = 4
// 63 / 51; 12 x 12, six, k = 1 56 / 46; 20 x 20, one, k = 2 19 / 26, k = 4
// 24 / 23.  (16 x 16 blocks always take the matrix cores.)
template <typename T>
bool few_block_products(int64_t b, double entries, int64_t k) {
  const double products = (double)b * (double)k * (entries + 4.0);
  if (b == 16 || b >= 32)
    return false;
  if (sizeof(T) == 2)
    return products < 950.0;
  return b < 16 ? products < 1000.0 + 25.0 * entries
                : products < 4300.0 && entries <= 40.0;
}

template <typename T, typename TO>
int launch_bsr(const int32_t *bro, const int32_t *bcol, const T *bval,
               const T *rhs, TO *out, int64_t rows, int64_t cols, int64_t nnzb,
               int64_t k, int64_t b, const sw_options &o, hipStream_t st,
               bool mfma) {
  if (rows == 0 || k == 0)
    return SW_OK;
  mfma = mfma && !few_block_products<T>(
                     b, (double)nnzb * (double)(b * b) / (double)rows, k);
  const int nbr = (int)(rows / 16);
  // The matrix-core kernels' x must stay within one grid dimension's
  // 2^32 - 1 work-items; past it the thread-per-output kernel below, whose
  // launch folds, computes the product.
  const bool b16 = mfma && b == 16 && rows / 16 <= sw::grid_row(512) &&
                   (reinterpret_cast<uintptr_t>(bval) &
                    (4 * sizeof(T) - 1)) == 0;
  if (b16 && k > (int64_t)65535 * 128)
    return sw::fail(SW_ERR_INVALID_SHAPE, "rhs has too many columns");
  // The kernels for 16 x 16 blocks whose values are aligned to four elements
  // (they read A rows as 16-byte (fp32) or 8-byte (bf16) vectors) take 64 <
  // k <= 128; on both sides of that bsr_mfma is faster (us, fp32 k = 64
  // 68.9 against 66.0 us, k = 128 125.5 / 126.7, k = 256 289 / 266; bf16
  // k = 64 53 / 38, k = 128 57.4 / 55.6, k = 200 118 / 94: a narrow strip
  // leaves most of their lanes idle, and their strips of one block row lie
  // a whole grid apart)
  const bool mfma_ok = b16 && k > 64 && k <= 128;
  if constexpr (sizeof(T) == 4) {
    // fp32 with k % 4 == 0 takes the column-interleaved kernel
    if (mfma_ok && k % 4 == 0 && sw::aligned16(rhs) && sw::aligned16(out)) {
      hipLaunchKernelGGL((bsr16_mfma_f32_x4<kF32Batch, kF32Split>),
                         dim3((unsigned)nbr), dim3(64 * kF32Strips * kF32Split),
                         0, st, bro, bcol, bval, rhs, out, k, nbr);
      return sw::launch_check("BSR MFMA kernel");
    }
  } else {
    // k % 8 == 0: eight interleaved tiles per workgroup, 128-bit RHS loads
    if (mfma_ok && k % 8 == 0 && sw::aligned16(rhs) && sw::aligned16(out)) {
      hipLaunchKernelGGL((bsr16_mfma_bf16_x8<kBf16Batch, kBf16Split, TO>),
                         dim3((unsigned)nbr), dim3(64 * kBf16Split), 0, st, bro,
                         bcol, bval, rhs, out, k, nbr);
      return sw::launch_check("BSR MFMA kernel");
    }
  }
  // Every other shape with b a multiple of 4; a launch that one grid
  // dimension cannot hold takes the thread-per-output kernel below.  Sweeps
  // (us, mean blocks per block row in parentheses):
  // * bf16, waves per strip group 1 / 2 / 4: 32 x 32 blocks, 2,048 block
  //   rows (9.25), k = 200 41.1 / 34.5 / 40.2; k = 64 (columns per lane 4)
  //   20.7 / 15.4 / 17.8; 16 x 16, 16,384 block rows (8), k = 200 122.9 /
  //   93.7 / 97.0, k = 30 29.5 / 29.4 / 33.5.
  // * bf16, columns per lane 8 / 4: k = 61 44.2 / 38.6, k = 100 47.8 / 82.4
  //   (two strips): 4 where one strip of 64 columns holds k.
  // * fp32, 2 / 4 waves: 32 x 32, k = 200 137.7 / 127.2; 16 x 16, k = 256
  //   268.7 / 266.2; 8 x 8 (half the steps), k = 45 31.8 / 35.4.
  const int64_t N = sizeof(T) == 2 && k > 64 ? 8 : 4;
  const int64_t SPL = sizeof(T) == 2 || b < 16 ? 2 : 4;
  const int64_t gy = sw::ceil_div(k, 16 * N);
  const int64_t groups = sw::ceil_div(b, 32);
  const int64_t x = rows / b * groups, row = sw::grid_row(64 * SPL);
  if (mfma && b % 4 == 0 && b <= (1 << 24) && x <= row &&
      (gy <= 65535 || gy <= row / x)) {
    // one grid dimension where it holds them all
    const int64_t strips = gy <= row / x ? gy : 1;
    const bool vec = k % N == 0 && sw::aligned16(rhs) && sw::aligned16(out) &&
                     (reinterpret_cast<uintptr_t>(bval) &
                      (4 * sizeof(T) - 1)) == 0;
    const dim3 grid((unsigned)(x * strips), (unsigned)(gy / strips));
#define SW_BSR_ANY(MS, N, SPL)                                                \
  do {                                                                        \
    if (vec)                                                                  \
      hipLaunchKernelGGL((bsr_mfma<T, TO, MS, N, SPL, true>), grid,           \
                         dim3(64 * SPL), 0, st, bro, bcol, bval, rhs, out, k, \
                         (int32_t)b, (int32_t)groups, (int32_t)strips,        \
                         cols * k);                                           \
    else                                                                      \
      hipLaunchKernelGGL((bsr_mfma<T, TO, MS, N, SPL, false>), grid,          \
                         dim3(64 * SPL), 0, st, bro, bcol, bval, rhs, out, k, \
                         (int32_t)b, (int32_t)groups, (int32_t)strips,        \
                         cols * k);                                           \
  } while (0)
    if constexpr (sizeof(T) == 4) {
      if (b > 16)
        SW_BSR_ANY(2, 4, 4);
      else if (b == 16)
        SW_BSR_ANY(1, 4, 4);
      else
        SW_BSR_ANY(1, 4, 2);
    } else {
      if (b > 16 && N == 8)
        SW_BSR_ANY(2, 8, 2);
      else if (b > 16)
        SW_BSR_ANY(2, 4, 2);
      else if (N == 8)
        SW_BSR_ANY(1, 8, 2);
      else
        SW_BSR_ANY(1, 4, 2);
    }
#undef SW_BSR_ANY
    return sw::launch_check("BSR MFMA kernel");
  }
  const int64_t B = o.spmm_block_size;
  int64_t grid = std::max<int64_t>(sw::ceil_div(rows * k, B), 1);
  int rc = sw::check_grid(grid, B, "BSR SpMM");
  if (rc)
    return rc;
  const bool by_row = k % 64 == 0 && B % 64 == 0 && rows <= INT32_MAX;
#define SW_BSR_TPO(BS, ROW)                                                   \
  hipLaunchKernelGGL((bsr_thread_per_output<T, TO, BS, ROW>),                 \
                     sw::grid_dim(grid, B), dim3((unsigned)B), 0, st, bro,   \
                     bcol, bval, rhs, out, rows, k, (int32_t)b)
  if (b == 16 && by_row)
    SW_BSR_TPO(16, true);
  else if (b == 16)
    SW_BSR_TPO(16, false);
  else if (by_row)
    SW_BSR_TPO(0, true);
  else
    SW_BSR_TPO(0, false);
#undef SW_BSR_TPO
  return sw::launch_check("thread-per-output BSR SpMM kernel");
}

template <typename T, typename TO>
int bsr_entry(const int32_t *block_row_offsets,
              const int32_t *block_column_indices, const T *block_values,
              const T *rhs, TO *output, int64_t rows, int64_t cols,
              int64_t nnzb, int64_t k, int64_t block_size,
              const sw_options *opts, void *stream) {
  sw::clear_error();
  sw_options o;
  int rc = sw::resolve_options(opts, &o);
  if (rc)
    return rc;
  rc = check_bsr(block_row_offsets, block_column_indices, block_values, rhs,
                 output, rows, cols, nnzb, k, block_size);
  if (rc)
    return rc;
  rc = sw::check_value_alignment(sizeof(T), {block_values, rhs});
  if (!rc)
    rc = sw::check_value_alignment(sizeof(TO), {output});
  if (rc)
    return rc;
  return launch_bsr<T, TO>(block_row_offsets, block_column_indices,
                           block_values, rhs, output, rows, cols, nnzb, k,
                           block_size, o, sw::as_stream(stream),
                           o.bsr_use_mfma != 0);
}

// The slab floor: the MFMA kernel launch_bsr would run for these operands,
// in its FLOOR form.
template <typename T, typename TO>
int launch_slab_floor(const int32_t *bro, const int32_t *bcol, const T *bval,
                      const T *rhs, TO *out, int64_t rows, int64_t k,
                      hipStream_t st) {
  if (rows == 0 || k == 0)
    return SW_OK;
  const int nbr = (int)(rows / 16);
  if constexpr (sizeof(T) == 4) {
    const int64_t strips = std::min<int64_t>(kF32Strips, sw::ceil_div(k, 64));
    const int64_t gy = sw::ceil_div(k, 64 * strips);
    if (gy > 65535)
      return sw::fail(SW_ERR_INVALID_SHAPE, "rhs has too many columns");
    const int rc = sw::check_flat_grid(nbr, 64 * strips * kF32Split,
                                       "BSR slab floor kernel");
    if (rc)
      return rc;
    hipLaunchKernelGGL((bsr16_mfma_f32_x4<kF32Batch, kF32Split, true>),
                       dim3((unsigned)nbr, (unsigned)gy),
                       dim3((unsigned)(64 * strips * kF32Split)), 0, st, bro,
                       bcol, bval, rhs, out, k, nbr);
  } else {
    const int64_t gy = sw::ceil_div(k, 128);
    if (gy > 65535)
      return sw::fail(SW_ERR_INVALID_SHAPE, "rhs has too many columns");
    const int rc =
        sw::check_flat_grid(nbr, 64 * kBf16Split, "BSR slab floor kernel");
    if (rc)
      return rc;
    hipLaunchKernelGGL((bsr16_mfma_bf16_x8<kBf16Batch, kBf16Split, TO, true>),
                       dim3((unsigned)nbr, (unsigned)gy), dim3(64 * kBf16Split),
                       0, st, bro, bcol, bval, rhs, out, k, nbr);
  }
  return sw::launch_check("BSR slab floor kernel");
}

} // namespace

extern "C" int sw_bsr_slab_floor(const int32_t *block_row_offsets,
                                 const int32_t *block_column_indices,
                                 const void *block_values, const void *rhs,
                                 void *output, int64_t rows, int64_t cols,
                                 int64_t nnzb, int64_t k, int value_bytes,
                                 int output_bytes, void *stream) {
  sw::clear_error();
  int rc = check_bsr(block_row_offsets, block_column_indices, block_values,
                     rhs, output, rows, cols, nnzb, k, 16);
  if (rc)
    return rc;
  const bool f32 = value_bytes == 4 && output_bytes == 4;
  const bool b16 = value_bytes == 2 && (output_bytes == 2 || output_bytes == 4);
  if (!f32 && !b16)
    return sw::fail(SW_ERR_INVALID_ARGUMENT,
                    "slab floor value / output bytes must be 4 / 4, 2 / 2 or "
                    "2 / 4, but got %d / %d", value_bytes, output_bytes);
  // the floor runs where the MFMA kernels run: 16-byte aligned rhs and
  // output, block values aligned to four elements, k % 4 (fp32) or k % 8
  const uintptr_t va = reinterpret_cast<uintptr_t>(block_values);
  if (k % (f32 ? 4 : 8) != 0 || !sw::aligned16(rhs) ||
      !sw::aligned16(output) || (va & (4u * value_bytes - 1)) != 0)
    return sw::fail(SW_ERR_INVALID_ARGUMENT,
                    "the slab floor needs the MFMA kernels' shapes: k a "
                    "multiple of %d, 16-byte aligned rhs and output, block "
                    "values aligned to %d bytes", f32 ? 4 : 8,
                    4 * value_bytes);
  hipStream_t st = sw::as_stream(stream);
  if (f32)
    return launch_slab_floor<float, float>(
        block_row_offsets, block_column_indices,
        static_cast<const float *>(block_values),
        static_cast<const float *>(rhs), static_cast<float *>(output), rows,
        k, st);
  if (output_bytes == 2)
    return launch_slab_floor<uint16_t, uint16_t>(
        block_row_offsets, block_column_indices,
        static_cast<const uint16_t *>(block_values),
        static_cast<const uint16_t *>(rhs), static_cast<uint16_t *>(output),
        rows, k, st);
  return launch_slab_floor<uint16_t, float>(
      block_row_offsets, block_column_indices,
      static_cast<const uint16_t *>(block_values),
      static_cast<const uint16_t *>(rhs), static_cast<float *>(output), rows,
      k, st);
}

extern "C" int sw_bsr_spmm_f32(const int32_t *block_row_offsets,
                               const int32_t *block_column_indices,
                               const float *block_values, const float *rhs,
                               float *output, int64_t rows, int64_t cols,
                               int64_t nnzb, int64_t k, int64_t block_size,
                               const sw_options *opts, void *stream) {
  return bsr_entry<float, float>(block_row_offsets, block_column_indices,
                                 block_values, rhs, output, rows, cols, nnzb,
                                 k, block_size, opts, stream);
}

extern "C" int sw_bsr_spmm_bf16(const int32_t *block_row_offsets,
                                const int32_t *block_column_indices,
                                const uint16_t *block_values,
                                const uint16_t *rhs, uint16_t *output,
                                int64_t rows, int64_t cols, int64_t nnzb,
                                int64_t k, int64_t block_size,
                                const sw_options *opts, void *stream) {
  return bsr_entry<uint16_t, uint16_t>(block_row_offsets,
                                       block_column_indices, block_values, rhs,
                                       output, rows, cols, nnzb, k, block_size,
                                       opts, stream);
}

extern "C" int sw_bsr_spmm_bf16_f32out(const int32_t *block_row_offsets,
                                       const int32_t *block_column_indices,
                                       const uint16_t *block_values,
                                       const uint16_t *rhs, float *output,
                                       int64_t rows, int64_t cols,
                                       int64_t nnzb, int64_t k,
                                       int64_t block_size,
                                       const sw_options *opts, void *stream) {
  return bsr_entry<uint16_t, float>(block_row_offsets, block_column_indices,
                                    block_values, rhs, output, rows, cols,
                                    nnzb, k, block_size, opts, stream);
}
