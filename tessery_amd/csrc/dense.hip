// fp32 dense projections and elementwise kernels of tessery's BERT (BGE) layer on gfx950.
//
// matmul_f32<BIAS>: out[r][n] = sum_k a[r][k] * bt[n][k] (+ bias[n]) for rows [row0, row1), any
// K and N: the matmul_f32 / matmul_f32_tiled / matmul_f32_chunk32 / matmul_bias_f32 /
// matmul_bias_f32_chunk32 routes (kernels.metal:306-322, 396-487). Weights stay [N, K] as in the
// reference ("transposed weight"). Products accumulate in K32 partial sums added to the total
// (the chunk32 order, kernels.metal:416-436), and the bias is added once after the last one. Every
// route runs the same kernels: matmul_planes and matmul_x3 on bf16 MFMA where K % 32 == 0 (below),
// matmul_f32 for the rest.
// add_bias, gelu_f32 and layer_norm follow kernels.metal:362-394.
#include <algorithm>

#include "common.h"
#include "kernels.h"
#include "lds_dma.h"

namespace tessery {

// 256 threads = 4 wavefronts; tile 64 rows x 128 columns: wavefront w owns columns 32w..32w+31
// of both 32-row halves, so every weight it loads feeds two 32x32 MFMA tiles. The K loop walks
// 64 columns at a time. v_mfma_f32_32x32x2_f32 with lane (column n = l%32, k-slot h = l/32):
// k-step t of a 32-wide half pairs k = 32h + t, so each lane holds 32 consecutive weights of its
// row per 64-column chunk. Columns past K and rows / weight rows past their ends read as zero.
constexpr int kDenseRows = 64;

// erf-form GELU, x * (1 + erf(x / sqrt 2)) / 2, with erf by Abramowitz & Stegun 7.1.26 (absolute
// error below 1.5e-7), the approximation tessery's kernel uses (kernels.metal:381-394). The
// gelu_f32 route and the fused projection epilogue share it, so both give the same bits.
__device__ __forceinline__ float gelu_value(float value) {
  const float z = fabsf(value) * 0.70710678118654752f;
  const float t = 1.0f / (1.0f + 0.3275911f * z);
  const float poly =
      ((((1.061405429f * t - 1.453152027f) * t + 1.421413741f) * t - 0.284496736f) * t +
       0.254829592f) * t;
  const float tail = poly * expf(-z * z);  // 1 - erf(z)
  return 0.5f * value * (value < 0.0f ? tail : 2.0f - tail);
}

// x . w over k inputs as fp32 products: for a result of the split-operand kernels that isn't finite. An
// infinite operand splits into NaN terms there, and a finite sum may overflow on its way.
__device__ __forceinline__ float fp32_dot(const float* x, const float* w, int k) {
  float y = 0.0f;
  for (int i = 0; i < k; i += 32) {
    float part = 0.0f;
    for (int j = i; j < min(i + 32, k); ++j) part = fmaf(x[j], w[j], part);
    y += part;
  }
  return y;
}
__device__ __forceinline__ bool is_finite(float y) { return fabsf(y) <= 3.402823466e38f; }

// PARTIAL: workgroup z sums chunks [z * per, (z + 1) * per) only and stores its raw sums to
// out + z * (row1 - row0) * cols (rows relative to row0), for dense_reduce to add in z order.
template <bool BIAS, bool GELU, bool PARTIAL>
__global__ __launch_bounds__(256) void matmul_f32(const float* __restrict__ a,
                                                  const float* __restrict__ bt,
                                                  const float* __restrict__ bias,
                                                  float* __restrict__ out, int row0, int row1,
                                                  int cols, int k, int per) {
  constexpr int XROW = 64 + 4;
  __shared__ __attribute__((aligned(16))) float xs[kDenseRows * XROW];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int rbase = row0 + blockIdx.x * kDenseRows;
  const int n = blockIdx.y * 128 + wave * 32 + l32;
  const bool nvalid = n < cols;
  const bool vec = (k & 3) == 0;  // rows start 16-byte aligned: float4 loads
  const int all_chunks = (k + 63) / 64;
  const int c_begin = PARTIAL ? static_cast<int>(blockIdx.z) * per : 0;
  const int c_end = PARTIAL ? min(c_begin + per, all_chunks) : all_chunks;
  floatx16 acc[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[rt][e] = 0.0f;
  // x chunks are loaded into registers one chunk ahead and written to LDS after the barrier that
  // retires the previous chunk's reads; the lane's weights are loaded before that barrier
  constexpr int XV = kDenseRows * 16 / 256;  // four-float x pieces per thread per chunk
  floatx4 xr[XV];
  auto load_x = [&](int k0) {
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int c = tid + 256 * i;  // four-float pieces: 64 rows x 16
      const int r = c / 16, kk = k0 + 4 * (c % 16);
      floatx4 t = {0.f, 0.f, 0.f, 0.f};
      if (rbase + r < row1 && kk < k) {
        const float* src = a + static_cast<size_t>(rbase + r) * k + kk;
        if (vec && kk + 4 <= k) {
          t = *reinterpret_cast<const floatx4*>(src);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) t[j] = kk + j < k ? src[j] : 0.0f;
        }
      }
      xr[i] = t;
    }
  };
  load_x(c_begin * 64);
  for (int ci = c_begin; ci < c_end; ++ci) {
    const int k0 = ci * 64;
    float wv[32];
    {
      const int kw = k0 + 32 * hh;
      const float* src = bt + static_cast<size_t>(n) * k + kw;
      if (nvalid && vec && kw + 32 <= k) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const floatx4 t = *reinterpret_cast<const floatx4*>(src + 4 * j);
          wv[4 * j] = t[0];
          wv[4 * j + 1] = t[1];
          wv[4 * j + 2] = t[2];
          wv[4 * j + 3] = t[3];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 32; ++j) wv[j] = nvalid && kw + j < k ? src[j] : 0.0f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int c = tid + 256 * i;
      *reinterpret_cast<floatx4*>(&xs[(c / 16) * XROW + 4 * (c % 16)]) = xr[i];
    }
    __syncthreads();
    if (ci + 1 < c_end) load_x(k0 + 64);
    // K32 partial sums per 32-row tile, each added to its total (the chunk32 order)
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        floatx16 part;
#pragma unroll
        for (int e = 0; e < 16; ++e) part[e] = 0.0f;
#pragma unroll
        for (int c4 = 4 * half; c4 < 4 * half + 4; ++c4) {
          const floatx4 xa =
              *reinterpret_cast<const floatx4*>(&xs[(32 * rt + l32) * XROW + 32 * hh + 4 * c4]);
#pragma unroll
          for (int t = 0; t < 4; ++t)
            part = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[t], wv[4 * c4 + t], part, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[rt][e] += part[e];
      }
  }
  if (!nvalid) return;
  const float b = BIAS ? bias[n] : 0.0f;
  // rows of a partial are counted from row0
  float* const dst = PARTIAL ? out + static_cast<size_t>(blockIdx.z) * (row1 - row0) * cols : out;
  const int rfirst = PARTIAL ? row0 : 0;
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int r = rbase + 32 * rt + 8 * (e >> 2) + 4 * hh + (e & 3);
      if (r < row1) {
        const size_t at = static_cast<size_t>(r - rfirst) * cols + n;
        if constexpr (PARTIAL) {
          dst[at] = acc[rt][e];
        } else {
          const float y = BIAS ? acc[rt][e] + b : acc[rt][e];
          dst[at] = GELU ? gelu_value(y) : y;
        }
      }
    }
}

// matmul_x3<BIAS, GELU>: the same product on bf16 MFMA (K % 32 == 0, N % 128 == 0): a and bt are
// split exactly into three bf16 planes each (split3x8) and every fp32 product is taken as the six
// terms b_i c_j with i + j <= 4, or (EXACT) the eight with i + j <= 5, on v_mfma_f32_32x32x16_bf16
// in fp32 (the bf16 rate is 16x the fp32 one, so six products cost well under half the fp32
// instructions; what they leave out is at most 2^-21 of the product, eight 2^-30, and EXACT sums
// the leading products apart from the others, so that only they round at the magnitude of the
// result). Tile 64 rows x 128 columns; wavefront w owns rows 32 (w >> 1) .. +31 and columns 64 (w &
// 1) .. +63 (two 32x32 tiles). Per 32-wide K chunk every thread loads 8 floats of one x row and 16
// of one weight row into registers (one chunk ahead), splits them after the barrier that retires
// the previous chunk's reads, and stores the three planes to LDS as rows of 64 bytes (four 16-byte
// chunks, chunk c of row r at c ^ ((r >> 1) & 3): conflict-free for the 16-lane reads and the
// 8-lane writes on gfx950). As in matmul_f32, each 32-wide chunk's products form a partial sum
// added to the total (the chunk32 order), and the bias and GELU are applied the same way. Rows past
// row1 read row0 and are never stored.
constexpr int kX3Rows = 64;

__device__ __forceinline__ int x3sw(int row) { return (row >> 1) & 3; }

// PARTIAL: as in matmul_f32, workgroup z sums K chunks [z * per, (z + 1) * per) (of 32 here) and
// stores its raw sums for dense_reduce.
template <bool BIAS, bool GELU, bool PARTIAL, bool EXACT>
__global__ __launch_bounds__(256, 3) void matmul_x3(const float* __restrict__ a,
                                                   const float* __restrict__ bt,
                                                   const float* __restrict__ bias,
                                                   float* __restrict__ out, int row0, int row1,
                                                   int cols, int k, int per) {
  __shared__ __attribute__((aligned(16))) uint16_t as[3][kX3Rows * 32];
  __shared__ __attribute__((aligned(16))) uint16_t bs[3][128 * 32];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wr = wave >> 1, wc = wave & 1;
  const int rbase = row0 + blockIdx.x * kX3Rows;
  const int nbase = blockIdx.y * 128;
  // load roles: x row tid / 4, floats 8 (tid % 4) .. +7 of the chunk; weight row tid / 2,
  // floats 16 (tid % 2) .. +15
  const int arow = tid >> 2, apart = tid & 3;
  const int brow = tid >> 1, bpart = tid & 1;
  const int agrow = rbase + arow < row1 ? rbase + arow : row0;
  const float* const asrc = a + static_cast<size_t>(agrow) * k + 8 * apart;
  const float* const bsrc = bt + static_cast<size_t>(nbase + brow) * k + 16 * bpart;
  floatx4 ar[2], br[4];
  auto load = [&](int k0) {
    ar[0] = *reinterpret_cast<const floatx4*>(asrc + k0);
    ar[1] = *reinterpret_cast<const floatx4*>(asrc + k0 + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) br[j] = *reinterpret_cast<const floatx4*>(bsrc + k0 + 4 * j);
  };
  const int aslot = arow * 32 + 8 * (apart ^ x3sw(arow));
  const int bslot0 = brow * 32 + 8 * ((2 * bpart) ^ x3sw(brow));
  const int bslot1 = brow * 32 + 8 * ((2 * bpart + 1) ^ x3sw(brow));
  // operand rows of this lane: x row 32 wr + l32, weight rows 64 wc + 32 j + l32
  const int orow = 32 * wr + l32;
  floatx16 acc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;
  const int k_begin = PARTIAL ? static_cast<int>(blockIdx.z) * per * 32 : 0;
  const int k_end = PARTIAL ? min(k_begin + per * 32, k) : k;
  load(k_begin);
  for (int k0 = k_begin; k0 < k_end; k0 += 32) {
    {
      uint4v p1, p2, p3;
      split3x8(ar[0], ar[1], p1, p2, p3);
      *reinterpret_cast<uint4v*>(&as[0][aslot]) = p1;
      *reinterpret_cast<uint4v*>(&as[1][aslot]) = p2;
      *reinterpret_cast<uint4v*>(&as[2][aslot]) = p3;
      split3x8(br[0], br[1], p1, p2, p3);
      *reinterpret_cast<uint4v*>(&bs[0][bslot0]) = p1;
      *reinterpret_cast<uint4v*>(&bs[1][bslot0]) = p2;
      *reinterpret_cast<uint4v*>(&bs[2][bslot0]) = p3;
      split3x8(br[2], br[3], p1, p2, p3);
      *reinterpret_cast<uint4v*>(&bs[0][bslot1]) = p1;
      *reinterpret_cast<uint4v*>(&bs[1][bslot1]) = p2;
      *reinterpret_cast<uint4v*>(&bs[2][bslot1]) = p3;
    }
    __syncthreads();  // this chunk's planes are in LDS
    if (k0 + 32 < k_end) load(k0 + 32);
    // the chunk's 32-wide partial sum of each tile, then added to its total (the chunk32 order)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int wrow = 64 * wc + 32 * j + l32;
      floatx16 c, lo;  // lo: with EXACT, all but the leading products
#pragma unroll
      for (int e = 0; e < 16; ++e) c[e] = lo[e] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int chunk = 2 * ks + hh;
        const int ao = orow * 32 + 8 * (chunk ^ x3sw(orow));
        const int bo = wrow * 32 + 8 * (chunk ^ x3sw(wrow));
        const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(&as[0][ao]);
        const bf16x8 a2 = *reinterpret_cast<const bf16x8*>(&as[1][ao]);
        const bf16x8 a3 = *reinterpret_cast<const bf16x8*>(&as[2][ao]);
        const bf16x8 b1 = *reinterpret_cast<const bf16x8*>(&bs[0][bo]);
        const bf16x8 b2 = *reinterpret_cast<const bf16x8*>(&bs[1][bo]);
        const bf16x8 b3 = *reinterpret_cast<const bf16x8*>(&bs[2][bo]);
        floatx16& l = EXACT ? lo : c;
        if constexpr (EXACT) {
          l = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a3, b2, l, 0, 0, 0);
          l = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2, b3, l, 0, 0, 0);
        }
        l = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a3, b1, l, 0, 0, 0);
        l = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2, b2, l, 0, 0, 0);
        l = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b3, l, 0, 0, 0);
        l = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2, b1, l, 0, 0, 0);
        l = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b2, l, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b1, c, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] += EXACT ? c[e] + lo[e] : c[e];
    }
    __syncthreads();  // every wavefront has read this chunk's planes
  }
  // rows of a partial are counted from row0
  float* const dst = PARTIAL ? out + static_cast<size_t>(blockIdx.z) * (row1 - row0) * cols : out;
  const int rfirst = PARTIAL ? row0 : 0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = nbase + 64 * wc + 32 * j + l32;
    const float b = BIAS ? bias[n] : 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int r = rbase + 32 * wr + 8 * (e >> 2) + 4 * hh + (e & 3);
      if (r < row1) {
        const size_t at = static_cast<size_t>(r - rfirst) * cols + n;
        if constexpr (PARTIAL) {
          dst[at] = acc[j][e];
        } else {
          const float y = BIAS ? acc[j][e] + b : acc[j][e];
          dst[at] = GELU ? gelu_value(y) : y;
        }
      }
    }
  }
}

// ---- the same product with operands split beforehand (K % 32 == 0, K <= 512) ----
//
// split_dense makes the three bf16 terms of x and of the weights once, laid out as MFMA operands, for
// all the projections of one x in one launch:
// [row tile of 32][k-step of 16][term][lane][8], lane = row % 32 + 32 h holding inputs
// 16 step + 8 h .. + 7. matmul_planes then only copies operands to LDS (global_load_lds_dwordx4:
// whole KiB pieces, read back by lane, no bank conflicts) and multiplies, all of K in one workgroup:
// no partial sums, and q, k and v in one launch. Measured, q, k and v of 1024 rows of 384: 19.3 us,
// 47.5 as three split-K launches with their reductions; of 4096: 36.8 us, 72.0 on matmul_x3.
//
// Eight products (EXACT), all but that of the two smallest terms (below 2^-30 of the whole): nothing
// is lost against fp32 products. Shapes that matmul_x3 would take on six products, K split, take six
// here too (eight cost a forward of 4096 tokens 3%). K order: two halves, each with its leading
// products in one sum and the smaller ones in another (only the leading ones round at the magnitude
// of the result), added at the end. It is the same for every tile shape, so a row's bits depend on
// no projection beside it.
constexpr int kDenseStep = 3 * 64 * 8;  // bf16 words of a row tile's k-step

struct SplitArgs {
  const float* src[4];  // x, then up to three weight matrices, rows of k floats
  int row0[4], rows[4], tiles[4];
  int count, k;
  uint16_t* planes;  // the operands' planes, one after the other
};

// A workgroup splits 32 rows x 64 inputs of one operand: thread (row tid / 8, chunk tid % 8) 8 of
// them. Rows past the last one repeat it.
__global__ __launch_bounds__(256) void split_dense(SplitArgs a) {
  int tile = blockIdx.x, which = 0;
  size_t base = 0;
  while (which + 1 < a.count && tile >= a.tiles[which]) {
    tile -= a.tiles[which];
    base += a.tiles[which];
    ++which;
  }
  const int row = threadIdx.x >> 3, c = threadIdx.x & 7, kk = 64 * blockIdx.y + 8 * c;
  if (kk >= a.k) return;
  const int at = min(32 * tile + row, a.rows[which] - 1);
  const float* const src = a.src[which] + static_cast<size_t>(a.row0[which] + at) * a.k + kk;
  const floatx4 u = *reinterpret_cast<const floatx4*>(src);
  const floatx4 v = *reinterpret_cast<const floatx4*>(src + 4);
  uint4v t[3];
  split3x8(u, v, t[0], t[1], t[2]);
  uint16_t* const dst = a.planes + ((base + tile) * (a.k >> 4) + (kk >> 4)) * kDenseStep +
                        (row + 32 * (c & 1)) * 8;
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4v*>(dst + i * 512) = t[i];
}

struct PlanesSet {
  const float* bt;    // the weights as they came
  const float* bias;  // null: none
  float* out;
  int cols;
  int tile0;  // first 32-column tile of its weights
};
struct PlanesArgs {
  const uint16_t* x;
  const uint16_t* w;
  const float* a;  // the inputs as they came
  PlanesSet set[3];
  int count, row0, row1, k;
};

// The outputs of a 32 x 32 tile at `row`, `col` of set `which`, from the sums over the halves of K.
template <bool GELU>
__device__ __forceinline__ void store_halves(const PlanesArgs& a, int which, int row, int col,
                                             const floatx16& first, const floatx16& second) {
  const PlanesSet set = a.set[which];
  const int lane = threadIdx.x & 63, hh = lane >> 5;
  col += lane & 31;
  if (col >= set.cols) return;
  const float bias = set.bias ? set.bias[col] : 0.0f;
  auto row_of = [&](int e) { return row + 8 * (e >> 2) + 4 * hh + (e & 3); };
  auto store = [&](int r, float y) {
    if (set.bias) y += bias;
    set.out[static_cast<size_t>(r) * set.cols + col] = GELU ? gelu_value(y) : y;
  };
  uint32_t again = 0;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const float y = first[e] + second[e];
    if (row_of(e) >= a.row1) continue;
    store(row_of(e), y);
    again |= is_finite(y) ? 0u : 1u << e;
  }
  for (; again; again &= again - 1) {
    const int r = row_of(__builtin_ctz(again));
    store(r, fp32_dot(a.a + static_cast<size_t>(r) * a.k, set.bt + static_cast<size_t>(col) * a.k,
                      a.k));
  }
}

// The products of two operands' terms that are taken: the smaller ones, then the leading one.
template <bool EXACT>
struct Terms;
template <>
struct Terms<true> {
  static constexpr int n = 8, at[8][2] = {{2, 0}, {1, 1}, {2, 1}, {0, 2},
                                          {1, 2}, {1, 0}, {0, 1}, {0, 0}};
};
template <>
struct Terms<false> {
  static constexpr int n = 6, at[6][2] = {{2, 0}, {1, 1}, {0, 2}, {1, 0}, {0, 1}, {0, 0}};
};

// Tile 64 x 64, 4 wavefronts of 32 x 32 each. Two LDS stages of a 32-input chunk. While a chunk's
// products run, its wavefront reads the operands of the next one from LDS and copies those of the
// one after, one instruction between two products (issued together they cost as much as the
// products). Bound: L2 (13 TB/s for q, k and v of 4096 rows). Tiles of 64 x 128 and 128 x 128, which
// ask it for less, or more stages leave too few wavefronts on a CU to hide a chunk's latency: 16384 x
// 1152 outputs 97 and 194 us, 130 with three stages, against 94. Workgroups are numbered so that
// an XCD takes all columns of a row tile in turn, from its own L2.
template <bool GELU, bool EXACT>
__global__ __launch_bounds__(256, 3) void matmul_planes(PlanesArgs a, int row_tiles,
                                                        int col_tiles) {
  using T = Terms<EXACT>;
  constexpr int STAGE = 24 * 512;  // bf16 words: 12 KiB of x, then 12 KiB of weights
  constexpr int COPIES = 6, READS = 12;
  __shared__ __attribute__((aligned(1024))) uint16_t mem[2 * STAGE];
  const int block = blockIdx.x, turn = block >> 3;
  const int rt = (block & 7) + 8 * (turn / col_tiles);
  if (rt >= row_tiles) return;
  int ct = turn % col_tiles, which = 0;
  while (which + 1 < a.count && ct >= (a.set[which].cols + 63) / 64) {
    ct -= (a.set[which].cols + 63) / 64;
    ++which;
  }
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wr = wave >> 1, wc = wave & 1;
  const int ksteps = a.k >> 4, chunks = a.k >> 5, half = chunks >> 1;
  // A wavefront copies the 6 KiB of one operand tile: row tiles 0 and 1, column tiles 0 and 1.
  // Row tiles past the last one read it again (their rows aren't stored).
  const int last = (a.row1 - a.row0 - 1) >> 5;
  const int from = wave < 2 ? min(2 * rt + wave, last) : a.set[which].tile0 + 2 * ct + wave - 2;
  const uint16_t* const src =
      (wave < 2 ? a.x : a.w) + static_cast<size_t>(from) * ksteps * kDenseStep;
  auto copy = [&](int i, int buf, int chunk) {
    dma16_at(src + static_cast<size_t>(chunk) * (2 * kDenseStep) + i * 512, 16u * lane,
             reinterpret_cast<_Float16*>(mem + buf * STAGE + (6 * wave + i) * 512));
  };
  struct Operands {
    bf16x8 x[2][3], y[2][3];
  };
  // read i of a chunk's operands, in the order the products need them: terms (2, 0), (1, 1), (0, 2)
  auto read = [&](Operands& f, int i, int buf) {
    const uint16_t* const at = mem + buf * STAGE + lane * 8;
    const int t = i / 4, ks = (i >> 1) & 1;
    if (i & 1)
      f.y[ks][t] = *reinterpret_cast<const bf16x8*>(at + ((2 + wc) * 6 + ks * 3 + t) * 512);
    else
      f.x[ks][2 - t] = *reinterpret_cast<const bf16x8*>(at + (wr * 6 + ks * 3 + 2 - t) * 512);
  };

  floatx16 hi, lo, first;
#pragma unroll
  for (int e = 0; e < 16; ++e) hi[e] = lo[e] = first[e] = 0.0f;
  Operands even, odd;
#pragma unroll
  for (int i = 0; i < COPIES; ++i) copy(i, 0, 0);
  wait_vmcnt<0>();
  stage_barrier();
  if (chunks > 1) {
#pragma unroll
    for (int i = 0; i < COPIES; ++i) copy(i, 1, 1);
  }
#pragma unroll
  for (int i = 0; i < READS; ++i) read(even, i, 0);
  // chunk `step` from `now`; `next` takes the one after
  auto chunk = [&](int step, int buf, const Operands& now, Operands& next) {
    // the next chunk's copy has landed, and every wavefront has read this one's stage
    wait_vmcnt<0>();
    wait_lgkmcnt<0>();
    stage_barrier();
    const bool more = step + 2 < chunks;
#pragma unroll
    for (int i = 0; i < 2 * T::n; ++i) {
      const int ks = i & 1, t = i >> 1;
      floatx16& c = t < T::n - 1 ? lo : hi;
      c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(now.x[ks][T::at[t][0]], now.y[ks][T::at[t][1]], c,
                                                  0, 0, 0);
      if (i < READS) read(next, i, buf ^ 1);  // stale data after the last chunk, unused
      if (more && i < 2 * COPIES && (i & 1)) copy(i >> 1, buf, step + 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (step + 1 == half) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        first[e] = hi[e] + lo[e];
        hi[e] = lo[e] = 0.0f;
      }
    }
  };
  for (int step = 0; step < chunks; step += 2) {
    chunk(step, 0, even, odd);
    if (step + 1 < chunks) chunk(step + 1, 1, odd, even);
  }
  floatx16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = hi[e] + lo[e];
  wait_lgkmcnt<0>();  // the last chunk's reads ahead have landed before the kernel ends
  store_halves<GELU>(a, which, a.row0 + rt * 64 + 32 * wr, ct * 64 + 32 * wc, first, acc);
}

// The same for few tiles, with the same bits, straight from the operands as they came. A workgroup makes
// a tile of 32 x 32, a wavefront one half of K; each splits the operands of the next chunk in
// registers beside the products of this one, loaded a chunk before. Bound: the latency of that chain
// (deeper loads ahead only lengthen its start: 9.1 us for 24 to 656 rows of 384 x 384 with four chunks
// ahead, 8.3 with two, 9.4 with splits and products in turn). Per launch, against the pass that splits
// and matmul_planes, and matmul_f32 with its reduction: 24 x 384 outputs of K = 384 7.7, 11.6 and 8.8
// us, 128 x 1536 8.3, 16.3 and 11.3, 64 x 512 of K = 512 9.1, 14.5 and 10.3; q, k and v of 128 rows
// 8.5, 15.2 and 29.4.
template <bool GELU, bool EXACT>
__global__ __launch_bounds__(128) void matmul_direct(PlanesArgs a) {
  using T = Terms<EXACT>;
  constexpr int DEPTH = 2;  // chunks loaded ahead
  __shared__ __attribute__((aligned(16))) float sums[4 * 64 * 4];
  int ct = blockIdx.y, which = 0;
  while (which + 1 < a.count && ct >= (a.set[which].cols + 31) / 32) {
    ct -= (a.set[which].cols + 31) / 32;
    ++which;
  }
  const int tid = threadIdx.x, half = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5, k = a.k;
  const int row = a.row0 + 32 * static_cast<int>(blockIdx.x), chunks = k >> 5;
  const int begin = half ? chunks >> 1 : 0, end = half ? chunks : chunks >> 1;
  // rows and columns past the last one repeat it (they aren't stored)
  const float* const x = a.a + static_cast<size_t>(min(row + l32, a.row1 - 1)) * k + 8 * hh;
  const float* const w =
      a.set[which].bt + static_cast<size_t>(min(32 * ct + l32, a.set[which].cols - 1)) * k + 8 * hh;

  struct Chunk {
    floatx4 x[2][2], w[2][2];
  };
  auto load = [&](Chunk& c, int at) {
    const int from = 32 * min(at, end - 1);  // past the last one it again, unused
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        c.x[ks][i] = *reinterpret_cast<const floatx4*>(x + from + 16 * ks + 4 * i);
        c.w[ks][i] = *reinterpret_cast<const floatx4*>(w + from + 16 * ks + 4 * i);
      }
  };
  floatx16 hi, lo;
#pragma unroll
  for (int e = 0; e < 16; ++e) hi[e] = lo[e] = 0.0f;
  struct Operands {
    bf16x8 x[2][3], w[2][3];
  };
  auto split = [&](Operands& o, const Chunk& c) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      uint4v t[3];
      split3x8(c.x[ks][0], c.x[ks][1], t[0], t[1], t[2]);
#pragma unroll
      for (int i = 0; i < 3; ++i) o.x[ks][i] = __builtin_bit_cast(bf16x8, t[i]);
      split3x8(c.w[ks][0], c.w[ks][1], t[0], t[1], t[2]);
#pragma unroll
      for (int i = 0; i < 3; ++i) o.w[ks][i] = __builtin_bit_cast(bf16x8, t[i]);
    }
  };
  auto multiply = [&](const Operands& o) {
#pragma unroll
    for (int i = 0; i < 2 * T::n; ++i) {
      const int ks = i & 1, t = i >> 1;
      floatx16& sum = t < T::n - 1 ? lo : hi;
      sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(o.x[ks][T::at[t][0]], o.w[ks][T::at[t][1]], sum,
                                                    0, 0, 0);
    }
  };
  if (begin < end) {
    Chunk ring[DEPTH];
    Operands now[2];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) load(ring[i], begin + i);
    split(now[0], ring[0]);
    for (int at = begin; at < end; at += DEPTH) {
#pragma unroll
      for (int i = 0; i < DEPTH; ++i) {
        if (at + i >= end) break;
        load(ring[i], at + i + DEPTH);
        __builtin_amdgcn_sched_barrier(0);
        multiply(now[i & 1]);
        split(now[(i + 1) & 1], ring[(i + 1) % DEPTH]);
#pragma unroll
        for (int m = 0; m < 2 * T::n; ++m) {  // an MFMA, then the splitting that fits beside it
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, 176 / (2 * T::n), 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  floatx16 acc, second;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = hi[e] + lo[e];
  floatx4* const at = reinterpret_cast<floatx4*>(sums) + lane;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (half) at[q * 64] = floatx4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  __syncthreads();
  if (half) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const floatx4 s = at[q * 64];
#pragma unroll
    for (int j = 0; j < 4; ++j) second[4 * q + j] = s[j];
  }
  store_halves<GELU>(a, which, row, 32 * ct, acc, second);
}

// Split-K epilogue: out[r][n] = sum over z in order of part[z][r - row0][n] (+ bias, GELU). With a (split
// operands): a result that isn't finite is made again from rows of a and bt.
template <bool BIAS, bool GELU>
__global__ __launch_bounds__(256) void dense_reduce(const float* __restrict__ part,
                                                    const float* __restrict__ bias,
                                                    float* __restrict__ out, int row0, int rows,
                                                    int cols, int splits, const float* a,
                                                    const float* bt, int k) {
  const size_t i = blockIdx.x * 256ull + threadIdx.x, total = static_cast<size_t>(rows) * cols;
  if (i >= total) return;
  float y = part[i];
  for (int z = 1; z < splits; ++z) y += part[static_cast<size_t>(z) * total + i];
  if (a && !is_finite(y))
    y = fp32_dot(a + (static_cast<size_t>(row0) + i / cols) * k, bt + (i % cols) * k, k);
  if (BIAS) y += bias[i % cols];
  out[static_cast<size_t>(row0) * cols + i] = GELU ? gelu_value(y) : y;
}

// x[i] += bias[i % cols] (kernels.metal:376-379)
__global__ __launch_bounds__(256) void add_bias_f32(float* __restrict__ x,
                                                    const float* __restrict__ bias, uint32_t n,
                                                    uint32_t cols) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) x[i] += bias[i % cols];
}

__global__ __launch_bounds__(256) void gelu_f32(float* __restrict__ x, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) x[i] = gelu_value(x[i]);
}

// LayerNorm over rows of `cols` floats: (x - mean) / sqrt(var + eps) * w + bias, mean and variance
// in fp32 (kernels.metal:362-374). One wavefront per row; out may alias x.
// RESIDUAL: x is first replaced by x + r (tessery's add, kernels.metal:300-304) and the row is
// normalized in place, the pair add(x, r -> x), layer_norm(x -> x) in one pass.
template <bool RESIDUAL>
__global__ __launch_bounds__(256) void layer_norm_f32(float* x, const float* r,
                                                      const float* __restrict__ w,
                                                      const float* __restrict__ bias, float* out,
                                                      int rows, int cols, float eps) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  float* xr = x + static_cast<size_t>(row) * cols;
  if (cols % 64 == 0 && cols <= 512 && (!RESIDUAL || out == x)) {
    // the row in registers (one load of x and r): the sums below add the same values in the
    // same order as the loop further down, so both give the same bits
    const int nv = cols / 64;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i < nv) {
        v[i] = xr[lane + 64 * i];
        if constexpr (RESIDUAL) v[i] = v[i] + r[static_cast<size_t>(row) * cols + lane + 64 * i];
      }
    }
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < nv) total += v[i];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) total += __shfl_xor(total, off);
    const float mean = total / static_cast<float>(cols);
    float squares = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i < nv) {
        const float d = v[i] - mean;
        squares += d * d;
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) squares += __shfl_xor(squares, off);
    const float inv = __frsqrt_rn(squares / static_cast<float>(cols) + eps);
    float* orow = out + static_cast<size_t>(row) * cols;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i < nv) {
        const int c = lane + 64 * i;
        orow[c] = (v[i] - mean) * inv * w[c] + bias[c];
      }
    }
    return;
  }
  if constexpr (RESIDUAL) {
    const float* rr = r + static_cast<size_t>(row) * cols;
    for (int c = lane; c < cols; c += 64) xr[c] = xr[c] + rr[c];
  }
  float total = 0.0f;
  for (int c = lane; c < cols; c += 64) total += xr[c];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) total += __shfl_xor(total, off);
  const float mean = total / static_cast<float>(cols);
  float squares = 0.0f;
  for (int c = lane; c < cols; c += 64) {
    const float d = xr[c] - mean;
    squares += d * d;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) squares += __shfl_xor(squares, off);
  const float inv = __frsqrt_rn(squares / static_cast<float>(cols) + eps);
  float* orow = out + static_cast<size_t>(row) * cols;
  for (int c = lane; c < cols; c += 64) orow[c] = (xr[c] - mean) * inv * w[c] + bias[c];
}

int dense_splits(int rows, int cols, int k, size_t scratch_floats) {
  const int tiles = ((rows + kDenseRows - 1) / kDenseRows) * ((cols + 127) / 128);
  const int chunks = (k + 63) / 64;
  // Under one tile per CU (256 CUs) the CUs that hold a tile run it with one wavefront per SIMD,
  // too few to cover the MFMA chains' latency: split K so every CU holds several workgroups
  // (about 256 in all below 128 tiles, about 768 from 128 to 255 tiles, e.g. 4096 x 384 outputs).
  if (tiles >= 256 || chunks < 4) return 1;
  const int target = tiles < 128 ? 256 : 768;
  int splits = std::min(chunks, (target + tiles - 1) / tiles);
  const int per = (chunks + splits - 1) / splits;
  splits = (chunks + per - 1) / per;  // no empty split
  if (static_cast<size_t>(splits) * rows * cols > scratch_floats) return 1;
  return splits;
}

// Workgroups along K for matmul_x3: 1 from 512 tiles of 64 x 128; from 64 tiles, enough splits of at
// least two 32-wide chunks for about 768 workgroups; fewer tiles, for about 256 workgroups of at
// least four chunks (656 x 384 outputs of K = 1536: 17.3 us with 7 to 12 splits, 20.8 with 4, 21.8
// with 24, and 24.9 on matmul_f32), below K = 1024 of two (64 x 384 outputs of K = 544: 10.0 us, 11.8
// with four and 10.9 on matmul_f32); 0 (the fp32 kernel) where the partial sums do not fit the
// scratch or K is short. Every split holds at least one chunk.
constexpr int kX3WideTiles = 64;  // fewer take eight products, as precise as matmul_f32 in their place
static int x3_split_count(int rows, int cols, int k, int tiles, size_t scratch_floats) {
  if (tiles >= 512) return 1;
  const int chunks32 = k / 32;
  if (tiles < 1 || chunks32 < (tiles < kX3WideTiles ? 8 : 4)) return 0;
  int splits = tiles < kX3WideTiles ? std::min(chunks32 / (chunks32 < 32 ? 2 : 4), 256 / tiles)
                                    : std::min(chunks32 / 2, (768 + tiles - 1) / tiles);
  const int per = (chunks32 + splits - 1) / splits;
  splits = (chunks32 + per - 1) / per;
  if (splits < 2 || static_cast<size_t>(splits) * rows * cols > scratch_floats) return 0;
  return splits;
}

template <bool EXACT>
static void run_planes(const PlanesArgs& a, bool gelu, hipStream_t st) {
  const int row_tiles = (a.row1 - a.row0 + 63) / 64;
  int col_tiles = 0;
  for (int i = 0; i < a.count; ++i) col_tiles += (a.set[i].cols + 63) / 64;
  const unsigned grid = 8u * static_cast<unsigned>((row_tiles + 7) / 8) *
                        static_cast<unsigned>(col_tiles);
  if (gelu)
    matmul_planes<true, EXACT><<<grid, 256, 0, st>>>(a, row_tiles, col_tiles);
  else
    matmul_planes<false, EXACT><<<grid, 256, 0, st>>>(a, row_tiles, col_tiles);
}

template <bool EXACT>
static void run_direct(const PlanesArgs& a, bool gelu, hipStream_t st) {
  unsigned col_tiles = 0;
  for (int i = 0; i < a.count; ++i) col_tiles += static_cast<unsigned>((a.set[i].cols + 31) / 32);
  const dim3 grid(static_cast<unsigned>((a.row1 - a.row0 + 31) / 32), col_tiles);
  if (gelu)
    matmul_direct<true, EXACT><<<grid, 128, 0, st>>>(a);
  else
    matmul_direct<false, EXACT><<<grid, 128, 0, st>>>(a);
}

static size_t dense_planes_bytes(int64_t rows, int k) {
  return static_cast<size_t>((rows + 31) / 32) * static_cast<size_t>(k / 16) * kDenseStep * 2;
}

// K % 32 == 0 and 16-byte rows. Up to K = 512: beyond, one workgroup's walk over K is longer than
// split-K launches and their reduction (656 x 384 outputs of K = 1536: 4.6 + 22 us against 17). Up
// to 512 tiles of 64 x 128, where matmul_x3 fills the chip without split K and splits nothing
// beforehand (16384 x 384 outputs of K = 384: 16 + 35 us against 40, 4096 x 1536: 8 + 38 against 42).
static bool split_shape(const DenseJob& j, size_t planes_bytes) {
  const int64_t tiles = static_cast<int64_t>((j.row1 - j.row0 + 63) / 64) * ((j.cols + 127) / 128);
  return j.k > 0 && j.k % 32 == 0 && j.k <= 512 && j.cols > 0 && tiles < 512 &&
         dense_planes_bytes(64, j.k) * static_cast<size_t>((j.row1 - j.row0 + 63) / 64 +
                                                           3 * ((j.cols + 63) / 64)) <= planes_bytes &&
         ((reinterpret_cast<uintptr_t>(j.a) | reinterpret_cast<uintptr_t>(j.bt)) & 15) == 0;
}

// matmul_direct reads its operands while other workgroups write outputs.
static bool output_apart(const DenseJob& j) { return j.out != j.a && j.out != j.bt; }

// matmul_direct up to this many tiles of 32 x 32, three a CU, matmul_planes after split_dense beyond: 768
// tiles (512 x 1536 outputs of K = 384) 16.8 and 19.4 us, 800 (800 x 1024) 20.2 and 18.4, 1024 (1000 x
// 1024) 20.7 and 18.8; of K = 512 19.5 and 22.2, 23.7 and 21.8, 24.3 and 22.4.
constexpr int64_t kDirectTiles = 768;

static int64_t direct_tiles(const DenseJob& j) {
  return static_cast<int64_t>((j.row1 - j.row0 + 31) / 32) * ((j.cols + 31) / 32);
}

bool matmul_reads_planes(const DenseJob& j, size_t planes_bytes) {
  return split_shape(j, planes_bytes) && (3 * direct_tiles(j) > kDirectTiles || !output_apart(j));
}

bool matmul_on_planes(const DenseJob& j, const DenseScratch& scratch) {
  return split_shape(j, scratch.planes_bytes) && (scratch.planes || output_apart(j));
}

// The shapes (under 512 tiles) that matmul_x3 would take on six products, K split.
static bool x3_takes_six(const DenseJob& j, const DenseScratch& scratch) {
  const int rows = j.row1 - j.row0, tiles = ((rows + kX3Rows - 1) / kX3Rows) * (j.cols / 128);
  return j.cols % 128 == 0 && tiles >= kX3WideTiles &&
         x3_split_count(rows, j.cols, j.k, tiles, scratch.sums_floats) > 0;
}

bool matmul_joins(const DenseJob& a, const DenseJob& b, const DenseScratch& scratch) {
  return b.a == a.a && b.row0 == a.row0 && b.row1 == a.row1 && b.k == a.k &&
         matmul_on_planes(a, scratch) && matmul_on_planes(b, scratch) &&
         x3_takes_six(a, scratch) == x3_takes_six(b, scratch);
}

hipError_t launch_matmul_planes(const DenseJob* jobs, int count, bool gelu,
                                const DenseScratch& scratch, hipStream_t st) {
  if (count < 1 || count > 3) return hipErrorInvalidValue;
  const DenseJob& j = jobs[0];
  for (int i = 0; i < count; ++i)
    if (!matmul_joins(j, jobs[i], scratch)) return hipErrorInvalidValue;
  if (j.row1 <= j.row0) return hipSuccess;
  const int rows = j.row1 - j.row0;
  PlanesArgs p{};
  p.a = j.a;
  p.row0 = j.row0;
  p.row1 = j.row1;
  p.k = j.k;
  p.count = count;
  int wtiles = 0;
  int64_t tiles = 0;
  bool direct = true;
  const bool exact = !x3_takes_six(j, scratch);
  for (int i = 0; i < count; ++i) {
    p.set[i] = PlanesSet{jobs[i].bt, jobs[i].bias, jobs[i].out, jobs[i].cols, wtiles};
    wtiles += (jobs[i].cols + 63) / 64 * 2;  // whole 64-column tiles
    tiles += direct_tiles(jobs[i]);
    direct = direct && output_apart(jobs[i]);
  }
  const int xtiles = (rows + 31) / 32;
  if (!scratch.planes || (direct && tiles <= kDirectTiles)) {
    exact ? run_direct<true>(p, gelu, st) : run_direct<false>(p, gelu, st);
    return hipGetLastError();
  }
  // every job fits the scratch with three times its own weights, so three of equal width do
  if (dense_planes_bytes(32 * (static_cast<int64_t>(xtiles) + wtiles), j.k) > scratch.planes_bytes) {
    for (int i = 0; i < count; ++i) {
      const hipError_t e = launch_matmul_planes(jobs + i, 1, gelu, scratch, st);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  SplitArgs s{};
  s.k = j.k;
  s.planes = static_cast<uint16_t*>(scratch.planes);
  s.count = count + 1;
  s.src[0] = j.a;
  s.row0[0] = j.row0;
  s.rows[0] = rows;
  s.tiles[0] = xtiles;
  p.x = s.planes;
  p.w = s.planes + static_cast<size_t>(xtiles) * (j.k / 16) * kDenseStep;
  for (int i = 0; i < count; ++i) {
    s.src[i + 1] = jobs[i].bt;
    s.rows[i + 1] = jobs[i].cols;
    s.tiles[i + 1] = (jobs[i].cols + 63) / 64 * 2;
  }
  split_dense<<<dim3(static_cast<unsigned>(xtiles + wtiles), (j.k + 63) / 64), 256, 0, st>>>(s);
  exact ? run_planes<true>(p, gelu, st) : run_planes<false>(p, gelu, st);
  return hipGetLastError();
}

// again: results that aren't finite are made again (split operands in place of fp32 MFMA).
static void run_reduce(const DenseJob& j, bool gelu, const float* part, int splits, bool again,
                       hipStream_t st) {
  const int rows = j.row1 - j.row0;
  const unsigned blocks = static_cast<unsigned>((static_cast<size_t>(rows) * j.cols + 255) / 256);
  const float* const a = again ? j.a : nullptr;
  auto run = [&](auto kernel) {
    kernel<<<blocks, 256, 0, st>>>(part, j.bias, j.out, j.row0, rows, j.cols, splits, a, j.bt, j.k);
  };
  if (j.bias)
    gelu ? run(dense_reduce<true, true>) : run(dense_reduce<true, false>);
  else
    gelu ? run(dense_reduce<false, true>) : run(dense_reduce<false, false>);
}

hipError_t launch_matmul_f32(const DenseJob& j, bool gelu, const DenseScratch& dense,
                             hipStream_t st) {
  if (j.row1 <= j.row0 || j.cols <= 0) return hipSuccess;
  if (j.k <= 0) return hipErrorInvalidValue;
  if (matmul_on_planes(j, dense)) return launch_matmul_planes(&j, 1, gelu, dense, st);
  const float *a = j.a, *bt = j.bt, *bias = j.bias;
  float *out = j.out, *scratch = dense.sums;
  const int row0 = j.row0, row1 = j.row1, cols = j.cols, k = j.k;
  const size_t scratch_floats = dense.sums_floats;
  const int rows = row1 - row0, chunks = (k + 63) / 64;
  // bf16 MFMA (split x3), with 16-byte rows: at least two tiles per CU, or K split over workgroups
  // into partial sums
  const int x3_tiles = ((rows + kX3Rows - 1) / kX3Rows) * (cols / 128);
  const int x3_splits = k % 32 == 0 && cols % 128 == 0 &&
                                ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(bt)) &
                                 15) == 0
                            ? x3_split_count(rows, cols, k, x3_tiles, scratch ? scratch_floats : 0)
                            : 0;
  if (x3_splits == 1) {
    dim3 grid((rows + kX3Rows - 1) / kX3Rows, cols / 128);
    if (bias && gelu)
      matmul_x3<true, true, false, false><<<grid, 256, 0, st>>>(a, bt, bias, out, row0, row1, cols,
                                                             k, 0);
    else if (bias)
      matmul_x3<true, false, false, false><<<grid, 256, 0, st>>>(a, bt, bias, out, row0, row1, cols,
                                                             k, 0);
    else if (gelu)
      matmul_x3<false, true, false, false><<<grid, 256, 0, st>>>(a, bt, nullptr, out, row0, row1, cols,
                                                             k, 0);
    else
      matmul_x3<false, false, false, false><<<grid, 256, 0, st>>>(a, bt, nullptr, out, row0, row1, cols,
                                                           k, 0);
    return hipGetLastError();
  }
  if (x3_splits > 1) {
    const int chunks32 = k / 32, per = (chunks32 + x3_splits - 1) / x3_splits;
    dim3 grid((rows + kX3Rows - 1) / kX3Rows, cols / 128, x3_splits);
    if (x3_tiles < kX3WideTiles)
      matmul_x3<false, false, true, true><<<grid, 256, 0, st>>>(a, bt, nullptr, scratch, row0, row1,
                                                                cols, k, per);
    else
      matmul_x3<false, false, true, false><<<grid, 256, 0, st>>>(a, bt, nullptr, scratch, row0,
                                                                 row1, cols, k, per);
    run_reduce(j, gelu, scratch, x3_splits, x3_tiles < kX3WideTiles, st);
    return hipGetLastError();
  }
  const int splits = scratch ? dense_splits(rows, cols, k, scratch_floats) : 1;
  if (splits > 1) {
    // few output tiles (small batches): K split over workgroups, partial sums added in order
    const int per = (chunks + splits - 1) / splits;
    dim3 grid((rows + kDenseRows - 1) / kDenseRows, (cols + 127) / 128, splits);
    matmul_f32<false, false, true><<<grid, 256, 0, st>>>(a, bt, nullptr, scratch, row0, row1,
                                                         cols, k, per);
    run_reduce(j, gelu, scratch, splits, false, st);
    return hipGetLastError();
  }
  dim3 grid((rows + kDenseRows - 1) / kDenseRows, (cols + 127) / 128);
  if (bias && gelu)
    matmul_f32<true, true, false><<<grid, 256, 0, st>>>(a, bt, bias, out, row0, row1, cols, k, 0);
  else if (bias)
    matmul_f32<true, false, false><<<grid, 256, 0, st>>>(a, bt, bias, out, row0, row1, cols, k, 0);
  else if (gelu)
    matmul_f32<false, true, false><<<grid, 256, 0, st>>>(a, bt, nullptr, out, row0, row1, cols, k, 0);
  else
    matmul_f32<false, false, false><<<grid, 256, 0, st>>>(a, bt, nullptr, out, row0, row1, cols, k, 0);
  return hipGetLastError();
}

hipError_t launch_add_bias_f32(float* x, const float* bias, uint32_t n, uint32_t cols,
                               hipStream_t st) {
  if (!n) return hipSuccess;
  add_bias_f32<<<(n + 255) / 256, 256, 0, st>>>(x, bias, n, cols);
  return hipGetLastError();
}

hipError_t launch_gelu_f32(float* x, uint32_t n, hipStream_t st) {
  if (!n) return hipSuccess;
  gelu_f32<<<(n + 255) / 256, 256, 0, st>>>(x, n);
  return hipGetLastError();
}

hipError_t launch_layer_norm_f32(const float* x, const float* w, const float* bias, float* out,
                                 int rows, int cols, float eps, hipStream_t st) {
  if (rows <= 0) return hipSuccess;
  layer_norm_f32<false><<<(rows + 3) / 4, 256, 0, st>>>(const_cast<float*>(x), nullptr, w, bias,
                                                       out, rows, cols, eps);
  return hipGetLastError();
}

hipError_t launch_add_layer_norm_f32(float* x, const float* r, const float* w, const float* bias,
                                     int rows, int cols, float eps, hipStream_t st) {
  if (rows <= 0) return hipSuccess;
  layer_norm_f32<true><<<(rows + 3) / 4, 256, 0, st>>>(x, r, w, bias, x, rows, cols, eps);
  return hipGetLastError();
}

}  // namespace tessery
