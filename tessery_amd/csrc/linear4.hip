// uint4 affine group-64 projections of fp32 activations for gfx950.
//
// Weight format (tessery weight4, kernels.metal:11-19): W packed u32[N, K/8]; nibble j of word
// (n, k/8) is column 8*(k/8)+j, little-nibble first; group g = n*(K/64) + k/64;
// w[n][k] = code * scale[g] + bias[g], scale/bias bfloat16 words [N, K/64].
// y[t][n] = sum_k x[t][k] * w[n][k].
//
// linear4_rows serves every tessery linear4 route name (linear4, linear4_tiled, linear4_tail,
// linear4_16x32_k64, linear4_32x32_k64, linear4_small3) below kLinear4HiloRows rows, and any
// shape linear4_hilo does not tile: one reduction order per output element, whatever the launch's
// rows, its tile shape and the projections beside it, so every route over a row produces
// bit-identical results.
//
// The gated form runs it over two weight sets (gate and up) with the SwiGLU epilogue
// out = silu(gate) * up (kernels.metal:609-656, 687-731); each projection keeps the linear4
// reduction order and the epilogue is silu_gate's expression, so the fused routes are
// bit-identical to linear4 + linear4 + silu_gate over the same rows.
#include <algorithm>

#include "common.h"
#include "kernels.h"
#include "lds_dma.h"
#include "planes.h"

namespace tessery {

namespace {

// Per group of 64 inputs, with c' = c - z and b' = z scale + bias (w = scale c' + b'), z being the whole
// number of 0 .. 15 nearest to -bias / scale, for each column and group:
//     y[m][n] += scale[n] * sum_k x[m][k] c'[n][k] + b'[n] * sum_k x[m][k]
// x is split exactly into three bf16 terms (split3x8) and c' is exact in bf16, so every product on
// v_mfma_f32_32x32x16_bf16 is exact and the sums are fp32, at three bf16 MFMAs of 32 cycles per 16
// inputs where fp32 MFMA takes eight of 64. The second term is one more MFMA per group, its two
// factors split into three bf16 terms each: eight of their nine products fill the lane's eight
// k-slots, and the ninth (the two smallest terms) is below 2^-30 of the whole.
//
// z keeps both terms as small as w: where it is not cut off, |b'| <= |scale| / 2, so that
// |scale c'| <= 2 |w| and |b'| <= |w| for every code; where it is, both terms have one sign. With one
// z for all groups (8), a group whose codes sit at one end against a bias that cancels them lost
// the result in the difference of two large sums: codes 0 with bias 2^-12 scale, 5.8e-4 of
// sum |x| |w| instead of 1e-7.
//
// K order: eight partitions of consecutive groups (partition p: groups [p G / 8, (p + 1) G / 8)),
// each summed on its own, then added as a balanced tree.
//
// x comes as planes (planes.h), so no workgroup splits it again. linear4_rows (few tiles): operands go
// straight from L1 to registers, with no LDS and no barrier before the end; a workgroup makes a
// tile of 32 x 32 with one partition a wavefront, and their sums meet in LDS, so no partial sums
// leave it. Bound: the loads. A wavefront reads 12 KiB of x for a group and fetches whole lines of
// weights and scales, which is why it takes four groups of those at a time. Measured, the o
// projection (K = 2048) of 24 rows: 7.4 us, 9.3 us with every workgroup splitting x itself; down
// (K = 3072) 9.2 and 12.8 us.
constexpr int kL4Parts = 8;
constexpr int kRedRow = 40;  // floats per staged result row: the lane halves' rows r, r + 4 on
                             // opposite halves of the banks

struct L4Set {
  const uint32_t* w;
  const uint16_t* s;
  const uint16_t* b;
  float* out;
  int cols;
};

// Up to three projections of the same x, or (GATED) gate and up of equal width: out of set 0 takes
// silu(gate) * up, out of set 1 (may be null) the up projection.
struct L4Args {
  Planes x;  // of rows row0 .. row1 - 1
  const float* rows;  // the whole x as it came
  L4Set set[3];
  int row0, row1, k;
  int vec;      // every out 16-byte aligned and every width a multiple of 4
  Planes next;  // GATED: the planes of the output (terms null: none), row0 = 0
};

// z of a column's group, and -(2^(23 - 4 i) + z) for the codes at bits 4 i of a word.
struct Centre {
  float z, base[5];
};
__device__ __forceinline__ Centre centre_of(float scale, float bias) {
  Centre c;
  // any z is exact; the nearest one (within the reciprocal's rounding) is well conditioned. scale 0
  // gives 0 or 15
  c.z = __builtin_rintf(
      __builtin_amdgcn_fmed3f(-bias * __builtin_amdgcn_rcpf(scale), 0.0f, 15.0f));
#pragma unroll
  for (int i = 0; i < 5; ++i) c.base[i] = -static_cast<float>(1 << (23 - 4 * i)) - c.z;
  return c;
}

// c - z of the eight codes of a weight word as bf16, in natural order. A code at bits 4 i .. 4 i + 3 of
// the significand of 2.0 makes 2 + c 2^(4 i - 22), and one fma c - z: two full-rate instructions a code
// (masks and factors in scalar registers, 2.0 inline), where v_cvt_off_f32_i4 alone takes 16 cycles.
__device__ __forceinline__ bf16x8 decode_centred(uint32_t word, const Centre& c) {
  const uint32_t late = word >> 12;  // codes 5, 6 and 7 where 2, 3 and 4 were
  uint32_t f[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int i = j < 5 ? j : j - 3;
    uint32_t mask = 15u << (4 * i);
    asm("" : "+s"(mask));  // a register, so that the mask and 2.0 fit one instruction
    const uint32_t bits = ((j < 5 ? word : late) & mask) | 0x40000000u;
    f[j] = __float_as_uint(
        fmaf(__uint_as_float(bits), static_cast<float>(1 << (22 - 4 * i)), c.base[i]));
  }
  uint4v r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = __builtin_amdgcn_perm(f[2 * j + 1], f[2 * j], 0x07060302u);
  return __builtin_bit_cast(bf16x8, r);
}

// Planes of rows row0 .. of x: a workgroup splits one row tile's group, thread (row tid / 8, chunk
// tid % 8) 8 inputs; the 8 rows of a wavefront make 128-byte pieces.
__global__ __launch_bounds__(256) void split_planes(const float* __restrict__ x, Planes p,
                                                    int row0, int row1, int k) {
  const int groups = k >> 6, g = blockIdx.y, row = threadIdx.x >> 3, c = threadIdx.x & 7;
  const int at = static_cast<int>(blockIdx.x) * kPlaneRows + row;
  if (row0 + at >= row1) return;
  const float* const src = x + static_cast<size_t>(row0 + at) * k + 64 * g + 8 * c;
  const floatx4 u = *reinterpret_cast<const floatx4*>(src);
  const floatx4 v = *reinterpret_cast<const floatx4*>(src + 4);
  const size_t tile = static_cast<size_t>(blockIdx.x) * groups + g;
  const int lane = row + 32 * (c >> 2);
  uint4v t[3];
  split3x8(u, v, t[0], t[1], t[2]);
#pragma unroll
  for (int i = 0; i < 3; ++i)
    *reinterpret_cast<uint4v*>(p.terms + tile * kPlaneGroup + i * kPlaneTerm + (c & 3) * 512 +
                               lane * 8) = t[i];
  float sum = ((u[0] + u[1]) + (u[2] + u[3])) + ((v[0] + v[1]) + (v[2] + v[3]));
  sum += __shfl_xor(sum, 1);
  sum += __shfl_xor(sum, 2);
  if ((c & 3) == 0) p.sums[tile * kPlaneSums + lane] = sum;
}

typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t resource(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
}

// Weight words, scales and biases of a lane's column for N consecutive groups: a column's groups lie
// side by side, so four of them fill the line that one would fetch. Scales and biases are 2-byte
// words at any parity: whole dwords from the aligned one below, shifted by the lane. Groups past
// the last one read the next column's, or zero past the end (the caller uses none of them).
template <int N>
struct Words {
  uint4v w[N];
  uint32_t s[N / 2 + 1], b[N / 2 + 1];
};
struct ColumnWords {
  rsrc_t wres, sres, bres;
  uint32_t woff, soff, groups;

  __device__ __forceinline__ ColumnWords(const L4Set& set, int n, int hh, int K) {
    const uint32_t half = static_cast<uint32_t>(K >> 1), cols = static_cast<uint32_t>(set.cols);
    groups = static_cast<uint32_t>(K >> 6);
    // scales and biases in whole dwords: an odd count is followed by padding of its allocation
    const uint32_t bytes = (cols * groups * 2u + 3u) & ~3u;
    wres = resource(set.w, cols * half);
    sres = resource(set.s, bytes);
    bres = resource(set.b, bytes);
    woff = static_cast<uint32_t>(n) * half + 16u * static_cast<uint32_t>(hh);
    soff = static_cast<uint32_t>(n) * groups * 2u;
  }
  template <int N>
  __device__ __forceinline__ void load(Words<N>& r, int at) const {
    const uint32_t g = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
    for (int j = 0; j < N; ++j)
      r.w[j] = __builtin_amdgcn_raw_buffer_load_b128(wres, woff + 32u * j, 32u * g, 0);
    const uint32_t off = (soff + 2u * g) & ~3u;
    if constexpr (N == 4) {
      const uint3v s = __builtin_amdgcn_raw_buffer_load_b96(sres, off, 0, 0);
      const uint3v b = __builtin_amdgcn_raw_buffer_load_b96(bres, off, 0, 0);
#pragma unroll
      for (int j = 0; j < 3; ++j) r.s[j] = s[j], r.b[j] = b[j];
    } else {
      static_assert(N == 2, "two or four groups");
      const uint2v s = __builtin_amdgcn_raw_buffer_load_b64(sres, off, 0, 0);
      const uint2v b = __builtin_amdgcn_raw_buffer_load_b64(bres, off, 0, 0);
#pragma unroll
      for (int j = 0; j < 2; ++j) r.s[j] = s[j], r.b[j] = b[j];
    }
  }
  // the words as loaded for `at` -> scales and biases of groups 2 i, 2 i + 1 in s[i] and b[i]
  template <int N>
  __device__ __forceinline__ void align(Words<N>& r, int at) const {
    const uint32_t shift = ((soff + 2u * static_cast<uint32_t>(at)) & 2u) * 8u;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      r.s[i] = __builtin_amdgcn_alignbit(r.s[i + 1], r.s[i], shift);
      r.b[i] = __builtin_amdgcn_alignbit(r.b[i + 1], r.b[i], shift);
    }
  }
};

// Column tile t of a launch -> the weight set it belongs to and the tile's place in it.
__device__ __forceinline__ void column_tile(const L4Args& a, int width, int& tile, int& set) {
  while (set < 2 && tile >= (a.set[set].cols + width - 1) / width) {
    tile -= (a.set[set].cols + width - 1) / width;
    ++set;
  }
}

// What a 32-column block needs of one group's words: the codes, the bias operand (b' in the lane's
// k-slots, against the terms of its half-group sum) and the scale.
struct Prepared {
  bf16x8 codes[4], bias;
  float scale;
};
// of group j (a constant after unrolling) of aligned words
template <int N>
__device__ __forceinline__ Prepared prepare_group(const Words<N>& words, int j) {
  auto upper = [&](uint32_t v) { return __uint_as_float(j & 1 ? v & 0xffff0000u : v << 16); };
  const float scale = upper(words.s[j / 2]), bias = upper(words.b[j / 2]);
  const Centre centre = centre_of(scale, bias);
  Prepared r;
#pragma unroll
  for (int s4 = 0; s4 < 4; ++s4) r.codes[s4] = decode_centred(words.w[j][s4], centre);
  const Split3 bs = split3(fmaf(centre.z, scale, bias));
  const uint32_t b12 = upper_pair(bs.t[0], bs.t[1]);
  r.bias = __builtin_bit_cast(bf16x8, uint4v{b12, b12, upper_pair(bs.t[2], bs.t[0]),
                                             upper_pair(bs.t[2], bs.t[1])});
  r.scale = scale;
  return r;
}

// acc += the group's products for one 32 x 32 tile; x(t, s4): the operand of term t, k-step s4.
template <typename X>
__device__ __forceinline__ void multiply_group(const Prepared& w, X x, float xsum, floatx16& acc) {
  // bias term: the products of the terms of the lane's half-group sum and b' but the smallest one
  const Split3 xs = split3(xsum);
  const bf16x8 xa = __builtin_bit_cast(
      bf16x8, uint4v{upper_pair(xs.t[0], xs.t[0]), upper_pair(xs.t[1], xs.t[1]),
                     upper_pair(xs.t[0], xs.t[2]), upper_pair(xs.t[1], xs.t[2])});
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa, w.bias, acc, 0, 0, 0);
  floatx16 p;
#pragma unroll
  for (int e = 0; e < 16; ++e) p[e] = 0.0f;
#pragma unroll
  for (int t = 2; t >= 0; --t)  // the smallest terms first
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
      p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x(t, s4), w.codes[s4], p, 0, 0, 0);
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = fmaf(w.scale, p[e], acc[e]);
}

// x . w of one row and column as fp32 products: for a result that isn't finite. An infinite x splits
// into NaN terms, and so does an infinite scale or bias.
__device__ __forceinline__ float fp32_dot(const L4Args& a, const L4Set& set, int row, int col) {
  const int groups = a.k >> 6;
  const float* x = a.rows + static_cast<size_t>(row) * a.k;
  const uint32_t* w = set.w + static_cast<size_t>(col) * (a.k >> 3);
  float y = 0.0f;
  for (int g = 0; g < groups; ++g) {
    const size_t at = static_cast<size_t>(col) * groups + g;
    const float scale = bf16_to_float(set.s[at]), bias = bf16_to_float(set.b[at]);
    float part = 0.0f;
    for (int i = 0; i < 64; ++i) {
      const uint32_t code = w[8 * g + (i >> 3)] >> (4 * (i & 7)) & 15u;
      part = fmaf(x[64 * g + i], fmaf(static_cast<float>(code), scale, bias), part);
    }
    y += part;
  }
  return y;
}

// The end of a tile of BLOCKS column blocks (GATED: the gate's, then the up projection's), one a
// wavefront: the sums of the SLOTS slots meet in LDS (`red`, free by now), then whole-row stores.
template <int BLOCKS, int SLOTS, bool GATED>
__device__ __forceinline__ void store_tile(const L4Args& a, float* red,
                                           const floatx16& total, int slot, int own, int first,
                                           int tile, int rbase) {
  constexpr int TC = GATED ? 16 * BLOCKS : 32 * BLOCKS, THREADS = 64 * SLOTS * BLOCKS;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int e = 0; e < 16; ++e)
    red[((slot * BLOCKS + own) * 32 + 8 * (e >> 2) + 4 * hh + (e & 3)) * kRedRow + l32] = total[e];
  wait_lgkmcnt<0>();
  stage_barrier();
  auto sum4 = [&](int block, int row, int col) {
    auto at = [&](int s) {
      return *reinterpret_cast<const floatx4*>(
          &red[((s * BLOCKS + block) * 32 + row) * kRedRow + col]);
    };
    auto add = [](const floatx4& u, const floatx4& v) {
      return floatx4{u[0] + v[0], u[1] + v[1], u[2] + v[2], u[3] + v[3]};
    };
    if constexpr (SLOTS == 8)
      return add(add(add(at(0), at(1)), add(at(2), at(3))),
                 add(add(at(4), at(5)), add(at(6), at(7))));
    else if constexpr (SLOTS == 4)
      return add(add(at(0), at(1)), add(at(2), at(3)));
    else
      return add(at(0), at(1));
  };
  auto made_again = [&](const L4Set& set, int row, int c0, floatx4& y) {
    uint32_t again = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      again |= fabsf(y[j]) <= 3.402823466e38f || c0 + j >= set.cols ? 0u : 1u << j;
    for (; again; again &= again - 1) {
      const int at = __builtin_ctz(again);
      const float dot = fp32_dot(a, set, row, c0 + at);
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = j == at ? dot : y[j];
    }
  };
  auto store = [&](const L4Set& set, int row, int c0, const floatx4& y) {
    float* const dst = set.out + static_cast<size_t>(row) * set.cols + c0;
    if (a.vec && c0 + 4 <= set.cols) {
      *reinterpret_cast<floatx4*>(dst) = y;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c0 + j < set.cols) dst[j] = y[j];
    }
  };
  for (int i = tid; i < 32 * TC / 4; i += THREADS) {
    const int row = i / (TC / 4), c = 4 * (i % (TC / 4)), block = c >> 5;
    if (rbase + row >= a.row1) break;  // rows ascend with i
    floatx4 y = sum4(block, row, c & 31);
    made_again(a.set[GATED ? 0 : first], rbase + row, tile * TC + c, y);
    if constexpr (GATED) {
      floatx4 up = sum4(block + BLOCKS / 2, row, c & 31);
      made_again(a.set[1], rbase + row, tile * TC + c, up);
      if (a.set[1].out) store(a.set[1], rbase + row, tile * TC + c, up);
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = silu_times(y[j], up[j]);
      if (a.next.terms && tile * TC + c < a.set[0].cols)
        store_planes4(a.next, rbase + row, tile * TC + c, a.set[0].cols >> 6, y);
    }
    store(a.set[GATED ? 0 : first], rbase + row, tile * TC + c, y);
  }
}

// A 32 x 32 tile, one partition a wavefront.
__global__ __launch_bounds__(512, 2) void linear4_rows(L4Args a) {
  __shared__ __attribute__((aligned(16))) float red[8 * 32 * kRedRow];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int groups = a.k >> 6;
  const int rbase = a.row0 + static_cast<int>(blockIdx.x) * kPlaneRows;
  int tile = blockIdx.y, first = 0;
  column_tile(a, 32, tile, first);
  // clamped columns aren't stored
  const ColumnWords column(a.set[first], min(tile * 32 + l32, a.set[first].cols - 1), hh, a.k);

  // Rows past the last one, and a group past the wavefront's last one, are asked for at kNowhere,
  // out of the resource's range: no memory access, and no branch around the loads, which keeps the
  // compiler's waits exact.
  constexpr uint32_t kNowhere = 0xc0000000u;
  const uint32_t norow = rbase + l32 < a.row1 ? 0u : kNowhere;
  const size_t xtile = static_cast<size_t>(blockIdx.x) * groups;
  const rsrc_t xres = resource(a.x.terms + xtile * kPlaneGroup,
                               static_cast<uint32_t>(groups) * (kPlaneGroup * 2u));
  const rsrc_t xsres = resource(a.x.sums + xtile * kPlaneSums,
                                static_cast<uint32_t>(groups) * (kPlaneSums * 4u));
  struct Group {
    bf16x8 x[3][4];
    float sum;
  };
  int g = wave * groups / kL4Parts;
  const int end = (wave + 1) * groups / kL4Parts;
  auto load = [&](Group& r, int at) {
    const uint32_t past = at < end ? norow : kNowhere;
    const uint32_t gx = __builtin_amdgcn_readfirstlane(at < end ? at : 0);
    r.sum = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                          xsres, (4u * lane) | past, 4u * kPlaneSums * gx, 0));
#pragma unroll
    for (int t = 2; t >= 0; --t)
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
        r.x[t][s4] = __builtin_bit_cast(
            bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                        xres, ((16u * lane) | past) + 1024u * s4,
                        2u * kPlaneGroup * gx + 2u * kPlaneTerm * t, 0));
    asm volatile("" ::: "memory");  // issued here, before the product that runs meanwhile
    __builtin_amdgcn_sched_barrier(0);
  };
  // every sum started from +0, as in the other tile shape
  floatx16 total;
#pragma unroll
  for (int e = 0; e < 16; ++e) total[e] = 0.0f;
  if (g < end) {
    Group x[2];
    Words<4> words;
    column.load(words, g);
    load(x[0], g);
    bool more = true;
    while (more) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j == 0) column.align(words, g);
        const Prepared w = prepare_group(words, j);
        if (j == 3) column.load(words, g + 4);
        load(x[(j + 1) & 1], g + j + 1);
        const Group& r = x[j & 1];
        multiply_group(w, [&](int t, int s4) { return r.x[t][s4]; }, r.sum, total);
        if (g + j + 1 >= end) {
          more = false;
          break;
        }
      }
      g += 4;
    }
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) total[e] += 0.0f;
  store_tile<1, 8, false>(a, red, total, wave, 0, first, tile, rbase);
}

// The same with x shared: 8 wavefronts = WC column blocks of 32 x WK slots of 8 / WK partitions
// (GATED: half of the blocks are the gate's columns, half the up projection's). One group of x a
// slot at a time is copied to LDS (two stages, the copy of the next group under way while this one
// is multiplied) and read by the slot's WC wavefronts. Bound: the issue of VALU instructions
// (decoding and folding, about 150 beside 13 MFMAs) and a step's barrier and waits. Measured: q, k
// and v of 308 rows 18.1 us, gate and up 20.9; with x split in every workgroup 22 and 26.
template <int WC, bool GATED>
__global__ __launch_bounds__(512, WC == 4 ? 4 : 2) void linear4_rows_shared(L4Args a) {
  constexpr int WK = 8 / WC, NP = kL4Parts / WK;  // partitions of a slot
  constexpr int TC = GATED ? 16 * WC : 32 * WC;   // columns of a tile in each of its sets
  constexpr int STAGES = 2 * WK * kPlaneGroup * 2, RED = 8 * 32 * kRedRow * 4;
  __shared__ __attribute__((aligned(1024))) char mem[STAGES > RED ? STAGES : RED];

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wc = wave % WC, slot = wave / WC;
  const int groups = a.k >> 6;
  const int rbase = a.row0 + static_cast<int>(blockIdx.x) * kPlaneRows;
  int tile = blockIdx.y, first = 0;
  if constexpr (!GATED) column_tile(a, TC, tile, first);
  const L4Set set = a.set[GATED ? (wc >= WC / 2) : first];
  const int n = tile * TC + 32 * (GATED ? wc % (WC / 2) : wc) + l32;
  const ColumnWords column(set, min(n, set.cols - 1), hh, a.k);  // clamped columns aren't stored
  const size_t xtile = static_cast<size_t>(blockIdx.x) * groups;

  auto stage = [&](int buf) {
    return reinterpret_cast<_Float16*>(mem) + (buf * WK + slot) * kPlaneGroup;
  };
  float sum;
  auto load = [&](int buf, int g) {
    sum = a.x.sums[(xtile + g) * kPlaneSums + lane];
    const uint16_t* const src = a.x.terms + (xtile + g) * kPlaneGroup;
#pragma unroll
    for (int i = 0; i < 12 / WC; ++i) {
      const int piece = wc * (12 / WC) + i;
      dma16_at(src + piece * 512, 16u * lane, stage(buf) + piece * 512);
    }
  };

  floatx16 acc, pair, total;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = pair[e] = total[e] = 0.0f;
  const int p0 = slot * NP;
  auto bound = [&](int p) { return p * groups / kL4Parts; };
  int g = bound(p0), part = 0, pend = bound(p0 + 1);
  const int end = bound(p0 + NP);
  // closes partition `part` of the slot: balanced-tree sums, every one started from +0
  auto close = [&]() {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if constexpr (NP == 4) {
        const bool second = part & 1;
        total[e] = second ? total[e] + (pair[e] + acc[e]) : total[e];
        pair[e] = second ? pair[e] : acc[e];
      } else {
        total[e] += acc[e];
      }
      acc[e] = 0.0f;
    }
    ++part;
    pend = bound(p0 + part + 1);
  };
  int steps = 0;  // of the slot with the most groups: barriers are for all wavefronts
#pragma unroll
  for (int s = 0; s < WK; ++s) steps = max(steps, bound((s + 1) * NP) - bound(s * NP));

  constexpr int N = WC == 4 ? 2 : 4;  // registers: 128 at WC = 4, for two workgroups on a CU
  Words<N> words;
  column.load(words, g);
  if (g < end) load(0, g);
  for (int step = 0; step < steps; step += N, g += N) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (step + j >= steps) break;
      // this step's copy and words have landed; every wavefront is done with the other stage
      wait_vmcnt<0>();
      stage_barrier();
      if (j == 0) column.align(words, g);
      const Prepared w = prepare_group(words, j);
      const float xsum = sum;
      if (j == N - 1) column.load(words, g + N);
      if (g + j + 1 < end) load((j + 1) & 1, g + j + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (g + j >= end) continue;
      while (part + 1 < NP && g + j >= pend) close();
      const _Float16* const src = stage(j & 1) + lane * 8;
      multiply_group(w,
                     [&](int t, int s4) {
                       return *reinterpret_cast<const bf16x8*>(src + t * kPlaneTerm + s4 * 512);
                     },
                     xsum, acc);
    }
  }
  while (part < NP) close();
  wait_vmcnt<0>();
  wait_lgkmcnt<0>();
  stage_barrier();  // the stages are free
  store_tile<WC, WK, GATED>(a, reinterpret_cast<float*>(mem), total, slot, wc, first, tile, rbase);
}

template <int WIDTH>
dim3 l4_grid(const L4Args& a, int sets) {
  unsigned tiles = 0;
  for (int i = 0; i < sets; ++i)
    tiles += static_cast<unsigned>((a.set[i].cols + WIDTH - 1) / WIDTH);
  return dim3(static_cast<unsigned>((a.row1 - a.row0 + kPlaneRows - 1) / kPlaneRows), tiles);
}

void run_rows(const L4Args& a, int sets, hipStream_t st) {
  linear4_rows<<<l4_grid<32>(a, sets), 512, 0, st>>>(a);
}

template <int WC, bool GATED>
void run_shared(const L4Args& a, int sets, hipStream_t st) {
  linear4_rows_shared<WC, GATED>
      <<<l4_grid<GATED ? 16 * WC : 32 * WC>(a, GATED ? 1 : sets), 512, 0, st>>>(a);
}

hipError_t launch_rows(const Linear4Job* jobs, int count, bool gated, const Planes& x, int row0,
                       int row1, const Planes& next, hipStream_t st) {
  L4Args a{};
  a.x = x;
  a.rows = jobs[0].x;
  a.row0 = row0;
  a.row1 = row1;
  a.k = jobs[0].k;
  a.vec = 1;
  a.next = next;
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i) {
    a.set[i] = L4Set{jobs[i].w, jobs[i].scales, jobs[i].biases, jobs[i].out, jobs[i].cols};
    if (jobs[i].cols % 4 || (reinterpret_cast<uintptr_t>(jobs[i].out) & 15)) a.vec = 0;
    tiles += (jobs[i].cols + 31) / 32;
  }
  tiles *= (row1 - row0 + kPlaneRows - 1) / kPlaneRows;
  // the widest tile that still has a workgroup for (nearly) every CU: one 32 x 32 tile each up to
  // 256 (q, k and v of 48 rows 6.0 us, 8.1 with two blocks), two up to 512 (o of 308 rows 12.1 us,
  // 14.3 with one and 18.8 with four), else four (gate and up of 1000 rows 55 us, 86 with two)
  if (tiles > 512)
    gated ? run_shared<4, true>(a, count, st) : run_shared<4, false>(a, count, st);
  else if (gated)
    run_shared<2, true>(a, count, st);
  else if (tiles > 256)
    run_shared<2, false>(a, count, st);
  else
    run_rows(a, count, st);
  return hipGetLastError();
}

// large batches: fp16 MFMA on row-scaled hi + lo activations (fp32-grade, several times the fp32 MFMA
// rate)
bool runs_hilo(const Linear4Job& j, const float* scratch, size_t scratch_floats) {
  return linear4_hilo_fits(j.row1 - j.row0, j.cols, j.k, j.x + static_cast<size_t>(j.row0) * j.k,
                           j.out + static_cast<size_t>(j.row0) * j.cols, scratch, scratch_floats);
}

__global__ __launch_bounds__(256) void silu_gate_f32(float* __restrict__ gate,
                                                     const float* __restrict__ up, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) gate[i] = silu_times(gate[i], up[i]);
}

}  // namespace

bool linear4_on_rows(const Linear4Job& j, const float* scratch, size_t scratch_floats) {
  return !runs_hilo(j, scratch, scratch_floats);
}

hipError_t launch_linear4_rows(const Linear4Job* jobs, int count, bool gated,
                               const PlanesScratch& scratch, bool prepared, bool keep,
                               hipStream_t st) {
  if (count < 1 || count > 3 || (gated && (count != 2 || jobs[0].cols != jobs[1].cols)))
    return hipErrorInvalidValue;
  const Linear4Job& j = jobs[0];
  for (int i = 0; i < count; ++i)
    if (jobs[i].x != j.x || jobs[i].row0 != j.row0 || jobs[i].row1 != j.row1 ||
        jobs[i].k != j.k || jobs[i].cols <= 0 || j.k <= 0 || j.k % 64 || j.k > 65536)
      return hipErrorInvalidValue;
  if (j.row1 <= j.row0) return hipSuccess;
  const int rows = j.row1 - j.row0;
  Planes next{};
  if (keep) {
    if (!gated || j.row0 || j.cols % 64 || planes_bytes(rows, j.cols) > scratch.bytes)
      return hipErrorInvalidValue;
    next = planes_at(scratch.out, rows, j.cols);
  }
  if (prepared) {
    if (j.row0 || planes_bytes(rows, j.k) > scratch.bytes) return hipErrorInvalidValue;
    return launch_rows(jobs, count, gated, planes_at(scratch.in, rows, j.k), 0, j.row1, next, st);
  }
  // x in ranges of whole row tiles whose planes fit the scratch (one range for most shapes; an
  // output kept as planes is within it)
  const size_t tile_bytes = planes_bytes(kPlaneRows, j.k);
  const int64_t fit = static_cast<int64_t>(scratch.bytes / tile_bytes);
  if (fit < 1) return hipErrorInvalidValue;
  const int step = static_cast<int>(std::min<int64_t>(fit * kPlaneRows, 1 << 20));
  if (keep && step < rows) return hipErrorInvalidValue;
  for (int r = j.row0; r < j.row1; r += std::min(step, j.row1 - r)) {
    const int end = r + std::min(step, j.row1 - r);
    const Planes x = planes_at(scratch.in, end - r, j.k);
    const dim3 grid((end - r + kPlaneRows - 1) / kPlaneRows, j.k / 64);
    split_planes<<<grid, 256, 0, st>>>(j.x, x, r, end, j.k);
    const hipError_t e = launch_rows(jobs, count, gated, x, r, end, next, st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_linear4_f32(const Linear4Job& j, float* scratch, size_t scratch_floats,
                              bool scaled, const PlanesScratch& planes, hipStream_t st) {
  if (j.row1 <= j.row0 || j.cols <= 0) return hipSuccess;
  if (runs_hilo(j, scratch, scratch_floats))
    return launch_linear4_hilo_f32(j.x + static_cast<size_t>(j.row0) * j.k, j.w, j.scales, j.biases,
                                   j.out + static_cast<size_t>(j.row0) * j.cols, j.row1 - j.row0,
                                   j.cols, j.k, scratch, scratch_floats, scaled, st);
  return launch_linear4_rows(&j, 1, false, planes, false, false, st);
}

hipError_t launch_silu_gate_f32(float* gate, const float* up, uint32_t n, hipStream_t st) {
  if (!n) return hipSuccess;
  silu_gate_f32<<<(n + 255) / 256, 256, 0, st>>>(gate, up, n);
  return hipGetLastError();
}

}  // namespace tessery
