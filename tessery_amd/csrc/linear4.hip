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

namespace tessery {

namespace {

// Per group of 64 inputs, with c' = c - 8 and b' = 8 scale + bias (w = scale c' + b'):
//     y[m][n] += 16 scale[n] * sum_k x[m][k] (c'[n][k] / 16) + b'[n] * sum_k x[m][k]
// x is split exactly into three bf16 terms (split3x8) and c' / 16 is exact in bf16, so every
// product on v_mfma_f32_32x32x16_bf16 is exact and the sums are fp32: nothing is rounded that the
// fp32 product would keep, at three bf16 MFMAs of 32 cycles per 16 inputs where fp32 MFMA takes
// eight of 64. The second term is one more MFMA per group, its two factors split into three bf16
// terms each. Centred codes keep the sums as small as the result (uncentred ones cancel against
// the bias term).
//
// K order: eight partitions of consecutive groups (partition p: groups [p G / 8, (p + 1) G / 8)),
// each summed on its own, then added as a balanced tree.
//
// Layout: 8 wavefronts = WC column blocks of 32 x WK slots of 8 / WK consecutive partitions; a
// workgroup makes a tile of 32 rows x 32 WC columns. The WC wavefronts of a slot stage one group
// of x at a time (32 x 64 floats -> three bf16 planes in LDS, the next group's x and weights in
// registers meanwhile); the slots' sums meet in LDS at the end, so no partial sums leave the
// workgroup. Bound: with few rows the latency of one pass over K (loads, split, MFMA chain, the
// sum over slots) and the splitting of x, which every workgroup repeats; with many rows the VALU
// (split, decode, fold), about as many cycles as the MFMAs at WC = 4.
// LDS planes are rows of 128 bytes, 16-byte chunk c of row r at c ^ ((r >> 1) & 7): the 16 rows one
// read group takes land on different banks, and 8 lanes write one row.
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
  const float* x;
  L4Set set[3];
  int row0, row1, k;
  int vec;  // every out 16-byte aligned and every width a multiple of 4
};

// (c - 8) / 16 of the eight codes of a weight word as bf16, in natural order
__device__ __forceinline__ bf16x8 decode_centred(uint32_t word) {
  const uint32_t even = word ^ 0x88888888u, odd = even >> 4;
  uint4v r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t e = __float_as_uint(__builtin_amdgcn_cvt_off_f32_i4((even >> (8 * j)) & 0xffu));
    const uint32_t o = __float_as_uint(__builtin_amdgcn_cvt_off_f32_i4((odd >> (8 * j)) & 0xffu));
    r[j] = __builtin_amdgcn_perm(o, e, 0x07060302u);
  }
  return __builtin_bit_cast(bf16x8, r);
}

struct Split3 {
  uint32_t t[3];  // the three bf16 terms, each in the upper half of its word
};
__device__ __forceinline__ Split3 split3(float x) {
  Split3 r;
  r.t[0] = __float_as_uint(x);
  const float r1 = x - __uint_as_float(r.t[0] & 0xffff0000u);
  r.t[1] = __float_as_uint(r1);
  r.t[2] = __float_as_uint(r1 - __uint_as_float(r.t[1] & 0xffff0000u));
  return r;
}
__device__ __forceinline__ uint32_t upper_pair(uint32_t first, uint32_t second) {
  return __builtin_amdgcn_perm(second, first, 0x07060302u);
}

template <int WC, int WK, bool GATED>
__global__ __launch_bounds__(512, WC == 1 ? 2 : 4) void linear4_rows(L4Args a) {
  static_assert(WC * WK == 8 && kL4Parts % WK == 0 && (!GATED || WC > 1), "eight wavefronts");
  constexpr int NP = kL4Parts / WK;     // partitions of a slot
  constexpr int NBUF = WC == 4 ? 2 : 1;  // x stages of a slot
  constexpr int CPT = 4 / WC;           // 8-float chunks of x a thread stages per group
  constexpr int PLANE = 32 * 64;
  constexpr int STAGE = NBUF * WK * 3 * PLANE * 2, RED = 8 * 32 * kRedRow * 4;
  __shared__ __attribute__((aligned(1024))) char mem[STAGE > RED ? STAGE : RED];
  __shared__ float xg[NBUF][WK][2][32];  // sums of 32 inputs (half a group) per row
  uint16_t* const planes = reinterpret_cast<uint16_t*>(mem);

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wc = wave % WC, slot = wave / WC;
  const int K = a.k, groups = K >> 6;
  const int rbase = a.row0 + static_cast<int>(blockIdx.x) * 32;

  // column tile -> weight set and the wavefront's first column in it
  constexpr int TC = GATED ? 16 * WC : 32 * WC;  // columns of a tile in each of its sets
  int tile = blockIdx.y, first = 0;
  if constexpr (!GATED)
    while (first < 2 && tile >= (a.set[first].cols + TC - 1) / TC) {
      tile -= (a.set[first].cols + TC - 1) / TC;
      ++first;
    }
  const L4Set& mine = a.set[GATED ? (wc >= WC / 2) : first];
  const int cblock = GATED ? wc % (WC / 2) : wc;
  const int n = min(tile * TC + 32 * cblock + l32, mine.cols - 1);  // clamped columns aren't stored
  // wave-uniform bases, 32-bit lane offsets (cols, K <= 65536)
  const uint32_t woff = static_cast<uint32_t>(n) * static_cast<uint32_t>(K >> 3) + 4u * hh;
  const uint32_t soff = static_cast<uint32_t>(n) * static_cast<uint32_t>(groups);

  // staging role: chunk (row, c) = floats 8c .. 8c + 7 of the group
  const int st = wc * 64 + lane, srow = st >> 3, sc = st & 7;
  const float* const xbase = a.x + static_cast<size_t>(rbase) * K;
  uint32_t xoff[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i)
    xoff[i] = static_cast<uint32_t>(min(srow + 8 * WC * i, a.row1 - 1 - rbase)) *
                  static_cast<uint32_t>(K) + 8u * sc;

  floatx4 xr[CPT][2];
  uint4v wd;
  uint16_t sw, bw;
  auto load = [&](int g) {
    wd = *reinterpret_cast<const uint4v*>(mine.w + 8 * g + woff);
    sw = (mine.s + g)[soff];
    bw = (mine.b + g)[soff];
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const floatx4* src = reinterpret_cast<const floatx4*>(xbase + 64 * g + xoff[i]);
      xr[i][0] = src[0];
      xr[i][1] = src[1];
    }
  };
  // the group in xr -> planes and half-group sums of stage buf
  auto stage = [&](int buf) {
    uint16_t* const dst = planes + (buf * WK + slot) * 3 * PLANE;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const floatx4 u = xr[i][0], v = xr[i][1];
      const int row = srow + 8 * WC * i;
      uint4v p1, p2, p3;
      split3x8(u, v, p1, p2, p3);
      const int at = row * 64 + 8 * (sc ^ ((row >> 1) & 7));
      *reinterpret_cast<uint4v*>(dst + at) = p1;
      *reinterpret_cast<uint4v*>(dst + PLANE + at) = p2;
      *reinterpret_cast<uint4v*>(dst + 2 * PLANE + at) = p3;
      // a half group is one lane quad: DPP quad permutations (lane ^ 1, then lane ^ 2)
      float sum = ((u[0] + u[1]) + (u[2] + u[3])) + ((v[0] + v[1]) + (v[2] + v[3]));
      sum += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sum), 0xB1, 0xf, 0xf, false));
      sum += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sum), 0x4E, 0xf, 0xf, false));
      xg[buf][slot][sc >> 2][row] = sum;  // the quad's lanes hold the same sum
    }
  };

  floatx16 acc, pair, total;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = pair[e] = total[e] = 0.0f;
  const int p0 = slot * NP;
  auto bound = [&](int p) { return p * groups / kL4Parts; };
  int g = bound(p0), part = 0, pend = bound(p0 + 1);
  const int gend = bound(p0 + NP);
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

  if (g < gend) load(g);
  for (int step = 0; step < steps; ++step, ++g) {
    const int buf = NBUF == 2 ? step & 1 : 0;
    const bool live = g < gend;
    if (NBUF == 1 && WC > 1 && step) stage_barrier();  // the group before has been read
    uint4v wcur = wd;
    const float scale = bf16_to_float(sw), bias = bf16_to_float(bw);
    if (live) stage(buf);
    if (g + 1 < gend) load(g + 1);
    if constexpr (WC > 1) {
      wait_lgkmcnt<0>();
      stage_barrier();
    } else {
      __builtin_amdgcn_wave_barrier();
    }
    if (!live) continue;
    while (part + 1 < NP && g >= pend) close();
    const uint16_t* const src = planes + (buf * WK + slot) * 3 * PLANE;
    const int arow = l32 * 64;
    // bias term: the lane's half-group sum X and b', six products of their terms in the lane's
    // k-slots
    const Split3 xs = split3(xg[buf][slot][hh][l32]), bs = split3(fmaf(8.0f, scale, bias));
    const uint32_t b12 = upper_pair(bs.t[0], bs.t[1]);
    const bf16x8 xa = __builtin_bit_cast(
        bf16x8, uint4v{upper_pair(xs.t[0], xs.t[0]), upper_pair(xs.t[1], xs.t[1]),
                       upper_pair(xs.t[0], xs.t[2]), 0u});
    const bf16x8 xb =
        __builtin_bit_cast(bf16x8, uint4v{b12, b12, upper_pair(bs.t[2], bs.t[0]), 0u});
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa, xb, acc, 0, 0, 0);
    floatx16 p;
#pragma unroll
    for (int e = 0; e < 16; ++e) p[e] = 0.0f;
    bf16x8 bq[4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) bq[s4] = decode_centred(wcur[s4]);
#pragma unroll
    for (int plane = 2; plane >= 0; --plane)  // the smallest terms first
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const bf16x8 av = *reinterpret_cast<const bf16x8*>(
            src + plane * PLANE + arow + 8 * ((4 * hh + s4) ^ ((l32 >> 1) & 7)));
        p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bq[s4], p, 0, 0, 0);
      }
    const float s16 = 16.0f * scale;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = fmaf(s16, p[e], acc[e]);
    if constexpr (WC == 1) __builtin_amdgcn_wave_barrier();
  }
  while (part < NP) close();

  // ---- sum over the slots in LDS, then whole-row stores ----
  wait_lgkmcnt<0>();
  stage_barrier();  // the x stages are free
  float* const red = reinterpret_cast<float*>(mem);
#pragma unroll
  for (int e = 0; e < 16; ++e)
    red[(wave * 32 + 8 * (e >> 2) + 4 * hh + (e & 3)) * kRedRow + l32] = total[e];
  wait_lgkmcnt<0>();
  stage_barrier();
  // V consecutive columns of a row from column block cb
  constexpr int V = TC * 32 / 512 < 4 ? TC * 32 / 512 : 4;
  auto sum_slots = [&](int cb, int row, int col, float (&y)[V]) {
    auto at = [&](int s, int j) { return red[((s * WC + cb) * 32 + row) * kRedRow + col + j]; };
#pragma unroll
    for (int j = 0; j < V; ++j) {
      if constexpr (WK == 8)
        y[j] = ((at(0, j) + at(1, j)) + (at(2, j) + at(3, j))) +
               ((at(4, j) + at(5, j)) + (at(6, j) + at(7, j)));
      else if constexpr (WK == 4)
        y[j] = (at(0, j) + at(1, j)) + (at(2, j) + at(3, j));
      else
        y[j] = at(0, j) + at(1, j);
    }
  };
  auto store = [&](const L4Set& set, int row, int c0, const float (&y)[V]) {
    float* const dst = set.out + static_cast<size_t>(row) * set.cols + c0;
    if (a.vec && V == 4 && c0 + V <= set.cols) {
      *reinterpret_cast<floatx4*>(dst) = floatx4{y[0], y[1], y[V > 2 ? 2 : 0], y[V > 2 ? 3 : 0]};
    } else if (a.vec && V == 2 && c0 + V <= set.cols) {
      *reinterpret_cast<float2v*>(dst) = float2v{y[0], y[1]};
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j)
        if (c0 + j < set.cols) dst[j] = y[j];
    }
  };
#pragma unroll
  for (int i = 0; i < TC * 32 / (512 * V); ++i) {
    const int at = V * (tid + 512 * i), row = at / TC, c = at % TC;
    if (rbase + row >= a.row1) continue;
    float y[V];
    sum_slots(c >> 5, row, c & 31, y);
    if constexpr (GATED) {
      float up[V];
      sum_slots((c >> 5) + WC / 2, row, c & 31, up);
      if (a.set[1].out) store(a.set[1], rbase + row, tile * TC + c, up);
#pragma unroll
      for (int j = 0; j < V; ++j) y[j] = silu_times(y[j], up[j]);
    }
    store(a.set[GATED ? 0 : first], rbase + row, tile * TC + c, y);
  }
}

// Column blocks per workgroup for `tiles` 32 x 32 output tiles.
int l4_blocks(int64_t tiles) { return tiles >= 2048 ? 4 : tiles >= 512 ? 2 : 1; }

template <int WC, bool GATED>
void run_rows(const L4Args& a, int sets, hipStream_t st) {
  constexpr int TC = GATED ? 16 * WC : 32 * WC;
  unsigned tiles = 0;
  for (int i = 0; i < (GATED ? 1 : sets); ++i)
    tiles += static_cast<unsigned>((a.set[i].cols + TC - 1) / TC);
  const dim3 grid(static_cast<unsigned>((a.row1 - a.row0 + 31) / 32), tiles);
  linear4_rows<WC, 8 / WC, GATED><<<grid, 512, 0, st>>>(a);
}

hipError_t launch_rows(const Linear4Job* jobs, int count, bool gated, hipStream_t st) {
  const Linear4Job& j = jobs[0];
  L4Args a{};
  a.x = j.x;
  a.row0 = j.row0;
  a.row1 = j.row1;
  a.k = j.k;
  a.vec = 1;
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i) {
    a.set[i] = L4Set{jobs[i].w, jobs[i].scales, jobs[i].biases, jobs[i].out, jobs[i].cols};
    if (jobs[i].cols % 4 || (reinterpret_cast<uintptr_t>(jobs[i].out) & 15)) a.vec = 0;
    tiles += (jobs[i].cols + 31) / 32;
  }
  tiles *= (j.row1 - j.row0 + 31) / 32;
  const int wc = l4_blocks(tiles);
  if (gated) {
    if (wc == 4)
      run_rows<4, true>(a, count, st);
    else
      run_rows<2, true>(a, count, st);
  } else if (wc == 4) {
    run_rows<4, false>(a, count, st);
  } else if (wc == 2) {
    run_rows<2, false>(a, count, st);
  } else {
    run_rows<1, false>(a, count, st);
  }
  return hipGetLastError();
}

bool runs_hilo(const Linear4Job& j, const float* scratch, size_t scratch_floats) {
  // large batches: fp16 MFMA on row-scaled hi + lo activations (fp32-grade, several times the
  // fp32 MFMA rate)
  const int rows = j.row1 - j.row0;
  const float* xr = j.x + static_cast<size_t>(j.row0) * j.k;
  const float* yr = j.out + static_cast<size_t>(j.row0) * j.cols;
  return rows >= kLinear4HiloRows && j.cols % 128 == 0 && scratch &&
         static_cast<size_t>(rows) <= scratch_floats &&
         ((reinterpret_cast<uintptr_t>(xr) | reinterpret_cast<uintptr_t>(yr)) & 15) == 0;
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

hipError_t launch_linear4_rows(const Linear4Job* jobs, int count, bool gated, hipStream_t st) {
  if (count < 1 || count > 3 || (gated && (count != 2 || jobs[0].cols != jobs[1].cols)))
    return hipErrorInvalidValue;
  for (int i = 0; i < count; ++i)
    if (jobs[i].x != jobs[0].x || jobs[i].row0 != jobs[0].row0 || jobs[i].row1 != jobs[0].row1 ||
        jobs[i].k != jobs[0].k || jobs[i].cols <= 0 || jobs[i].k <= 0 || jobs[i].k % 64)
      return hipErrorInvalidValue;
  if (jobs[0].row1 <= jobs[0].row0) return hipSuccess;
  return launch_rows(jobs, count, gated, st);
}

hipError_t launch_linear4_f32(const Linear4Job& j, float* scratch, size_t scratch_floats,
                              hipStream_t st) {
  if (j.row1 <= j.row0 || j.cols <= 0) return hipSuccess;
  if (runs_hilo(j, scratch, scratch_floats))
    return launch_linear4_hilo_f32(j.x + static_cast<size_t>(j.row0) * j.k, j.w, j.scales, j.biases,
                                   j.out + static_cast<size_t>(j.row0) * j.cols, j.row1 - j.row0,
                                   j.cols, j.k, scratch, scratch_floats, st);
  return launch_linear4_rows(&j, 1, false, st);
}

hipError_t launch_silu_gate_f32(float* gate, const float* up, uint32_t n, hipStream_t st) {
  if (!n) return hipSuccess;
  silu_gate_f32<<<(n + 255) / 256, 256, 0, st>>>(gate, up, n);
  return hipGetLastError();
}

}  // namespace tessery
