// C-ABI runtime of libtessery_hip.so: the HIP counterpart of tessery's Metal bridge
// (src/metal_inference/native/runtime.mm). See include/tessery_hip.h for the contract of every
// exported function.
//
// Design (MI355X): one HIP stream per runtime at default priority, device-resident buffers,
// commands recorded on the host and launched back to back at mi_finish (so an aborted command
// launches nothing), HIP events for command and per-dispatch timing. Routes are selected by
// tessery's kernel names; each route decodes the 64-byte Params block, derives its batch size
// from the reference thread formula and checks every buffer size before it may be queued.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <tuple>
#include <utility>
#include <vector>

#include "kernels.h"
#include "planes.h"
#include "tessery_hip.h"

using tessery::Params;

namespace {

constexpr int kAbiVersion = 2;
constexpr uint32_t kMaxBuffers = 8;
constexpr size_t kMaxProfiled = 2048;  // runtime.mm:118 (4096 timestamp samples, 2 per dispatch)
constexpr size_t kMaxPlanOps = 2048;   // runtime.mm:166

enum Route : int {
  R_ATTENTION,
  R_ATTENTION_TILED,
  R_ATTENTION_TAIL_32,
  R_ATTENTION_TAIL_128,
  R_ATTENTION_F16,
  R_ATTENTION_F16_SCALAR,
  R_ATTENTION_F16_NORM_ROPE,
  R_NORM_ROPE_F16,
  R_RMS_NORM,
  R_ROPE,
  R_LINEAR4,
  R_LINEAR4_TILED,
  R_LINEAR4_TAIL,
  R_LINEAR4_16X32,
  R_LINEAR4_32X32,
  R_LINEAR4_SMALL3,
  R_QKV4_F16,
  R_GATED4_16X32,
  R_GATED4_8X32,
  R_SILU_GATE,
  R_MATMUL,
  R_MATMUL_TILED,
  R_MATMUL_CHUNK32,
  R_MATMUL_BIAS,
  R_MATMUL_BIAS_CHUNK32,
  R_ADD_BIAS,
  R_GELU,
  R_LAYER_NORM,
  R_ADD,
  R_EMBEDDING4,
  R_EMBEDDING_POSITION,
  R_POOL_PROJECT,
  R_COPY,
  R_NONE
};

struct RouteName {
  const char* name;
  Route route;
  uint32_t buffers;
};

const RouteName kRoutes[] = {
    {"attention", R_ATTENTION, 5},
    {"attention_tiled", R_ATTENTION_TILED, 5},
    {"attention_tail_32", R_ATTENTION_TAIL_32, 5},
    {"attention_tail_128", R_ATTENTION_TAIL_128, 5},
    {"attention_f16", R_ATTENTION_F16, 5},
    {"attention_f16_scalar", R_ATTENTION_F16_SCALAR, 5},
    {"attention_f16_norm_rope", R_ATTENTION_F16_NORM_ROPE, 6},
    {"norm_rope_f16", R_NORM_ROPE_F16, 4},
    {"rms_norm", R_RMS_NORM, 3},
    {"rope", R_ROPE, 1},
    {"linear4", R_LINEAR4, 5},
    {"linear4_tiled", R_LINEAR4_TILED, 5},
    {"linear4_tail", R_LINEAR4_TAIL, 5},
    {"linear4_16x32_k64", R_LINEAR4_16X32, 5},
    {"linear4_32x32_k64", R_LINEAR4_32X32, 5},
    {"linear4_small3", R_LINEAR4_SMALL3, 5},
    {"qkv4_f16", R_QKV4_F16, 7},
    {"gated4_16x32_k64", R_GATED4_16X32, 8},
    {"gated4_8x32", R_GATED4_8X32, 8},
    {"silu_gate", R_SILU_GATE, 2},
    {"matmul_f32", R_MATMUL, 3},
    {"matmul_f32_tiled", R_MATMUL_TILED, 3},
    {"matmul_f32_chunk32", R_MATMUL_CHUNK32, 3},
    {"matmul_bias_f32", R_MATMUL_BIAS, 4},
    {"matmul_bias_f32_chunk32", R_MATMUL_BIAS_CHUNK32, 4},
    {"add_bias", R_ADD_BIAS, 2},
    {"gelu_f32", R_GELU, 1},
    {"layer_norm", R_LAYER_NORM, 4},
    {"add", R_ADD, 3},
    {"embedding4", R_EMBEDDING4, 5},
    {"embedding_position", R_EMBEDDING_POSITION, 5},
    {"pool_project", R_POOL_PROJECT, 3},
    {"copy", R_COPY, 2},
};

Route find_route(const char* name, uint32_t* nbuf) {
  if (!name) return R_NONE;
  for (const auto& r : kRoutes)
    if (std::strcmp(r.name, name) == 0) {
      *nbuf = r.buffers;
      return r.route;
    }
  return R_NONE;
}

struct Runtime;
struct Plan;

struct Buffer {
  void* ptr;
  uint64_t size;
  Runtime* owner;
};

struct Op {
  Route route;
  Params p;
  uint64_t threads;
  uint32_t group;
  uint32_t count;
  std::array<void*, kMaxBuffers> ptr;
  std::array<uint64_t, kMaxBuffers> size;
};

struct RopeTable {
  float* cos;
  float* sin;
};

// Ops [first, first + count) of the queued command came from one plan replay bound to `key` (the
// device pointers of the plan's slots).
struct Segment {
  size_t first, count;
  Plan* plan;
  std::vector<void*> key;
};

struct Runtime {
  int device = 0;
  bool graphs = true;  // replay plans through cached HIP graphs (TESSERY_HIP_GRAPHS=0 disables)
  uint64_t graph_launches = 0, graph_builds = 0;
  uint64_t fused_pairs = 0, fused_gated = 0;  // launch-time fusions (diagnostics)
  float* dense_scratch = nullptr;  // split-K partial sums of dense projections, row scales of uint4
  void* dense_planes = nullptr;    // split operands of fp32 projections
  void* planes[2] = {};  // planes of the activations uint4 projections read, and of their output
  void* wide_planes = nullptr;  // of activations beyond those
  std::vector<Segment> segments;
  hipStream_t stream = nullptr;
  hipEvent_t ev_start = nullptr, ev_end = nullptr;
  bool recording = false;
  std::vector<Op> ops;
  double last_gpu = -1.0;
  bool profiling = false;
  std::vector<hipEvent_t> prof_events;
  std::vector<double> profile_seconds;
  // per profiled op: 1 when it ran inside the kernel of the op before it (a launch-time fusion),
  // so its events enclose no work of its own
  std::vector<uint8_t> profile_fused;
  std::map<std::tuple<uint32_t, uint32_t, uint32_t>, RopeTable> rope;
  // Device allocations whose buffers were freed while a command was open: queued launches may
  // still name them, so they are released only after the command has finished or aborted.
  std::vector<void*> pending_free;
};

struct PlanOp {
  Route route;
  Params p;
  uint64_t threads;
  uint32_t group;
  uint32_t count;
  std::array<uint32_t, kMaxBuffers> slots;
};

// Launch-time fusions made while queuing a range of ops (see launch_range).
struct FusionCount {
  uint64_t pairs = 0, gated = 0;
  size_t launches = 0;  // steps of launch_next (a few are two or three kernels)
};

// An instantiated HIP graph of a plan's launches for one binding of its slots, with the fusions
// its captured launches made (added to the runtime's counts on every replay).
struct CachedGraph {
  std::vector<void*> key;
  hipGraphExec_t exec;
  FusionCount fused;
};

struct Plan {
  Runtime* owner;
  std::vector<uint64_t> sizes;
  std::vector<PlanOp> ops;
  std::vector<CachedGraph> graphs;  // most recently used last, at most kPlanGraphs
  bool direct = false;              // too short for a graph (see kGraphLaunches)
};

constexpr size_t kPlanGraphs = 4;
// A plan of fewer launches is replayed launch by launch: up to five launches start at once, the sixth
// costs 10 to 17 us more, and from there on a graph costs less. Measured per replay, as a graph and
// directly: attention of one 24-token query 4 launches 58.8 and 45.6 us, 5 62.0 and 51.5, 6 66.6 and
// 68.8, 7 73.4 and 76.9, 9 89.0 and 94.3; projection and attention of 24 tokens 4 launches 84.7 and
// 72.6, 6 109.6 and 111.5; of a 32 x 464 batch, attention 5 launches 490.6 and 485.6, 6 610.7 and 609.9;
// 10 launches of a decoder layer 87.8 and 96.5.
constexpr size_t kGraphLaunches = 6;

inline uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// ---- shape derivation -------------------------------------------------------------------------

struct AttnShape {
  uint64_t B, S, H, KV, D;
  int in_f16, out_f16;
};

constexpr uint64_t kMaxTokens = 0x7fffffffull;  // launchers take row counts as int
// Row-per-wavefront kernels (rms_norm, layer_norm, pool_project) launch 64 lanes per row on a
// 1-D grid, and elementwise kernels round n up to whole 256-lane workgroups in 32-bit arithmetic.
constexpr uint64_t kMaxWaveRows = (1ull << 26) - 4;
constexpr uint64_t kMaxElements = (1ull << 32) - 256;

bool attn_shape(Route r, const Params& p, uint64_t threads, uint32_t group, AttnShape* s) {
  const uint64_t H = p.heads, KV = p.kv_heads, S = p.seq, D = p.dim;
  if (!H || !KV || H % KV || !S || !D || H > 1024 || D > 1024 || S > (1u << 20)) return false;
  uint64_t tokens = 0;
  s->in_f16 = 0;
  s->out_f16 = 0;
  switch (r) {
    case R_ATTENTION:  // metal.py:560-569, scalar: tokens*heads*32 threads, groups of 32
      if (group != 32 || threads % (H * 32) || D > 256) return false;
      tokens = threads / (H * 32);
      break;
    case R_ATTENTION_TILED:  // (tokens/8)*heads*128 threads, groups of 128
      if (group != 128 || threads % (H * 128) || S % 8 || (D != 32 && D != 64 && D != 128))
        return false;
      tokens = threads / (H * 128) * 8;
      break;
    case R_ATTENTION_TAIL_32:
    case R_ATTENTION_TAIL_128: {  // metal.py:544-555: B*ceil(S/8)*heads*128 threads
      const uint64_t want = r == R_ATTENTION_TAIL_32 ? 32 : 128;
      const uint64_t per = ceil_div(S, 8) * H * 128;
      if (group != 128 || D != want || threads % per) return false;
      tokens = threads / per * S;
      break;
    }
    case R_ATTENTION_F16:
    case R_ATTENTION_F16_NORM_ROPE:
      if (group != 256 || (D != 64 && D != 128)) return false;
      tokens = threads;
      s->in_f16 = 1;
      s->out_f16 = p.u1 & 1u;
      break;
    case R_ATTENTION_F16_SCALAR:
      if (group != 64 || D > 256) return false;
      tokens = threads;
      s->in_f16 = 1;
      s->out_f16 = p.u1 & 1u;
      break;
    default:
      return false;
  }
  if (!tokens || tokens % S || tokens > kMaxTokens) return false;
  s->B = tokens / S;
  s->S = S;
  s->H = H;
  s->KV = KV;
  s->D = D;
  return true;
}

bool attn_sizes(const AttnShape& s, const uint64_t* sz) {
  const uint64_t ein = s.in_f16 ? 2 : 4, eout = s.out_f16 ? 2 : 4;
  const uint64_t qn = s.B * s.S * s.H * s.D, kn = s.B * s.S * s.KV * s.D;
  return qn * ein <= sz[0] && kn * ein <= sz[1] && kn * ein <= sz[2] && s.B * 4 <= sz[3] &&
         qn * eout <= sz[4];
}

struct RowRange {
  uint64_t r0, r1;
};

bool linear4_range(Route r, const Params& p, uint64_t threads, uint32_t group, RowRange* out) {
  const uint64_t rows = p.rows, cols = p.cols, k = p.k, n = p.n;
  if (!rows || !cols || !k || k % 64 || rows > kMaxTokens || cols > 65536 || k > 65536)
    return false;
  switch (r) {
    case R_LINEAR4: {  // kernels.metal:32-51: rows n + 4*(threadgroup / cols) + t
      if (group != 32 || threads % (cols * 32)) return false;
      const uint64_t blocks = threads / (cols * 32);
      out->r0 = n;
      out->r1 = std::min(n + 4 * blocks, rows);
      break;
    }
    case R_LINEAR4_TILED: {  // kernels.metal:489-520: 8-row tiles from row n
      const uint64_t per = (cols / 32) * 128;
      if (group != 128 || cols % 32 || threads % per) return false;
      out->r0 = n;
      out->r1 = n + 8 * (threads / per);
      if (out->r1 > rows) return false;
      break;
    }
    case R_LINEAR4_TAIL:  // kernels.metal:560-605: one partial 8-row tile from row n
      if (group != 128 || cols % 32 || threads != (cols / 32) * 128) return false;
      out->r0 = n;
      out->r1 = std::min(n + 8, rows);
      break;
    case R_LINEAR4_16X32:  // kernels.metal:522-558: 16-row tiles from row 0
    case R_LINEAR4_32X32: {  // kernels.metal:733-773: 32-row tiles from row 0
      const uint64_t tile = r == R_LINEAR4_16X32 ? 16 : 32;
      const uint64_t per = (cols / 32) * 256;
      if (group != 256 || cols % 32 || threads % per) return false;
      out->r0 = 0;
      out->r1 = tile * (threads / per);
      if (out->r1 > rows) return false;
      break;
    }
    case R_LINEAR4_SMALL3:  // kernels.metal:655-684: exactly three rows
      if (group != 32 || threads != cols * 32 || rows != 3) return false;
      out->r0 = 0;
      out->r1 = 3;
      break;
    default:
      return false;
  }
  return out->r0 < out->r1;
}

// Rows of a fused gate/up launch: gated4_16x32_k64 runs 16-row tiles from row 0
// (kernels.metal:609-616), gated4_8x32 one complete 8-row tile from row n (kernels.metal:687-694).
bool gated4_range(Route r, const Params& p, uint64_t threads, uint32_t group, RowRange* out) {
  const uint64_t rows = p.rows, cols = p.cols, k = p.k, n = p.n;
  if (!rows || !cols || !k || k % 64 || cols % 32 || rows > kMaxTokens || cols > 65536 ||
      k > 65536)
    return false;
  if (r == R_GATED4_16X32) {
    const uint64_t per = (cols / 32) * 256;
    if (group != 256 || threads % per) return false;
    out->r0 = 0;
    out->r1 = 16 * (threads / per);
  } else {
    if (group != 128 || threads != (cols / 32) * 128) return false;
    out->r0 = n;
    out->r1 = n + 8;
  }
  return out->r0 < out->r1 && out->r1 <= rows;
}

// Rows of an fp32 dense projection: the scalar routes cover rows n + 4 * (group / cols) + t
// (kernels.metal:306-322, 438-455), the tiled ones 8-row tiles from row 0 (kernels.metal:396-436,
// 457-487).
bool matmul_range(Route r, const Params& p, uint64_t threads, uint32_t group, RowRange* out) {
  const uint64_t rows = p.rows, cols = p.cols, k = p.k, n = p.n;
  if (!rows || !cols || !k || rows > kMaxTokens || cols > 65536 || k > 65536) return false;
  if (r == R_MATMUL || r == R_MATMUL_BIAS) {
    if (group != 32 || threads % (cols * 32)) return false;
    out->r0 = n;
    out->r1 = std::min(n + 4 * (threads / (cols * 32)), rows);
  } else {
    const uint64_t per = (cols / 32) * 128;
    if (group != 128 || cols % 32 || threads % per) return false;
    out->r0 = 0;
    out->r1 = 8 * (threads / per);
    if (out->r1 > rows) return false;
  }
  return out->r0 < out->r1;
}

// Validates one launch against the buffer sizes it would touch. Pure: no allocation.
bool validate(Route r, const Params& p, uint64_t threads, uint32_t group, const uint64_t* sz,
              uint32_t count, uint32_t nbuf) {
  if (count != nbuf || !threads || !group) return false;
  switch (r) {
    case R_ATTENTION:
    case R_ATTENTION_TILED:
    case R_ATTENTION_TAIL_32:
    case R_ATTENTION_TAIL_128:
    case R_ATTENTION_F16:
    case R_ATTENTION_F16_SCALAR:
    case R_ATTENTION_F16_NORM_ROPE: {
      AttnShape s;
      if (!attn_shape(r, p, threads, group, &s) || !attn_sizes(s, sz)) return false;
      const int B = static_cast<int>(s.B), S = static_cast<int>(s.S), H = static_cast<int>(s.H),
                KV = static_cast<int>(s.KV), D = static_cast<int>(s.D);
      if (r == R_ATTENTION || r == R_ATTENTION_F16_SCALAR) {
        if (!tessery::attention_scalar_fits(s.B, s.S, s.H)) return false;
      } else if (r == R_ATTENTION_F16 || r == R_ATTENTION_F16_NORM_ROPE) {
        if (!tessery::attention_f16_fits(B, S, H, KV, D)) return false;
      } else if (!tessery::attention_f32_fits(B, S, H, KV)) {
        return false;
      }
      if (r == R_ATTENTION_F16_NORM_ROPE)  // k holds hi and lo planes
          return sz[1] >= 2 * s.B * s.S * s.KV * s.D * 2 && sz[5] >= s.D * 2 && p.theta > 0.0f &&
               p.eps >= 0.0f && std::isfinite(p.theta) && tessery::rope_tables_fit(S, D);
      return true;
    }
    case R_NORM_ROPE_F16: {  // buffers: x, gamma, lengths, y; u1 bit 0: y gets hi + lo planes
      const uint64_t heads = p.heads, S = p.seq, D = p.dim, tokens = threads;
      if (group != 256 || !heads || heads > 1024 || !S || tokens % S || tokens > kMaxTokens ||
          (D != 32 && D != 64 && D != 128) || !(p.theta > 0.0f) || !std::isfinite(p.theta))
        return false;
      if (!tessery::norm_rope_f16_fits(static_cast<int>(tokens / S), static_cast<int>(S),
                                       static_cast<int>(heads), static_cast<int>(D)) ||
          !tessery::rope_tables_fit(static_cast<int>(S), static_cast<int>(D)))
        return false;
      const uint64_t bytes = tokens * heads * D * 2;
      const uint64_t planes = (p.u1 & 1u) ? 2 : 1;
      return sz[0] >= bytes && sz[1] >= D * 2 && sz[2] >= tokens / S * 4 &&
             sz[3] >= planes * bytes;
    }
    case R_RMS_NORM: {  // kernels.metal:53-63: rows*32 threads, groups of 32
      const uint64_t cols = p.cols;
      if (group != 32 || threads % 32 || !cols || cols > 65536) return false;
      const uint64_t rows = threads / 32;
      if (rows > kMaxWaveRows) return false;
      return sz[0] >= rows * cols * 4 && sz[1] >= cols * 2 && sz[2] >= rows * cols * 4;
    }
    case R_ROPE: {  // kernels.metal:65-74: n threads, n = tokens*heads*dim/2
      const uint64_t n = p.n, D = p.dim;
      if (!n || !D || D % 2 || D > 1024 || !p.heads || !p.seq || n % (D / 2) ||
          n > kMaxElements || !(p.theta > 0.0f) || !std::isfinite(p.theta) ||
          !tessery::rope_tables_fit(static_cast<int>(p.seq), static_cast<int>(D)))
        return false;
      return sz[0] >= n * 2 * 4;
    }
    case R_LINEAR4:
    case R_LINEAR4_TILED:
    case R_LINEAR4_TAIL:
    case R_LINEAR4_16X32:
    case R_LINEAR4_32X32:
    case R_LINEAR4_SMALL3: {
      RowRange rr;
      if (!linear4_range(r, p, threads, group, &rr)) return false;
      const uint64_t cols = p.cols, k = p.k;
      return sz[0] >= rr.r1 * k * 4 && sz[1] >= cols * (k / 8) * 4 &&
             sz[2] >= cols * (k / 64) * 2 && sz[3] >= cols * (k / 64) * 2 &&
             sz[4] >= rr.r1 * cols * 4;
    }
    case R_QKV4_F16: {  // buffers: x, w_qkv, s_qkv, b_qkv, yq, yk, yv (weights concatenated on N)
      const uint64_t M = p.rows, K = p.k, nq = p.cols, nkv = p.n, ntot = nq + 2 * nkv;
      if (group != 256 || threads != M || !M || M > kMaxTokens || !K || K % 64 || K > 65536 ||
          !nq || nq % 128 || !nkv || nkv % 128 || ntot > 65536)
        return false;
      const int widths[3] = {static_cast<int>(nq), static_cast<int>(nkv), static_cast<int>(nkv)};
      if (!tessery::qkv4_f16_fits(static_cast<int>(M), static_cast<int>(K), widths)) return false;
      return sz[0] >= M * K * 2 && sz[1] >= ntot * (K / 8) * 4 && sz[2] >= ntot * (K / 64) * 2 &&
             sz[3] >= ntot * (K / 64) * 2 && sz[4] >= M * nq * 2 && sz[5] >= M * nkv * 2 &&
             sz[6] >= M * nkv * 2;
    }
    case R_GATED4_16X32:
    case R_GATED4_8X32: {  // buffers: x, w, s, b, up w, up s, up b, out
      RowRange rr;
      if (!gated4_range(r, p, threads, group, &rr)) return false;
      const uint64_t cols = p.cols, k = p.k;
      const uint64_t wb = cols * (k / 8) * 4, sb = cols * (k / 64) * 2;
      return sz[0] >= rr.r1 * k * 4 && sz[1] >= wb && sz[2] >= sb && sz[3] >= sb &&
             sz[4] >= wb && sz[5] >= sb && sz[6] >= sb && sz[7] >= rr.r1 * cols * 4;
    }
    case R_MATMUL:
    case R_MATMUL_TILED:
    case R_MATMUL_CHUNK32:
    case R_MATMUL_BIAS:
    case R_MATMUL_BIAS_CHUNK32: {  // buffers: a [rows, k], bt [cols, k], out [rows, cols], bias
      RowRange rr;
      if (!matmul_range(r, p, threads, group, &rr)) return false;
      const uint64_t cols = p.cols, k = p.k;
      const bool bias = r == R_MATMUL_BIAS || r == R_MATMUL_BIAS_CHUNK32;
      return sz[0] >= rr.r1 * k * 4 && sz[1] >= cols * k * 4 && sz[2] >= rr.r1 * cols * 4 &&
             (!bias || sz[3] >= cols * 4);
    }
    case R_ADD_BIAS: {  // kernels.metal:376-379: x, bias
      const uint64_t n = p.n, cols = p.cols;
      return n && cols && n <= (1ull << 32) - 256 && sz[0] >= n * 4 &&
             sz[1] >= std::min(n, cols) * 4;
    }
    case R_GELU: {  // kernels.metal:381-394
      const uint64_t n = p.n;
      return n && n <= (1ull << 32) - 256 && sz[0] >= n * 4;
    }
    case R_LAYER_NORM: {  // kernels.metal:362-374: rows*32 threads, groups of 32; x, w, bias, out
      const uint64_t cols = p.cols;
      if (group != 32 || threads % 32 || !cols || cols > 65536) return false;
      const uint64_t rows = threads / 32;
      if (rows > kMaxWaveRows) return false;
      return sz[0] >= rows * cols * 4 && sz[1] >= cols * 4 && sz[2] >= cols * 4 &&
             sz[3] >= rows * cols * 4;
    }
    case R_SILU_GATE: {  // kernels.metal:334-337: gate, up
      const uint64_t n = p.n;
      return n && n <= (1ull << 32) - 256 && sz[0] >= n * 4 && sz[1] >= n * 4;
    }
    case R_ADD: {  // kernels.metal:300-304
      const uint64_t n = p.n;
      return n && n <= kMaxElements && sz[0] >= n * 4 && sz[1] >= n * 4 && sz[2] >= n * 4;
    }
    case R_EMBEDDING4: {  // kernels.metal:21-30: ids, w, scales, biases, out; n = tokens*cols
      const uint64_t n = p.n, cols = p.cols;
      if (!n || !cols || cols % 64 || cols > 65536 || n % cols || n / cols > kMaxTokens * 16)
        return false;
      const uint64_t vocab = sz[1] / (cols / 2);
      return vocab && vocab <= 0xffffffffull && sz[0] >= n / cols * 4 &&
             sz[2] >= vocab * (cols / 64) * 2 && sz[3] >= vocab * (cols / 64) * 2 &&
             sz[4] >= n * 4;
    }
    case R_EMBEDDING_POSITION: {  // kernels.metal:351-360: ids, words, positions, types, out
      const uint64_t n = p.n, cols = p.cols, seq = p.seq;
      if (!n || !cols || cols > 65536 || n % cols || !seq || n / cols > kMaxTokens * 16)
        return false;
      const uint64_t vocab = sz[1] / (cols * 4);
      return vocab && vocab <= 0xffffffffull && sz[0] >= n / cols * 4 &&
             sz[2] >= seq * cols * 4 && sz[3] >= cols * 4 && sz[4] >= n * 4;
    }
    case R_POOL_PROJECT: {  // kernels.metal:339-349: x, lengths, out; batch*32 threads
      const uint64_t cols = p.cols, seq = p.seq, dim = p.dim;
      if (group != 32 || !threads || threads % 32 || !cols || !seq || !dim || dim > cols)
        return false;
      const uint64_t batch = threads / 32;
      if (batch > kMaxWaveRows) return false;
      return sz[0] >= batch * seq * cols * 4 && (p.u1 || sz[1] >= batch * 4) &&
             sz[2] >= batch * dim * 4;
    }
    case R_COPY:
      return threads % 16 == 0 && sz[0] >= threads && sz[1] >= threads;
    default:
      return false;
  }
}

// ---- RoPE tables ------------------------------------------------------------------------------

uint32_t float_bits(float f) {
  uint32_t u;
  std::memcpy(&u, &f, sizeof u);
  return u;
}

// cos/sin[pos][c] = cos/sin(pos * theta^(-2c/D)), evaluated in float64 and rounded once, by a
// kernel on the runtime stream: queued launches of the open command run after it.
bool ensure_rope(Runtime* rt, uint32_t seq, uint32_t dim, float theta) {
  const auto key = std::make_tuple(seq, dim, float_bits(theta));
  if (rt->rope.count(key)) return true;
  const size_t bytes = static_cast<size_t>(seq) * (dim / 2) * sizeof(float);
  RopeTable t{nullptr, nullptr};
  if (hipMalloc(&t.cos, bytes) != hipSuccess) return false;
  if (hipMalloc(&t.sin, bytes) != hipSuccess) {
    (void)hipFree(t.cos);
    return false;
  }
  if (tessery::launch_rope_tables(t.cos, t.sin, static_cast<int>(seq), static_cast<int>(dim),
                                  theta, rt->stream) != hipSuccess) {
    (void)hipStreamSynchronize(rt->stream);
    (void)hipFree(t.cos);
    (void)hipFree(t.sin);
    return false;
  }
  rt->rope[key] = t;
  return true;
}

bool is_linear4(Route r) {
  return r == R_LINEAR4 || r == R_LINEAR4_TILED || r == R_LINEAR4_TAIL || r == R_LINEAR4_16X32 ||
         r == R_LINEAR4_32X32 || r == R_LINEAR4_SMALL3;
}

bool is_gated4(Route r) { return r == R_GATED4_16X32 || r == R_GATED4_8X32; }

bool is_dense(Route r) {
  return r == R_MATMUL || r == R_MATMUL_TILED || r == R_MATMUL_CHUNK32 || r == R_MATMUL_BIAS ||
         r == R_MATMUL_BIAS_CHUNK32;
}

// Scratch is allocated by the first op that runs on it and kept for the runtime's life (a captured graph
// keeps pointing at it). Split-K partial sums of dense projections, and the row scales that the
// fp16-MFMA uint4 projections read:
constexpr size_t kDenseScratchFloats = size_t{8} << 20;  // 32 MiB
// Split operands of the dense projections: at most 512 tiles of 64 x 128 outputs (more run on
// matmul_x3), which is 96 MiB where they are one column of tiles of K = 512.
constexpr size_t kDensePlanesBytes = size_t{104} << 20;
// Each of the two planes scratches: 1023 rows (more run on linear4_hilo) of 3072 inputs, Qwen3's
// widest, in 18.4 MiB.
constexpr size_t kPlanesBytes = size_t{20} << 20;
// Wider inputs: 1023 rows of 8192. What exceeds it goes through in row ranges, one after the other,
// each too few tiles for the chip where the columns are few (1000 x 64 outputs of K = 8192: 100.4 us
// in three ranges of 20 MiB, 39.1 in one; of K = 4096 43.2 and 23.3).
constexpr size_t kWidePlanesBytes = size_t{49} << 20;

const RopeTable* rope_of(Runtime* rt, const Params& p) {
  auto it = rt->rope.find(std::make_tuple(p.seq, p.dim, float_bits(p.theta)));
  return it == rt->rope.end() ? nullptr : &it->second;
}

// ---- launch -----------------------------------------------------------------------------------

// Kernel arguments of a qkv4_f16 op: buffers x, w_qkv, s_qkv, b_qkv, yq, yk, yv with the three
// weight sets concatenated on N (q first); no k prologue.
tessery::Qkv4Args qkv4_args(const Op& op) {
  const Params& p = op.p;
  tessery::Qkv4Args a{};
  const int K = static_cast<int>(p.k);
  const int nq = static_cast<int>(p.cols), nkv = static_cast<int>(p.n);
  const int offsets[3] = {0, nq, nq + nkv};
  a.x = static_cast<const _Float16*>(op.ptr[0]);
  for (int i = 0; i < 3; ++i) {
    a.w[i] = static_cast<const uint32_t*>(op.ptr[1]) + static_cast<size_t>(offsets[i]) * (K / 8);
    a.s[i] = static_cast<const uint16_t*>(op.ptr[2]) + static_cast<size_t>(offsets[i]) * (K / 64);
    a.b[i] = static_cast<const uint16_t*>(op.ptr[3]) + static_cast<size_t>(offsets[i]) * (K / 64);
    a.y[i] = static_cast<_Float16*>(op.ptr[4 + i]);
    a.n[i] = i == 0 ? nq : nkv;
  }
  a.M = static_cast<int>(p.rows);
  a.K = K;
  a.scale_bf16 = p.u1 & 1u;
  return a;
}

// Kernel arguments of an attention-family op (buffers q, k, v, lengths, out [, q_norm]).
bool attention_args(Runtime* rt, const Op& op, tessery::AttnArgs* out) {
  const Params& p = op.p;
  AttnShape s;
  if (!attn_shape(op.route, p, op.threads, op.group, &s)) return false;
  tessery::AttnArgs a{};
  a.q = op.ptr[0];
  a.k = op.ptr[1];
  a.v = op.ptr[2];
  a.lengths = static_cast<const uint32_t*>(op.ptr[3]);
  a.out = op.ptr[4];
  a.B = static_cast<int>(s.B);
  a.S = static_cast<int>(s.S);
  a.H = static_cast<int>(s.H);
  a.KV = static_cast<int>(s.KV);
  a.D = static_cast<int>(s.D);
  a.scale = p.scale;
  a.bidi = p.u0 ? 1 : 0;
  a.in_f16 = s.in_f16;
  a.out_f16 = s.out_f16;
  a.eps = p.eps;
  if (op.route == R_ATTENTION_F16_NORM_ROPE) {
    const RopeTable* t = rope_of(rt, p);
    if (!t) return false;
    a.gamma_q = static_cast<const uint16_t*>(op.ptr[5]);
    a.rope_cos = t->cos;
    a.rope_sin = t->sin;
  }
  *out = a;
  return true;
}

// The projection of a linear4 op (buffers x, w, scales, biases, out).
bool linear4_job(const Op& op, tessery::Linear4Job* job) {
  RowRange rr;
  if (!is_linear4(op.route) || !linear4_range(op.route, op.p, op.threads, op.group, &rr))
    return false;
  *job = {static_cast<const float*>(op.ptr[0]),    static_cast<const uint32_t*>(op.ptr[1]),
          static_cast<const uint16_t*>(op.ptr[2]), static_cast<const uint16_t*>(op.ptr[3]),
          static_cast<float*>(op.ptr[4]),          static_cast<int>(rr.r0),
          static_cast<int>(rr.r1),                 static_cast<int>(op.p.cols),
          static_cast<int>(op.p.k)};
  return true;
}

// Gate and up projections of a gated4 op (buffers x, w, s, b, up w, up s, up b, out).
bool gated4_jobs(const Op& op, tessery::Linear4Job* jobs) {
  RowRange rr;
  if (!is_gated4(op.route) || !gated4_range(op.route, op.p, op.threads, op.group, &rr))
    return false;
  for (int i = 0; i < 2; ++i)
    jobs[i] = {static_cast<const float*>(op.ptr[0]),
               static_cast<const uint32_t*>(op.ptr[1 + 3 * i]),
               static_cast<const uint16_t*>(op.ptr[2 + 3 * i]),
               static_cast<const uint16_t*>(op.ptr[3 + 3 * i]),
               i == 0 ? static_cast<float*>(op.ptr[7]) : nullptr,
               static_cast<int>(rr.r0),
               static_cast<int>(rr.r1),
               static_cast<int>(op.p.cols),
               static_cast<int>(op.p.k)};
  return true;
}

// The projection of a dense op (buffers a, bt, out [, bias]).
bool dense_job(const Op& op, tessery::DenseJob* job) {
  RowRange rr;
  if (!is_dense(op.route) || !matmul_range(op.route, op.p, op.threads, op.group, &rr)) return false;
  const bool bias = op.route == R_MATMUL_BIAS || op.route == R_MATMUL_BIAS_CHUNK32;
  *job = {static_cast<const float*>(op.ptr[0]),
          static_cast<const float*>(op.ptr[1]),
          bias ? static_cast<const float*>(op.ptr[3]) : nullptr,
          static_cast<float*>(op.ptr[2]),
          static_cast<int>(rr.r0),
          static_cast<int>(rr.r1),
          static_cast<int>(op.p.cols),
          static_cast<int>(op.p.k)};
  return true;
}

tessery::DenseScratch dense_scratch(Runtime* rt) {
  return {rt->dense_scratch, kDenseScratchFloats, rt->dense_planes, kDensePlanesBytes};
}

// `in` is the planes scratch `slot`, `out` the other one.
tessery::PlanesScratch planes_scratch(Runtime* rt, int slot) {
  return {rt->planes[slot], rt->planes[1 - slot], kPlanesBytes};
}

// Allocates *block once; false (and no error left for the launches to find) when it cannot be had.
template <typename T>
bool have_scratch(T** block, size_t bytes) {
  if (!*block && hipMalloc(reinterpret_cast<void**>(block), bytes) != hipSuccess) {
    *block = nullptr;
    (void)hipGetLastError();
  }
  return *block;
}

// What op needs beside its buffers. A scratch that another kernel does without is left out when it
// cannot be had.
bool prepare(Runtime* rt, const Op& op) {
  const Params& p = op.p;
  const size_t sums_bytes = kDenseScratchFloats * sizeof(float);
  if (op.route == R_ATTENTION_F16_NORM_ROPE || op.route == R_NORM_ROPE_F16 || op.route == R_ROPE)
    return ensure_rope(rt, p.seq, p.dim, p.theta);
  tessery::DenseJob dense;
  if (dense_job(op, &dense)) {
    if (tessery::matmul_reads_planes(dense, kDensePlanesBytes))
      (void)have_scratch(&rt->dense_planes, kDensePlanesBytes);
    return have_scratch(&rt->dense_scratch, sums_bytes);
  }
  tessery::Linear4Job job, gated[2];
  if (linear4_job(op, &job)) {
    if (job.row1 - job.row0 >= tessery::kLinear4HiloRows &&
        have_scratch(&rt->dense_scratch, sums_bytes) &&
        !tessery::linear4_on_rows(job, rt->dense_scratch, kDenseScratchFloats))
      return true;
  } else if (gated4_jobs(op, gated)) {
    job = gated[0];
  } else {
    return true;
  }
  if (tessery::planes_bytes(job.row1 - job.row0, job.k) > kPlanesBytes)
    (void)have_scratch(&rt->wide_planes, kWidePlanesBytes);
  (void)have_scratch(&rt->planes[1], kPlanesBytes);
  return have_scratch(&rt->planes[0], kPlanesBytes);
}

// What a launch leaves and finds beside its op's buffers: where a rms_norm or an attention also puts
// its output as planes, where a rms_norm puts the row scales of its output (null: nowhere), and
// whether a projection finds the row scales of its input in the dense scratch.
struct Beside {
  void* planes = nullptr;
  float* scales = nullptr;
  bool scaled = false;
};

hipError_t launch(Runtime* rt, const Op& op, const Beside& beside) {
  hipStream_t st = rt->stream;
  const Params& p = op.p;
  switch (op.route) {
    case R_ATTENTION:
    case R_ATTENTION_TILED:
    case R_ATTENTION_TAIL_32:
    case R_ATTENTION_TAIL_128:
    case R_ATTENTION_F16:
    case R_ATTENTION_F16_SCALAR:
    case R_ATTENTION_F16_NORM_ROPE: {
      tessery::AttnArgs a{};
      if (!attention_args(rt, op, &a)) return hipErrorInvalidValue;
      a.planes = beside.planes;
      if (op.route == R_ATTENTION || op.route == R_ATTENTION_F16_SCALAR)
        return tessery::launch_attention_scalar(a, st);
      if (op.route == R_ATTENTION_F16 || op.route == R_ATTENTION_F16_NORM_ROPE)
        return tessery::launch_attention_f16(a, st);
      return tessery::launch_attention_f32(a, st);
    }
    case R_NORM_ROPE_F16: {
      const RopeTable* t = rope_of(rt, p);
      if (!t) return hipErrorInvalidValue;
      return tessery::launch_norm_rope_f16(
          static_cast<const _Float16*>(op.ptr[0]), static_cast<_Float16*>(op.ptr[3]),
          static_cast<const uint16_t*>(op.ptr[1]), t->cos, t->sin,
          static_cast<const uint32_t*>(op.ptr[2]), static_cast<int>(op.threads / p.seq),
          static_cast<int>(p.seq), static_cast<int>(p.heads), static_cast<int>(p.dim), p.eps,
          (p.u1 & 1u) != 0, st);
    }
    case R_RMS_NORM:
      return tessery::launch_rms_norm_f32(
          static_cast<const float*>(op.ptr[0]), static_cast<const uint16_t*>(op.ptr[1]),
          static_cast<float*>(op.ptr[2]), static_cast<int>(op.threads / 32),
          static_cast<int>(p.cols), p.eps, beside.planes, beside.scales, st);
    case R_ROPE: {
      const RopeTable* t = rope_of(rt, p);
      if (!t) return hipErrorInvalidValue;
      return tessery::launch_rope_f32(static_cast<float*>(op.ptr[0]), t->cos, t->sin, p.n,
                                      static_cast<int>(p.heads), static_cast<int>(p.seq),
                                      static_cast<int>(p.dim), st);
    }
    case R_LINEAR4:
    case R_LINEAR4_TILED:
    case R_LINEAR4_TAIL:
    case R_LINEAR4_16X32:
    case R_LINEAR4_32X32:
    case R_LINEAR4_SMALL3: {
      tessery::Linear4Job job;
      if (!linear4_job(op, &job)) return hipErrorInvalidValue;
      return tessery::launch_linear4_f32(job, rt->dense_scratch, kDenseScratchFloats, beside.scaled,
                                         planes_scratch(rt, 0), st);
    }
    case R_QKV4_F16:
      return tessery::launch_qkv4_f16(qkv4_args(op), st);
    case R_GATED4_16X32:
    case R_GATED4_8X32: {
      tessery::Linear4Job jobs[2];
      if (!gated4_jobs(op, jobs)) return hipErrorInvalidValue;
      return tessery::launch_linear4_rows(jobs, 2, true, planes_scratch(rt, 0), false, false, st);
    }
    case R_SILU_GATE:
      return tessery::launch_silu_gate_f32(static_cast<float*>(op.ptr[0]),
                                           static_cast<const float*>(op.ptr[1]), p.n, st);
    case R_MATMUL:
    case R_MATMUL_TILED:
    case R_MATMUL_CHUNK32:
    case R_MATMUL_BIAS:
    case R_MATMUL_BIAS_CHUNK32: {
      tessery::DenseJob job;
      if (!dense_job(op, &job)) return hipErrorInvalidValue;
      return tessery::launch_matmul_f32(job, false, dense_scratch(rt), st);
    }
    case R_ADD_BIAS:
      return tessery::launch_add_bias_f32(static_cast<float*>(op.ptr[0]),
                                          static_cast<const float*>(op.ptr[1]), p.n, p.cols, st);
    case R_GELU:
      return tessery::launch_gelu_f32(static_cast<float*>(op.ptr[0]), p.n, st);
    case R_LAYER_NORM:
      return tessery::launch_layer_norm_f32(
          static_cast<const float*>(op.ptr[0]), static_cast<const float*>(op.ptr[1]),
          static_cast<const float*>(op.ptr[2]), static_cast<float*>(op.ptr[3]),
          static_cast<int>(op.threads / 32), static_cast<int>(p.cols), p.eps, st);
    case R_ADD:
      return tessery::launch_add_f32(static_cast<const float*>(op.ptr[0]),
                                     static_cast<const float*>(op.ptr[1]),
                                     static_cast<float*>(op.ptr[2]), p.n, st);
    case R_EMBEDDING4:
      return tessery::launch_embedding4_f32(
          static_cast<const uint32_t*>(op.ptr[0]), static_cast<const uint32_t*>(op.ptr[1]),
          static_cast<const uint16_t*>(op.ptr[2]), static_cast<const uint16_t*>(op.ptr[3]),
          static_cast<float*>(op.ptr[4]), p.n, p.cols,
          static_cast<uint32_t>(op.size[1] / (p.cols / 2)), st);
    case R_EMBEDDING_POSITION:
      return tessery::launch_embedding_position_f32(
          static_cast<const uint32_t*>(op.ptr[0]), static_cast<const float*>(op.ptr[1]),
          static_cast<const float*>(op.ptr[2]), static_cast<const float*>(op.ptr[3]),
          static_cast<float*>(op.ptr[4]), p.n, p.cols, p.seq,
          static_cast<uint32_t>(op.size[1] / (static_cast<uint64_t>(p.cols) * 4)), st);
    case R_POOL_PROJECT:
      return tessery::launch_pool_project_f32(
          static_cast<const float*>(op.ptr[0]), static_cast<const uint32_t*>(op.ptr[1]),
          static_cast<float*>(op.ptr[2]), static_cast<uint32_t>(op.threads / 32), p.seq, p.cols,
          p.dim, p.u1 != 0, st);
    case R_COPY:
      return tessery::launch_copy(op.ptr[0], op.ptr[1], op.threads, st);
    default:
      return hipErrorInvalidValue;
  }
}

bool make_op(Route r, const Params& p, uint64_t threads, uint32_t group, void* const* ptrs,
             const uint64_t* sizes, uint32_t count, Op* op) {
  op->route = r;
  op->p = p;
  op->threads = threads;
  op->group = group;
  op->count = count;
  for (uint32_t i = 0; i < kMaxBuffers; ++i) {
    op->ptr[i] = i < count ? ptrs[i] : nullptr;
    op->size[i] = i < count ? sizes[i] : 0;
  }
  return true;
}

bool queue_op(Runtime* rt, const Op& op) {
  if (rt->profiling && rt->ops.size() >= kMaxProfiled) return false;
  rt->ops.push_back(op);
  return true;
}

void release_profile_events(Runtime* rt) {
  for (hipEvent_t e : rt->prof_events) (void)hipEventDestroy(e);
  rt->prof_events.clear();
}

// Frees the allocations of buffers released during the last command, once nothing launched on
// the stream can still use them.
void release_pending(Runtime* rt) {
  if (rt->pending_free.empty()) return;
  (void)hipStreamSynchronize(rt->stream);
  for (void* p : rt->pending_free) (void)hipFree(p);
  rt->pending_free.clear();
}

}  // namespace

extern "C" {

int mi_abi_version(void) { return kAbiVersion; }

void* mi_create(const char* /*source*/) {
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return nullptr;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return nullptr;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) return nullptr;
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return nullptr;
  auto rt = new Runtime();
  rt->device = device;
  const char* graphs = std::getenv("TESSERY_HIP_GRAPHS");
  rt->graphs = !(graphs && std::strcmp(graphs, "0") == 0);
  if (hipStreamCreateWithFlags(&rt->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&rt->ev_start) != hipSuccess || hipEventCreate(&rt->ev_end) != hipSuccess) {
    mi_destroy(rt);
    return nullptr;
  }
  return rt;
}

void mi_destroy(void* runtime) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt) return;
  (void)hipSetDevice(rt->device);
  if (rt->stream) (void)hipStreamSynchronize(rt->stream);
  for (void* p : rt->pending_free) (void)hipFree(p);
  for (auto& kv : rt->rope) {
    (void)hipFree(kv.second.cos);
    (void)hipFree(kv.second.sin);
  }
  if (rt->dense_scratch) (void)hipFree(rt->dense_scratch);
  if (rt->dense_planes) (void)hipFree(rt->dense_planes);
  for (void* p : rt->planes)
    if (p) (void)hipFree(p);
  if (rt->wide_planes) (void)hipFree(rt->wide_planes);
  release_profile_events(rt);
  if (rt->ev_start) (void)hipEventDestroy(rt->ev_start);
  if (rt->ev_end) (void)hipEventDestroy(rt->ev_end);
  if (rt->stream) (void)hipStreamDestroy(rt->stream);
  delete rt;
}

void* mi_buffer(void* runtime, const void* bytes, uint64_t size) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || !size) return nullptr;
  if (hipSetDevice(rt->device) != hipSuccess) return nullptr;
  void* ptr = nullptr;
  if (hipMalloc(&ptr, size) != hipSuccess) return nullptr;
  const hipError_t e = bytes ? hipMemcpy(ptr, bytes, size, hipMemcpyHostToDevice)
                             : hipMemset(ptr, 0, size);
  if (e != hipSuccess) {
    (void)hipFree(ptr);
    return nullptr;
  }
  return new Buffer{ptr, size, rt};
}

void mi_free(void* buffer) {
  auto b = static_cast<Buffer*>(buffer);
  if (!b) return;
  Runtime* rt = b->owner;
  if (rt->recording) {
    // the open command may have queued launches (or a plan replay) that use this memory: keep
    // it until mi_finish / mi_abort
    rt->pending_free.push_back(b->ptr);
  } else {
    (void)hipSetDevice(rt->device);
    (void)hipStreamSynchronize(rt->stream);
    (void)hipFree(b->ptr);
  }
  delete b;
}

int mi_read(void* buffer, void* output, uint64_t bytes) {
  auto b = static_cast<Buffer*>(buffer);
  if (!b || !output || bytes > b->size) return 1;
  if (hipSetDevice(b->owner->device) != hipSuccess) return 1;
  if (hipStreamSynchronize(b->owner->stream) != hipSuccess) return 1;
  return hipMemcpy(output, b->ptr, bytes, hipMemcpyDeviceToHost) == hipSuccess ? 0 : 1;
}

int mi_write(void* buffer, const void* bytes, uint64_t size) {
  auto b = static_cast<Buffer*>(buffer);
  if (!b || !bytes || size > b->size) return 1;
  if (hipSetDevice(b->owner->device) != hipSuccess) return 1;
  if (hipStreamSynchronize(b->owner->stream) != hipSuccess) return 1;
  return hipMemcpy(b->ptr, bytes, size, hipMemcpyHostToDevice) == hipSuccess ? 0 : 1;
}

int mi_begin(void* runtime) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || rt->recording) return 1;
  rt->recording = true;
  rt->ops.clear();
  rt->profile_seconds.clear();
  return 0;
}

int mi_dispatch(void* runtime, const char* name, void** buffers, uint32_t count,
                const void* parameters, uint32_t size, uint64_t threads, uint32_t group) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || !rt->recording || count > kMaxBuffers || size != sizeof(Params) || !parameters ||
      !threads || !group)
    return 1;
  uint32_t nbuf = 0;
  const Route r = find_route(name, &nbuf);
  if (r == R_NONE) return 1;
  Params p;
  std::memcpy(&p, parameters, sizeof p);
  void* ptrs[kMaxBuffers] = {};
  uint64_t sizes[kMaxBuffers] = {};
  for (uint32_t i = 0; i < count; ++i) {
    auto b = static_cast<Buffer*>(buffers ? buffers[i] : nullptr);
    if (!b || b->owner != rt) return 1;
    ptrs[i] = b->ptr;
    sizes[i] = b->size;
  }
  if (!validate(r, p, threads, group, sizes, count, nbuf)) return 1;
  Op op;
  make_op(r, p, threads, group, ptrs, sizes, count, &op);
  if (hipSetDevice(rt->device) != hipSuccess || !prepare(rt, op)) return 1;
  return queue_op(rt, op) ? 0 : 1;
}

hipError_t launch_fused_dual(Runtime* rt, const Op& a, const Op& b, bool gated, bool scaled);

// The rows of an in-place rms_norm whose rope follows.
bool norm_rope_rows(const Op& a, const Op& b, tessery::NormRopeRows* rows) {
  if (a.route != R_RMS_NORM || b.route != R_ROPE || a.ptr[2] != a.ptr[0] || b.ptr[0] != a.ptr[0] ||
      b.p.dim != a.p.cols || static_cast<uint64_t>(b.p.n) != (a.threads / 32) * (a.p.cols / 2))
    return false;
  *rows = {static_cast<float*>(a.ptr[0]), static_cast<const uint16_t*>(a.ptr[1]),
           static_cast<int>(a.threads / 32), static_cast<int>(b.p.heads), a.p.eps};
  return true;
}

// Two such pairs over different buffers of one dim, seq and theta (a layer's q, then k) as one
// launch of ops first .. first + 3; hipErrorNotReady when they are not that.
hipError_t launch_norm_rope_pairs(Runtime* rt, size_t first, size_t last) {
  tessery::NormRopeRows rows[2];
  if (first + 3 >= last) return hipErrorNotReady;
  const Op *a = &rt->ops[first], *b = a + 1, *c = a + 2, *d = a + 3;
  if (!norm_rope_rows(*a, *b, &rows[0]) || !norm_rope_rows(*c, *d, &rows[1]) ||
      a->p.cols != c->p.cols || b->p.seq != d->p.seq ||
      float_bits(b->p.theta) != float_bits(d->p.theta) || a->ptr[0] == c->ptr[0] ||
      a->ptr[1] == c->ptr[0] || c->ptr[1] == a->ptr[0])
    return hipErrorNotReady;
  const RopeTable* t = rope_of(rt, b->p);
  if (!t) return hipErrorNotReady;
  return tessery::launch_rms_norm_rope_f32(rows, 2, t->cos, t->sin, static_cast<int>(a->p.cols),
                                           static_cast<int>(b->p.seq), rt->stream);
}

// Pairs of queued launches that one kernel runs with the same bits (the second op of a pair is
// then not launched on its own):
//   add(a, b -> a), then layer_norm(a -> a) over the same rows
//     -> one pass that adds and normalizes in place;
//   add(a, b -> a), then rms_norm(a -> y) -> one pass (add_rms_norm_f32);
//   an in-place rms_norm, then rope on the same rows -> rms_norm_rope_f32;
//   qkv4_f16, then norm_rope_f16 over its k output (D = 128) -> the projection with the k
//     prologue in the k tiles' epilogue;
//   two uint4 projections of the same x with the same shape -> one fp16-MFMA launch
//     (launch_fused_dual);
//   attention_f16_norm_rope of one layer, then norm_rope_f16 (hi + lo planes) of another over the
//     same shape and lengths, neither writing a buffer of the other -> the attention launch with
//     the prologue in extra workgroups.
// Returns the launch status, or hipErrorNotReady when ops[i], ops[i + 1] are not such a pair.
hipError_t launch_fused_pair(Runtime* rt, const Op& a, const Op& b, const Beside& beside) {
  hipStream_t st = rt->stream;
  if (is_linear4(a.route)) return launch_fused_dual(rt, a, b, false, beside.scaled);
  if (a.route == R_ADD && b.route == R_LAYER_NORM && a.ptr[2] == a.ptr[0] &&
      b.ptr[0] == a.ptr[0] && b.ptr[3] == a.ptr[0] && a.ptr[1] != a.ptr[0] &&
      static_cast<uint64_t>(a.p.n) == (b.threads / 32) * b.p.cols) {
    return tessery::launch_add_layer_norm_f32(
        static_cast<float*>(a.ptr[0]), static_cast<const float*>(a.ptr[1]),
        static_cast<const float*>(b.ptr[1]), static_cast<const float*>(b.ptr[2]),
        static_cast<int>(b.threads / 32), static_cast<int>(b.p.cols), b.p.eps, st);
  }
  if (a.route == R_ADD && b.route == R_RMS_NORM && a.ptr[2] == a.ptr[0] &&
      a.ptr[1] != a.ptr[0] && b.ptr[0] == a.ptr[0] && b.ptr[2] != a.ptr[1] &&
      static_cast<uint64_t>(a.p.n) == (b.threads / 32) * b.p.cols) {
    return tessery::launch_add_rms_norm_f32(
        static_cast<float*>(a.ptr[0]), static_cast<const float*>(a.ptr[1]),
        static_cast<const uint16_t*>(b.ptr[1]), static_cast<float*>(b.ptr[2]),
        static_cast<int>(b.threads / 32), static_cast<int>(b.p.cols), b.p.eps, beside.planes, beside.scales, st);
  }
  if (a.route == R_QKV4_F16 && b.route == R_NORM_ROPE_F16 && b.ptr[0] == a.ptr[5] &&
      b.p.dim == 128 && static_cast<uint64_t>(b.p.heads) * 128 == a.p.n &&
      b.threads == a.p.rows) {
    // the projection's k output, then its k prologue (the fused attention's norm_rope_f16):
    // the k tiles finish with the prologue; the k output itself is still written
    for (int i = 0; i < 7; ++i)
      if (b.ptr[3] == a.ptr[i]) return hipErrorNotReady;
    for (int i = 4; i < 7; ++i)
      if (b.ptr[1] == a.ptr[i] || b.ptr[2] == a.ptr[i]) return hipErrorNotReady;
    const RopeTable* t = rope_of(rt, b.p);
    if (!t) return hipErrorNotReady;
    tessery::Qkv4Args q = qkv4_args(a);
    q.kn = static_cast<_Float16*>(b.ptr[3]);
    q.kn_split = (b.p.u1 & 1u) != 0;
    q.kn_gamma = static_cast<const uint16_t*>(b.ptr[1]);
    q.kn_cos = t->cos;
    q.kn_sin = t->sin;
    q.kn_lengths = static_cast<const uint32_t*>(b.ptr[2]);
    q.kn_S = static_cast<int>(b.p.seq);
    q.kn_eps = b.p.eps;
    return tessery::launch_qkv4_f16(q, st);
  }
  if (a.route == R_ATTENTION_F16_NORM_ROPE && b.route == R_NORM_ROPE_F16 && (b.p.u1 & 1u) &&
      b.ptr[2] == a.ptr[3]) {
    // the fused attention of one layer, then the k prologue of another (the next layer's, queued
    // right after it) over the same lengths and shape, with no buffer of one written by the
    // other: extra workgroups of the attention launch run the prologue, with its bits
    tessery::AttnArgs args;
    if (!attention_args(rt, a, &args) || b.p.dim != static_cast<uint32_t>(args.D) ||
        b.p.heads != static_cast<uint32_t>(args.KV) || b.p.seq != static_cast<uint32_t>(args.S) ||
        b.threads != static_cast<uint64_t>(args.B) * args.S ||
        !tessery::attention_f16_carries_prologue(args.B, args.S, args.H, args.KV, args.D))
      return hipErrorNotReady;
    for (int i = 0; i < 6; ++i)
      if (b.ptr[3] == a.ptr[i]) return hipErrorNotReady;
    for (int i = 0; i < 3; ++i)
      if (a.ptr[4] == b.ptr[i]) return hipErrorNotReady;
    const RopeTable* t = rope_of(rt, b.p);
    if (!t) return hipErrorNotReady;
    args.pro_x = static_cast<const _Float16*>(b.ptr[0]);
    args.pro_y = static_cast<_Float16*>(b.ptr[3]);
    args.pro_gamma = static_cast<const uint16_t*>(b.ptr[1]);
    args.pro_cos = t->cos;
    args.pro_sin = t->sin;
    args.pro_eps = b.p.eps;
    return tessery::launch_attention_f16(args, st);
  }
  tessery::NormRopeRows rows;
  if (norm_rope_rows(a, b, &rows)) {
    const RopeTable* t = rope_of(rt, b.p);
    if (!t) return hipErrorNotReady;
    return tessery::launch_rms_norm_rope_f32(&rows, 1, t->cos, t->sin, static_cast<int>(a.p.cols),
                                             static_cast<int>(b.p.seq), st);
  }
  return hipErrorNotReady;
}

// The gated MLP as the reference's unfused form queues it (metal.py:501-530): linear4(x -> g),
// linear4(x -> u) over the same rows, then silu_gate(g, u). When both projections cover all rows
// of their outputs and would run the fp16-MFMA kernel, one launch computes both from one staging
// of x and leaves the same bits in g and u. Returns the launch status, or hipErrorNotReady when
// ops[i .. i + 2] are not such a triple.
hipError_t launch_fused_gated(Runtime* rt, const Op& a, const Op& b, const Op& c, bool scaled) {
  if (c.route != R_SILU_GATE || c.ptr[0] != a.ptr[4] || c.ptr[1] != b.ptr[4] ||
      static_cast<uint64_t>(c.p.n) != static_cast<uint64_t>(a.p.rows) * a.p.cols)
    return hipErrorNotReady;
  return launch_fused_dual(rt, a, b, true, scaled);
}

// Two uint4 projections of the same x with the same shape (the k and v projections of a Qwen3
// layer, or the gated MLP's gate and up) as one launch of the fp16-MFMA kernel, with the bits of
// the two launches; with `gated` the first output receives silu(first) * second. Returns the
// launch status, or hipErrorNotReady when the pair does not qualify.
hipError_t launch_fused_dual(Runtime* rt, const Op& a, const Op& b, bool gated, bool scaled) {
  if (!is_linear4(a.route) || b.route != a.route) return hipErrorNotReady;
  const Params &pa = a.p, &pb = b.p;
  if (pa.rows != pb.rows || pa.cols != pb.cols || pa.k != pb.k || a.ptr[0] != b.ptr[0])
    return hipErrorNotReady;
  // outputs distinct from x, from each other and from the second projection's weights: the second
  // projection reads them after the first has written its output
  if (a.ptr[4] == a.ptr[0] || b.ptr[4] == a.ptr[0] || a.ptr[4] == b.ptr[4]) return hipErrorNotReady;
  // and the second output distinct from the first projection's weights, scales and biases: in one
  // kernel the second projection's stores overlap the first projection's reads
  for (int i = 1; i < 4; ++i)
    if (b.ptr[i] == a.ptr[4] || b.ptr[4] == a.ptr[i]) return hipErrorNotReady;
  RowRange ra, rb;
  if (!linear4_range(a.route, pa, a.threads, a.group, &ra) ||
      !linear4_range(b.route, pb, b.threads, b.group, &rb) || ra.r0 != 0 || ra.r1 != pa.rows ||
      rb.r0 != 0 || rb.r1 != pb.rows)
    return hipErrorNotReady;
  const int M = static_cast<int>(pa.rows), N = static_cast<int>(pa.cols),
            K = static_cast<int>(pa.k);
  if (!rt->dense_scratch || !tessery::linear4_hilo_dual_fits(M, N, K)) return hipErrorNotReady;
  const hipError_t e = tessery::launch_linear4_hilo_dual_f32(
      static_cast<const float*>(a.ptr[0]), static_cast<const uint32_t*>(a.ptr[1]),
      static_cast<const uint16_t*>(a.ptr[2]), static_cast<const uint16_t*>(a.ptr[3]),
      static_cast<float*>(a.ptr[4]), static_cast<const uint32_t*>(b.ptr[1]),
      static_cast<const uint16_t*>(b.ptr[2]), static_cast<const uint16_t*>(b.ptr[3]),
      static_cast<float*>(b.ptr[4]), gated, M, N, K, rt->dense_scratch, kDenseScratchFloats,
      scaled, rt->stream);
  // hipErrorInvalidValue: nothing was launched (alignment or sizes); the ops run as queued
  return e == hipErrorInvalidValue ? hipErrorNotReady : e;
}

// A uint4 projection over a run of queued ops: ops[first, end) are launches of one projection (the
// same buffers and shape) over consecutive row ranges, as linear4_plan partitions its rows.
struct Linear4Run {
  tessery::Linear4Job job;
  size_t end;
};

// The run that starts at op `first`; false unless linear4_rows runs it. Its results depend on no
// launch's rows, so one launch over the joined rows leaves the bits of the separate ones; a
// projection that fp16 MFMA takes (linear4_hilo) stays as queued.
bool linear4_run(Runtime* rt, size_t first, size_t last, Linear4Run* run) {
  if (!linear4_job(rt->ops[first], &run->job) ||
      !tessery::linear4_on_rows(run->job, rt->dense_scratch, kDenseScratchFloats))
    return false;
  run->end = first + 1;
  // a launch reads x and the weights that an output over them would have changed by then
  const Op& a = rt->ops[first];
  for (int i = 0; i < 4; ++i)
    if (a.ptr[i] == a.ptr[4]) return true;
  for (; run->end < last; ++run->end) {
    const Op& b = rt->ops[run->end];
    tessery::Linear4Job next;
    if (!linear4_job(b, &next) || b.p.rows != a.p.rows || next.cols != run->job.cols ||
        next.k != run->job.k || next.row0 != run->job.row1 ||
        !std::equal(a.ptr.begin(), a.ptr.begin() + 5, b.ptr.begin()) ||
        !tessery::linear4_on_rows(next, rt->dense_scratch, kDenseScratchFloats))
      break;
    run->job.row1 = next.row1;
  }
  return true;
}

// A linear4_rows launch over ops [first, end).
struct Projection {
  tessery::Linear4Job jobs[3];
  int count;
  bool gated;
  size_t end;
};

// The launch that starts at op `first`: up to three projections of the same rows of one x queued one
// after the other (q, k and v), two of them with the silu_gate that follows (gate and up), each
// over its whole run of row ranges, or the row ranges of a gated4 projection. False: op `first`
// is no projection that linear4_rows runs.
bool find_projection(Runtime* rt, size_t first, size_t last, Projection* p) {
  const Op& a = rt->ops[first];
  if (is_gated4(a.route)) {
    tessery::Linear4Job next[2];
    if (!gated4_jobs(a, p->jobs)) return false;
    p->count = 2;
    p->gated = true;
    p->end = first + 1;
    bool apart = true;  // the output is none of the inputs
    for (int i = 0; i < 7; ++i) apart = apart && a.ptr[i] != a.ptr[7];
    for (; apart && p->end < last; ++p->end) {
      const Op& b = rt->ops[p->end];
      if (!gated4_jobs(b, next) || a.ptr != b.ptr || b.p.rows != a.p.rows ||
          next[0].cols != p->jobs[0].cols || next[0].k != p->jobs[0].k ||
          next[0].row0 != p->jobs[0].row1)
        break;
      p->jobs[0].row1 = p->jobs[1].row1 = next[0].row1;
    }
    return true;
  }
  Linear4Run run;
  if (!is_linear4(a.route) || !linear4_run(rt, first, last, &run)) return false;
  p->jobs[0] = run.job;
  p->gated = false;
  p->count = 1;
  size_t ends[3] = {run.end, 0, 0};
  while (p->count < 3 && ends[p->count - 1] < last &&
         linear4_run(rt, ends[p->count - 1], last, &run)) {
    const tessery::Linear4Job& j = run.job;
    const tessery::Linear4Job& lead = p->jobs[0];
    bool joins = j.x == lead.x && j.k == lead.k && j.row0 == lead.row0 && j.row1 == lead.row1 &&
                 static_cast<const void*>(j.out) != j.x;
    // no output is an input or output of another projection of the launch
    for (int i = 0; i < p->count && joins; ++i) {
      const tessery::Linear4Job& o = p->jobs[i];
      for (const void* in : {static_cast<const void*>(j.x), static_cast<const void*>(j.w),
                             static_cast<const void*>(j.scales),
                             static_cast<const void*>(j.biases), static_cast<const void*>(j.out)})
        joins = joins && in != o.out;
      for (const void* in : {static_cast<const void*>(o.w), static_cast<const void*>(o.scales),
                             static_cast<const void*>(o.biases)})
        joins = joins && in != j.out;
    }
    if (!joins) break;
    p->jobs[p->count] = j;
    ends[p->count++] = run.end;
  }
  // gate, up, silu_gate(gate, up) over every row
  if (p->count >= 2 && ends[1] < last && p->jobs[0].cols == p->jobs[1].cols &&
      p->jobs[0].row0 == 0) {
    const Op& c = rt->ops[ends[1]];
    if (c.route == R_SILU_GATE && c.ptr[0] == p->jobs[0].out && c.ptr[1] == p->jobs[1].out &&
        static_cast<uint64_t>(c.p.n) ==
            static_cast<uint64_t>(p->jobs[0].row1) * static_cast<uint64_t>(p->jobs[0].cols)) {
      p->count = 2;
      p->gated = true;
      p->end = ends[1] + 1;
      return true;
    }
  }
  p->end = ends[p->count - 1];
  return true;
}

// A dense launch over ops [first, end).
struct DenseProjection {
  tessery::DenseJob jobs[3];
  int count;
  bool gelu;
  size_t end;
};

// One projection's launches over consecutive row ranges (as the planners partition its rows) from op
// `first`, joined; false when it is no dense projection.
bool dense_run(Runtime* rt, size_t first, size_t last, tessery::DenseJob* job, size_t* end) {
  if (!dense_job(rt->ops[first], job)) return false;
  *end = first + 1;
  const Op& a = rt->ops[first];
  for (uint32_t i = 0; i < a.count; ++i)
    if (i != 2 && a.ptr[i] == a.ptr[2]) return true;
  for (; *end < last; ++*end) {
    const Op& b = rt->ops[*end];
    tessery::DenseJob next;
    if (!dense_job(b, &next) || b.p.rows != a.p.rows || next.a != job->a || next.bt != job->bt ||
        next.bias != job->bias || next.out != job->out || next.cols != job->cols ||
        next.k != job->k || next.row0 != job->row1)
      break;
    job->row1 = next.row1;
  }
  return true;
}

// The launch that starts at op `first`: one projection, with the gelu_f32 over its whole output that
// follows, or up to three of the same rows of one input (q, k and v) on matmul_planes. False: op
// `first` is no dense projection.
bool find_dense(Runtime* rt, size_t first, size_t last, DenseProjection* p) {
  if (!is_dense(rt->ops[first].route) || !dense_run(rt, first, last, &p->jobs[0], &p->end))
    return false;
  p->count = 1;
  p->gelu = false;
  const tessery::DenseJob& lead = p->jobs[0];
  if (p->end < last) {
    const Op& b = rt->ops[p->end];
    if (b.route == R_GELU && b.ptr[0] == lead.out && lead.row0 == 0 &&
        static_cast<uint64_t>(lead.row1) == rt->ops[first].p.rows &&
        static_cast<uint64_t>(b.p.n) ==
            static_cast<uint64_t>(lead.row1) * static_cast<uint64_t>(lead.cols)) {
      p->gelu = true;
      ++p->end;
      return true;
    }
  }
  const tessery::DenseScratch scratch = dense_scratch(rt);
  while (p->count < 3 && p->end < last && tessery::matmul_on_planes(lead, scratch)) {
    tessery::DenseJob j;
    size_t end;
    if (!dense_run(rt, p->end, last, &j, &end) || !tessery::matmul_joins(lead, j, scratch) ||
        j.out == j.a)
      break;
    // no output is an input or output of another projection of the launch
    bool apart = true;
    for (int i = 0; i < p->count; ++i) {
      const tessery::DenseJob& o = p->jobs[i];
      apart = apart && o.out != j.a && o.out != j.bt && o.out != j.bias && o.out != j.out &&
              j.out != o.bt && j.out != o.bias;
    }
    // its own gelu_f32 runs with it
    const bool gelu = end < last && rt->ops[end].route == R_GELU && rt->ops[end].ptr[0] == j.out;
    if (!apart || gelu) break;
    p->jobs[p->count++] = j;
    p->end = end;
  }
  return true;
}

// What the launch before left for the next one: the planes of x [rows, k], in a planes scratch.
struct Ready {
  const void* x = nullptr;
  uint64_t rows = 0, k = 0;
  int slot = 0;
};

// Launches of one pass over the queue: their fusions, and what the last one left behind.
struct Pass {
  FusionCount fused;
  Ready ready;
  Ready scaled;  // the row scales of x [rows, k], in the dense scratch
};

// The projection of op `at` when it starts at row 0 and runs on linear4_hilo, which reads row scales.
bool reads_scales(Runtime* rt, size_t at, size_t last, tessery::Linear4Job* job) {
  return at < last && linear4_job(rt->ops[at], job) && job->row0 == 0 &&
         !tessery::linear4_on_rows(*job, rt->dense_scratch, kDenseScratchFloats);
}

// Whether op `at` starts a projection that reads all of x [rows, k] as planes the scratch holds.
bool reads_planes(Runtime* rt, size_t at, size_t last, const void* x, uint64_t rows, uint64_t k) {
  Projection p;
  return at < last && find_projection(rt, at, last, &p) && p.jobs[0].x == x &&
         p.jobs[0].row0 == 0 && static_cast<uint64_t>(p.jobs[0].row1) == rows &&
         static_cast<uint64_t>(p.jobs[0].k) == k && p.jobs[0].out != x &&
         tessery::planes_bytes(p.jobs[0].row1, p.jobs[0].k) <= kPlanesBytes;
}

// Launches op `first` and those after it (before op `last`) that run inside the same kernel: the
// projections find_projection takes, the triples of launch_fused_gated and the pairs of
// launch_fused_pair (the last two counted). A kernel whose output the next launch projects leaves
// its planes too. *taken: the ops launched.
hipError_t launch_next(Runtime* rt, size_t first, size_t last, size_t* taken, Pass* pass) {
  const Ready ready = pass->ready, scaled = pass->scaled;
  pass->ready = pass->scaled = {};
  const Op& op = rt->ops[first];
  Projection p;
  if (find_projection(rt, first, last, &p)) {
    const tessery::Linear4Job& j = p.jobs[0];
    const bool prepared = ready.x && ready.x == j.x && j.row0 == 0 &&
                          ready.rows == static_cast<uint64_t>(j.row1) &&
                          ready.k == static_cast<uint64_t>(j.k);
    const int slot = prepared ? ready.slot : 0;
    *taken = p.end - first;
    const bool keep = p.gated && j.row0 == 0 && j.out != j.x && rt->planes[1 - slot] &&
                      tessery::planes_bytes(j.row1, j.k) <= kPlanesBytes &&
                      reads_planes(rt, p.end, last, j.out, j.row1, j.cols);
    // its scratch is another one: the row scales of its input stay
    bool untouched = true;
    for (int i = 0; i < p.count; ++i) untouched = untouched && p.jobs[i].out != scaled.x;
    if (untouched) pass->scaled = scaled;
    if (keep)
      pass->ready = {j.out, static_cast<uint64_t>(j.row1), static_cast<uint64_t>(j.cols), 1 - slot};
    // too wide for a planes scratch: neither prepared nor kept
    const bool wide =
        rt->wide_planes && tessery::planes_bytes(j.row1 - j.row0, j.k) > kPlanesBytes;
    return tessery::launch_linear4_rows(
        p.jobs, p.count, p.gated,
        wide ? tessery::PlanesScratch{rt->wide_planes, nullptr, kWidePlanesBytes}
             : planes_scratch(rt, slot),
        prepared, keep, rt->stream);
  }
  DenseProjection d;
  if (find_dense(rt, first, last, &d)) {
    *taken = d.end - first;
    const hipError_t e =
        d.count > 1
            ? tessery::launch_matmul_planes(d.jobs, d.count, false, dense_scratch(rt), rt->stream)
            : tessery::launch_matmul_f32(d.jobs[0], d.gelu, dense_scratch(rt), rt->stream);
    pass->fused.pairs += d.gelu && e == hipSuccess;
    return e;
  }
  Beside beside;
  tessery::Linear4Job hilo;
  const bool on_hilo = reads_scales(rt, first, last, &hilo);
  if (on_hilo) {
    beside.scaled = scaled.x == hilo.x && scaled.rows >= static_cast<uint64_t>(hilo.row1) &&
                    scaled.k == static_cast<uint64_t>(hilo.k);
    // for the next projection of the same input
    if (hilo.out != hilo.x)
      pass->scaled = beside.scaled ? scaled
                                   : Ready{hilo.x, static_cast<uint64_t>(hilo.row1),
                                           static_cast<uint64_t>(hilo.k), 0};
  }
  const hipError_t gated =
      first + 2 < last
          ? launch_fused_gated(rt, op, rt->ops[first + 1], rt->ops[first + 2], beside.scaled)
          : hipErrorNotReady;
  if (gated != hipErrorNotReady) {
    pass->scaled = {};  // of no use to what follows the gated projections
    pass->fused.gated += gated == hipSuccess;
    *taken = 3;
    return gated;
  }
  const hipError_t pairs = launch_norm_rope_pairs(rt, first, last);
  if (pairs != hipErrorNotReady) {
    if (pairs == hipSuccess) pass->fused.pairs += 2;
    *taken = 4;
    return pairs;
  }
  // the planes of a rms_norm (alone, or after the add it runs with) that projections read
  auto norm_ready = [&](size_t at) {
    const Op& n = rt->ops[at];
    const uint64_t rows = n.threads / 32;
    if (n.route == R_RMS_NORM && reads_planes(rt, at + 1, last, n.ptr[2], rows, n.p.cols))
      return Ready{n.ptr[2], rows, n.p.cols, 0};
    return Ready{};
  };
  // the row scales of a rms_norm's output that a projection reads
  auto norm_scales = [&](size_t at) {
    const Op& n = rt->ops[at];
    const uint64_t rows = n.threads / 32;
    tessery::Linear4Job job;
    if (n.route == R_RMS_NORM && reads_scales(rt, at + 1, last, &job) && job.x == n.ptr[2] &&
        static_cast<uint64_t>(job.row1) <= rows && rows <= kDenseScratchFloats &&
        job.k == static_cast<int>(n.p.cols))
      return Ready{n.ptr[2], rows, n.p.cols, 0};
    return Ready{};
  };
  if (first + 1 < last) {
    Ready after, scales;
    if (op.route == R_ADD) {
      after = norm_ready(first + 1);
      scales = norm_scales(first + 1);
      beside.planes = after.x ? rt->planes[after.slot] : nullptr;
      beside.scales = scales.x ? rt->dense_scratch : nullptr;
    }
    const hipError_t pair = launch_fused_pair(rt, op, rt->ops[first + 1], beside);
    if (pair != hipErrorNotReady) {
      pass->fused.pairs += pair == hipSuccess;
      pass->ready = after;
      if (scales.x) pass->scaled = scales;
      // a second projection of the input: its output may be that input only in the pair itself
      if (on_hilo && rt->ops[first + 1].ptr[4] == hilo.x) pass->scaled = {};
      *taken = 2;
      return pair;
    }
  }
  *taken = 1;
  pass->ready = norm_ready(first);
  if (const Ready scales = norm_scales(first); scales.x) {
    pass->scaled = scales;
    beside.scales = rt->dense_scratch;
  }
  tessery::AttnArgs at{};
  if (attention_args(rt, op, &at) && tessery::attention_leaves_planes(at, op.route == R_ATTENTION)) {
    const uint64_t rows = static_cast<uint64_t>(at.B) * static_cast<uint64_t>(at.S);
    const uint64_t width = static_cast<uint64_t>(at.H) * static_cast<uint64_t>(at.D);
    if (reads_planes(rt, first + 1, last, at.out, rows, width))
      pass->ready = Ready{at.out, rows, width, 0};
  }
  beside.planes = pass->ready.x ? rt->planes[pass->ready.slot] : nullptr;
  return launch(rt, op, beside);
}

// Launches ops [first, last) in order; the fusions made are added to *fc. Under stream capture
// nothing runs yet, so the caller decides where the count goes (the runtime's totals for direct
// launches, the cached graph for a capture).
hipError_t launch_range(Runtime* rt, size_t first, size_t last, FusionCount* fc) {
  Pass pass;
  for (size_t i = first, taken = 0; i < last; i += taken) {
    const hipError_t e = launch_next(rt, i, last, &taken, &pass);
    if (e != hipSuccess) return e;
    ++fc->launches;
  }
  fc->pairs += pass.fused.pairs;
  fc->gated += pass.fused.gated;
  return hipSuccess;
}

void count_fusions(Runtime* rt, const FusionCount& fc) {
  rt->fused_pairs += fc.pairs;
  rt->fused_gated += fc.gated;
}

// A plan replay as one graph launch: the graph of this plan for this binding is instantiated the
// first time (stream capture of launch_range, which records the same kernels with the same
// arguments) and reused afterwards. Captured launches do not run, so on any capture error the
// caller launches the segment directly. hipErrorNotReady: graphs are off for this runtime, or the
// plan is a short one.
hipError_t launch_segment_graph(Runtime* rt, const Segment& seg) {
  if (!rt->graphs || seg.plan->direct) return hipErrorNotReady;
  auto& cache = seg.plan->graphs;
  for (size_t j = 0; j < cache.size(); ++j)
    if (cache[j].key == seg.key) {
      CachedGraph hit = cache[j];
      cache.erase(cache.begin() + static_cast<std::ptrdiff_t>(j));
      cache.push_back(hit);
      ++rt->graph_launches;
      const hipError_t e = hipGraphLaunch(hit.exec, rt->stream);
      if (e == hipSuccess) count_fusions(rt, hit.fused);
      return e;
    }
  if (hipStreamBeginCapture(rt->stream, hipStreamCaptureModeThreadLocal) != hipSuccess)
    return hipErrorNotReady;
  FusionCount fc;
  const hipError_t recorded = launch_range(rt, seg.first, seg.first + seg.count, &fc);
  hipGraph_t graph = nullptr;
  const hipError_t ended = hipStreamEndCapture(rt->stream, &graph);
  if (recorded != hipSuccess || ended != hipSuccess || !graph) {
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipGetLastError();
    return hipErrorNotReady;
  }
  if (fc.launches < kGraphLaunches) {
    seg.plan->direct = true;
    (void)hipGraphDestroy(graph);
    return hipErrorNotReady;
  }
  hipGraphExec_t exec = nullptr;
  const hipError_t made = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (made != hipSuccess || !exec) {
    (void)hipGetLastError();
    return hipErrorNotReady;
  }
  if (cache.size() >= kPlanGraphs) {
    (void)hipGraphExecDestroy(cache.front().exec);
    cache.erase(cache.begin());
  }
  cache.push_back(CachedGraph{seg.key, exec, fc});
  ++rt->graph_builds;
  ++rt->graph_launches;
  const hipError_t e = hipGraphLaunch(exec, rt->stream);
  if (e == hipSuccess) count_fusions(rt, fc);
  return e;
}

// Direct launches of ops [first, last), with their fusions counted.
hipError_t launch_direct(Runtime* rt, size_t first, size_t last) {
  FusionCount fc;
  const hipError_t e = launch_range(rt, first, last, &fc);
  if (e == hipSuccess) count_fusions(rt, fc);
  return e;
}

int mi_finish(void* runtime) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || !rt->recording) return 1;
  if (hipSetDevice(rt->device) != hipSuccess) return 1;
  int failed = 0;
  const size_t n = rt->ops.size();
  if (rt->profiling) {
    while (rt->prof_events.size() < 2 * n) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) return 1;
      rt->prof_events.push_back(e);
    }
  }
  if (hipEventRecord(rt->ev_start, rt->stream) != hipSuccess) failed = 1;
  if (!rt->profiling) {
    // plan replays run as cached graphs (plans are never replayed while profiling); the rest,
    // and any segment whose graph could not be made, launch one by one
    size_t i = 0;
    for (const Segment& seg : rt->segments) {
      if (failed) break;
      if (launch_direct(rt, i, seg.first) != hipSuccess) failed = 1;
      if (failed) break;
      const hipError_t g = launch_segment_graph(rt, seg);
      if (g == hipErrorNotReady) {
        if (launch_direct(rt, seg.first, seg.first + seg.count) != hipSuccess) failed = 1;
      } else if (g != hipSuccess) {
        failed = 1;
      }
      i = seg.first + seg.count;
    }
    if (!failed && launch_direct(rt, i, n) != hipSuccess) failed = 1;
  }
  if (rt->profiling) {
    // ops that run inside the kernel of one before them: the first one's events enclose that
    // kernel, the others' enclose no work
    rt->profile_fused.assign(n, 0);
    Pass pass;
    for (size_t i = 0, taken = 0; i < n && !failed; i += taken) {
      if (hipEventRecord(rt->prof_events[2 * i], rt->stream) != hipSuccess ||
          launch_next(rt, i, n, &taken, &pass) != hipSuccess ||
          hipEventRecord(rt->prof_events[2 * i + 1], rt->stream) != hipSuccess) {
        failed = 1;
        break;
      }
      for (size_t j = i + 1; j < i + taken && !failed; ++j) {
        rt->profile_fused[j] = 1;
        if (hipEventRecord(rt->prof_events[2 * j], rt->stream) != hipSuccess ||
            hipEventRecord(rt->prof_events[2 * j + 1], rt->stream) != hipSuccess)
          failed = 1;
      }
    }
    if (!failed) count_fusions(rt, pass.fused);
  }
  if (hipEventRecord(rt->ev_end, rt->stream) != hipSuccess) failed = 1;
  if (hipStreamSynchronize(rt->stream) != hipSuccess) failed = 1;
  rt->last_gpu = -1.0;
  float ms = 0.0f;
  if (!failed && hipEventElapsedTime(&ms, rt->ev_start, rt->ev_end) == hipSuccess)
    rt->last_gpu = ms * 1e-3;
  rt->profile_seconds.clear();
  if (!failed && rt->profiling) {
    for (size_t i = 0; i < n; ++i) {
      float t = 0.0f;
      if (hipEventElapsedTime(&t, rt->prof_events[2 * i], rt->prof_events[2 * i + 1]) !=
          hipSuccess) {
        failed = 1;
        break;
      }
      rt->profile_seconds.push_back(t * 1e-3);
    }
    if (failed) rt->profile_seconds.clear();
  }
  if (rt->profile_seconds.empty()) rt->profile_fused.clear();
  rt->ops.clear();
  rt->segments.clear();
  rt->recording = false;
  release_pending(rt);
  return failed;
}

double mi_gpu_seconds(void* runtime) {
  auto rt = static_cast<Runtime*>(runtime);
  return rt ? rt->last_gpu : -1.0;
}

void mi_abort(void* runtime) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt) return;
  rt->ops.clear();  // queued work was never launched
  rt->segments.clear();
  rt->recording = false;
  (void)hipSetDevice(rt->device);
  release_pending(rt);
}

int mi_profile_enable(void* runtime, int enabled) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || rt->recording) return 1;
  rt->profile_seconds.clear();
  rt->profile_fused.clear();
  rt->profiling = enabled != 0;
  if (!rt->profiling) release_profile_events(rt);
  return 0;
}

int mi_profile_read(void* runtime, double* seconds, uint32_t count) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || rt->recording || count != rt->profile_seconds.size()) return 1;
  if (count) std::memcpy(seconds, rt->profile_seconds.data(), count * sizeof(double));
  return 0;
}

int mi_profile_fused(void* runtime, uint8_t* fused, uint32_t count) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || rt->recording || count != rt->profile_fused.size()) return 1;
  if (count) std::memcpy(fused, rt->profile_fused.data(), count);
  return 0;
}

void* mi_plan_create(void* runtime, void** buffers, uint32_t count) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || !rt->recording || rt->profiling || !count || count > 2048 || !buffers) return nullptr;
  auto plan = new Plan{rt, {}, {}};
  for (uint32_t i = 0; i < count; ++i) {
    auto b = static_cast<Buffer*>(buffers[i]);
    if (!b || b->owner != rt) {
      delete plan;
      return nullptr;
    }
    plan->sizes.push_back(b->size);
  }
  return plan;
}

int mi_plan_add(void* plan, const char* name, const uint32_t* slots, uint32_t count,
                const void* params, uint64_t threads, uint32_t group) {
  auto pl = static_cast<Plan*>(plan);
  if (!pl || !pl->owner->recording || pl->owner->profiling || !count || count > kMaxBuffers ||
      !threads || !group || !params || !slots || pl->ops.size() >= kMaxPlanOps)
    return 1;
  uint32_t nbuf = 0;
  const Route r = find_route(name, &nbuf);
  if (r == R_NONE) return 1;
  PlanOp op{};
  std::memcpy(&op.p, params, sizeof(Params));
  uint64_t sizes[kMaxBuffers] = {};
  for (uint32_t i = 0; i < count; ++i) {
    if (slots[i] >= pl->sizes.size()) return 1;
    op.slots[i] = slots[i];
    sizes[i] = pl->sizes[slots[i]];
  }
  if (!validate(r, op.p, threads, group, sizes, count, nbuf)) return 1;
  op.route = r;
  op.threads = threads;
  op.group = group;
  op.count = count;
  pl->ops.push_back(op);
  return 0;
}

uint64_t mi_plan_bytes(void* plan) {
  auto pl = static_cast<Plan*>(plan);
  if (!pl) return 0;
  return sizeof(Plan) + pl->sizes.capacity() * sizeof(uint64_t) +
         pl->ops.capacity() * sizeof(PlanOp);
}

int mi_graph_counts(void* runtime, uint64_t* launches, uint64_t* builds) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || !launches || !builds) return 1;
  *launches = rt->graph_launches;
  *builds = rt->graph_builds;
  return 0;
}

int mi_fusion_counts(void* runtime, uint64_t* pairs, uint64_t* gated) {
  auto rt = static_cast<Runtime*>(runtime);
  if (!rt || !pairs || !gated) return 1;
  *pairs = rt->fused_pairs;
  *gated = rt->fused_gated;
  return 0;
}

void mi_plan_free(void* plan) {
  auto pl = static_cast<Plan*>(plan);
  if (!pl) return;
  // A replay of this plan may still be queued in the open command (a plan can be evicted while
  // another one is captured): its launches stay queued and run one by one.
  auto& segs = pl->owner->segments;
  for (size_t i = segs.size(); i-- > 0;)
    if (segs[i].plan == pl) segs.erase(segs.begin() + static_cast<std::ptrdiff_t>(i));
  for (auto& g : pl->graphs) (void)hipGraphExecDestroy(g.exec);
  delete pl;
}

int mi_plan_run(void* runtime, void* plan, void** buffers, uint32_t count) {
  auto rt = static_cast<Runtime*>(runtime);
  auto pl = static_cast<Plan*>(plan);
  if (!rt || !pl || pl->owner != rt || !rt->recording || rt->profiling ||
      count != pl->sizes.size() || pl->ops.empty() || !buffers)
    return 1;
  // Validate every slot before queueing any work (runtime.mm:198-202).
  for (uint32_t i = 0; i < count; ++i) {
    auto b = static_cast<Buffer*>(buffers[i]);
    if (!b || b->owner != rt || b->size != pl->sizes[i]) return 1;
  }
  if (hipSetDevice(rt->device) != hipSuccess) return 1;
  std::vector<Op> ops;
  ops.reserve(pl->ops.size());
  for (const auto& po : pl->ops) {
    void* ptrs[kMaxBuffers] = {};
    uint64_t sizes[kMaxBuffers] = {};
    for (uint32_t i = 0; i < po.count; ++i) {
      auto b = static_cast<Buffer*>(buffers[po.slots[i]]);
      ptrs[i] = b->ptr;
      sizes[i] = b->size;
    }
    Op op;
    make_op(po.route, po.p, po.threads, po.group, ptrs, sizes, po.count, &op);
    if (!prepare(rt, op)) return 1;
    ops.push_back(op);
  }
  rt->ops.insert(rt->ops.end(), ops.begin(), ops.end());
  Segment seg{rt->ops.size() - pl->ops.size(), pl->ops.size(), pl, {}};
  for (uint32_t i = 0; i < count; ++i) seg.key.push_back(static_cast<Buffer*>(buffers[i])->ptr);
  rt->segments.push_back(std::move(seg));
  return 0;
}

}  // extern "C"
