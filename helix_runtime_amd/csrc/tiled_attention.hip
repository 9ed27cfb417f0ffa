// Reference-shaped paged attention for any head size up to 256 and any page
// size, on the fp32 matrix cores (v_mfma_f32_16x16x4_f32): the calls whose
// geometry the head_dim-128 routes do not take.
//
// Work: one workgroup per (kv head, 16 query rows), the rows of a kv head
// being its query heads' positions, head major; its wavefronts take the
// 16-key tiles in turn (wavefront w: tiles w, w + waves, ...) with their own
// online softmax, and are merged through LDS.  Both products read K and V
// straight from global memory in operand order: a lane holds one key's dims
// 16 u + 4 g .. + 3 (g = lane / 16) for the scores, and four keys' dims
// 64 v + 4 c .. + 3 (c = lane % 16) for P.V, each a 16-byte load when rows
// are aligned.  The scores come out with 4 keys of one query row per lane,
// which is the P.V operand as it stands.  No scratch: the raw scores
// wait in the lane's registers where a wavefront has one tile
// (up to 256 keys, 128 past 64 dims), else in the caller's score workspace, and
// each lane turns its own entries into probabilities once the row's maximum
// and sum are known.
//
// The scalar kernel it replaces gave one query row to a workgroup and one
// key to a thread, so a wavefront's 64 loads touched 64 rows and every row
// re-read all of K and V: latency-bound.  8 heads of 64 dims, 128 query rows
// over 1024 keys: 390 us before, 27 us now; one row of the same 143 -> 23 us;
// 16/4 heads of 96 dims, 160 rows over 1660 keys 2.0 ms -> 66 us.  A call of
// a few keys is a chain of latencies: 4 heads of 16 dims over 65 keys 8.0 us for
// the scalar kernel, 8.2 with the scores through the workspace, 5.6 as it is
// (kernel alone).
#include "kernels.hpp"

#include "prefill_body.hpp"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <limits>

namespace helix::hip {
namespace {

using prefill_detail::exp2_ratio;
using prefill_detail::row_max;
using prefill_detail::row_sum;
using prefill_detail::v4f;

// Division by a value fixed for the launch, of 0 <= n < 2^31: multiplication
// by 2^(31 + l) / d rounded up, l = ceil(log2 d), which is exact there (T.
// Granlund and P. Montgomery, 1994).  The compiler's division is a chain of
// dozens of instructions, of which a call of a few keys ran several in a row
// before its first load.
struct Divisor {
  unsigned factor;
  int shift;
  __device__ __forceinline__ int operator()(int n) const {
    return static_cast<int>(static_cast<unsigned long long>(factor) * static_cast<unsigned>(n) >>
                            shift);
  }
};
Divisor divisor(std::size_t d) {  // 1 <= d < 2^31
  int l = 0;
  while ((std::size_t{1} << l) < d) ++l;
  return Divisor{static_cast<unsigned>(((1ull << (31 + l)) + d - 1) / d), 31 + l};
}

struct TiledArgs {
  GenericArgs g;
  int key_dim, value_dim, block_tokens, history, tail, keys, queries, rows, offset;
  bool quad;    // history is a multiple of 4
  bool vec_ws;  // workspace rows are 16-byte aligned
  Divisor by_block, by_queries, by_vectors;  // block_tokens, queries, value vectors
  float qscale;  // 1 / sqrt(key_dim); scores of calls past HELD also times log2(e)
};

// Wavefronts of a workgroup: the merge holds one 16 x DM output tile of each
// in LDS.
template <int DM>
constexpr int tiled_waves() {
  return DM <= 64 ? 16 : 8;
}

// exp(t) for t <= 0 (or NaN): 2^(t log2 e) with the rounding of the product
// and of log2 e put back in first order, for scores in natural units.  Over few
// keys this is what the outputs' error is made of (4 heads of 16 dims over 65
// keys, mean of 12 inputs against 64 bits: 1.58e-7 with scores in units of
// log2, 1.42e-7 so, 1.50e-7 for the scalar kernel); over many it costs 3 % and
// the order of the sums, in which this kernel is the better one, decides.
__device__ __forceinline__ float exp_of(float t) {
  constexpr float kL = 1.44269502162933349609375f;  // log2 e, fp32
  constexpr float kLow = 1.92596298909e-8f;         // what it leaves out
  t = t < -200.0f ? -200.0f : t;  // (keeps -inf out of the correction)
  const float hi = t * kL;
  const float lo = fmaf(t, kLow, fmaf(t, kL, -hi));
  const float e = __builtin_amdgcn_exp2f(hi);
  return fmaf(e, lo * 0.693147180559945309f, e);
}
template <bool NATURAL>
__device__ __forceinline__ float power(float t) {
  return NATURAL ? exp_of(t) : __builtin_amdgcn_exp2f(t);
}
template <bool NATURAL>
__device__ __forceinline__ float power_ratio(float a, float b) {
  return NATURAL ? (a == b ? 1.0f : exp_of(a - b)) : exp2_ratio(a, b);
}

// Four consecutive floats of a row from `at` on; entries past `dim` are 0.
template <bool VEC>
__device__ __forceinline__ float4 load4(const float* row, int at, int dim) {
  float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
  if (row == nullptr || at >= dim) return r;
  if constexpr (VEC) return *reinterpret_cast<const float4*>(row + at);
  r.x = row[at];
  if (at + 1 < dim) r.y = row[at + 1];
  if (at + 2 < dim) r.z = row[at + 2];
  if (at + 3 < dim) r.w = row[at + 3];
  return r;
}

// DM: the head sizes' upper bound (32, 64, 128 or 256).  VEC: head sizes are
// multiples of 4 and every tensor is 16-byte aligned.  HELD: the workgroup has
// a wavefront per tile of the keys, whose scores then stay in its registers.
template <int DM, bool VEC, bool HELD>
__global__ __launch_bounds__(tiled_waves<DM>() * 64) void tiled_attention_kernel(TiledArgs a) {
  constexpr int KC = DM / 16;                // 16-dim chunks of the score product
  constexpr int VC = DM <= 64 ? 1 : DM / 64; // 64-dim groups of the outputs
  constexpr int NW = tiled_waves<DM>();
  constexpr int OR = VC * 64 + 4;            // output row stride in LDS
  __shared__ __align__(16) float s_o[NW][16][OR];
  __shared__ float s_ml[NW][2][16];
  __shared__ float s_w[NW][16];
  __shared__ float s_fin[2][16];

  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int waves = static_cast<int>(blockDim.x) >> 6;
  const int col = lane & 15;
  const int grp = lane >> 4;
  const int kvh = static_cast<int>(blockIdx.y);
  const int heads = static_cast<int>(a.g.q_heads / a.g.kv_heads);
  const int T = a.queries;
  auto row_of = [&](int x) { return x - a.by_queries(x) * T; };
  const int r0 = static_cast<int>(blockIdx.x) * 16;
  const int r1 = min(r0 + 16, a.rows) - 1;

  // This lane's query row.
  const bool live = r0 + col < a.rows;
  const int r = live ? r0 + col : r1;
  const int t = row_of(r);
  const std::size_t qrow = (static_cast<std::size_t>(kvh) * heads + a.by_queries(r)) * T + t;
  const int qpos = a.offset + t;
  // Keys below `all` are seen by every row of the tile, keys from `seen` on
  // by none.
  const bool one_head = a.by_queries(r0) == a.by_queries(r1);
  const int all = min(a.keys, a.offset + (one_head ? row_of(r0) : 0) + 1);
  const int seen = min(a.keys, a.offset + (one_head ? row_of(r1) : T - 1) + 1);
  float* const srow = a.g.workspace + qrow * static_cast<std::size_t>(a.keys);

  float4 q[KC];
#pragma unroll
  for (int u = 0; u < KC; ++u) {
    q[u] = load4<VEC>(a.g.query + qrow * a.key_dim, 16 * u + 4 * grp, a.key_dim);
  }
  v4f acc[VC][4];
#pragma unroll
  for (int v = 0; v < VC; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[v][e] = v4f{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.0f;

  // Row index of key `key` in the pools (tail rows: -2 - row, past the keys:
  // -1), with its page checked.
  auto key_row = [&](int key, bool& bad) -> long long {
    bad = false;
    if (key >= seen) return -1;
    if (key >= a.history) return -2 - (static_cast<long long>(kvh) * a.tail + (key - a.history));
    const int page = a.by_block(key);
    const std::uint32_t phys = a.g.table[page];
    if (phys >= a.g.physical_blocks) {
      bad = true;
      return -1;
    }
    return (static_cast<long long>(phys) * a.g.kv_heads + kvh) * a.block_tokens +
           (key - page * a.block_tokens);
  };

  const int tiles = (seen + 15) / 16;
  float4 kept = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);  // HELD: the tile's scores
  bool bad = false;
  long long row = w < tiles ? key_row(w * 16 + col, bad) : -1;
  for (int kt = w; kt < tiles; kt += HELD ? tiles : waves) {
    const int k0 = kt * 16;
    const float* kp = row >= 0    ? a.g.key_blocks + row * a.key_dim
                      : row == -1 ? nullptr
                                  : a.g.tail_key + (-2 - row) * a.key_dim;
    const float* vp = row >= 0    ? a.g.value_blocks + row * a.value_dim
                      : row == -1 ? nullptr
                                  : a.g.tail_value + (-2 - row) * a.value_dim;
    const unsigned bad_keys = static_cast<unsigned>(__ballot(bad)) & 0xffffu;
    float4 k[KC];
#pragma unroll
    for (int u = 0; u < KC; ++u) k[u] = load4<VEC>(kp, 16 * u + 4 * grp, a.key_dim);
    // Value rows of keys k0 + 4 grp + i, this lane's dims 64 v + 4 col: on
    // their way during the scores, where the registers hold both.
    constexpr bool kAhead = DM <= 128;
    float4 val[VC][4];
    auto value_row = [&](int key) -> const float* {
      const auto p = reinterpret_cast<std::uintptr_t>(vp);
      const unsigned lo = __shfl(static_cast<unsigned>(p), key, 64);
      const unsigned hi = __shfl(static_cast<unsigned>(p >> 32), key, 64);
      return reinterpret_cast<const float*>(static_cast<std::uintptr_t>(hi) << 32 | lo);
    };
    auto load_values = [&]() {
      const float* first = value_row(4 * grp);
      // Four keys from a multiple of 4 on lie in one page (or in the tail)
      // wherever the page size and the history are multiples of 4; past
      // `seen` the rows differ (null).
      const bool together = (a.quad || k0 + 16 <= (a.history & ~3)) && k0 + 16 <= seen &&
                            a.block_tokens % 4 == 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float* vrow = i == 0 ? first
                            : !together ? value_row(4 * grp + i)
                            : first == nullptr ? nullptr : first + i * a.value_dim;
#pragma unroll
        for (int v = 0; v < VC; ++v) val[v][i] = load4<VEC>(vrow, 64 * v + 4 * col, a.value_dim);
      }
    };
    if constexpr (kAhead) load_values();
    // The next tile's table entry is on its way meanwhile.
    bool next_bad = false;
    const long long next =
        !HELD && kt + waves < tiles ? key_row((kt + waves) * 16 + col, next_bad) : -1;

    // Two accumulators: half the chain of dependent matrix instructions.
    v4f s0 = v4f{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int u = 0; u < KC; ++u) {
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u].x, q[u].x, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u].y, q[u].y, s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u].z, q[u].z, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u].w, q[u].w, s1, 0, 0, 0);
    }
    if constexpr (!kAhead) load_values();
    // Every row sees every key of the tile and its pages are good.
    const bool plain = k0 + 16 <= all && bad_keys == 0;
    float x[4], p[4];
    bool vis[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = (s0[i] + s1[i]) * a.qscale;
    if (!plain) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = k0 + 4 * grp + i;
        vis[i] = key <= qpos && key < seen;
        if ((bad_keys >> (4 * grp + i) & 1u) != 0) x[i] = NAN;
        if (!vis[i]) x[i] = -INFINITY;
      }
    }
    if constexpr (HELD) {
      kept = make_float4(x[0], x[1], x[2], x[3]);
    } else if (live) {
      float* const dst = srow + k0 + 4 * grp;
      if (a.vec_ws && k0 + 16 <= a.keys) {
        *reinterpret_cast<float4*>(dst) = make_float4(x[0], x[1], x[2], x[3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (k0 + 4 * grp + i < a.keys) dst[i] = x[i];
        }
      }
    }
    const float mn = fmaxf(m, row_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]))));
    const float alpha = power_ratio<HELD>(m, mn);
    if (plain && __ballot(!(fabsf(mn) < INFINITY)) == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = power<HELD>(x[i] - mn);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = plain || vis[i] ? power_ratio<HELD>(x[i], mn) : 0.0f;
    }
    l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
    m = mn;
#pragma unroll
    for (int v = 0; v < VC; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[v][e] *= alpha;

    // O^T += V^T P^T: output tile (v, e) holds dims 64 v + 4 (4 grp + i) + e
    // of row col; contraction step i is keys k0 + 4 grp + i.
    bool special = false;
    if (k0 + 16 > all) {  // some row masks a key here
#pragma unroll
      for (int v = 0; v < VC; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) special = special || !prefill_detail::finite4(val[v][i]);
    }
    if (__ballot(special) == 0) {
#pragma unroll
      for (int v = 0; v < VC; ++v) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[v][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(val[v][i].x, p[i], acc[v][0], 0, 0, 0);
          acc[v][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(val[v][i].y, p[i], acc[v][1], 0, 0, 0);
          acc[v][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(val[v][i].z, p[i], acc[v][2], 0, 0, 0);
          acc[v][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(val[v][i].w, p[i], acc[v][3], 0, 0, 0);
        }
      }
    } else {
      // A value row that is not finite must not reach rows that mask it
      // (0 * inf): key by key, each lane adding to its own outputs.
#pragma unroll 1
      for (int kk = 0; kk < 16; ++kk) {
        const float* vrow = value_row(kk);
        const int c = kk & 3;
        const float mine = c == 0 ? p[0] : c == 1 ? p[1] : c == 2 ? p[2] : p[3];
        const float pk = __shfl(mine, (kk >> 2) * 16 + col, 64);
        const bool sees = k0 + kk <= qpos && k0 + kk < seen;
        if (sees) {
#pragma unroll
          for (int v = 0; v < VC; ++v) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float4 y = load4<VEC>(vrow, 64 * v + 16 * grp + 4 * i, a.value_dim);
              acc[v][0][i] += pk * y.x;
              acc[v][1][i] += pk * y.y;
              acc[v][2][i] += pk * y.z;
              acc[v][3][i] += pk * y.w;
            }
          }
        }
      }
    }
    row = next;
    bad = next_bad;
  }

  // Merge of the wavefronts (one without tiles leaves m = -inf, l = 0, o = 0).
  l = row_sum(l);
#pragma unroll
  for (int v = 0; v < VC; ++v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<float4*>(&s_o[w][col][64 * v + 16 * grp + 4 * i]) =
          make_float4(acc[v][0][i], acc[v][1][i], acc[v][2][i], acc[v][3][i]);
    }
  }
  if (grp == 0) {
    s_ml[w][0][col] = m;
    s_ml[w][1][col] = l;
  }
  __syncthreads();
  // Each row's maximum and sum, and the wavefronts' weights in it: 16 lanes
  // per row, one wavefront's entry each.
  for (int e = static_cast<int>(threadIdx.x); e < 256; e += static_cast<int>(blockDim.x)) {
    const int rr = e >> 4;
    const int x = e & 15;
    const float xm = x < waves ? s_ml[x][0][rr] : -INFINITY;
    float fm = xm;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) fm = fmaxf(fm, __shfl_xor(fm, o, 16));
    const float wt = x < waves ? power_ratio<HELD>(xm, fm) : 0.0f;
    float fl = x < waves ? wt * s_ml[x][1][rr] : 0.0f;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) fl += __shfl_xor(fl, o, 16);
    if (x < waves) s_w[x][rr] = wt;
    if (x == 0) {
      s_fin[0][rr] = fm;
      s_fin[1][rr] = fl;
    }
  }
  __syncthreads();
  const int vectors = (a.value_dim + 3) / 4;
  for (int e = static_cast<int>(threadIdx.x); e < 16 * vectors; e += static_cast<int>(blockDim.x)) {
    const int rr = a.by_vectors(e);
    const int d = (e - rr * vectors) * 4;
    if (r0 + rr > r1) continue;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (int x = 0; x < waves; ++x) {
      const float wt = s_w[x][rr];
      const float4 y = *reinterpret_cast<const float4*>(&s_o[x][rr][d]);
      o.x += wt * y.x;
      o.y += wt * y.y;
      o.z += wt * y.z;
      o.w += wt * y.w;
    }
    const float inv = s_fin[0][rr] == -INFINITY ? NAN : 1.0f / s_fin[1][rr];
    const int rt = r0 + rr;
    float* const dst =
        a.g.out +
        ((static_cast<std::size_t>(kvh) * heads + a.by_queries(rt)) * T + row_of(rt)) * a.value_dim + d;
    if constexpr (VEC) {
      *reinterpret_cast<float4*>(dst) = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
    } else {
      dst[0] = o.x * inv;
      if (d + 1 < a.value_dim) dst[1] = o.y * inv;
      if (d + 2 < a.value_dim) dst[2] = o.z * inv;
      if (d + 3 < a.value_dim) dst[3] = o.w * inv;
    }
  }

  // Scores -> probabilities: each lane its own entries (and keys that no row
  // of the tile sees), kNorm tiles' loads together.
  if (!live) return;
  const float fm = s_fin[0][col];
  const float fl = s_fin[1][col];
  const bool nan_row = fm == -INFINITY || isnan(fl);
  constexpr int kNorm = HELD ? 1 : 4;
  for (int kt = w; kt * 16 < a.keys; kt += kNorm * waves) {
    float4 x[kNorm];
    auto whole = [&](int n) {  // uniform: 16-byte entries that every row sees
      const int k0 = (kt + n * waves) * 16;
      return a.vec_ws && k0 + 16 <= all;
    };
#pragma unroll
    for (int n = 0; n < kNorm; ++n) {
      const int key = (kt + n * waves) * 16 + 4 * grp;
      if constexpr (HELD) {
        x[n] = kept;
      } else if (whole(n)) {
        x[n] = *reinterpret_cast<const float4*>(srow + key);
      } else {
        x[n].x = key <= qpos && key < seen ? srow[key] : -INFINITY;
        x[n].y = key + 1 <= qpos && key + 1 < seen ? srow[key + 1] : -INFINITY;
        x[n].z = key + 2 <= qpos && key + 2 < seen ? srow[key + 2] : -INFINITY;
        x[n].w = key + 3 <= qpos && key + 3 < seen ? srow[key + 3] : -INFINITY;
      }
    }
#pragma unroll
    for (int n = 0; n < kNorm; ++n) {
      const int key = (kt + n * waves) * 16 + 4 * grp;
      const float y[4] = {x[n].x, x[n].y, x[n].z, x[n].w};
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool sees = key + i <= qpos && key + i < seen;
        p[i] = nan_row ? NAN : sees ? power_ratio<HELD>(y[i], fm) / fl : 0.0f;
      }
      if (whole(n)) {
        *reinterpret_cast<float4*>(srow + key) = make_float4(p[0], p[1], p[2], p[3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (key + i < a.keys) srow[key + i] = p[i];
        }
      }
    }
  }
}

bool aligned(const void* p) { return (reinterpret_cast<std::uintptr_t>(p) & 15u) == 0; }

}  // namespace

bool tiled_attention_fits(const GenericArgs& a) {
  constexpr std::size_t kMax = static_cast<std::size_t>(std::numeric_limits<std::int32_t>::max()) / 2;
  return a.key_dim >= 1 && a.key_dim <= 256 && a.value_dim >= 1 && a.value_dim <= 256 &&
         a.kv_heads >= 1 && a.kv_heads <= 65535 && a.q_heads % a.kv_heads == 0 &&
         a.block_tokens >= 1 && a.block_tokens <= kMax && a.history <= kMax &&
         a.tail <= kMax && a.offset <= kMax && a.queries <= kMax &&
         a.history + a.tail <= kMax && a.offset + a.queries <= kMax &&
         a.q_heads / a.kv_heads <= kMax / (a.queries == 0 ? 1 : a.queries);
}

hipError_t launch_tiled_attention(const GenericArgs& a, hipStream_t stream) {
  if (a.queries == 0 || a.q_heads == 0) return hipSuccess;
  TiledArgs k{};
  k.g = a;
  k.key_dim = static_cast<int>(a.key_dim);
  k.value_dim = static_cast<int>(a.value_dim);
  k.block_tokens = static_cast<int>(a.block_tokens);
  k.history = static_cast<int>(a.history);
  k.tail = static_cast<int>(a.tail);
  k.keys = static_cast<int>(a.history + a.tail);
  k.queries = static_cast<int>(a.queries);
  k.rows = static_cast<int>(a.q_heads / a.kv_heads * a.queries);
  k.offset = static_cast<int>(a.offset);
  k.quad = a.history % 4 == 0;
  k.vec_ws = (a.history + a.tail) % 4 == 0 && aligned(a.workspace);
  k.by_block = divisor(a.block_tokens);
  k.by_queries = divisor(a.queries);
  k.by_vectors = divisor((a.value_dim + 3) / 4);
  const bool vec = a.key_dim % 4 == 0 && a.value_dim % 4 == 0 && aligned(a.query) &&
                   aligned(a.key_blocks) && aligned(a.value_blocks) && aligned(a.tail_key) &&
                   aligned(a.tail_value) && aligned(a.out);
  const dim3 grid(static_cast<unsigned>((k.rows + 15) / 16), static_cast<unsigned>(a.kv_heads));
  const int key_tiles = (k.keys + 15) / 16;
  auto run = [&](auto dm) {
    constexpr int DM = decltype(dm)::value;
    constexpr int most = tiled_waves<DM>();
    const unsigned threads = 64u * static_cast<unsigned>(key_tiles < most ? key_tiles : most);
    const bool held = key_tiles <= most;
    k.qscale = (held ? 1.0f : 1.4426950408889634f) / sqrtf(static_cast<float>(a.key_dim));
    if (vec) {
      auto* const kernel =
          held ? tiled_attention_kernel<DM, true, true> : tiled_attention_kernel<DM, true, false>;
      kernel<<<grid, threads, 0, stream>>>(k);
    } else {
      auto* const kernel =
          held ? tiled_attention_kernel<DM, false, true> : tiled_attention_kernel<DM, false, false>;
      kernel<<<grid, threads, 0, stream>>>(k);
    }
  };
  const std::size_t dim = a.key_dim > a.value_dim ? a.key_dim : a.value_dim;
  if (dim <= 32) {
    run(std::integral_constant<int, 32>{});
  } else if (dim <= 64) {
    run(std::integral_constant<int, 64>{});
  } else if (dim <= 128) {
    run(std::integral_constant<int, 128>{});
  } else {
    run(std::integral_constant<int, 256>{});
  }
  return hipGetLastError();
}

}  // namespace helix::hip
