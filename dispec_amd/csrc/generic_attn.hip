// J3 / J4 for the shapes the tuned attention kernels leave out: fp32 caches, head_dim 8 (any
// power of two from 8 to 256), and 256-wide heads or GQA groups above 8 on decode where the
// tuned kernels' 16-byte vectors are not aligned or the keys come from a slot table.  The reference's
// Triton kernel takes any power-of-two HEAD_DIM and loads keys and values as fp32
// (dispec/engine/triton_attn.py:60-95, tl.arange(0, HEAD_DIM) at :71); its native path
// attends in whatever dtype the model runs (dispec/engine/model_runner.py:160-185).  fp32
// caches run on 16-row tiles of the fp32 matrix cores (f32_tile_kernel below); the 16-bit
// shapes on a general kernel, correct and coalesced:
//
//  * one wave per (query row, query head, key partition of P keys); lane d holds dims d,
//    d + 64, ..., so every K or V row is read by one coalesced load per 64 dims;
//  * eight keys per step: eight partial dot products reduced across the wave side by side
//    (DPP within rows of 16 lanes, then two lane permutes), an online softmax in base 2,
//    fp32 accumulation;
//  * query row i of sequence b's block sees keys j <= ctx_b - q_len_b + i (causal,
//    lower-right); decode is one row per sequence over its whole context;
//  * a row with more than one partition is merged by the second kernel (16 partitions'
//    partials in flight per lane).
//
// Grid x runs over B * max_q_len row slots z (b = z / max_q_len, i = z % max_q_len), as the
// tiled kernels' grids do: a sequence's rows beyond max_q_len are not computed.  Partial
// results go to ws row (z * Hq + h) * num_parts + part (B * max_q_len * Hq rows of
// num_parts partitions, then their (max, sum) pairs).
#include <float.h>

#include <type_traits>

#include "dsp_common.h"
#include "dsp_internal.h"

namespace {

struct GBf16 { using store = uint16_t; };
struct GF16 { using store = uint16_t; };
struct GF32 { using store = float; };

template <typename Tag>
__device__ __forceinline__ float ld1(const typename Tag::store* p) {
  if constexpr (std::is_same<Tag, GBf16>::value)
    return dsp_bf16lo(*p);
  else if constexpr (std::is_same<Tag, GF16>::value)
    return dsp_f16lo(*p);
  else
    return *p;
}

template <typename Tag>
__device__ __forceinline__ typename Tag::store st1(float f) {
  if constexpr (std::is_same<Tag, GBf16>::value)
    return dsp_f32_to_bf16(f);
  else if constexpr (std::is_same<Tag, GF16>::value)
    return dsp_f32_to_f16(f);
  else
    return f;
}

constexpr int kKeysPerStep = 8;
constexpr int kMergeBatch = 16;

// Where row slot z sits and how many keys it sees.
struct RowInfo {
  int b;         // sequence
  int64_t tok;   // packed row of q / out
  int vis;       // visible keys; 0 writes zeros
  bool live;     // false: slot beyond the sequence's q_len (nothing to write)
  bool counted;  // this slot reports the sequence's bad lengths (one slot per sequence)
};

__device__ __forceinline__ RowInfo row_info(const int32_t* __restrict__ cu_q,
                                            const int32_t* __restrict__ ctx_lens,
                                            int max_q_len, int max_ctx, int z) {
  RowInfo r;
  r.b = z / max_q_len;
  const int i = z - r.b * max_q_len;
  const int ctx = ctx_lens[r.b];
  if (cu_q == nullptr) {  // decode: one row per sequence, context clamped to [0, max_ctx]
    r.tok = r.b;
    r.live = true;
    r.vis = ctx < 0 ? 0 : (ctx > max_ctx ? max_ctx : ctx);
    r.counted = ctx < 0 || ctx > max_ctx;
    return r;
  }
  const int c0 = cu_q[r.b];
  const int qlen = cu_q[r.b + 1] - c0;
  r.tok = int64_t(c0) + i;
  r.live = i < qlen;
  const bool bad = qlen < 0 || ctx < qlen || ctx > max_ctx;
  r.vis = bad ? 0 : ctx - qlen + i + 1;
  r.counted = bad && i == 0;
  return r;
}

// Sum over all 64 lanes of the wave, every lane ending with the total.
__device__ __forceinline__ float wave_sum(float v) {
  v = dsp_group_sum<16>(v);
  v += dsp_shfl_xor(v, 16);
  return v + dsp_shfl_xor(v, 32);
}

template <typename Tag, int D>
__global__ __launch_bounds__(64) void generic_attn_kernel(
    const typename Tag::store* __restrict__ q, int64_t qst, int64_t qsh,
    const typename Tag::store* __restrict__ kc, const typename Tag::store* __restrict__ vc,
    int64_t num_slots, int64_t kvs_slot, int64_t kvs_head, const int32_t* __restrict__ table,
    int64_t table_stride, int32_t log2_bs, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ ctx_lens, int32_t G, int32_t max_ctx, int32_t max_q_len,
    float scale_log2, int32_t P, int32_t num_parts, float* __restrict__ ws_acc,
    float* __restrict__ ws_ml, typename Tag::store* __restrict__ out, int64_t ost, int64_t osh,
    int32_t* __restrict__ err_count) {
  constexpr int NV = D > 64 ? D / 64 : 1;  // dims per lane
  const int z = blockIdx.x, h = blockIdx.y, part = blockIdx.z, Hq = gridDim.y;
  const int lane = threadIdx.x;
  const bool act = lane < D;
  const RowInfo r = row_info(cu_q, ctx_lens, max_q_len, max_ctx, z);
  if (!r.live) return;
  if (r.counted && part == 0 && h == 0 && lane == 0 && err_count) atomicAdd(err_count, 1);
  const int vis = r.vis;
  const int nparts = vis > 0 ? (vis + P - 1) / P : 1;
  typename Tag::store* o = out + r.tok * ost + int64_t(h) * osh;
  if (vis <= 0) {  // no keys (an empty context or bad lengths): zeros
    if (part == 0 && act) {
#pragma unroll
      for (int j = 0; j < NV; ++j) o[lane + 64 * j] = st1<Tag>(0.f);
    }
    return;
  }
  if (part >= nparts) return;
  const int kbeg = part * P, kend = min(kbeg + P, vis);
  float qf[NV], acc[NV];
  const typename Tag::store* qrow = q + r.tok * qst + int64_t(h) * qsh;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    qf[j] = act ? ld1<Tag>(qrow + lane + 64 * j) * scale_log2 : 0.f;
    acc[j] = 0.f;
  }
  const int64_t head_off = int64_t(h / G) * kvs_head + (act ? lane : 0);
  const int32_t* trow = table + int64_t(r.b) * table_stride;
  float m = -INFINITY, l = 0.f;
  bool bad_slot = false;
  for (int k0 = kbeg; k0 < kend; k0 += kKeysPerStep) {
    float kv[kKeysPerStep][NV], vv[kKeysPerStep][NV], s[kKeysPerStep];
    bool ok[kKeysPerStep];
#pragma unroll
    for (int u = 0; u < kKeysPerStep; ++u) {
      const int key = k0 + u;
      int64_t sl = 0;
      if (key < kend) {
        sl = log2_bs >= 0 ? (int64_t(trow[key >> log2_bs]) << log2_bs) +
                                (key & ((1 << log2_bs) - 1))
                          : int64_t(trow[key]);
      }
      ok[u] = key < kend && sl >= 0 && sl < num_slots;
      bad_slot |= key < kend && !ok[u];
      const int64_t e = (ok[u] ? sl : 0) * kvs_slot + head_off;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        kv[u][j] = act && ok[u] ? ld1<Tag>(kc + e + 64 * j) : 0.f;
        vv[u][j] = act && ok[u] ? ld1<Tag>(vc + e + 64 * j) : 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < kKeysPerStep; ++u) {
      float p = 0.f;
#pragma unroll
      for (int j = 0; j < NV; ++j) p = fmaf(qf[j], kv[u][j], p);
      s[u] = wave_sum(p);
    }
    float mx = m;
#pragma unroll
    for (int u = 0; u < kKeysPerStep; ++u) {
      s[u] = ok[u] ? s[u] : -INFINITY;
      mx = fmaxf(mx, s[u]);
    }
    const float mu = mx == -INFINITY ? 0.f : mx;
    const float alpha = dsp_exp2(m - mu);
    l *= alpha;
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[j] *= alpha;
#pragma unroll
    for (int u = 0; u < kKeysPerStep; ++u) {
      const float p = dsp_exp2(s[u] - mu);
      l += p;
#pragma unroll
      for (int j = 0; j < NV; ++j) acc[j] = fmaf(p, vv[u][j], acc[j]);
    }
    m = mx;
  }
  if (bad_slot && lane == 0 && err_count) atomicAdd(err_count, 1);
  if (nparts == 1) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    if (act) {
#pragma unroll
      for (int j = 0; j < NV; ++j) o[lane + 64 * j] = st1<Tag>(acc[j] * inv);
    }
    return;
  }
  const int64_t row = (int64_t(z) * Hq + h) * num_parts + part;
  if (act) {
#pragma unroll
    for (int j = 0; j < NV; ++j) ws_acc[row * D + lane + 64 * j] = acc[j];
  }
  if (lane == 0) {
    ws_ml[2 * row] = m;
    ws_ml[2 * row + 1] = l;
  }
}

// fp32 caches: the same attention on the fp32 matrix cores (v_mfma_f32_16x16x4_f32).  A
// workgroup of 4 waves owns 16 packed rows (row r: query r / G, head r % G) of one (sequence,
// KV head) and one partition of its keys, so a key row is read once for the G heads and the
// queries of the tile (one wave per row re-read it for each: 8 decodes and a 128-token chunk
// of 14 heads over 1000-2000 keys took 379 us).  The waves take 16-key chunks in turn.
//  * S^T = K . Q^T: lane l holds row l % 16 of an operand and, per MFMA, one value of K index
//    l / 16; the dims are dealt so that a lane's values of 4 MFMAs are 4 consecutive floats
//    (MFMA 4j + e, K index g: dim 16j + 4g + e; D 8: MFMA e, dim 2g + e): K rows come straight
//    from memory in 16-byte loads (4-byte alignment is enough for them), Q stays in registers.
//    Four chains of MFMAs, added at the end: a chain's rounding grows with its length.
//  * S^T leaves lane l with keys 4 (l / 16) + j of row l % 16, the B operand of O^T = V^T . P^T
//    for the 4 keys {4g + j : g}: P stays in fp32 registers.  V^T's operand is dim index
//    l % 16 of a 16-dim tile; tile e of vector h holds dims 64h + 4 (l % 16) + e (D 32: 2 (l %
//    16) + e), so V rows too are read in 16-byte loads and nothing goes through LDS.
// Bound by the latency of its loads (slot, then K and V rows): that step's kernel takes 26 us
// (379 before), the error against 64 bits 2.3e-7 (3.3e-7).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

template <int N>
__device__ __forceinline__ void load_f32(const float* __restrict__ p, bool ok, float (&f)[N]) {
  if constexpr (N == 4) {
    f32x4u v = {0.f, 0.f, 0.f, 0.f};
    if (ok) v = *reinterpret_cast<const f32x4u*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = v[i];
  } else if constexpr (N == 2) {
    f32x2u v = {0.f, 0.f};
    if (ok) v = *reinterpret_cast<const f32x2u*>(p);
    f[0] = v[0];
    f[1] = v[1];
  } else {
    f[0] = ok ? *p : 0.f;
  }
}

constexpr int kTileWaves = 4;

template <int D>
__global__ __launch_bounds__(64 * kTileWaves) __attribute__((amdgpu_waves_per_eu(D > 128 ? 1 : 2))) void f32_tile_kernel(
    const float* __restrict__ q, int64_t qst, int64_t qsh, const float* __restrict__ kc,
    const float* __restrict__ vc, int64_t num_slots, int64_t kvs_slot, int64_t kvs_head,
    const int32_t* __restrict__ table, int64_t table_stride, int32_t log2_bs,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ ctx_lens, int32_t G,
    int32_t max_ctx, int32_t max_q_len, float scale_log2, int32_t P, int32_t num_parts,
    float* __restrict__ ws_acc, float* __restrict__ ws_ml, float* __restrict__ out, int64_t ost,
    int64_t osh, int32_t* __restrict__ err_count) {
  constexpr int KE = D >= 16 ? 4 : 2;          // floats per K load
  constexpr int KJ = D / (4 * KE);             // K loads per row and lane
  constexpr int VE = D >= 64 ? 4 : (D >= 32 ? 2 : 1);  // floats per V load
  constexpr int VH = D >= 64 ? D / 64 : 1;     // V loads per key and lane
  constexpr int NT = VE * VH;                  // 16-dim output tiles (D 8: half of one)
  __shared__ float s_acc[kTileWaves][16][D + 1];
  __shared__ float s_m[kTileWaves][16], s_l[kTileWaves][16];
  __shared__ int32_t s_bad[kTileWaves];        // first key of a bad slot each wave met
  const int part = blockIdx.x % num_parts, tile = blockIdx.x / num_parts;
  const int kvh = blockIdx.y, b = blockIdx.z, KVH = gridDim.y, Hq = KVH * G;
  const bool dec = cu_q == nullptr;
  const int q0 = dec ? b : cu_q[b];
  const int qlen = dec ? 1 : cu_q[b + 1] - q0;
  int ctx = ctx_lens[b];
  const int rows = min(qlen, max_q_len) * G, r0 = tile * 16;
  if (qlen <= 0 || r0 >= rows) return;
  const bool bad_len = dec ? ctx < 0 || ctx > max_ctx : ctx < qlen || ctx > max_ctx;
  if (bad_len && threadIdx.x == 0 && tile == 0 && part == 0 && kvh == 0 && err_count)
    atomicAdd(err_count, 1);
  if (dec) ctx = ctx < 0 ? 0 : (ctx > max_ctx ? max_ctx : ctx);
  // keys visible to row r: its query's position + 1 (none for bad lengths or no context)
  auto visible = [&](int r) { return !dec && bad_len ? 0 : ctx - qlen + r / G + 1; };
  const int kend = visible(min(r0 + 15, rows - 1)), vis0 = visible(r0);
  const int kbeg = part * P, kfin = min(kbeg + P, kend);
  if (kbeg >= kend && part > 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = lane & 15, grp = lane >> 4;
  const int r = r0 + n;
  const bool row_ok = r < rows;
  const int vis = row_ok ? visible(r) : 0;
  const float* qrow = q + int64_t(q0 + (row_ok ? r / G : 0)) * qst +
                      int64_t(kvh * G + (row_ok ? r % G : 0)) * qsh;
  float qf[KJ][KE];
#pragma unroll
  for (int j = 0; j < KJ; ++j) load_f32<KE>(qrow + 4 * KE * j + KE * grp, row_ok, qf[j]);
  const int32_t* trow = table + int64_t(b) * table_stride;
  const int64_t head_off = int64_t(kvh) * kvs_head;
  auto slot_of = [&](int key) -> int64_t {  // -1: past the partition, or outside the cache
    if (key >= kfin) return -1;
    const int64_t sl = log2_bs >= 0 ? (int64_t(trow[key >> log2_bs]) << log2_bs) +
                                          (key & ((1 << log2_bs) - 1))
                                    : int64_t(trow[key]);
    return sl >= 0 && sl < num_slots ? sl : -1;
  };
  float m = -INFINITY, l = 0.f;
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int first_bad = INT32_MAX;
  int64_t slot = slot_of(kbeg + 16 * wave + n);  // of this lane's key of the next chunk
  for (int t0 = kbeg + 16 * wave; t0 < kfin; t0 += 16 * kTileWaves) {
    const int64_t cur = slot;
    if (t0 + n < kfin && cur < 0 && first_bad == INT32_MAX) first_bad = t0 + n;
    float kf[KJ][KE], vf[4][VH][VE];
    const float* krow = kc + (cur < 0 ? 0 : cur) * kvs_slot + head_off + KE * grp;
#pragma unroll
    for (int j = 0; j < KJ; ++j) load_f32<KE>(krow + 4 * KE * j, cur >= 0, kf[j]);
    bool ok[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // keys 4 * grp + j: their slots sit in lanes 0..15
      const int src = 4 * grp + j;
      const int64_t sv = (int64_t(__shfl(int(cur >> 32), src)) << 32) |
                         uint32_t(__shfl(int(uint32_t(cur)), src));
      ok[j] = sv >= 0;
      const float* vrow = vc + (ok[j] ? sv : 0) * kvs_slot + head_off + VE * n;
#pragma unroll
      for (int h = 0; h < VH; ++h)
        load_f32<VE>(vrow + 64 * h, ok[j] && (D >= 16 || n < D), vf[j][h]);
    }
    slot = slot_of(t0 + 16 * kTileWaves + n);
    // scores of keys t0 + 4 * grp + j, row n: up to four chains
    constexpr int CH = KJ * KE < 4 ? KJ * KE : 4;
    f32x4 sc[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) sc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < KJ; ++j)
#pragma unroll
      for (int e = 0; e < KE; ++e)
        sc[(j * KE + e) % CH] =
            __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][e], qf[j][e], sc[(j * KE + e) % CH], 0, 0, 0);
#pragma unroll
    for (int c = 1; c < CH; ++c) sc[0] += sc[c];
    float p[4], mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      p[j] = ok[j] && t0 + 4 * grp + j < vis ? sc[0][j] * scale_log2 : -INFINITY;
      mx = fmaxf(mx, p[j]);
    }
    mx = fmaxf(mx, dsp_shfl_xor(mx, 16));
    mx = fmaxf(mx, dsp_shfl_xor(mx, 32));
    const float mn = fmaxf(m, mx), mu = mn == -INFINITY ? 0.f : mn;
    const float alpha = dsp_exp2(m - mu);
    m = mn;
    l *= alpha;
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] *= alpha;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      p[j] = dsp_exp2(p[j] - mu);
      l += p[j];
    }
    if (t0 + 16 > vis0) {  // a chunk that the tile's first row does not see whole (uniform)
      bool odd = false;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < VH; ++h)
#pragma unroll
          for (int e = 0; e < VE; ++e) odd |= !(fabsf(vf[j][h][e]) < INFINITY);
      if (__ballot(odd)) {  // rare
        // Infinities and NaN of V go to the rows that see their keys only (0 * inf is NaN):
        // kHuge * kHuge overflows to inf, -kHuge * kHuge to -inf, and NaN takes both (each
        // from a sum of its own: products are not rounded before they are added, and inf - 2^254
        // is inf).
        constexpr float kHuge = 0x1p127f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float seen = t0 + 4 * grp + j < vis ? kHuge : 0.f;
#pragma unroll
          for (int h = 0; h < VH; ++h)
#pragma unroll
            for (int e = 0; e < VE; ++e) {
              float& v = vf[j][h][e];
              f32x4& a = acc[h * VE + e];
              const bool nan = v != v;
              const f32x4 none = {0.f, 0.f, 0.f, 0.f};
              a += __builtin_amdgcn_mfma_f32_16x16x4f32(nan || v == INFINITY ? kHuge : 0.f, seen, none,
                                                        0, 0, 0);
              a += __builtin_amdgcn_mfma_f32_16x16x4f32(nan || v == -INFINITY ? -kHuge : 0.f, seen,
                                                        none, 0, 0, 0);
              v = fabsf(v) < INFINITY ? v : 0.f;
            }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int h = 0; h < VH; ++h)
#pragma unroll
        for (int e = 0; e < VE; ++e)
          acc[h * VE + e] =
              __builtin_amdgcn_mfma_f32_16x16x4f32(vf[j][h][e], p[j], acc[h * VE + e], 0, 0, 0);
  }
  l += dsp_shfl_xor(l, 16);
  l += dsp_shfl_xor(l, 32);
#pragma unroll
  for (int k = 1; k < 64; k <<= 1) first_bad = min(first_bad, __shfl_xor(first_bad, k));
  if (lane == 0) s_bad[wave] = first_bad;
  if (grp == 0) {
    s_m[wave][n] = m;
    s_l[wave][n] = l;
  }
  // acc tile (h, e), element j: dim index 4 * grp + j of the tile, row n
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = 64 * (t / VE) + VE * (4 * grp + j) + t % VE;
      if (D >= 16 || d < D) s_acc[wave][n][d] = acc[t][j];
    }
  __syncthreads();
  int bad_key = s_bad[0];
#pragma unroll
  for (int w = 1; w < kTileWaves; ++w) bad_key = min(bad_key, s_bad[w]);
  for (int idx = threadIdx.x; idx < 16 * D; idx += 64 * kTileWaves) {
    const int rr = idx / D, d = idx % D, row = r0 + rr;
    if (row >= rows) break;
    const int rvis = visible(row), np = rvis > 0 ? (rvis + P - 1) / P : 1;
    if (part >= np) continue;
    // counted once per (row, partition) that met a bad block id
    if (d == 0 && bad_key < rvis && err_count) atomicAdd(err_count, 1);
    float M = s_m[0][rr];
#pragma unroll
    for (int w = 1; w < kTileWaves; ++w) M = fmaxf(M, s_m[w][rr]);
    const float Mu = M == -INFINITY ? 0.f : M;
    float L = 0.f, A = 0.f;
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) {
      const float x = dsp_exp2(s_m[w][rr] - Mu);
      L = fmaf(s_l[w][rr], x, L);
      A = fmaf(s_acc[w][rr][d], x, A);
    }
    const int i = row / G, h = kvh * G + row % G;
    if (np == 1) {
      // (no keys: 0 * 0; a NaN score makes L and A NaN, and the row with them)
      out[int64_t(q0 + i) * ost + int64_t(h) * osh + d] = A * (L > 0.f ? 1.f / L : 0.f);
    } else {
      const int64_t w = ((int64_t(b) * max_q_len + i) * Hq + h) * num_parts + part;
      ws_acc[w * D + d] = A;
      if (d == 0) {
        ws_ml[2 * w] = M;
        ws_ml[2 * w + 1] = L;
      }
    }
  }
}

// Merge of a row's partitions: one wave per (row slot, head), four heads per workgroup (most row
// slots of a ragged batch are empty: a quarter of the workgroups to start and end); lane d
// folds dims d, d+64, ...
template <typename Tag, int D>
__global__ __launch_bounds__(256) void generic_merge_kernel(
    const float* __restrict__ ws_acc, const float* __restrict__ ws_ml,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ ctx_lens, int32_t max_ctx,
    int32_t max_q_len, int32_t P, int32_t num_parts, int32_t Hq,
    typename Tag::store* __restrict__ out, int64_t ost, int64_t osh) {
  constexpr int NV = D > 64 ? D / 64 : 1;
  const int z = blockIdx.x, h = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (h >= Hq) return;
  const RowInfo r = row_info(cu_q, ctx_lens, max_q_len, max_ctx, z);
  if (!r.live || r.vis <= P) return;  // one partition at most: written by the attention kernel
  const int nparts = (r.vis + P - 1) / P;
  const int64_t row0 = (int64_t(z) * Hq + h) * num_parts;
  const bool act = lane < D;
  float M = -INFINITY, L = 0.f, A[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) A[j] = 0.f;
  for (int p0 = 0; p0 < nparts; p0 += kMergeBatch) {
    const int n = min(nparts - p0, kMergeBatch);
    float vm[kMergeBatch], vl[kMergeBatch], va[kMergeBatch][NV];
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const int64_t rr = row0 + p0 + (u < n ? u : 0);
      vm[u] = u < n ? ws_ml[2 * rr] : -INFINITY;
      vl[u] = u < n ? ws_ml[2 * rr + 1] : 0.f;
#pragma unroll
      for (int j = 0; j < NV; ++j)
        va[u][j] = (u < n && act) ? ws_acc[rr * D + lane + 64 * j] : 0.f;
    }
    float bm = M;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) bm = fmaxf(bm, vm[u]);
    const float bmu = bm == -INFINITY ? 0.f : bm;
    const float keep = dsp_exp2(M - bmu);
    L *= keep;
#pragma unroll
    for (int j = 0; j < NV; ++j) A[j] *= keep;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const float w = dsp_exp2(vm[u] - bmu);
      L = fmaf(vl[u], w, L);
#pragma unroll
      for (int j = 0; j < NV; ++j) A[j] = fmaf(va[u][j], w, A[j]);
    }
    M = bm;
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  if (act) {
    typename Tag::store* o = out + r.tok * ost + int64_t(h) * osh;
#pragma unroll
    for (int j = 0; j < NV; ++j) o[lane + 64 * j] = st1<Tag>(A[j] * inv);
  }
}

struct GenericArgs {
  const void* q;
  int64_t qst, qsh;
  const void* kc;
  const void* vc;
  int64_t num_slots, kvs_slot, kvs_head;
  const int32_t* table;
  int64_t table_stride;
  int32_t log2_bs;
  const int32_t* cu_q;
  const int32_t* ctx_lens;
  int32_t G, Hq, max_ctx, max_q_len;
  float scale_log2;
  int32_t P, num_parts;
  float* ws_acc;
  float* ws_ml;
  void* out;
  int64_t ost, osh;
  int32_t* err_count;
};

template <typename Tag, int D>
int launch_generic_d(const GenericArgs& a, dim3 grid, dim3 mgrid, hipStream_t s) {
  using S = typename Tag::store;
  if constexpr (std::is_same<Tag, GF32>::value)
    f32_tile_kernel<D><<<grid, 64 * kTileWaves, 0, s>>>(
        static_cast<const S*>(a.q), a.qst, a.qsh, static_cast<const S*>(a.kc),
        static_cast<const S*>(a.vc), a.num_slots, a.kvs_slot, a.kvs_head, a.table, a.table_stride,
        a.log2_bs, a.cu_q, a.ctx_lens, a.G, a.max_ctx, a.max_q_len, a.scale_log2, a.P,
        a.num_parts, a.ws_acc, a.ws_ml, static_cast<S*>(a.out), a.ost, a.osh, a.err_count);
  else
    generic_attn_kernel<Tag, D><<<grid, 64, 0, s>>>(
        static_cast<const S*>(a.q), a.qst, a.qsh, static_cast<const S*>(a.kc),
        static_cast<const S*>(a.vc), a.num_slots, a.kvs_slot, a.kvs_head, a.table, a.table_stride,
        a.log2_bs, a.cu_q, a.ctx_lens, a.G, a.max_ctx, a.max_q_len, a.scale_log2, a.P,
        a.num_parts, a.ws_acc, a.ws_ml, static_cast<S*>(a.out), a.ost, a.osh, a.err_count);
  const int st = dsp_launch_status();
  if (st != DSP_OK || a.num_parts <= 1) return st;
  generic_merge_kernel<Tag, D><<<mgrid, 256, 0, s>>>(a.ws_acc, a.ws_ml, a.cu_q, a.ctx_lens,
                                                     a.max_ctx, a.max_q_len, a.P, a.num_parts,
                                                     a.Hq, static_cast<S*>(a.out), a.ost, a.osh);
  return dsp_launch_status();
}

template <typename Tag>
int launch_generic(int D, const GenericArgs& a, dim3 grid, dim3 mgrid, hipStream_t s) {
  switch (D) {
    case 8: return launch_generic_d<Tag, 8>(a, grid, mgrid, s);
    case 16: return launch_generic_d<Tag, 16>(a, grid, mgrid, s);
    case 32: return launch_generic_d<Tag, 32>(a, grid, mgrid, s);
    case 64: return launch_generic_d<Tag, 64>(a, grid, mgrid, s);
    case 128: return launch_generic_d<Tag, 128>(a, grid, mgrid, s);
    case 256: return launch_generic_d<Tag, 256>(a, grid, mgrid, s);
    default: return DSP_EUNSUPPORTED;
  }
}

}  // namespace

namespace dsp_detail {

bool generic_head_dim(int32_t D) {
  return D == 8 || D == 16 || D == 32 || D == 64 || D == 128 || D == 256;
}

size_t generic_workspace_bytes(int32_t B, int32_t Hq, int32_t D, int32_t max_q_len,
                               int32_t max_ctx, int32_t P) {
  if (B <= 0 || Hq <= 0 || max_q_len <= 0 || max_ctx <= 0 || P <= 0) return 0;
  const int64_t np = (int64_t(max_ctx) + P - 1) / P;
  if (np <= 1) return 0;
  return size_t(B) * max_q_len * Hq * np * (size_t(D) + 2) * sizeof(float);
}

int generic_attention(const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_cache,
                      const void* v_cache, int64_t num_slots, int64_t kv_stride_slot,
                      int64_t kv_stride_head, const int32_t* table, int64_t table_stride,
                      int32_t log2_bs, const int32_t* cu_q, const int32_t* ctx_lens, int32_t B,
                      int32_t Hq, int32_t KVH, int32_t D, float scale, int32_t max_q_len,
                      int32_t max_ctx, int32_t P, void* workspace, void* out,
                      int64_t o_stride_t, int64_t o_stride_h, int32_t dtype, int32_t* err_count,
                      hipStream_t s) {
  if (B == 0 || max_q_len == 0) return DSP_OK;
  const int32_t num_parts = max_ctx > 0 ? (max_ctx + P - 1) / P : 1;
  const int64_t rows = int64_t(B) * max_q_len;
  // grid: x row slots (a sequence's rows side by side: they read the same keys), y query
  // heads, z partitions
  if (rows > (int64_t(1) << 26) || Hq > 65535 || num_parts > 65535) return DSP_EUNSUPPORTED;
  float* ws_acc = static_cast<float*>(workspace);
  GenericArgs a{q, q_stride_t, q_stride_h, k_cache, v_cache, num_slots, kv_stride_slot,
                kv_stride_head, table, table_stride, log2_bs, cu_q, ctx_lens, Hq / KVH, Hq,
                max_ctx, max_q_len, scale * 1.4426950408889634f, P, num_parts, ws_acc,
                num_parts > 1 ? ws_acc + rows * Hq * num_parts * D : nullptr, out, o_stride_t,
                o_stride_h, err_count};
  dim3 grid(static_cast<unsigned>(rows), static_cast<unsigned>(Hq),
            static_cast<unsigned>(num_parts));
  dim3 mgrid(static_cast<unsigned>(rows), static_cast<unsigned>((Hq + 3) / 4));
  if (dtype == DSP_F32) {
    // 16-row tiles: x (tile, partition), y KV heads, z sequences
    const int64_t tiles = (int64_t(max_q_len) * (Hq / KVH) + 15) / 16;
    if (tiles * num_parts >= (int64_t(1) << 31) || KVH > 65535 || B > 65535)
      return DSP_EUNSUPPORTED;
    grid = dim3(static_cast<unsigned>(tiles * num_parts), static_cast<unsigned>(KVH),
                static_cast<unsigned>(B));
  }
  switch (dtype) {
    case DSP_BF16: return launch_generic<GBf16>(D, a, grid, mgrid, s);
    case DSP_F16: return launch_generic<GF16>(D, a, grid, mgrid, s);
    case DSP_F32: return launch_generic<GF32>(D, a, grid, mgrid, s);
    default: return DSP_EUNSUPPORTED;
  }
}

}  // namespace dsp_detail
