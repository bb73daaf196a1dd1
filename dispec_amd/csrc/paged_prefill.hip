// J4 for long query blocks (chunked prefill over the paged cache): a FlashAttention-style
// tile of 128 packed rows per workgroup on v_mfma_f32_32x32x16.
//
// Semantics are dsp_paged_mq_attention's (ModelRunner._attention's native branch,
// dispec/engine/model_runner.py:160-185): per sequence, SDPA over the paged context with
// causal_lower_right(q_len, ctx) and GQA; packed row r of a (sequence, KV head) is query
// r / G of query head kvh*G + r % G.
//
// Why a second kernel: the multi-query kernel of paged_mq.hip gives each workgroup 16 rows
// and streams K/V through registers, which suits verify (q_len <= 16 / G) but caps a
// 512-token prefill chunk at ~200 TFLOP/s: every 16-row tile re-reads the whole context
// from L2 (16 flop per K/V byte).  Here four waves share each 64-key chunk of K and V,
// loaded once per workgroup straight into LDS (global_load_lds_dwordx4, double-buffered,
// 64 KiB: two workgroups per CU), so a chunk feeds 128 rows.
//
// Per wave (32 rows) and chunk:
//  * S^T = K . Q^T: 2 (keys) x D/16 (dims) MFMAs 32x32x16; K rows come from LDS as the A
//    operand (16-byte chunks XOR-swizzled by row: conflict-free), Q^T stays in registers.
//  * Lane l holds row l % 32 and, per 16-key step, keys 4*(l/32) + {0..3, 8..11} -- exactly
//    the B operand of O^T += V^T . P^T for a 16-key step whose K index is permuted the same
//    way, so P never leaves registers; V^T is read from LDS 2 bytes at a time in that
//    order (rows swizzled so the two lane groups hit different banks).
//  * Online softmax in base 2 per row; the row max needs one exchange between the lane
//    halves.
// Partials go to the multi-query kernel's workspace layout (16-row tiles), so its merge
// kernel combines the key partitions.
#include <float.h>

#include "dsp_common.h"
#include "dsp_internal.h"
#include "dsp_mfma.h"

namespace {

using namespace dsp_mfma;

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWaves = 4, kThreads = 64 * kWaves;
constexpr int kRows = 32 * kWaves;  // packed rows per workgroup
constexpr int kChunk = 64;          // keys per LDS chunk
constexpr int kMaxSharedSeqs = 1024;  // sequences of a shared-prefix launch (cu_q in LDS)

template <typename Tag>
__device__ __forceinline__ f32x16 mfma32x32(dsp_u32x4 a, dsp_u32x4 b, f32x16 c) {
  if constexpr (std::is_same<Tag, Bf16Tag>::value)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

typedef __attribute__((address_space(3))) void lds_void_t;

// One LDS DMA (global_load_lds_dwordx4): 16 bytes per lane from sbase + voff into LDS at
// m0 + 16 * lane.  It is issued from inline assembly so that the compiler does not make
// later LDS reads wait for it: its waitcnt pass cannot tell the DMA's target buffer from
// the one being read and would wait for the whole DMA.  The kernel waits for it itself
// (vmcnt) before the barrier that publishes the chunk.  M0 has no other user here.
// kNonTemporal marks the load nt: a shared-prefix launch reads most of its keys once (the
// prefix by one or a few packed tiles, each suffix by its sequence's tiles), so keeping them
// in the caches only evicts what other launches reuse (fork decode 23.5-23.8 -> 21.4 us
// per layer, verify unchanged).  An unshared prefill re-reads a sequence's keys from every
// 128-row tile of its queries and keeps the ordinary load (nt costs it 3-8 %).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool kNonTemporal>
__device__ __forceinline__ void dma16(const void* sbase, uint32_t voff, uint32_t m0) {
  if constexpr (kNonTemporal)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
                 :
                 : "v"(voff), "s"(sbase), "s"(m0)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(sbase), "s"(m0)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16_t;

// The V^T operand of 16-key step ps of a chunk in LDS: dim 32*dt + col, K index 8*hl + i <-> key
// 16*ps + 8*(i/4) + 4*hl + i%4 (the P^T order; col and hl as in attend_chunks).  In
// ds_read_b64_tr_b16, lane g + 4a + e of each 16-lane group g receives element e of the
// 4-element segments addressed by lanes g + a + 4j (j = 0..3); so lane s addresses key 16*ps +
// 8*inst + 4*hl + (s%16)/4, dims 32*dt + 16*((s/16)%2) + 4*(s%4) .. +3, for inst = 0, 1.
template <int D>
__device__ __forceinline__ dsp_u32x4 load_vt(const char* vs_lds, int ps, int dt) {
  const int lane = threadIdx.x & 63, hl = lane >> 5;
  v4i16 vh[2];
#pragma unroll
  for (int inst = 0; inst < 2; ++inst) {
    const int kr = 16 * ps + 8 * inst + 4 * hl + ((lane & 15) >> 2);
    const int dim0 = 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    const int swz = D >= 128 ? 4 * (kr & 3) : 4 * ((kr >> 1) & 1);
    vh[inst] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(
        vs_lds + kr * 2 * D + 16 * ((dim0 >> 3) ^ swz) + 2 * (dim0 & 7)));
  }
  return __builtin_bit_cast(dsp_u32x4, vh);
}

// One workgroup's keys [kbeg, kfin) of one (sequence, KV head), in 64-key chunks, for the rows
// whose Q^T operands are in qop: the running (max, sum, accumulator) of each row is updated.
// lim: the last key this lane's row sees; lim_min: the least of them in the wave, tile_lim in the
// workgroup (uniform).
// blk_first / blk_second: this wave's block ids of the first two chunks, loaded early and
// unclamped.  Every wave of the workgroup calls it (it has barriers).
template <typename Tag, int D, bool kNonTemporal, bool kMaskBad, int kTerms, typename Lds>
__device__ __forceinline__ void attend_chunks(
    Lds& lds, int32_t (&s_bad)[2][kWaves], int32_t (&s_odd)[2][kWaves],
    const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, int64_t num_slots, int64_t kvs_slot, int64_t head_off,
    const int32_t* __restrict__ bt, int64_t bt_row, int32_t log2_bs, int kbeg, int kfin, int lim,
    int lim_min, int tile_lim, bool wave_has_rows, const dsp_u32x4 (&qop)[D / 16], float scale_log2,
    int32_t blk_first, int32_t blk_second, float& m, float& lpart, f32x16 (&acc)[D / 32],
    bool& any_bad) {
  constexpr int NKS = D / 16;        // 16-dim steps of the score MFMA
  constexpr int NDT = D / 32;        // 32-dim output tiles
  constexpr int CPR = D / 8;         // 16-byte chunks per K/V row
  constexpr int ROWB = 2 * D;        // bytes per K/V row
  constexpr int SLAB = kChunk * ROWB;            // one K (or V) chunk
  constexpr int RPI = 1024 / ROWB;               // rows per 1-KiB DMA load
  constexpr int LPW = SLAB / 1024 / kWaves;      // DMA loads per wave per slab
  // kMaskBad: s_bad says which 16-key groups of each buffer's chunk have a block id outside the
  // cache (their keys are skipped, as on the 16-row tiles of 256-wide heads and on the generic
  // kernel: scores masked, V zeroed), no slot past kfin is read, and infinities and NaN of V reach
  // the rows that see their keys only: s_odd says which groups of a chunk that some row of the tile
  // does not see whole hold any.
  // kTerms: the 16-bit operands that hold a probability (pack8).  Three, i.e. fp32, at D 256 (as
  // on the generic kernel; one moves the error against 64 bits from 2.8e-3 to 3.3e-3), whose
  // 128 KiB of LDS leave one workgroup per CU, a wave's accumulators in AGPRs.
  static_assert(LPW >= 1, "every wave loads part of a chunk");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hl = lane >> 5;        // lane half: key sub-range of the operands
  const int col = lane & 31;       // this lane's row within the wave
  const int bmask = (1 << log2_bs) - 1;

  // K/V chunk rows into LDS: load j of this wave covers rows (wave*LPW + j)*RPI ..; lane l
  // fills slot l % CPR of row l / CPR with global chunk slot ^ swz(row).  K rows are
  // swizzled by (row & (CPR-1)) for the A-operand reads (32 rows, one 16-byte chunk each);
  // V rows by whole 64-byte groups (4 chunks): 4*(row & 3) at D 128 and 4*((row >> 1) & 1)
  // at D 64, so each half-wave of a transposing read (4 consecutive rows x 64 bytes) covers
  // all 64 banks once.
  auto kswz = [](int row) { return row & (CPR - 1); };
  auto vswz = [](int row) { return D >= 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1); };
  // Wave w loads rows 16*w .. 16*w + 15 of each chunk.  Chunks start at multiples of 64
  // keys and blocks hold a multiple of 16 tokens, so those rows lie in one block: its id
  // is wave-uniform and the addresses are a scalar base plus per-lane constants.  Rows past
  // kfin, masked, read other slots of the same block, with kMaskBad the last key's again; an
  // out-of-range block reads slots 0..15 (with kMaskBad its V is zeroed then).
  static_assert(LPW * RPI == 16, "16 rows per wave per chunk");
  uint32_t koff[LPW], voff[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int rw = j * RPI + lane / CPR, row = 16 * wave + rw, sl = lane % CPR;
    koff[j] = uint32_t(rw * kvs_slot * 2 + 16 * (sl ^ kswz(row)));
    voff[j] = uint32_t(rw * kvs_slot * 2 + 16 * (sl ^ vswz(row)));
  }
  const uint32_t lds_base = uint32_t(reinterpret_cast<uintptr_t>((lds_void_t*)&lds[0][0][0]));
  auto load_blk = [&](int t0) {
    return bt[bt_row + (min(t0 + 16 * wave, kfin - 1) >> log2_bs)];
  };
  bool bad_rows = false;  // kMaskBad: the rows this wave loaded last have a bad block id (uniform)
  auto issue = [&](int buf, int t0, int32_t blk_v) {
    const int32_t blk = __builtin_amdgcn_readfirstlane(blk_v);
    // kMaskBad: rows past kfin repeat the last key's (a stale row there may hold anything)
    const int first = kMaskBad ? min(t0 + 16 * wave, kfin - 1) : t0 + 16 * wave;
    int64_t slot0 = int64_t(blk) * (bmask + 1) + (first & bmask);
    if (blk < 0 || (int64_t(blk) + 1) * (bmask + 1) > num_slots) {
      slot0 = 0;
      any_bad |= t0 + 16 * wave < kfin;
      bad_rows = true;
    } else {
      bad_rows = false;
    }
    if constexpr (kMaskBad) s_bad[buf][wave] = bad_rows;
    const int64_t e = slot0 * kvs_slot + head_off;
    const char* kb = reinterpret_cast<const char*>(kc + e);
    const char* vb = reinterpret_cast<const char*>(vc + e);
    const uint32_t m0 = lds_base + uint32_t(buf * 2 * SLAB + wave * LPW * 1024);
    if constexpr (kMaskBad) {
      if (t0 + kChunk > kfin) {
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
          const int rw = j * RPI + lane / CPR, row = 16 * wave + rw, sl = lane % CPR;
          const uint32_t ro = uint32_t(min(rw, kfin - 1 - first) * kvs_slot * 2);
          dma16<kNonTemporal>(kb, ro + 16 * (sl ^ kswz(row)), m0 + j * 1024);
          dma16<kNonTemporal>(vb, ro + 16 * (sl ^ vswz(row)), m0 + SLAB + j * 1024);
        }
        return;
      }
    }
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
      dma16<kNonTemporal>(kb, koff[j], m0 + j * 1024);
      dma16<kNonTemporal>(vb, voff[j], m0 + SLAB + j * 1024);
    }
  };

  const int nch = (kfin - kbeg + kChunk - 1) / kChunk;
  // block ids run one chunk ahead of the DMAs, which run one chunk ahead of the MFMAs; the
  // first two were loaded at entry for the unclamped keys, which load_blk would clamp to
  // kfin - 1 only for a wave whose rows start past kfin (then reloaded, as load_blk does)
  if (kbeg + 16 * wave > kfin - 1) blk_first = load_blk(kbeg);
  issue(0, kbeg, blk_first);
  int32_t blk = blk_second;
  if (nch > 1 && kbeg + kChunk + 16 * wave > kfin - 1) blk = load_blk(kbeg + kChunk);
  for (int c = 0; c < nch; ++c) {
    const int t0 = kbeg + c * kChunk;
    // this wave's DMAs of chunk c (and the block ids of chunk c + 1) are in; after the
    // barrier every wave's are, and every wave is done reading chunk c - 1, whose buffer
    // the next DMA overwrites
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(dsp_waitcnt_vm<0>());
    char* const my_v = &lds[c & 1][1][wave * LPW * 1024];  // the V rows this wave loaded
    const bool edge = kMaskBad && t0 + kChunk - 1 > tile_lim;
    if (kMaskBad && bad_rows) zero_rows<CPR, LPW>(my_v, 0);
    if (edge) {
      __builtin_amdgcn_sched_barrier(0);
      s_odd[c & 1][wave] = any_nonfinite<Tag, LPW>(my_v);
    }
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    bool odd = false;  // rare: see below (uniform in the workgroup)
    if (edge)
      odd = __builtin_amdgcn_readfirstlane(s_odd[c & 1][0] | s_odd[c & 1][1] | s_odd[c & 1][2] |
                                           s_odd[c & 1][3]) != 0;
    auto clear_odd = [&] {
      __syncthreads();  // every wave has taken the chunk's infinities and NaN
      clear_nonfinite<Tag, LPW>(my_v);
      __syncthreads();
    };
    if (c + 1 < nch) {
      issue((c + 1) & 1, t0 + kChunk, blk);
      if (c + 2 < nch) blk = load_blk(t0 + 2 * kChunk);
    }
    // A wave whose 32 rows all lie past the tile's rows (a short query block: a verify
    // tile of 10 rows leaves three of four waves empty) only loads its share of each chunk.
    if (!wave_has_rows) {
      if (odd) clear_odd();
      continue;
    }
    const char* ks_lds = &lds[c & 1][0][0];
    const char* vs_lds = &lds[c & 1][1][0];

    // ---- scores S^T (keys x rows): two 32-key halves
    f32x16 sc[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
      for (int j = 0; j < 16; ++j) sc[mt][j] = 0.f;
      const int krow = 32 * mt + col;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const dsp_u32x4 kop = *reinterpret_cast<const dsp_u32x4*>(
            ks_lds + krow * ROWB + 16 * ((2 * ks + hl) ^ kswz(krow)));
        sc[mt] = mfma32x32<Tag>(kop, qop[ks], sc[mt]);
      }
    }
    // ---- mask (only chunks that reach past a row's causal limit or past kfin), row max.
    // sc[mt][j] is key 32*mt + 8*(j/4) + 4*hl + j%4 of this lane's row.
    if (t0 + kChunk - 1 > lim_min) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int key = t0 + 32 * mt + 8 * (j >> 2) + 4 * hl + (j & 3);
          sc[mt][j] = key <= lim ? sc[mt][j] : -INFINITY;
        }
    }
    if constexpr (kMaskBad) {
      // sc[mt][j] lies in the chunk's 16-key group 2*mt + j/8, the rows one wave loaded
      const int32_t* bad = s_bad[c & 1];
#pragma unroll
      for (int g16 = 0; g16 < 4; ++g16)
        if (__builtin_amdgcn_readfirstlane(bad[g16])) {
#pragma unroll
          for (int j = 0; j < 8; ++j) sc[g16 >> 1][8 * (g16 & 1) + j] = -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int j = 0; j < 16; ++j) mx = fmaxf(mx, sc[mt][j]);
    mx = fmaxf(mx, dsp_shfl_xor(mx, 32)) * scale_log2;  // base-2 units; -inf stays -inf
    // Lazy rescale: the running max m only moves when some row's chunk max exceeds it by
    // more than 8 (so p <= 2^8); the result is exact either way, since l and acc share m.
    // (Where pack8 takes p <= 1 at most, m is the exact maximum.)
    constexpr float kLag = p_scale<Tag, kTerms>() > 128.f ? 0.f : 8.f;
    if (__builtin_amdgcn_ballot_w64(mx > m + kLag) != 0) {
      const float m_new = fmaxf(m, mx);
      const float alpha = m_new == -INFINITY ? 1.f : dsp_exp2(m - m_new);
      m = m_new;
      lpart *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) acc[dt] *= alpha;
    }
    const float neg_m = m == -INFINITY ? 0.f : -m;
    // P^T operands of the four 16-key steps: step ps = 2*mt + half takes registers
    // j = 8*half .. 8*half + 7, i.e. keys 16*ps + 4*hl + {0..3, 8..11}.
    // Three terms are formed step by step in the loop below: all four steps' would take 48
    // registers, the probabilities themselves 32.
    dsp_u32x4 pop[4][kTerms];
    float p8[4][8];
#pragma unroll
    for (int ps = 0; ps < 4; ++ps) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p8[ps][i] = dsp_exp2(fmaf(sc[ps >> 1][8 * (ps & 1) + i], scale_log2, neg_m)) *
                    p_scale<Tag, kTerms>();
        lpart += p8[ps][i];
      }
      if constexpr (kTerms < 3) pack8<Tag, kTerms>(p8[ps], pop[ps]);
    }

    // (rare) infinities and NaN of V to the rows that see them
    if (kMaskBad && odd) {
#pragma unroll 1
      for (int ps = 0; ps < 4; ++ps) {
        dsp_u32x4 seen;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = t0 + 16 * ps + 8 * (i >> 1) + 4 * hl + 2 * (i & 1);
          seen[i] = (key <= lim ? kHuge : 0u) | (key < lim ? kHuge << 16 : 0u);
        }
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          __builtin_amdgcn_sched_barrier(0);  // one tile's operands at a time: registers
          const dsp_u32x4 v = load_vt<D>(vs_lds, ps, dt);
          acc[dt] = mfma32x32<Bf16Tag>(odd_operand<Tag>(v, false), seen, acc[dt]);
          acc[dt] = mfma32x32<Bf16Tag>(odd_operand<Tag>(v, true), seen, acc[dt]);
        }
      }
      clear_odd();
    }
    // ---- O^T += V^T . P^T
#pragma unroll
    for (int ps = 0; ps < 4; ++ps) {
      if constexpr (kTerms == 3) pack8<Tag, kTerms>(p8[ps], pop[ps]);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        if constexpr (D > 128) {
          const dsp_u32x4 vop = load_vt<D>(vs_lds, ps, dt);
#pragma unroll
          for (int k = 0; k < kTerms; ++k) acc[dt] = mfma32x32<Tag>(vop, pop[ps][k], acc[dt]);
        } else {
          // load_vt written out: as a call the compiler keeps fewer addresses in registers, which
          // costs D 128 5 % (4 x 512 tokens over 4096: 154 -> 161 us) and saves D 256 6 %
          v4i16 vh[2];
#pragma unroll
          for (int inst = 0; inst < 2; ++inst) {
            const int kr = 16 * ps + 8 * inst + 4 * hl + ((lane & 15) >> 2);
            const int dim0 = 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
            vh[inst] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(
                vs_lds + kr * ROWB + 16 * ((dim0 >> 3) ^ vswz(kr)) + 2 * (dim0 & 7)));
          }
#pragma unroll
          for (int k = 0; k < kTerms; ++k)
            acc[dt] = mfma32x32<Tag>(__builtin_bit_cast(dsp_u32x4, vh), pop[ps][k], acc[dt]);
        }
      }
    }
  }
}

// kShared: a shared-prefix (cascade) launch, two kinds of workgroup in one grid.  For
// x < prefix_x (per KV head) a workgroup is a prefix tile: packed row r is token r / G of
// the whole batch (every sequence's queries), query head kvh*G + r % G; the keys are the
// first prefix_tokens of block-table row 0, which every sequence shares and every query
// sees whole (no mask); partition `part` covers keys [part*P, part*P + P) and is written,
// for every row, to that row's own (sequence, 16-row tile) slot of the merge layout.  The
// other workgroups are suffix tiles: one sequence's rows over one partition of P of its
// keys from prefix_tokens on (causal), numbered on from the prefix's partitions (keys
// [part*P, part*P + P) again).  Both kinds run side by side; the merge then folds every
// partition up to a row's last visible key, as for an unshared launch.
template <typename Tag, int D, bool kShared>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(D > 128 ? 1 : 2))) void paged_prefill_kernel(
    const uint16_t* __restrict__ q, int64_t qst, int64_t qsh, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, int64_t num_slots, int64_t kvs_slot, int64_t kvs_head,
    const int32_t* __restrict__ bt, int64_t bt_stride, int32_t log2_bs,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ ctx_lens, int32_t max_ctx,
    int32_t G, float scale_log2, int32_t P, int32_t num_parts, int32_t tiles16_max,
    float* __restrict__ ws_acc, float* __restrict__ ws_ml, uint16_t* __restrict__ out,
    int64_t ost, int64_t osh, int32_t* __restrict__ err_count, int32_t nseq,
    int32_t prefix_tokens, int32_t ws_parts, int32_t prefix_x) {
  constexpr int NKS = D / 16;        // 16-dim steps of the score MFMA
  constexpr int NDT = D / 32;        // 32-dim output tiles
  constexpr int SLAB = kChunk * 2 * D;  // one K (or V) chunk
  __shared__ __attribute__((aligned(1024))) char lds[2][2][SLAB];  // [buffer][K | V]
  __shared__ int32_t s_cu[kShared ? kMaxSharedSeqs + 1 : 1];         // cu_q, prefix pass
  __shared__ int32_t s_bad[2][kWaves], s_odd[2][kWaves];

  // XCD-aware order: the dispatcher hands workgroup `lin` to XCD lin % 8.  Each XCD gets a
  // contiguous range of logical ids, so the tiles of one (sequence, KV head) -- which read
  // the same K/V -- run on one XCD and share its L2.  Within a (sequence, KV head) the
  // heaviest tiles (the last rows see the most keys) come first.
  const int X = gridDim.x, KVH = gridDim.y;
  const int64_t nwg = int64_t(X) * KVH * gridDim.z;
  const int64_t lin = blockIdx.x + int64_t(X) * (blockIdx.y + int64_t(KVH) * blockIdx.z);
  const int64_t q8 = nwg / 8, r8 = nwg % 8, xcd = lin % 8, pos = lin / 8;
  const int64_t lg = xcd < r8 ? xcd * (q8 + 1) + pos : r8 * (q8 + 1) + (xcd - r8) * q8 + pos;
  const int xl = int(lg % X);
  const int kvh = int((lg / X) % KVH);
  int b = int(lg / X / KVH), part, tile;
  bool pre = false;  // a prefix tile of a shared-prefix launch
  if constexpr (kShared) {
    pre = xl < prefix_x;
    if (pre) {
      part = xl % num_parts;
      tile = prefix_x / num_parts - 1 - xl / num_parts;
    } else {
      // suffix tiles: per sequence tiles_s row tiles x nsp partitions of its keys past the
      // prefix (partition index continues the prefix's: key range [part*P, part*P + P))
      const int first = prefix_tokens / P, nsp = ws_parts - first;
      const int per_seq = (X - prefix_x) / nseq, idx = xl - prefix_x;
      const int tiles_s = per_seq / nsp, k = idx % per_seq;
      b = idx / per_seq;
      tile = tiles_s - 1 - k / nsp;
      part = first + k % nsp;
    }
  } else {
    const int ntiles = X / num_parts;
    part = xl % num_parts;
    tile = ntiles - 1 - xl / num_parts;
  }
  // The first two chunks' block ids are loaded now, beside the lengths below: chunk keys
  // start at part * P whatever the lengths are (clamped into the table's width here; a
  // wave whose rows turn out to start past the partition's end reloads its id below).
  const int wave_e = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t bt_row_e = int64_t(b) * bt_stride;
  const int key_cap = max(max_ctx - 1, 0);
  auto early_blk = [&](int t) {
    return bt[bt_row_e + (min(t + 16 * wave_e, key_cap) >> log2_bs)];
  };
  int32_t blk_first = early_blk(part * P), blk_second = early_blk(part * P + kChunk);
  int q0, qlen, ctx, kend = 0;
  if (pre) {
    // all tokens of the batch; the causal limit never binds (ctx - qlen + qi >= max_ctx)
    q0 = 0;
    qlen = cu_q[nseq];
    ctx = qlen + max_ctx;
    kend = prefix_tokens;
    // staged for the epilogue's row -> sequence search (published by the first chunk's
    // barrier: every workgroup that gets past the checks below runs at least one chunk)
    for (int i = threadIdx.x; i <= nseq; i += kThreads) s_cu[i] = cu_q[i];
  } else {
    q0 = cu_q[b];
    qlen = cu_q[b + 1] - q0;
    ctx = ctx_lens[b];
  }
  const int rows = qlen * G;
  const int r0 = tile * kRows;
  if (qlen <= 0 || r0 >= rows) return;
  if (!pre) {
    // bad lengths (and, in a shared-prefix launch, queries that start inside the prefix):
    // counted once, the rows are zeros
    if (ctx > max_ctx || ctx < qlen || (kShared && ctx - qlen < prefix_tokens)) {
      if (!kShared && part != 0) return;
      if (threadIdx.x == 0 && tile == 0 && kvh == 0 && err_count) atomicAdd(err_count, 1);
      for (int i = threadIdx.x; i < kRows * D; i += kThreads) {
        const int rr = r0 + i / D;
        if (rr < rows)
          out[int64_t(q0 + rr / G) * ost + int64_t(kvh * G + rr % G) * osh + i % D] = 0;
      }
      return;
    }
    const int r_last = min(r0 + kRows - 1, rows - 1);
    kend = ctx - qlen + r_last / G + 1;  // keys any row of the tile sees
  }
  // partition `part` covers keys [part*P, part*P + P) of the tile's visible range (a
  // suffix tile's partitions start at the prefix's end, which is a multiple of P)
  const int kbeg = part * P;
  if (kbeg >= kend) return;
  const int kfin = min(kbeg + P, kend);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hl = lane >> 5;        // lane half: key sub-range of the operands
  const int col = lane & 31;       // this lane's row within the wave
  const int r = r0 + 32 * wave + col;
  const bool row_ok = r < rows;
  const bool wave_has_rows = r0 + 32 * wave < rows;  // wave-uniform
  const int qi = row_ok ? r / G : 0;
  const int h = kvh * G + (row_ok ? r % G : 0);
  // Keys 0..lim are visible to this row (causal limit, and the partition's end); lim_min
  // is the smallest limit among the wave's rows (its first row), wave-uniform.  Rows past
  // `rows` have q = 0: finite scores, never stored.
  const int lim = min(ctx - qlen + qi, kfin - 1);
  const int lim_min = min(ctx - qlen + (r0 + 32 * wave) / G, kfin - 1);
  const int tile_lim = min(ctx - qlen + r0 / G, kfin - 1);
  const int64_t bt_row = int64_t(b) * bt_stride;
  const int64_t head_off = int64_t(kvh) * kvs_head;

  // Q^T (B operand): lane holds dims 16*ks + 8*hl .. +8 of its row.
  dsp_u32x4 qop[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    qop[ks] = row_ok ? *reinterpret_cast<const dsp_u32x4*>(q + int64_t(q0 + qi) * qst +
                                                           int64_t(h) * qsh + 16 * ks + 8 * hl)
                     : dsp_u32x4{0u, 0u, 0u, 0u};

  bool any_bad = false;  // (wave-uniform) a block id of visible keys lay outside the cache
  float m = -INFINITY, lpart = 0.f;
  f32x16 acc[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;
  attend_chunks<Tag, D, kShared, (D > 128), (D > 128 ? 3 : 1)>(lds, s_bad, s_odd, kc, vc, num_slots, kvs_slot, head_off, bt, bt_row,
                                 log2_bs, kbeg, kfin, lim, lim_min, tile_lim, wave_has_rows, qop, scale_log2,
                                 blk_first, blk_second, m, lpart, acc, any_bad);

  if (err_count && any_bad && lane == 0) atomicAdd(err_count, 1);  // once per wave

  // ---- epilogue: row sums over the two lane halves; acc[dt][j] = O[row col][dim 32*dt +
  // 8*(j/4) + 4*hl + j%4]
  lpart += dsp_shfl_xor(lpart, 32);
  if (!row_ok) return;
  int sb = b, lr = r;  // the row's sequence and its packed row there
  if (pre) {
    int lo = 0, hi = nseq - 1;  // last sequence whose first token is <= qi
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_cu[mid] <= qi) lo = mid; else hi = mid - 1;
    }
    sb = lo;
    lr = (qi - s_cu[lo]) * G + (r % G);
  }
  const int st = lr / 16, rr = lr % 16;                  // 16-row tile of the merge layout
  if (st >= tiles16_max) return;  // q_len past the caller's max_q_len: rows not covered
  if constexpr (!kShared) {
    const int r_last16 = min(st * 16 + 15, rows - 1);
    const int kend16 = ctx - qlen + r_last16 / G + 1;
    const int nparts16 = (kend16 + P - 1) / P;
    if (part >= nparts16) return;  // the merge for this 16-row tile does not read it
    if (nparts16 == 1) {
      const float inv = lpart > 0.f ? 1.f / lpart : 0.f;
      uint16_t* o = out + int64_t(q0 + qi) * ost + int64_t(h) * osh;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j)
          o[32 * dt + 8 * (j >> 2) + 4 * hl + (j & 3)] = narrow<Tag>(acc[dt][j] * inv);
      return;
    }
  }
  const int64_t slot = ((int64_t(sb) * KVH + kvh) * tiles16_max + st) * ws_parts + part;
  float* a = ws_acc + (slot * 16 + rr) * D;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int j4 = 0; j4 < 4; ++j4)
      *reinterpret_cast<f32x4*>(a + 32 * dt + 8 * j4 + 4 * hl) =
          f32x4{acc[dt][4 * j4], acc[dt][4 * j4 + 1], acc[dt][4 * j4 + 2], acc[dt][4 * j4 + 3]};
  if (hl == 0) {
    ws_ml[2 * (slot * 16 + rr)] = m;
    ws_ml[2 * (slot * 16 + rr) + 1] = lpart;
  }
}

// ---- equal shares of a ragged batch ------------------------------------------------------
// A batch that mixes prompt chunks with decodes has few 128-row tiles for the size of its grid
// (which the longest query block sizes for every sequence), and their keys differ widely: one
// chunk's tiles and 24 one-row tiles, each walking its context alone, leave most of the chip
// idle behind the longest.  Here the work is the list of (sequence, KV head, tile, 64-key
// chunk) units, in that order, and each of W workgroups -- as many as fit the chip at once --
// takes an equal run of it, computed on the device from the lengths (as decode_balanced.hip
// does, so nothing waits for the host).  A tile inside one run is normalised and written; a
// tile that crosses runs leaves a partial (128 rows' max, sum and accumulator) per run in the
// workspace: slot 2w for worker w's first piece when it continues a tile, 2w + 1 for its last
// when it begins one; the merge kernel's workgroup w folds the tile that worker w began.
// Verifies of 17 to 127 rows, whose 16-row tiles would each read the keys: 32 of 5 over 500-4000
// keys 93 -> 48 us (28 heads over 4).
// 24 decodes of 100-2860 keys beside a 700-token chunk over 1501 keys: 117 -> 58 us a layer with
// the merge (28 heads over 4 of 128), 46 -> 31 (14 over 2 of 64), 150 -> 71 (32 over 8).  The
// merge is 8-13 us of it: a partial is 64 KiB a tile at D 128.
constexpr int kMinChunks = 2;       // a worker gets at least this many chunks
// Run ends this many chunks from a tile's end or less move onto it: 2 decodes and a 1000-token
// prompt 45 -> 41 us at 2, 42 at 4, where batches of short contexts lose (4 decodes and 64
// tokens 17 -> 19 at 2, 23 at 4).
constexpr int kSnap = 2;
constexpr int kMaxRaggedSeqs = 512; // every wave scans the lengths

// Division by the launch's G (values below 2^24): a reciprocal and one correction step, a few
// instructions where the compiler's division is tens; every worker runs a chain of them before
// its first load.
struct DivG {
  int G;
  float inv;
  __device__ __forceinline__ explicit DivG(int g) : G(g), inv(1.f / float(g)) {}
  __device__ __forceinline__ int div(int x) const {
    int q = int(float(x) * inv);
    const int r = x - q * G;
    return r < 0 ? q - 1 : (r >= G ? q + 1 : q);
  }
  // sum of floor(k / G) over 0 <= k < x
  __device__ __forceinline__ int floors(int x) const {
    const int q = div(x);
    return G * (q * (q - 1) / 2) + q * (x - q * G);
  }
  // sum of floor((a + 2 t) / G) over 0 <= t < n.  The sum over every k in [a, a + 2n) is this
  // one plus the sum over the odd steps, floor((a + 2 t + 1) / G), which exceeds this one by 1
  // where G divides a + 2 t + 1: for odd G every G-th t from t0 on; for even G every G/2-th t
  // where a is odd, none where it is even.
  __device__ __forceinline__ int every_other(int a, int n) const {
    const int all = floors(a + 2 * n) - floors(a);
    const int r = a + 1 - div(a + 1) * G;      // (a + 1) mod G
    const int miss = r == 0 ? 0 : G - r;       // 2 t0 = miss (mod G)
    int hits = 0;
    if (G & 1) {
      const int t0 = (miss & 1) ? (miss + G) / 2 : miss / 2;   // below G
      hits = t0 < n ? div(n - 1 - t0) + 1 : 0;
    } else if (!(miss & 1)) {
      const int t0 = miss / 2;
      hits = t0 < n ? div(2 * (n - 1 - t0)) + 1 : 0;
    }
    return (all - hits) / 2;
  }
};

// One sequence's tiles: `tiles` of 128 packed rows (the first max_q_len queries); tile t but
// the last sees ceil((c0 + (128 t + 127) / G + 1) / 64) = floor((a + 2 t) / G) chunks.
struct RaggedSeq {
  int q0, qlen, ctx, rows, tiles, a, last, units;
  __device__ __forceinline__ int before(int t, const DivG& g) const {
    return t > 0 ? g.every_other(a, t) : 0;
  }
  __device__ __forceinline__ int chunks(int t, const DivG& g) const {
    return t + 1 < tiles ? g.div(a + 2 * t) : last;
  }
};
__device__ __forceinline__ bool ragged_bad(int qlen, int ctx, int max_ctx) {
  return qlen > 0 && (ctx < qlen || ctx > max_ctx);
}
__device__ __forceinline__ RaggedSeq ragged_seq(int q0, int q1, int ctx, const DivG& g,
                                                int max_q_len, int max_ctx) {
  RaggedSeq s;
  s.q0 = q0;
  s.qlen = q1 - q0;
  s.ctx = ctx;
  const bool none = s.qlen <= 0 || ragged_bad(s.qlen, s.ctx, max_ctx);
  s.rows = none ? 0 : min(s.qlen, max_q_len) * g.G;
  s.tiles = (s.rows + kRows - 1) / kRows;
  const int c0 = none ? 0 : s.ctx - s.qlen;
  s.a = (g.G * (c0 + kChunk) + kRows - 1) / kChunk;
  s.last = none ? 0 : (c0 + min(s.qlen, max_q_len) - 1 + kChunk) / kChunk;
  s.units = none ? 0 : s.before(s.tiles - 1, g) + s.last;
  return s;
}
__device__ __forceinline__ RaggedSeq lane_seq(const RaggedSeq& s, int l) {
  RaggedSeq r;
  r.q0 = __builtin_amdgcn_readlane(s.q0, l);
  r.qlen = __builtin_amdgcn_readlane(s.qlen, l);
  r.ctx = __builtin_amdgcn_readlane(s.ctx, l);
  r.rows = __builtin_amdgcn_readlane(s.rows, l);
  r.tiles = __builtin_amdgcn_readlane(s.tiles, l);
  r.a = __builtin_amdgcn_readlane(s.a, l);
  r.last = __builtin_amdgcn_readlane(s.last, l);
  r.units = __builtin_amdgcn_readlane(s.units, l);
  return r;
}
__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = __lane_id();
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d);
    if (lane >= d) v += o;
  }
  return v;
}

// kTerms: the operands of a probability (attend_chunks).  Two for blocks below 128 rows
// (verify), which the 16-row tiles would serve: their running maximum is exact, here it lags by
// up to 2^8, and one 16-bit probability would err 4 % more (3.1e-3 -> 3.2e-3 against 64 bits, 32
// verifies of 28 heads over 4).
template <typename Tag, int D, int kTerms>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(D > 128 ? 1 : D > 64 ? 2 : 3))) void prefill_ragged_kernel(
    const uint16_t* __restrict__ q, int64_t qst, int64_t qsh, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, int64_t num_slots, int64_t kvs_slot, int64_t kvs_head,
    const int32_t* __restrict__ bt, int64_t bt_stride, int32_t log2_bs,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ ctx_lens, int32_t B, int32_t KVH,
    int32_t G, int32_t max_q_len, int32_t max_ctx, float scale_log2, float* __restrict__ ws_acc,
    float* __restrict__ ws_ml, int32_t* __restrict__ ws_desc, uint16_t* __restrict__ out,
    int64_t ost, int64_t osh, int32_t* __restrict__ err_count) {
  constexpr int NKS = D / 16, NDT = D / 32, SLAB = kChunk * 2 * D;
  __shared__ __attribute__((aligned(1024))) char lds[2][2][SLAB];
  __shared__ int32_t s_bad[2][kWaves], s_odd[2][kWaves];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const int lin = blockIdx.x;

  // Lane l holds sequence b0 + l of the 64 the wave looks at; most batches are one such group,
  // whose lanes' values serve the whole kernel.
  const DivG g(G);
  int b0 = 0;
  RaggedSeq lane_s;
  int incl = 0;
  auto look = [&](int first) {
    b0 = first;
    const int b = min(b0 + lane, B - 1);
    lane_s = ragged_seq(cu_q[b], cu_q[b + 1], ctx_lens[b], g, max_q_len, max_ctx);
    if (b0 + lane >= B) lane_s.units = 0;
    incl = wave_incl_scan(lane_s.units);
  };
  int total = 0;  // units per KV head
  for (int first = 0; first < B; first += 64) {
    look(first);
    total += __builtin_amdgcn_readlane(incl, 63);
    // bad lengths: counted once, the rows written as zeros, one sequence per workgroup
    for (int b = lin; b < B; b += gridDim.x) {
      if (b < first || b >= first + 64) continue;
      const int l = b - first, qa = __builtin_amdgcn_readlane(lane_s.q0, l);
      const int ql = __builtin_amdgcn_readlane(lane_s.qlen, l);
      if (!ragged_bad(ql, __builtin_amdgcn_readlane(lane_s.ctx, l), max_ctx)) continue;
      if (threadIdx.x == 0 && err_count) atomicAdd(err_count, 1);
      const int row = KVH * G * D, n = min(ql, max_q_len);
      for (int i = 0; i < n; ++i)
        for (int e = threadIdx.x; e < row; e += kThreads)
          out[int64_t(qa + i) * ost + int64_t(e / D) * osh + e % D] = 0;
    }
  }
  const int C = total * KVH;
  const int W = min((C + kMinChunks - 1) / kMinChunks, int(gridDim.x));
  if (lin >= W) {
    if (threadIdx.x == 0) ws_desc[4 * lin + 3] = 0;
    return;
  }
  // XCD-aware: workgroup lin runs on XCD lin % 8; each XCD takes a contiguous run of workers,
  // so that the tiles of one (sequence, KV head) share an L2
  const int q8 = W / 8, r8 = W % 8, xcd = lin % 8, pos = lin / 8;
  const int w = xcd < r8 ? xcd * (q8 + 1) + pos : r8 * (q8 + 1) + (xcd - r8) * q8 + pos;
  // worker w's run starts at unit floor(w * C / W) (C = share * W + extra)
  const int share = C / W, extra = C - share * W;
  const int U = w * share + w * extra / W;
  int left = (w + 1) * share + (w + 1) * extra / W - U;
  int b = 0, base = 0;  // base: units (of all KV heads) before sequence b
  for (int first = 0, pre = 0; first < B; first += 64) {
    if (first != b0 || B > 64) look(first);
    const uint64_t hit = __ballot(KVH * (pre + incl) > U);
    if (hit) {
      const int f = __builtin_amdgcn_readfirstlane(__ffsll(static_cast<unsigned long long>(hit)) - 1);
      b = first + f;
      base = KVH * (pre + __builtin_amdgcn_readlane(incl, f) -
                    __builtin_amdgcn_readlane(lane_s.units, f));
      break;
    }
    pre += __builtin_amdgcn_readlane(incl, 63);
  }
  RaggedSeq sq = lane_seq(lane_s, b - b0);
  int kvh = 0, u = U - base;
  for (; u >= sq.units; u -= sq.units) ++kvh;
  // the tile of unit u: 64 candidates a step
  int tile = 0;
  for (int step = (sq.tiles + 63) / 64;; step = 1) {
    const int t = tile + lane * step;
    const bool at = t < sq.tiles && sq.before(t, g) <= u;
    tile += (__popcll(__ballot(at)) - 1) * step;
    if (step == 1) break;
  }
  tile = __builtin_amdgcn_readfirstlane(tile);
  // Run ends within kSnap chunks of a tile's either end move onto it: a piece of one or two
  // chunks costs its start-up and a partial of the whole tile.  (Both neighbours move their
  // common end alike: first the beginning, then the end of the tile.)
  int c0 = u - sq.before(tile, g);
  // the next tile, KV head or sequence with units (false: none is left)
  auto next_tile = [&]() {
    c0 = 0;
    if (++tile < sq.tiles) return true;
    tile = 0;
    if (++kvh < KVH) return true;
    kvh = 0;
    base += KVH * sq.units;
    while (++b < B) {
      sq = ragged_seq(cu_q[b], cu_q[b + 1], ctx_lens[b], g, max_q_len, max_ctx);
      if (sq.units > 0) return true;
    }
    return false;
  };
  bool work = true;
  if (c0 <= kSnap) {
    left += c0;
    c0 = 0;
  } else if (sq.chunks(tile, g) - c0 <= kSnap) {
    left -= sq.chunks(tile, g) - c0;
    work = left > 0 && next_tile();
  }
  int32_t d_b = 0, d_kvh = 0, d_tile = 0, d_np = 0;
  bool any_bad = false;
  for (bool again = false; work; again = true) {
    const int nch = sq.chunks(tile, g);
    int c1 = min(nch, c0 + left);
    if (c1 < nch) {
      if (c1 <= kSnap) break;  // the next worker's
      if (nch - c1 <= kSnap) c1 = nch;
    }
    const int r0 = tile * kRows, rows = sq.rows;
    const int r_last = min(r0 + kRows - 1, rows - 1);
    const int kend = sq.ctx - sq.qlen + r_last / G + 1;
    const int kbeg = c0 * kChunk, kfin = min(c1 * kChunk, kend);
    const int64_t bt_row = int64_t(b) * bt_stride;
    const int32_t blk0 = bt[bt_row + (min(kbeg + 16 * wave, kfin - 1) >> log2_bs)];
    const int32_t blk1 = bt[bt_row + (min(kbeg + kChunk + 16 * wave, kfin - 1) >> log2_bs)];
    const int r = r0 + 32 * wave + col;
    const bool row_ok = r < rows;
    const bool wave_has_rows = r0 + 32 * wave < rows;
    const int qi = row_ok ? r / G : 0;
    const int h = kvh * G + (row_ok ? r % G : 0);
    const int lim = min(sq.ctx - sq.qlen + qi, kfin - 1);
    const int lim_min = min(sq.ctx - sq.qlen + (r0 + 32 * wave) / G, kfin - 1);
    const int tile_lim = min(sq.ctx - sq.qlen + r0 / G, kfin - 1);
    dsp_u32x4 qop[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
      qop[ks] = row_ok ? *reinterpret_cast<const dsp_u32x4*>(q + int64_t(sq.q0 + qi) * qst +
                                                             int64_t(h) * qsh + 16 * ks + 8 * hl)
                       : dsp_u32x4{0u, 0u, 0u, 0u};
    float m = -INFINITY, lpart = 0.f;
    f32x16 acc[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;
    if (again) __syncthreads();  // every wave is done with the previous piece's buffers
    attend_chunks<Tag, D, false, true, kTerms>(lds, s_bad, s_odd, kc, vc, num_slots, kvs_slot,
                                 int64_t(kvh) * kvs_head, bt, bt_row, log2_bs, kbeg, kfin, lim,
                                 lim_min, tile_lim, wave_has_rows, qop, scale_log2, blk0, blk1, m, lpart, acc,
                                 any_bad);
    lpart += dsp_shfl_xor(lpart, 32);
    if (c0 == 0 && c1 == nch) {
      const float inv = lpart > 0.f ? 1.f / lpart : 0.f;
      if (row_ok) {
        uint16_t* o = out + int64_t(sq.q0 + qi) * ost + int64_t(h) * osh;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int j = 0; j < 16; ++j)
            o[32 * dt + 8 * (j >> 2) + 4 * hl + (j & 3)] = narrow<Tag>(acc[dt][j] * inv);
      }
    } else {
      const int64_t wrow = int64_t(2 * w + (c0 == 0 ? 1 : 0)) * kRows + 32 * wave + col;
      if (row_ok) {
        float* dst = ws_acc + wrow * D;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int j4 = 0; j4 < 4; ++j4)
            *reinterpret_cast<f32x4*>(dst + 32 * dt + 8 * j4 + 4 * hl) =
                f32x4{acc[dt][4 * j4], acc[dt][4 * j4 + 1], acc[dt][4 * j4 + 2],
                      acc[dt][4 * j4 + 3]};
        if (hl == 0) {
          ws_ml[2 * wrow] = m;
          ws_ml[2 * wrow + 1] = lpart;
        }
      }
      if (c0 == 0) {  // this worker began the tile: its merge is described here
        const int end = base + kvh * sq.units + sq.before(tile, g) + nch;
        d_b = b;
        d_kvh = kvh;
        d_tile = tile;
        // the last worker whose run begins before the tile's end (less the chunks it would skip)
        d_np = int32_t((int64_t(end - kSnap) * W - 1) / C) - w + 1;
      }
    }
    left -= c1 - c0;
    work = left > 0 && next_tile();
  }
  if (err_count && any_bad && lane == 0) atomicAdd(err_count, 1);  // once per wave
  if (threadIdx.x == 0) {
    int32_t* d = ws_desc + 4 * w;
    d[0] = d_b;
    d[1] = d_kvh;
    d[2] = d_tile;
    d[3] = d_np;
  }
}

// Grid (workers, 128 / R): R rows of the tile that worker x began and did not finish, one
// thread per (row, 4 dims); its pieces are loaded 16 at a time before they are folded.
constexpr int ragged_merge_rows(int D) { return 1024 / D; }

template <typename Tag, int D>
__global__ __launch_bounds__(256) void prefill_ragged_merge_kernel(
    const float* __restrict__ ws_acc, const float* __restrict__ ws_ml,
    const int32_t* __restrict__ ws_desc, const int32_t* __restrict__ cu_q, int32_t G,
    int32_t max_q_len, uint16_t* __restrict__ out, int64_t ost, int64_t osh) {
  constexpr int TPR = D / 4, R = ragged_merge_rows(D), kBatch = 16;
  const int64_t w = blockIdx.x;
  const int32_t* desc = ws_desc + 4 * w;
  const int b = desc[0], kvh = desc[1], tile = desc[2], np = desc[3];
  if (np <= 0) return;
  const int q0 = cu_q[b], rows = min(cu_q[b + 1] - q0, max_q_len) * G;
  const int lr = blockIdx.y * R + threadIdx.x / TPR, d = 4 * (threadIdx.x % TPR);
  const int r = tile * kRows + lr;
  if (r >= rows) return;
  float M = -INFINITY, L = 0.f;
  f32x4 A = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < np; p0 += kBatch) {
    const int n = min(np - p0, kBatch);
    f32x4 va[kBatch];
    float vm[kBatch], vl[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i)
      if (i < n) {
        const int p = p0 + i;
        const int64_t row = (p == 0 ? 2 * w + 1 : 2 * (w + p)) * kRows + lr;
        va[i] = *reinterpret_cast<const f32x4*>(ws_acc + row * D + d);
        vm[i] = ws_ml[2 * row];
        vl[i] = ws_ml[2 * row + 1];
      }
    float bm = M;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) bm = i < n ? fmaxf(bm, vm[i]) : bm;
    const float Mu = bm == -INFINITY ? 0.f : bm;
    const float keep = dsp_exp2(M - Mu);
    L *= keep;
    A *= keep;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const float x = i < n ? dsp_exp2(vm[i] - Mu) : 0.f;
      L = fmaf(i < n ? vl[i] : 0.f, x, L);
#pragma unroll
      for (int e = 0; e < 4; ++e) A[e] = fmaf(i < n ? va[i][e] : 0.f, x, A[e]);
    }
    M = bm;
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  uint16_t* o = out + int64_t(q0 + r / G) * ost + int64_t(kvh * G + r % G) * osh + d;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = narrow<Tag>(A[e] * inv);
}

template <typename Tag, int D>
int launch_ragged(int W, hipStream_t s, const uint16_t* q, int64_t qst, int64_t qsh,
                  const uint16_t* kc, const uint16_t* vc, int64_t num_slots, int64_t kvs_slot,
                  int64_t kvs_head, const int32_t* bt, int64_t bt_stride, int32_t log2_bs,
                  const int32_t* cu_q, const int32_t* ctx_lens, int32_t B, int32_t KVH, int32_t G,
                  int32_t max_q_len, int32_t max_ctx, float scale_log2, float* ws, uint16_t* out,
                  int64_t ost, int64_t osh, int32_t* err_count) {
  float* ws_ml = ws + int64_t(2) * W * kRows * D;
  int32_t* ws_desc = reinterpret_cast<int32_t*>(ws_ml + int64_t(4) * W * kRows);
  auto launch = [&](auto kernel) {
    kernel<<<W, kThreads, 0, s>>>(q, qst, qsh, kc, vc, num_slots, kvs_slot, kvs_head, bt, bt_stride,
                                  log2_bs, cu_q, ctx_lens, B, KVH, G, max_q_len, max_ctx, scale_log2,
                                  ws, ws_ml, ws_desc, out, ost, osh, err_count);
  };
  if (D > 128 || int64_t(max_q_len) * G < kRows)
    launch(prefill_ragged_kernel<Tag, D, (D > 128 ? 3 : 2)>);
  else
    launch(prefill_ragged_kernel<Tag, D, (D > 128 ? 3 : 1)>);
  const int st = dsp_launch_status();
  if (st != DSP_OK) return st;
  prefill_ragged_merge_kernel<Tag, D><<<dim3(W, kRows / ragged_merge_rows(D)), 256, 0, s>>>(
      ws, ws_ml, ws_desc, cu_q, G, max_q_len, out, ost, osh);
  return dsp_launch_status();
}

template <bool kShared, typename... A>
int launch_prefill(int D, bool f16, dim3 grid, hipStream_t s, A... args) {
  if constexpr (!kShared) {
    if (D == 256) {
      if (f16) paged_prefill_kernel<F16Tag, 256, false><<<grid, kThreads, 0, s>>>(args...);
      else paged_prefill_kernel<Bf16Tag, 256, false><<<grid, kThreads, 0, s>>>(args...);
      return dsp_launch_status();
    }
  }
  if (D == 128) {
    if (f16) paged_prefill_kernel<F16Tag, 128, kShared><<<grid, kThreads, 0, s>>>(args...);
    else paged_prefill_kernel<Bf16Tag, 128, kShared><<<grid, kThreads, 0, s>>>(args...);
  } else {
    if (f16) paged_prefill_kernel<F16Tag, 64, kShared><<<grid, kThreads, 0, s>>>(args...);
    else paged_prefill_kernel<Bf16Tag, 64, kShared><<<grid, kThreads, 0, s>>>(args...);
  }
  return dsp_launch_status();
}

}  // namespace

namespace dsp_detail {

bool prefill_applies(int32_t D, int32_t block_size, int64_t max_rows, int64_t num_slots,
                     int64_t kv_stride_slot) {
  return (D == 64 || D == 128 || D == 256) && block_size >= 16 && max_rows >= kRows &&
         num_slots >= 16 &&
         kv_stride_slot < (int64_t(1) << 25);  // 16-row lane offsets fit 32 bits
}

int64_t prefill_tiles(int32_t max_q_len, int32_t G) {
  return (int64_t(max_q_len) * G + kRows - 1) / kRows;
}

int prefill_attention(const uint16_t* q, int64_t q_stride_t, int64_t q_stride_h,
                      const uint16_t* k_cache, const uint16_t* v_cache, int64_t num_slots,
                      int64_t kv_stride_slot, int64_t kv_stride_head, const int32_t* block_table,
                      int64_t bt_stride, int32_t log2_bs, const int32_t* cu_q,
                      const int32_t* ctx_lens, int32_t B, int32_t KVH, int32_t G, int32_t D,
                      float scale_log2, int32_t max_q_len, int32_t max_ctx, int32_t P,
                      int32_t num_parts, int32_t tiles16_max, float* ws_acc, float* ws_ml,
                      uint16_t* out, int64_t o_stride_t, int64_t o_stride_h, bool f16,
                      int32_t* err_count, hipStream_t s) {
  const int64_t tiles = prefill_tiles(max_q_len, G);
  dim3 grid(static_cast<unsigned>(tiles * num_parts), static_cast<unsigned>(KVH),
            static_cast<unsigned>(B));
  return launch_prefill<false>(D, f16, grid, s, q, q_stride_t, q_stride_h, k_cache, v_cache,
                               num_slots, kv_stride_slot, kv_stride_head, block_table, bt_stride,
                               log2_bs, cu_q, ctx_lens, max_ctx, G, scale_log2, P, num_parts,
                               tiles16_max, ws_acc, ws_ml, out, o_stride_t, o_stride_h,
                               err_count, B, int32_t(0), num_parts, int32_t(0));
}

int prefill_shared_prefix(const uint16_t* q, int64_t q_stride_t, int64_t q_stride_h,
                          const uint16_t* k_cache, const uint16_t* v_cache, int64_t num_slots,
                          int64_t kv_stride_slot, int64_t kv_stride_head,
                          const int32_t* block_table, int64_t bt_stride, int32_t log2_bs,
                          const int32_t* cu_q, const int32_t* ctx_lens, int32_t B, int32_t KVH,
                          int32_t G, int32_t D, float scale_log2, int32_t max_q_len,
                          int32_t max_ctx, int32_t P, int32_t tiles16_max,
                          int32_t prefix_tokens, float* ws_acc, float* ws_ml, uint16_t* out,
                          int64_t o_stride_t, int64_t o_stride_h, bool f16, int32_t* err_count,
                          hipStream_t s) {
  const int32_t prefix_parts = prefix_tokens / P;
  const int32_t suffix_parts = (max_ctx - prefix_tokens + P - 1) / P;
  const int64_t tiles_p = (int64_t(B) * max_q_len * G + kRows - 1) / kRows;
  const int64_t prefix_x = tiles_p * prefix_parts;
  const int64_t suffix_x = int64_t(B) * prefill_tiles(max_q_len, G) * suffix_parts;
  dim3 grid(static_cast<unsigned>(prefix_x + suffix_x), static_cast<unsigned>(KVH), 1u);
  return launch_prefill<true>(D, f16, grid, s, q, q_stride_t, q_stride_h, k_cache, v_cache,
                              num_slots, kv_stride_slot, kv_stride_head, block_table, bt_stride,
                              log2_bs, cu_q, ctx_lens, max_ctx, G, scale_log2, P, prefix_parts,
                              tiles16_max, ws_acc, ws_ml, out, o_stride_t, o_stride_h, err_count,
                              B, prefix_tokens, prefix_parts + suffix_parts,
                              static_cast<int32_t>(prefix_x));
}

int64_t shared_prefix_grid(int32_t B, int32_t G, int32_t max_q_len, int32_t max_ctx, int32_t P,
                           int32_t prefix_tokens) {
  const int64_t tiles_p = (int64_t(B) * max_q_len * G + kRows - 1) / kRows;
  return tiles_p * (prefix_tokens / P) +
         int64_t(B) * prefill_tiles(max_q_len, G) * ((max_ctx - prefix_tokens + P - 1) / P);
}

bool shared_prefix_applies(int32_t D, int32_t block_size, int32_t B, int64_t num_slots,
                           int64_t kv_stride_slot) {
  return (D == 64 || D == 128) && block_size >= 16 && B >= 1 && B <= kMaxSharedSeqs &&
         num_slots >= 16 && kv_stride_slot < (int64_t(1) << 25);
}

namespace {

// Workgroups that fit the chip at once: registers hold three per CU at D 64 (the kernel is
// compiled for three waves per SIMD), two at D 128, LDS one at D 256.  (Four at D 64, as the plain
// tile has, leave a quarter of the shares for a second round: 5700 random batches of prompt
// chunks, decodes and verifies 7 % slower on average, one in twenty by 23 % or more.)
int32_t ragged_workers(int32_t D) {
  return (D <= 64 ? 3 : D <= 128 ? 2 : 1) * dsp_detail::device_cus();
}

bool ragged_applies(int32_t B, int32_t KVH, int32_t G, int32_t D, int32_t max_q_len,
                    int32_t max_ctx) {
  // the launch's units stay inside 31 bits, the numbers DivG divides inside 24 and their sums
  // of floors inside 31, the tile search inside 64 steps of 64 tiles
  const int64_t tiles = prefill_tiles(max_q_len, G);
  const int64_t chunks = (int64_t(max_ctx) + kChunk - 1) / kChunk;
  const int64_t reach = G * (chunks + 2) + 2 * tiles + 2;
  return (D == 64 || D == 128 || D == 256) && B >= 1 && B <= kMaxRaggedSeqs && KVH >= 1 &&
         max_q_len >= 1 && max_ctx >= 1 && tiles <= 4096 &&
         reach < (int64_t(1) << 24) && reach / G * reach < (int64_t(1) << 31) &&
         (int64_t(max_ctx) + 2 * kChunk) * G < (int64_t(1) << 31) &&
         tiles * chunks * B * KVH < (int64_t(1) << 31);
}

}  // namespace

size_t ragged_workspace_bytes(int32_t B, int32_t KVH, int32_t G, int32_t D, int32_t max_q_len,
                              int32_t max_ctx) {
  if (!ragged_applies(B, KVH, G, D, max_q_len, max_ctx)) return 0;
  return size_t(ragged_workers(D)) * (size_t(2) * kRows * (D + 2) + 4) * sizeof(float);
}

int prefill_ragged(const uint16_t* q, int64_t q_stride_t, int64_t q_stride_h,
                   const uint16_t* k_cache, const uint16_t* v_cache, int64_t num_slots,
                   int64_t kv_stride_slot, int64_t kv_stride_head, const int32_t* block_table,
                   int64_t bt_stride, int32_t block_size, const int32_t* cu_q,
                   const int32_t* ctx_lens, int32_t B, int32_t KVH, int32_t G, int32_t D,
                   float scale_log2, int32_t max_q_len, int32_t max_ctx, float* workspace,
                   uint16_t* out, int64_t o_stride_t, int64_t o_stride_h, bool f16,
                   int32_t* err_count, hipStream_t s) {
  if (!ragged_applies(B, KVH, G, D, max_q_len, max_ctx) ||
      !prefill_applies(D, block_size, kRows, num_slots, kv_stride_slot) ||
      (D == 256 && num_slots % block_size != 0))
    return DSP_EUNSUPPORTED;
  auto launch = [&](auto fn) {
    return fn(ragged_workers(D), s, q, q_stride_t, q_stride_h, k_cache, v_cache, num_slots,
              kv_stride_slot, kv_stride_head, block_table, bt_stride, dsp_log2i(block_size), cu_q,
              ctx_lens, B, KVH, G, max_q_len, max_ctx, scale_log2, workspace, out, o_stride_t,
              o_stride_h, err_count);
  };
#define DSP_RAGGED(DD)                                                                \
  return f16 ? launch([](auto... a) { return launch_ragged<F16Tag, DD>(a...); })      \
             : launch([](auto... a) { return launch_ragged<Bf16Tag, DD>(a...); })
  if (D == 64) DSP_RAGGED(64);
  if (D == 128) DSP_RAGGED(128);
  DSP_RAGGED(256);
#undef DSP_RAGGED
}

}  // namespace dsp_detail
