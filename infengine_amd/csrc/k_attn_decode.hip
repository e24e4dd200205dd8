// GQA decode attention for one new token per sequence.
//
// Reference: decode_attn (kernels/attn.cu:373-439) runs QK^T and A.V as two
// cuBLAS batched GEMVs over device pointer arrays plus a separate row softmax
// (softmax.cu:109-160) with half-precision intermediates.  Here softmax(q.K^T /
// sqrt(128)) . V for all 32 q heads runs as split-context ("flash decoding")
// attention on MFMA:
//
//   batch 1: grid = (max_splits, 8 kv heads), 8 waves
//   split s of kv head g owns a contiguous run of the context 0..S-1 (at most 256 positions,
//   while the split cap allows), cut into tiles of 32 keys that its waves take in turn
//   batched: 12 waves, workgroups walk an item list (sequence, kv head, run of 384-key rounds)
//   a wave stages its tile's K and V rows in LDS (K by direct-to-LDS loads; V likewise at
//   batch 1, through registers in the batched form), and
//   computes, with
//   v_mfma_f32_16x16x32_bf16, S^T = K . Q^T for the 4 GQA q heads of the kv head (GQA: q head h
//   reads kv head h/4, attn.cu:51-53) as 4 of the 16 MFMA columns, an online softmax per head,
//   and O^T += V^T . P^T with P^T taken straight from the S^T accumulators and V^T read with
//   ds_read_b64_tr_b16, as in the prefill kernel.  The waves are merged in LDS and the split
//   writes one partial (m, l, o) per q head.
//
// Batch 1: the partials of the ns splits are merged either by the O projection itself (its
// input-staging prologue reads them; decode with max_splits = 4, no extra launch) or by a small
// merge kernel writing bf16 [h][128] (attn.cu:433-438) for long contexts (max_splits = 32).
// Batched: the last run of a (sequence, kv head) to arrive merges them, handed over by
// device-scope stores without a fence (whose L2 write-back and invalidate on this multi-XCD part
// cost more than a launch).
#include <algorithm>

#include "ie_kernels.h"

namespace ie {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) short4_t lds_short4;

constexpr int kSplitWaves = 8, kBatchedWaves = 12;  // waves a workgroup: batch 1, batched
constexpr int kKeys = 32;                           // keys per wave tile (a page holds two)
constexpr int kRowBytes = kHeadDim * 2;
constexpr int kBufferFlags = 0x00020000;   // buffer descriptor word 3 (raw 32-bit access)
static_assert(kAttnTile % kKeys == 0, "a wave tile lies in one page");

// chunk c of key r of a tile at slot c ^ (r & 15) (LDS bank spread for the fragment reads)
__device__ __forceinline__ int kv_slot(int r, int c) { return r * 16 + (c ^ (r & 15)); }

static_assert(kAttnSplits <= 64, "the merge gives each split one lane");
// A wave preloads the page ids of its tiles, one per lane: with kAttnSplits splits of kSplitWaves
// waves the longest context keeps that within 64 tiles per wave; a batched run has at most 5 rounds
// more than kAttnSplits runs of kBatchedWaves waves need (run_rounds).
static_assert(kMaxLongCtx / kKeys <= 64 * kAttnSplits * kSplitWaves &&
                  kMaxLongCtx / kKeys <= (64 - 6) * kAttnSplits * kBatchedWaves,
              "page ids per wave exceed a wave");

// A workgroup's LDS, each array its own variable (the compiler then sees that the tile loads do not
// write the partials): per wave its K tile (then V over it) and V tile, and the 4 heads' partials.
template <bool VREG>
using KvSlice = u32x4_t[VREG ? 1 : 2][kKeys * 16];
using PartO = float[kGQA][kHeadDim];
using PartMl = float[kGQA][2];

// The tiles t0 .. t1-1 (kKeys keys each) of (sequence b, kv head g) with S positions: the NW waves
// take every NW-th tile and leave their partials (m, l, o) of the 4 q heads in xo / xml
// (a barrier ends it).  VREG: one LDS slice per wave, K through it and V staged in registers then
// written over K (120 KiB for the 12-wave form); otherwise K and V each have a slice (136 KiB, one
// workgroup per CU; 0.7% faster per decode step at batch 1 than K fragments loaded straight into
// registers).
// 32-key tiles: with 12 waves (batched: 3 per SIMD within the registers) a context of 17-24 half
// tiles is two rounds of half the work: 10.6 against 11.8 us per layer for 8 waves on 64-key
// tiles at bs = 16, S = 517-564, where one wave's ninth full tile ended each workgroup ~3 us after
// the others.  The batch-1 split form likewise runs 8 waves on 32-key tiles (the same tiles per
// split, half the work per wave): 4.85 against 5.07 us at S = 550-610.
// AUX: the loads' cache policy (0, or 2: nontemporal).
template <bool VREG, int NW, int AUX>
__device__ __forceinline__ void attend_tiles(const AttnDecodeParams& p, int tid, int b, int g, int S,
                                             int t0, int t1, KvSlice<VREG>* kv, PartO* xo,
                                             PartMl* xml) {
  static_assert(kKeys == 32, "one P.V contraction per tile");
  constexpr int KB = kKeys / 16;  // 16-key MFMA blocks per tile
  constexpr int NJ = kKeys / 4;   // 1 KiB loads per tile (4 rows each)
  // wave id made provably uniform: the tile indices and buffer descriptors derived from it stay
  // in SGPRs (otherwise every buffer load becomes a readfirstlane loop)
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, G = lane >> 4;
  const uint16_t* Kh = p.k_cache + (size_t)b * p.cache_batch_stride + (size_t)g * kKVPlane;
  const uint16_t* Vh = p.v_cache + (size_t)b * p.cache_batch_stride + (size_t)g * kKVPlane;
  // rows past S read as zero (buffer bounds) and are masked below
  const __amdgpu_buffer_rsrc_t krs_seq =
      __builtin_amdgcn_make_buffer_rsrc((void*)Kh, 0, S * kRowBytes, kBufferFlags);
  const __amdgpu_buffer_rsrc_t vrs_seq =
      __builtin_amdgcn_make_buffer_rsrc((void*)Vh, 0, S * kRowBytes, kBufferFlags);

  // Q^T fragments: MFMA column fr is q head 4g + fr for fr < 4 (zero elsewhere); lane supplies
  // dims 32 ks + 8 G .. +8
  bf16x8_t qf[4];
  {
    const u32x4_t* qrow = reinterpret_cast<const u32x4_t*>(
        p.q + ((size_t)b * kQHeads + g * kGQA + min(fr, kGQA - 1)) * kHeadDim);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const u32x4_t v = qrow[4 * ks + G];
      qf[ks] = __builtin_bit_cast(bf16x8_t, fr < kGQA ? v : u32x4_t{0u, 0u, 0u, 0u});
    }
  }
  const float scale = 0.08838834764831845f;  // 1/sqrt(128), softmax.cu:79
  float m = -INFINITY, l = 0.f;
  f32x4_t o[8];
#pragma unroll
  for (int db = 0; db < 8; ++db) o[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t* kt = kv[wave][0];
  u32x4_t* vt = kv[wave][VREG ? 0 : 1];

  // paged KV: lane i holds the page of this wave's i-th tile (one load ahead of the loop)
  const bool paged = p.block_table != nullptr;
  int page_of = 0;
  if (paged) {
    const int t = t0 + wave + NW * lane;
    page_of = t < t1 ? p.block_table[(size_t)b * p.table_stride + t * kKeys / kAttnTile] : -1;
  }
  int it = 0;
  for (int t = t0 + wave; t < t1; t += NW, ++it) {
    const int key0 = t * kKeys;
    // the tile's buffers: rows key0.. of the sequence's cache, or rows 0.. of its page (a page
    // id outside the pool reads as zero)
    __amdgpu_buffer_rsrc_t krs = krs_seq, vrs = vrs_seq;
    int kr0 = key0;
    if (paged) {
      const int page = __builtin_amdgcn_readlane(page_of, it);
      const bool ok = page >= 0 && page < p.n_pages;
      const size_t base = (size_t)(ok ? page : 0) * kPageElems + (size_t)g * kPageHead;
      kr0 = key0 % kAttnTile;  // the tile's first row in its page
      const int bytes = ok ? min(kAttnTile, S - (key0 - kr0)) * kRowBytes : 0;
      krs = __builtin_amdgcn_make_buffer_rsrc((void*)(p.k_cache + base), 0, bytes, kBufferFlags);
      vrs = __builtin_amdgcn_make_buffer_rsrc((void*)(p.v_cache + base), 0, bytes, kBufferFlags);
    }
    // Tile to LDS: load j fills rows 4j .. 4j+3; lane fills slot lane%16 of row 4j + lane/16
    // with global chunk (lane%16) ^ (row & 15).  The wave only reads its own slice, so its own
    // vmcnt wait is the whole synchronisation.  VREG (the batched forms, one slice per
    // wave): K goes through the slice by direct-to-LDS loads while V is loaded into registers,
    // row-contiguous, and written over K once the K fragments are in registers.  (Loading the
    // K fragments straight from memory instead reads 64-byte pieces of 16 rows per lane
    // quad and issued ~3x slower than row-contiguous loads.)
    u32x4_t vv[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = 4 * j + G;
      const uint32_t off = (uint32_t)((kr0 + r) * kRowBytes + ((fr ^ (r & 15)) * 16));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(krs, (lds_void*)&kt[64 * j], 16, off, 0, 0, AUX);
      if constexpr (!VREG)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (lds_void*)&vt[64 * j], 16, off, 0, 0, 0);
    }
    if constexpr (VREG) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        vv[j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
            vrs, (uint32_t)((kr0 + 4 * j + G) * kRowBytes + fr * 16), 0, AUX));
    }
    // K fragments kk[kb][ks] = K[key0 + 16 kb + fr][32 ks + 8 G .. +8] from the LDS tile
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(VREG ? NJ : 0) : "memory");
    u32x4_t kk[KB][4];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) kk[kb][ks] = kt[kv_slot(16 * kb + fr, 4 * ks + G)];

    // ---- S^T blocks: s[kb][r] = S[q head 4g + fr][key key0 + 16 kb + 4 G + r]
    f32x4_t s[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      s[kb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kk[kb][ks]),
                                                        qf[ks], s[kb], 0, 0, 0);
    }
    // ---- online softmax per q column (spread over lanes fr, fr+16, fr+32, fr+48)
    float mt = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = key0 + 16 * kb + 4 * G + r;
        const float v = key < S ? s[kb][r] * scale : -INFINITY;
        s[kb][r] = v;
        mt = fmaxf(mt, v);
      }
    mt = xor32_max(xor16_max(mt));   // finite: key key0 < S is in every processed tile
    const float mn = fmaxf(m, mt);
    const float alpha = __expf(m - mn);
    float ls = 0.f;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __expf(s[kb][r] - mn);
        s[kb][r] = e;
        ls += e;
      }
    l = l * alpha + xor32_sum(xor16_sum(ls));
    m = mn;
#pragma unroll
    for (int db = 0; db < 8; ++db) o[db] *= alpha;
    // P^T fragment: slot 8 G + r <-> key 4 G + r, slot 8 G + 4 + r <-> key 16 + 4 G + r
    const u32x4_t pw = {pack_bf2(s[0][0], s[0][1]), pack_bf2(s[0][2], s[0][3]),
                        pack_bf2(s[1][0], s[1][1]), pack_bf2(s[1][2], s[1][3])};
    const bf16x8_t pb = __builtin_bit_cast(bf16x8_t, pw);
    // ---- O^T[d][q] += V^T[d][keys] . P^T[keys][q]; V^T by transposed LDS reads (source lane
    //      s of a 16-lane group reads V[key0 + s/4][d0 + 4 (s%4) .. +3])
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the V tile has landed (LDS or registers)
    if constexpr (VREG) {
      // every K fragment read has returned (the MFMAs above consumed them): V over K
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int j = 0; j < NJ; ++j) vt[kv_slot(4 * j + G, fr)] = vv[j];
    }
    const int kr = fr >> 2, dq = fr & 3;
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      const int c = 2 * db + (dq >> 1), hb = (dq & 1) * 8;
      const char* va = reinterpret_cast<const char*>(&vt[kv_slot(4 * G + kr, c)]) + hb;
      const char* vb = reinterpret_cast<const char*>(&vt[kv_slot(4 * G + kr + 16, c)]) + hb;
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)va);
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)vb);
      const short4_t both[2] = {lo, hi};
      o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, both), pb, o[db],
                                                      0, 0, 0);
    }
    // the next tile's loads overwrite this slice: every read of it has returned
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  // ---- this wave's partial: o[db][r] = O^T[d = 16 db + 4 G + r][head fr] (fr < 4); a wave
  //      without tiles has l = 0 (weight 0 in the merge)
  if (fr < kGQA) {
#pragma unroll
    for (int db = 0; db < 8; ++db)
      *reinterpret_cast<float4*>(&xo[wave][fr][16 * db + 4 * G]) =
          make_float4(o[db][0], o[db][1], o[db][2], o[db][3]);
    if (G == 0) {
      xml[wave][fr][0] = m;
      xml[wave][fr][1] = l;
    }
  }
  __syncthreads();
}

// Wave h (of the first 4) merges the waves' partials of q head 4g + h: lane d receives the
// unnormalised dims 2d, 2d+1, and the max and sum.
struct AttnMerged {
  float o0, o1, M, L;
};
template <int NW>
__device__ __forceinline__ AttnMerged merge_waves(const PartO* xo, const PartMl* xml, int h, int lane) {
  const float mw = lane < NW ? xml[lane][h][0] : -INFINITY;
  const float lw = lane < NW ? xml[lane][h][1] : 0.f;
  AttnMerged r{0.f, 0.f, wave_max(mw), 0.f};
  const float wl = lw > 0.f ? __expf(mw - r.M) : 0.f;
  r.L = wave_sum(lw * wl);
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float ww = readlane_f(wl, w);
    r.o0 = fmaf(xo[w][h][2 * lane], ww, r.o0);
    r.o1 = fmaf(xo[w][h][2 * lane + 1], ww, r.o1);
  }
  return r;
}

// Batch 1, phase 1: split s of kv head g attends its run of tiles and writes the unnormalised
// partial (m, l, o) of each of the 4 q heads.  Splits are counted in 64-key tiles, as the merge and
// the O projection count them.
__global__ __launch_bounds__(kSplitWaves * 64) void attn_decode_split_kernel(AttnDecodeParams p) {
  constexpr int NW = kSplitWaves;
  __shared__ KvSlice<false> kv[NW];
  __shared__ PartO xo[NW];
  __shared__ PartMl xml[NW];
  const int split = blockIdx.x, g = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (the arguments in one go, as in the batched kernel: decode steps over states in turn took 2746,
  // 2750 and 2742 us without, 2744, 2740 and 2741 with; over one state there is no difference)
  asm volatile("" ::"s"(p.q), "s"(p.k_cache), "s"(p.v_cache), "s"(p.block_table), "s"(p.n_pages),
               "s"(p.part_o), "s"(p.part_ml), "s"(p.d_seq_len), "s"(p.seq_len), "s"(p.max_splits));
  const int S = p.d_seq_len ? p.d_seq_len[0] : p.seq_len;
  const int ntiles = (S + kKeys - 1) / kKeys;
  const int ns = attn_decode_splits((S + kAttnTile - 1) / kAttnTile, p.max_splits);
  if (split >= ns) return;  // whole workgroup: nobody reads a partial past ns
  const int tps = (ntiles + ns - 1) / ns;
  const int t0 = split * tps, t1 = min(ntiles, t0 + tps);
  attend_tiles<false, NW, 0>(p, threadIdx.x, 0, g, S, t0, t1, kv, xo, xml);
  if (wave >= kGQA) return;  // waves past the 4 q heads only contribute partials
  const AttnMerged r = merge_waves<NW>(xo, xml, wave, lane);
  const size_t slot = ((size_t)g * kAttnSplits + split) * kGQA + wave;
  *reinterpret_cast<float2*>(p.part_o + slot * kHeadDim + 2 * lane) = make_float2(r.o0, r.o1);
  if (lane == 0) *reinterpret_cast<float2*>(p.part_ml + slot * 2) = make_float2(r.M, r.L);
}

template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

// Two floats to / from memory past the XCDs' L2s (device-scope accesses): what one workgroup hands
// to another within a launch.
__device__ __forceinline__ void agent_store2(float* p, float a, float b) {
  const uint64_t v = (uint64_t)__float_as_uint(b) << 32 | __float_as_uint(a);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 agent_load2(const float* p) {
  const uint64_t v = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}

// The partials of q head 4g + h of (sequence, kv head) bg merged in run order; every lane's loads
// of 8 runs in flight at a time (indices clamped to the last run).
__device__ __forceinline__ AttnMerged merge_runs(const AttnDecodeParams& p, size_t bg, int h,
                                                 int lane, int ns) {
  const size_t slot0 = bg * kAttnSplits * kGQA + h;
  const float2 ml = agent_load2(p.part_ml + (slot0 + (size_t)min(lane, ns - 1) * kGQA) * 2);
  const float ms = lane < ns ? ml.x : -INFINITY, ls = lane < ns ? ml.y : 0.f;
  AttnMerged r{0.f, 0.f, wave_max(ms), 0.f};
  const float wl = ls > 0.f ? __expf(ms - r.M) : 0.f;
  r.L = wave_sum(ls * wl);
  for (int s0 = 0; s0 < ns; s0 += 8) {
    float2 ov[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      ov[u] = agent_load2(p.part_o + (slot0 + (size_t)min(s0 + u, ns - 1) * kGQA) * kHeadDim + 2 * lane);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float ww = s0 + u < ns ? __shfl(wl, s0 + u, 64) : 0.f;
      r.o0 = fmaf(ov[u].x, ww, r.o0);
      r.o1 = fmaf(ov[u].y, ww, r.o1);
    }
  }
  return r;
}

// Rounds of the waves in a run (of one (sequence, kv head)'s tiles), for a lane's sequence of
// ntiles tiles.  SHORT (no sequence past kAttnShortMaxCtx): by the sequence's own length, so that
// its result does not depend on what shares its step: two rounds where one such run covers it (a
// second run of a short context costs more than its round), else one (more workgroups at once: 2
// sequences of 225-1800 take 11 us, 21 in one run each).  That serves few sequences and mixed lengths
// at the cost of full batches of one length, whose 3 or 4 runs are two turns of the chip: a step of 16 of
// 769-1200 takes 3561-3669 us, 3374-3568 in one run each; of 2 of 800-2048 3059-3040 and 3101-3478.  (One
// run of three rounds to 1024 positions, and two runs past them, mended the full batches and cost
// 2-8 sequences 2-7%.)  Otherwise one for the whole batch, so that a row's rounding then depends on
// the lengths that share its step: the candidate with the least (workgroups' turns, half counted whole) x (rounds + 0.5, an item's
// own cost) whose longest sequence has at most kAttnSplits runs.  Measured / fixed at 1, 2, 3, 4, 6
// rounds, us a layer: 16 sequences of 2850-7000 85, 70, 68, 75, 73; 6 of 2500-20000 60 (2 rounds
// at the longest), 66, 66, 57, 67; 2 of 20000 37, 37, 43, 31, 35.
template <bool SHORT, int NW>
__device__ __forceinline__ int run_rounds(int ntiles) {
  if constexpr (SHORT) return ntiles <= 2 * NW ? 2 : 1;
  int most = ntiles;
  most = max(most, dpp_i<kDppQuadXor1>(most));
  most = max(most, dpp_i<kDppQuadXor2>(most));
  most = max(most, dpp_i<kDppRowHalfMirror>(most));
  most = max(most, dpp_i<kDppRowMirror>(most));
  const int r0 = max(1, (most + kAttnSplits * NW - 1) / (kAttnSplits * NW));  // (1: unused lanes)
  int best = r0, best_cost = 0x7fffffff;
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    const int r = r0 + c;
    int items = (ntiles + r * NW - 1) / (r * NW);
    items += dpp_i<kDppQuadXor1>(items);
    items += dpp_i<kDppQuadXor2>(items);
    items += dpp_i<kDppRowHalfMirror>(items);
    items += dpp_i<kDppRowMirror>(items);
    items *= kKVHeads;
    const int cost = ((items + 255) / 256 * 256 + items) * (2 * r + 1);
    if (cost < best_cost) best = r, best_cost = cost;
  }
  return best;
}

// Batched: one launch over the work items (sequence, kv head, run of its tiles; run_rounds).  A
// sequence of one run writes its output; the others' partials go out by device-scope stores and
// the last run of a (sequence, kv head) to arrive (a device-scope counter, reset by it) merges them
// in run order -- no workgroup waits, and no merge launch.
// Workgroups (one a CU: 120 KiB of LDS) walk the items a grid apart; an item list, since a grid of
// (most runs) x 8 x batch would hold mostly idle workgroups, which take their turns on the CUs.
// Bound by the K/V loads as a wave takes them, one tile at a time (a copy without the arithmetic that
// kept these turns took the same time; nothing of a wave's next tile is in flight while it computes):
// 5.0-5.6 TB/s past 100 MB a layer.  Before (one 12-wave workgroup per (sequence, kv head) up to 2048 positions, else
// up to 32 splits of 4-wave workgroups and a merge launch), us a layer with the K/V from HBM: 16
// sequences of 225-1800 25.3, now 23.2; 2 of them 20.7, 11.5; 16 of 375-3000 37, 33; 16 of
// 2850-7000 86, 69; 6 of 2500-20000 67, 57.
// NT: nontemporal K/V loads, for K/V that cannot stay in the 256 MB cache until the next step.
template <bool SHORT, bool NT>
__global__ __launch_bounds__(kBatchedWaves * 64) void attn_decode_batched_kernel(
    AttnDecodeParams p, unsigned int* counters, int batch) {
  constexpr int NW = kBatchedWaves;
  __shared__ KvSlice<true> kv[NW];
  __shared__ PartO xo[NW];
  __shared__ PartMl xml[NW];
  __shared__ int s_last;
  __shared__ int2 s_seq[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (the arguments in one go: a cache line of them first touched later is a wait of its own: steps of
  // 8 and 16 sequences of 500-600 took 3091-3289 us without, 3073-3275 with)
  asm volatile("" ::"s"(p.q), "s"(p.d_seq_len), "s"(p.block_table), "s"(counters), "s"(batch));
  // lane b: sequence b's length and the runs of the sequences up to it.  The first item takes
  // them from registers; LDS keeps them for the next ones (through the tiles they would cost
  // registers that those need)
  int len = lane < batch ? p.d_seq_len[lane] : 0;
  const int nt = (len + kKeys - 1) / kKeys;
  int rounds = run_rounds<SHORT, NW>(nt);
  if constexpr (!SHORT) rounds = __builtin_amdgcn_readlane(rounds, 0);  // (one for the batch)
  int upto = lane < batch ? (nt + rounds * NW - 1) / (rounds * NW) : 0;
  upto += dpp_i<0x111>(upto);  // row_shr 1, 2, 4, 8: inclusive scan of 16 lanes
  upto += dpp_i<0x112>(upto);
  upto += dpp_i<0x114>(upto);
  upto += dpp_i<0x118>(upto);
  if (threadIdx.x < 16) s_seq[threadIdx.x] = make_int2(upto, len);  // (read past a barrier)
  const int total = __builtin_amdgcn_readlane(upto, 15) * kKVHeads;
  for (int w = blockIdx.x; w < total; w += gridDim.x) {
    const int b = __popcll(__ballot(lane < batch && upto * kKVHeads <= w));
    const int S = __builtin_amdgcn_readlane(len, b);
    const int ntiles = (S + kKeys - 1) / kKeys;
    const int tps = NW * (SHORT ? run_rounds<SHORT, NW>(ntiles) : rounds);
    const int ns = (ntiles + tps - 1) / tps;
    const int i = w - (__builtin_amdgcn_readlane(upto, b) - ns) * kKVHeads;
    const int g = i % kKVHeads, split = i / kKVHeads;
    // (the thread id made opaque per item: what is derived from it is not kept across the loop)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    attend_tiles<true, NW, NT ? 2 : 0>(p, tid, b, g, S, split * tps, min(ntiles, split * tps + tps),
                                             kv, xo, xml);
    const size_t bg = (size_t)b * kKVHeads + g;
    AttnMerged r{};
    if (wave < kGQA) {
      r = merge_waves<NW>(xo, xml, wave, lane);
      if (ns > 1) {
        const size_t slot = (bg * kAttnSplits + split) * kGQA + wave;
        agent_store2(p.part_o + slot * kHeadDim + 2 * lane, r.o0, r.o1);
        if (lane == 0) agent_store2(p.part_ml + slot * 2, r.M, r.L);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // performed, before the arrival counts
      }
    }
    bool mine = true;
    if (ns > 1) {
      __syncthreads();
      if (threadIdx.x == 0) {
        unsigned int* cnt = counters + bg * kCntStride;
        const unsigned int old = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = old == (unsigned)(ns - 1);
        if (s_last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      mine = s_last != 0;
      if (mine && wave < kGQA) r = merge_runs(p, bg, wave, lane, ns);
    }
    if (mine && wave < kGQA) {
      // (attn.cu:433-438)
      const float inv = 1.0f / r.L;
      uint32_t* dst = reinterpret_cast<uint32_t*>(p.out + (bg * kGQA + wave) * kHeadDim);
      dst[lane] = pack_bf2(r.o0 * inv, r.o1 * inv);
    }
    __syncthreads();  // the LDS is the next item's
    upto = s_seq[lane & 15].x;
    len = s_seq[lane & 15].y;
  }
}

// Batch 1, phase 2 (next kernel on the stream, so phase 1's writes are visible): one
// workgroup per kv head, wave w merges q head 4g + w.  Lane s holds
// split s's (m, l); every partial load is issued up front (one memory latency).
__global__ __launch_bounds__(256) void attn_decode_merge_kernel(AttnDecodeParams p) {
  const int g = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = g * kGQA + wave;
  const int S = p.d_seq_len ? p.d_seq_len[0] : p.seq_len;
  const int ns = attn_decode_splits((S + kAttnTile - 1) / kAttnTile, p.max_splits);
  __shared__ float wsh[4][64];
  const size_t slot0 = (size_t)g * kAttnSplits * kGQA + wave;
  float ms = -INFINITY, ls = 0.f;
  if (lane < ns) {
    const float2 v = *reinterpret_cast<const float2*>(p.part_ml + (slot0 + lane * kGQA) * 2);
    ms = v.x;
    ls = v.y;
  }
  float2 ov[kAttnSplits];
#pragma unroll
  for (int sp = 0; sp < kAttnSplits; ++sp)
    ov[sp] = sp < ns ? *reinterpret_cast<const float2*>(p.part_o + (slot0 + sp * kGQA) * kHeadDim +
                                                        2 * lane)
                     : make_float2(0.f, 0.f);
  const float M = wave_max(ms);
  const float wl = (ls > 0.f) ? __expf(ms - M) : 0.f;
  const float L = wave_sum(ls * wl);
  wsh[wave][lane] = wl;
  __syncthreads();
  float o0 = 0.f, o1 = 0.f;
#pragma unroll
  for (int sp = 0; sp < kAttnSplits; ++sp) {
    const float w = wsh[wave][sp];
    o0 = fmaf(ov[sp].x, w, o0);
    o1 = fmaf(ov[sp].y, w, o1);
  }
  const float inv = 1.0f / L;
  uint32_t* dst = reinterpret_cast<uint32_t*>(p.out + (size_t)h * kHeadDim);
  dst[lane] = pack_bf2(o0 * inv, o1 * inv);
}

}  // namespace

size_t attn_decode_partials_bytes(int batch) {
  const size_t slots = (size_t)batch * kKVHeads * kAttnSplits * kGQA;
  return slots * kHeadDim * sizeof(float) + slots * 2 * sizeof(float);
}

int launch_attn_decode(const AttnDecodeParams& p, bool merge, hipStream_t st) {
  // (a host-side length; the paged cache holds up to kMaxLongCtx positions)
  IE_REQUIRE(p.d_seq_len || (p.seq_len >= 1 && p.seq_len <= (p.block_table ? kMaxLongCtx : kMaxCtx)),
             "attn_decode: seq_len %d out of range [1,%d]", p.seq_len,
             p.block_table ? kMaxLongCtx : kMaxCtx);
  IE_REQUIRE(p.max_splits > 1 && p.max_splits <= kAttnSplits, "attn_decode: max_splits %d",
             p.max_splits);
  // one workgroup per possible split: idle ones would still cost dispatch
  hipLaunchKernelGGL(attn_decode_split_kernel, dim3(p.max_splits, kKVHeads),
                     dim3(kSplitWaves * 64), 0, st, p);
  IE_CHECK_LAUNCH();
  if (merge) {
    IE_REQUIRE(p.out, "attn_decode: merge needs an output buffer");
    hipLaunchKernelGGL(attn_decode_merge_kernel, dim3(kKVHeads), dim3(256), 0, st, p);
    IE_CHECK_LAUNCH();
  }
  return IE_OK;
}

int launch_attn_decode_batched(const AttnDecodeParams& p, unsigned int* counters, int batch,
                               int max_len, bool nt, hipStream_t st) {
  IE_REQUIRE(batch >= 1 && batch <= 16, "attn_decode: batch %d out of range [1,16]", batch);
  IE_REQUIRE(p.d_seq_len && p.out && counters && max_len >= 1 && max_len <= kMaxLongCtx,
             "attn_decode: batched lengths, output and counters");
  // the most items: a run of one round per kBatchedWaves tiles, at most kAttnSplits of them
  const int runs = std::min((max_len + kKeys * kBatchedWaves - 1) / (kKeys * kBatchedWaves), kAttnSplits);
  const dim3 grid(std::min(runs * kKVHeads * batch, 256)), block(kBatchedWaves * 64);
#define IE_ATTN(SHORT, NT) \
  hipLaunchKernelGGL((attn_decode_batched_kernel<SHORT, NT>), grid, block, 0, st, p, counters, batch)
  if (max_len <= kAttnShortMaxCtx) {
    if (nt) IE_ATTN(true, true);
    else IE_ATTN(true, false);
  } else {
    if (nt) IE_ATTN(false, true);
    else IE_ATTN(false, false);
  }
#undef IE_ATTN
  IE_CHECK_LAUNCH();
  return IE_OK;
}

}  // namespace ie
