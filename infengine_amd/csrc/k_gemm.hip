// MFMA bf16 GEMM for prefill (and any multi-row multiply_by_weight):
//   Y[M, N] = X[M, K] . W[N, K]^T      (X, W row-major, K contiguous; fp32 accumulate)
//
// Reference: every prefill matmul is cublasGemmEx / cublasGemmStridedBatchedEx
// with fp32 compute (kernels/ffn.cu:7-33, kernels/attn.cu:12-39, 265-293).
//
// Kernels of this file by the product's rows M (launch_gemm; M <= 16 goes to the skinny GEMM of
// k_gemm_skinny.hip):
//   17-128   gemm_mid_kernel: a workgroup streams 64 (or 128) weight rows, loaded nontemporal,
//            against all X rows; K split into fp32 partial planes summed by a split reduction
//            (RoPE + K/V write, residual + RMSNorm, SwiGLU or bf16), or unsplit with the
//            epilogue in the kernel.
//   beyond   launch_tiled: the ping-pong gemm_pp_kernel on the tile shape (128 or 256 W rows by
//            128 - 256 X rows; 192 for the fused QKV) and K split that a fitted cost model
//            picks (plan_tiles), or gemm_pp_dual_kernel; gemm_wide_kernel (direct-to-LDS ring) is
//            the same products' A/B form, and the 128 x 128 gemm_kernel described next takes
//            operands off 16 bytes.
//
// Tile: 128 W-rows x 128 X-rows x 64 k per workgroup of 4 waves; each wave owns
// a 64 x 64 block as 4 x 4 v_mfma_f32_16x16x32_bf16 tiles.  The MFMA computes
// D = W_tile . X_tile^T, so a lane's 4 accumulator values are 4 consecutive
// output columns of one output row (one 8-byte store).  Both operands are
// K-contiguous in HBM, so every fragment is one 16-byte LDS read.
//
// LDS: two stages x (W tile + X tile) x 16 KiB = 64 KiB.  A 16-byte chunk c of
// tile row r is stored at chunk slot c ^ (r & 7), so the 16 rows a fragment read
// touches land in distinct bank groups.  Global loads for stage k+1 are issued
// into registers before the MFMAs of stage k and written to the other LDS stage
// afterwards: one barrier per k-step.
//
// Workgroup -> tile mapping is XCD-aware: workgroups are dealt round-robin to
// the 8 XCDs, so workgroup b is given logical tile (b % 8) * (nb / 8) + b / 8,
// which hands each XCD a contiguous run of tiles that share W rows (column-major
// sweep over M inside one W tile) and keeps those rows in that XCD's L2.
//
// Epilogues: bf16 store, fp32 store, residual add (Y = bf16(Y + bf16(acc)),
// residual_add.cu:17-19), and SwiGLU over a gate/up pair of weights in which the
// 128 W rows of a tile are [32 gate | 32 up | 32 gate | 32 up] for 64 output
// columns, so each lane holds gate and up for the same output element.
#include <algorithm>

#include "ie_kernels.h"

namespace ie {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int BM = 128;  // X rows per tile
constexpr int BN = 128;  // W rows per tile
constexpr int BK = 64;

template <int EPI>
__device__ __forceinline__ const uint16_t* w_row(const GemmParams& p, int ntile, int r) {
  if constexpr (EPI == kGemmSwiglu) {
    // local row r -> [32 gate | 32 up] x 2; output columns ntile*64 + (r/64)*32 + (r%32)
    const int half = r >> 6, within = r & 63;
    const int col = ntile * 64 + half * 32 + (within & 31);
    const int c = col < p.N ? col : p.N - 1;
    return (within < 32 ? p.w0 : p.w1) + (size_t)c * p.K;
  } else {
    int R = ntile * BN + r;
    if (R >= p.N) R = p.N - 1;
    if (R < p.n0) return p.w0 + (size_t)R * p.K;
    if (R < p.n0 + p.n1) return p.w1 + (size_t)(R - p.n0) * p.K;
    return p.w2 + (size_t)(R - p.n0 - p.n1) * p.K;
  }
}

template <int EPI>
__global__ __launch_bounds__(256) void gemm_kernel(GemmParams p, int m_tiles) {
  __shared__ u32x4_t smem[2][2][BN * (BK / 8)];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wn = wave >> 1, wm = wave & 1;
  const int nb = gridDim.x, b = blockIdx.x;
  const int t = (nb % 8 == 0) ? (b % 8) * (nb / 8) + b / 8 : b;
  const int mtile = t % m_tiles, ntile = t / m_tiles;
  const int m0 = mtile * BM;

  // each thread moves 4 chunks of W and 4 chunks of X per k-step
  const uint16_t* wsrc[4];
  const uint16_t* xsrc[4];
  int slot[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int idx = tid + i * 256, r = idx >> 3, c = idx & 7;
    wsrc[i] = w_row<EPI>(p, ntile, r) + c * 8;
    const int xr = min(m0 + r, p.M - 1);
    xsrc[i] = p.x + (size_t)xr * p.K + c * 8;
    slot[i] = r * 8 + (c ^ (r & 7));
  }

  u32x4_t rw[4], rx[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    rw[i] = *reinterpret_cast<const u32x4_t*>(wsrc[i]);
    rx[i] = *reinterpret_cast<const u32x4_t*>(xsrc[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    smem[0][0][slot[i]] = rw[i];
    smem[0][1][slot[i]] = rx[i];
  }
  __syncthreads();

  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int KT = p.K / BK;
  const int fr = lane & 15, fq = lane >> 4, sw = lane & 7;
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < KT;
    if (more) {
      const int ko = (kt + 1) * BK;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        rw[i] = *reinterpret_cast<const u32x4_t*>(wsrc[i] + ko);
        rx[i] = *reinterpret_cast<const u32x4_t*>(xsrc[i] + ko);
      }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int ch = (ks * 4 + fq) ^ sw;
      bf16x8_t af[4], bf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = wn * 64 + i * 16 + fr;
        af[i] = __builtin_bit_cast(bf16x8_t, smem[cur][0][row * 8 + ch]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = wm * 64 + j * 16 + fr;
        bf[j] = __builtin_bit_cast(bf16x8_t, smem[cur][1][row * 8 + ch]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
    }
    if (more) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        smem[cur ^ 1][0][slot[i]] = rw[i];
        smem[cur ^ 1][1][slot[i]] = rx[i];
      }
    }
    __syncthreads();
  }

  // ---- epilogue: lane holds rows m = m0 + wm*64 + j*16 + fr, cols n = base + i*16 + 4*fq + q
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int m = m0 + wm * 64 + j * 16 + fr;
    if (m >= p.M) continue;
    if constexpr (EPI == kGemmSwiglu) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int n = ntile * 64 + wn * 32 + i * 16 + 4 * fq;
        if (n >= p.N) continue;
        uint32_t o[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float v[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float g = bf2f(f2bf(acc[i][j][2 * q + e]));
            const float u = bf2f(f2bf(acc[i + 2][j][2 * q + e]));
            v[e] = g * (1.0f / (1.0f + expf(-g))) * u;
          }
          o[q] = pack_bf2(v[0], v[1]);
        }
        *reinterpret_cast<uint2*>(p.y + (size_t)m * p.ldy + n) = make_uint2(o[0], o[1]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = ntile * BN + wn * 64 + i * 16 + 4 * fq;
        if (n >= p.N) continue;
        const f32x4_t a = acc[i][j];
        if constexpr (EPI == kGemmF32) {
          *reinterpret_cast<float4*>(p.yf + (size_t)m * p.ldy + n) =
              make_float4(a[0], a[1], a[2], a[3]);
        } else if constexpr (EPI == kGemmResid) {
          uint2* dst = reinterpret_cast<uint2*>(p.y + (size_t)m * p.ldy + n);
          const uint2 old = *dst;
          *dst = make_uint2(pack_bf2(bf_lo(old.x) + bf2f(f2bf(a[0])), bf_hi(old.x) + bf2f(f2bf(a[1]))),
                            pack_bf2(bf_lo(old.y) + bf2f(f2bf(a[2])), bf_hi(old.y) + bf2f(f2bf(a[3]))));
        } else {
          *reinterpret_cast<uint2*>(p.y + (size_t)m * p.ldy + n) =
              make_uint2(pack_bf2(a[0], a[1]), pack_bf2(a[2], a[3]));
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// DMA-ring kernel (ie_tune_gemm_schedule 0 and 1): 256 W rows x 256 X rows x 64 k per workgroup
// of 8 waves; each wave owns 128 W rows x 64 X rows as 4 x 2 tiles of
// v_mfma_f32_32x32x16_bf16 (128 fp32 accumulators per lane).
//
// Operands reach LDS by direct-to-LDS buffer loads (buffer_load_dwordx4 ... lds:
// lane i of a wave writes 16 bytes at LDS base + 16 i), through a 2-stage ring
// of 64 KiB stages, so the loads for k-step kt+1 are in flight while k-step kt
// is multiplied.  Each load covers 8 tile rows through its own buffer descriptor
// (base = the group's first row, size = the rows left in its matrix), so rows
// past the end of a matrix read as zero, and the k offset is a scalar operand.
// (The buffer form, not global_load_lds: a FLAT-encoded LDS load makes the
// compiler treat every later LDS wait as unordered, i.e. lgkmcnt(0).)  The LDS destination of a load is fixed by the lane index, so
// the bank swizzle is applied on the global side: LDS chunk slot s of tile row r
// holds global chunk s ^ swz(r).  swz(r) = ((r >> 1) & 7) ^ ((r >> 4) & 1) makes
// the 16 (or 32) rows that one ds_read_b128 phase touches land in distinct
// 16-byte bank groups for both a 64-bank and a 128-bank LDS.
//
// The loads are counted by vmcnt; the compiler does not track them, so every
// k-step's last sub-step starts with an explicit "s_waitcnt vmcnt(0); s_barrier".
// No other vector-memory instruction is issued inside the loop.
namespace wide {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kBufferFlags = 0x00020000;  // buffer descriptor word 3 (raw 32-bit access)

// Tile geometry: BN W rows x BM X rows x BK k, in a ring of STAGES LDS stages.  Every wave owns
// BN / 2 W rows x 64 X rows (NI = BN / 64 blocks of 32 W rows).
struct Cfg {
  static constexpr int BN = 256, BM = 256, BK = 64, STAGES = 2;
  static constexpr int WTN = BN / 2;                 // W rows per wave
  static constexpr int NI = WTN / 32;                // 32-row MFMA blocks per wave
  static constexpr int NT = 2 * NI;                  // MFMAs per k16 sub-step
  static constexpr int WM = BM / 64;                 // waves along X
  static constexpr int NW = 2 * WM;                  // waves
  static constexpr int THREADS = 64 * NW;
  static constexpr int CPR = BK / 8;                 // 16-byte chunks per tile row
  static constexpr int RPL = 64 / CPR;               // tile rows per wave-wide load
  static constexpr int W_CHUNKS = BN * CPR;
  static constexpr int X_CHUNKS = BM * CPR;
  static constexpr int STAGE = W_CHUNKS + X_CHUNKS;  // chunks per stage
  static constexpr int W_LOADS = W_CHUNKS / THREADS; // loads per thread per stage
  static constexpr int X_LOADS = X_CHUNKS / THREADS;
  static constexpr int LOADS = W_LOADS + X_LOADS;
  static constexpr int KSUB = BK / 16;               // MFMA k16 sub-steps per stage
  static_assert(KSUB % 2 == 0, "fragment double buffer alternates within a k-step");
  static_assert(W_CHUNKS % THREADS == 0 && X_CHUNKS % THREADS == 0, "loads per thread");
  static_assert(STAGES * STAGE * 16 <= 160 * 1024, "LDS");
  // Chunk slot s of row r holds global chunk s ^ swz(r): the 16 (or 32) consecutive rows one
  // ds_read_b128 phase touches fall in distinct 16-byte bank groups (64- or 128-bank LDS).
  static __device__ __forceinline__ int swz(int r) { return ((r >> 1) & 7) ^ ((r >> 4) & 1); }
};

// Buffer descriptor for the `rows` W rows starting at tile-local row r (all in one matrix).
template <int EPI, int BN>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t w_group(const GemmParams& p, int ntile, int r,
                                                          int k0 = 0) {
  const uint16_t* base;
  long long rows;
  if constexpr (EPI == kGemmSwiglu) {
    // local row r -> [32 gate | 32 up] x (BN / 64); output column ntile*BN/2 + (r/64)*32 + r%32
    const int col = ntile * (BN / 2) + (r >> 6) * 32 + (r & 31);
    base = ((r & 63) < 32 ? p.w0 : p.w1) + (size_t)col * p.K;
    rows = p.N - col;
  } else {
    int R = ntile * BN + r;
    if constexpr (EPI == kGemmQkvRope) {
      // tile rows 0..95: the first halves (dims 0..63) of RoPE pairs P = 96 ntile + r, rows
      // 96..191 the second halves (dims 64..127) of the same pairs; pair P is dim P % 64 of head
      // P / 64 of [q|k|v] (a group of 8 rows stays within one half-head: consecutive rows)
      static_assert(BN == 192, "QKV + RoPE tiles hold 96 pairs");
      const int half = r >= 96 ? 1 : 0, P = ntile * 96 + r - 96 * half;
      R = (P >> 6) * kHeadDim + 64 * half + (P & 63);
    }
    const int e0 = min(p.n0, p.N), e1 = min(p.n0 + p.n1, p.N);
    if (R < e0) {
      base = p.w0 + (size_t)R * p.K;
      rows = e0 - R;
    } else if (R < e1) {
      base = p.w1 + (size_t)(R - e0) * p.K;
      rows = e1 - R;
    } else if (R < p.N) {
      base = p.w2 + (size_t)(R - e1) * p.K;
      rows = p.N - R;
    } else {
      base = p.w0;
      rows = 0;
    }
  }
  // (split K: the buffer starts at column k0 of its first row and ends where the rows end)
  const long long bytes = rows > 0 ? rows * p.K * 2 - 2LL * k0 : 0;
  return __builtin_amdgcn_make_buffer_rsrc((void*)(base + k0), 0, (int)min(bytes, 0x7fffffffLL),
                                           kBufferFlags);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t x_group(const GemmParams& p, int m0, int r,
                                                          int k0 = 0) {
  const int R = m0 + r;
  const long long rows = p.M - R;
  const long long bytes = rows > 0 ? rows * p.K * 2 - 2LL * k0 : 0;
  return __builtin_amdgcn_make_buffer_rsrc((void*)(p.x + (size_t)min(R, p.M - 1) * p.K + k0), 0,
                                           (int)min(bytes, 0x7fffffffLL), kBufferFlags);
}

// Direct-to-LDS loads of k-step kt into ring slot `stage`.  (Plain device functions, not
// lambdas: a lambda around the amdgcn builtin inside a kernel template stops the host pass
// from emitting the kernel's launch stub.)
using C = Cfg;
__device__ __forceinline__ void issue_load(u32x4_t* lds, const __amdgpu_buffer_rsrc_t* rsrc,
                                           const uint32_t* voff, int wv, int kt, int stage, int j) {
  const bool is_w = j < C::W_LOADS;
  const int g = wv + C::NW * (is_w ? j : j - C::W_LOADS);
  u32x4_t* dst = &lds[stage * C::STAGE + (is_w ? 0 : C::W_CHUNKS) + g * 64];
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc[j], (lds_void*)dst, 16, voff[j],
                                           (uint32_t)(kt * C::BK * 2), 0, 0);
}

__device__ __forceinline__ void issue_stage(u32x4_t* lds, const __amdgpu_buffer_rsrc_t* rsrc,
                                            const uint32_t* voff, int wv, int kt, int stage) {
#pragma unroll
  for (int j = 0; j < C::LOADS; ++j) issue_load(lds, rsrc, voff, wv, kt, stage, j);
}

// Operand fragment n (0..NI+1) of a k16 sub-step, in the order the sub-step's MFMAs first use
// them: X0 W0 X1 W1 W2 (W3).  Lane l supplies tile row base + l%32 at k chunk ch (2*kk + l/32,
// swizzled).
__device__ __forceinline__ void read_frag(const u32x4_t* src, int a_row, int b_row, int ch, int n,
                                          bf16x8_t* af, bf16x8_t* bfr) {
  if (n == 0 || n == 2) {
    bfr[n / 2] = __builtin_bit_cast(bf16x8_t, src[b_row + (n / 2) * 32 * C::CPR + ch]);
  } else {
    const int i = n == 1 ? 0 : n - 2;
    af[i] = __builtin_bit_cast(bf16x8_t, src[a_row + i * 32 * C::CPR + ch]);
  }
}

// 8 bf16 at dst (8-byte aligned; 16-byte aligned when a16)
__device__ __forceinline__ void store16(uint16_t* dst, uint2 lo, uint2 hi, bool a16) {
  if (a16) {
    *reinterpret_cast<uint4*>(dst) = make_uint4(lo.x, lo.y, hi.x, hi.y);
  } else {
    reinterpret_cast<uint2*>(dst)[0] = lo;
    reinterpret_cast<uint2*>(dst)[1] = hi;
  }
}

// Wait until every load in flight has landed and this wave's LDS reads have returned, then
// barrier: after it the stage is visible to every wave and no wave still reads the ring slot the
// next loads overwrite.
__device__ __forceinline__ void wait_stage() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Logical tile of workgroup b.  Workgroups are dealt round-robin to the 8 XCDs, so each XCD
// is handed a contiguous range of W tiles (n_tiles / 8); inside it the range is swept in
// one W tile x all X tiles at a time, so the 32 tiles an XCD runs at once share W rows and X rows
// in its L2.
__device__ __forceinline__ void tile_of(int b, int nb, int m_tiles, int& mtile, int& ntile) {
  const int n_tiles = nb / m_tiles;
  if (nb % 8 == 0 && n_tiles % 8 == 0) {
    const int x = b % 8, local = b / 8;
    ntile = x * (n_tiles / 8) + local / m_tiles;
    mtile = local % m_tiles;
  } else {
    const int t = (nb % 8 == 0) ? (b % 8) * (nb / 8) + b / 8 : b;
    mtile = t % m_tiles;
    ntile = t / m_tiles;
  }
}

// One k-step on ring slot kt % STAGES, as 4 MFMA sub-steps of k16.  The fragments of the next
// sub-step are read one after each MFMA of the current one, so that their issue hides under the
// MFMAs (the scheduling fences keep this order: left alone the scheduler groups the reads and
// moves each just before its use).  The last sub-step waits for stage kt+1 and reads its first
// fragments, so no k-step starts on an LDS latency; with NEW it refills slot kt % STAGES (free
// once every wave has passed that sub-step's barrier) with stage kt+STAGES.
template <bool NEW>
__device__ __forceinline__ void k_step(f32x16_t (&acc)[C::NI][2], bf16x8_t (&af)[2][C::NI],
                                       bf16x8_t (&bfr)[2][2], u32x4_t* lds,
                                       const __amdgpu_buffer_rsrc_t* rsrc, const uint32_t* voff,
                                       int wv, int a_row, int b_row, int fh, int fs, int kt, int KT) {
  const u32x4_t* st = &lds[(kt % C::STAGES) * C::STAGE];
  const u32x4_t* nst = &lds[((kt + 1) % C::STAGES) * C::STAGE];
#pragma unroll
  for (int kk = 0; kk < C::KSUB; ++kk) {
    const int cur = kk & 1;
    const bool last = kk + 1 == C::KSUB;
    const bool rd = !last || kt + 1 < KT;
    if (last && rd) wait_stage();
    const u32x4_t* src = last ? nst : st;
    const int ch = (2 * (last ? 0 : kk + 1) + fh) ^ fs;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < C::NT; ++t) {
      acc[t / 2][t % 2] =
          __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[cur][t / 2], bfr[cur][t % 2], acc[t / 2][t % 2], 0, 0, 0);
      if (rd && t < C::NI + 2) read_frag(src, a_row, b_row, ch, t, af[cur ^ 1], bfr[cur ^ 1]);
      if (last && NEW) {
#pragma unroll
        for (int j = 0; j < C::LOADS; ++j)
          if (j * C::NT / C::LOADS == t)
            issue_load(lds, rsrc, voff, wv, kt + C::STAGES, kt % C::STAGES, j);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Output-tile swizzle: 8-byte unit u of row r (32 or 64 units a row) sits at slot
// u ^ (r % 32): the 32 rows one write instruction touches land in distinct 8-byte bank pairs.
__device__ __forceinline__ int swz_out(int u, int r) { return u ^ (r & 31); }

// Copy-out of a bf16 output tile staged in LDS as [BM][UPR] 8-byte units (unit u of row r at
// swz(u, r)): 16 bytes (8 columns) per thread, consecutive threads along a row; the residual
// epilogue adds the tile to y.
template <int THREADS, int BM, int UPR, int EPI, class SW>
__device__ __forceinline__ void tile_copy_out(const GemmParams& p, const uint2* ot, uint16_t* y,
                                              int m0, int n_base, int tid, SW swz) {
  const bool ld16 = (p.ldy & 7) == 0;  // rows 16-byte aligned: one 16-byte store per thread
#pragma unroll 4
  for (int P = tid; P < BM * UPR / 2; P += THREADS) {
    const int r = P / (UPR / 2), c2 = P % (UPR / 2);
    const int m = m0 + r, n = n_base + 8 * c2;
    if (m >= p.M || n >= p.N) continue;
    const uint2 lo = ot[r * UPR + swz(2 * c2, r)], hi = ot[r * UPR + swz(2 * c2 + 1, r)];
    uint16_t* dst = y + (size_t)m * p.ldy + n;
    if constexpr (EPI == kGemmResid) {
      // y = bf16(y + bf16(acc)) (residual_add.cu:17-19); the LDS tile holds bf16(acc)
      const uint2 a = *reinterpret_cast<const uint2*>(dst);
      const uint2 o0 = make_uint2(pack_bf2(bf_lo(a.x) + bf_lo(lo.x), bf_hi(a.x) + bf_hi(lo.x)),
                                  pack_bf2(bf_lo(a.y) + bf_lo(lo.y), bf_hi(a.y) + bf_hi(lo.y)));
      if (n + 8 <= p.N) {
        const uint2 b = *reinterpret_cast<const uint2*>(dst + 4);
        const uint2 o1 = make_uint2(pack_bf2(bf_lo(b.x) + bf_lo(hi.x), bf_hi(b.x) + bf_hi(hi.x)),
                                    pack_bf2(bf_lo(b.y) + bf_lo(hi.y), bf_hi(b.y) + bf_hi(hi.y)));
        store16(dst, o0, o1, ld16);
      } else {
        *reinterpret_cast<uint2*>(dst) = o0;
      }
    } else {
      if (n + 8 <= p.N) store16(dst, lo, hi, ld16);
      else *reinterpret_cast<uint2*>(dst) = lo;
    }
  }
}

// Copy-out of the prefill QKV + RoPE tile staged in LDS as [BM][48] 8-byte units: unit u < 24
// holds the first halves of pairs 96 ntile + 4u .. +3 (pair P: head P / 64, dims P % 64 and
// P % 64 + 64), unit 24 + u their second halves.  Each thread takes 4 pairs of one row: RoPE at
// position start_pos + m on q and k (the scatter kernel's pairing and roundings, on the same
// bf16 values), q to y [M][32][128], k and v to this layer's cache planes (or pages).
template <int THREADS, int BM, class SW>
__device__ __forceinline__ void rope_copy_out(const GemmParams& p, const uint2* ot, int m0,
                                              int ntile, int tid, SW swz) {
  constexpr int UPR = 48, QUADS = 24;
#pragma unroll 4
  for (int it = tid; it < BM * QUADS; it += THREADS) {
    const int r = it / QUADS, u = it % QUADS;
    const int m = m0 + r;
    if (m >= p.M) continue;
    const uint2 lo = ot[r * UPR + swz(u, r)], hi = ot[r * UPR + swz(QUADS + u, r)];
    const int P = ntile * 96 + 4 * u;
    const int head = P >> 6, j = P & 63;
    const int pos = p.start_pos + m;
    uint2 o0 = lo, o1 = hi;
    if (head < kQHeads + kKVHeads) {
      const float4 c = *reinterpret_cast<const float4*>(p.rope_cos + (size_t)pos * 64 + j);
      const float4 sn = *reinterpret_cast<const float4*>(p.rope_sin + (size_t)pos * 64 + j);
      const float a[4] = {bf_lo(lo.x), bf_hi(lo.x), bf_lo(lo.y), bf_hi(lo.y)};
      const float b[4] = {bf_lo(hi.x), bf_hi(hi.x), bf_lo(hi.y), bf_hi(hi.y)};
      const float cc[4] = {c.x, c.y, c.z, c.w}, ss[4] = {sn.x, sn.y, sn.z, sn.w};
      float va[4], vb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        va[e] = rope_lo(a[e], b[e], cc[e], ss[e]);
        vb[e] = rope_hi(a[e], b[e], cc[e], ss[e]);
      }
      o0 = make_uint2(pack_bf2(va[0], va[1]), pack_bf2(va[2], va[3]));
      o1 = make_uint2(pack_bf2(vb[0], vb[1]), pack_bf2(vb[2], vb[3]));
    }
    uint16_t* dst;
    if (head < kQHeads) {
      dst = p.y + ((size_t)m * kQHeads + head) * kHeadDim;
    } else {
      const bool is_k = head < kQHeads + kKVHeads;
      const int kvh = head - kQHeads - (is_k ? 0 : kKVHeads);
      uint16_t* const plane = is_k ? p.k_cache : p.v_cache;
      if (p.block_table) {  // paged: row pos % kPagePos of the page holding block pos / kPagePos
        const int page = p.block_table[pos / kPagePos];
        if (page < 0 || page >= p.n_pages) continue;
        dst = plane + (size_t)page * kPageElems + ((size_t)kvh * kPagePos + pos % kPagePos) * kHeadDim;
      } else {
        dst = plane + ((size_t)kvh * kMaxCtx + pos) * kHeadDim;
      }
    }
    *reinterpret_cast<uint2*>(dst + j) = o0;
    *reinterpret_cast<uint2*>(dst + j + 64) = o1;
  }
}

struct WideOutSwz {
  __device__ __forceinline__ int operator()(int u, int r) const { return swz_out(u, r); }
};

// The epilogue of the ring kernel's tile: wave (wn, wm) holds accumulator element 4*g + q of tile
// (i, j) = W row wn*WTN + 32*i + 8*g + 4*(lane/32) + q, X row m0 + wm*64 + 32*j + lane%32.  fp32
// results go straight to global memory; bf16 ones are staged through the LDS ring as a [BM][OUTN]
// tile and stored as whole row segments.
template <int EPI>
__device__ __forceinline__ void wide_epilogue(const GemmParams& p, f32x16_t (&acc)[C::NI][2],
                                              u32x4_t* lds, uint16_t* y, float* yf, int m0,
                                              int ntile, int wn, int wm, int lane, int tid) {
  constexpr int BM = C::BM, BN = C::BN, STAGES = C::STAGES;
  const int fr = lane & 31, fh = lane >> 5;
  if constexpr (EPI == kGemmF32) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = m0 + wm * 64 + j * 32 + fr;
      if (m >= p.M) continue;
#pragma unroll
      for (int i = 0; i < C::NI; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int n = ntile * BN + wn * C::WTN + i * 32 + 8 * g + 4 * fh;
          if (n < p.N)
            *reinterpret_cast<float4*>(yf + (size_t)m * p.ldy + n) =
                make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
        }
    }
  } else {
    // bf16 results go through LDS so that the global stores are whole, coalesced row segments
    // (a lane's accumulators are 4 columns of 32 different rows; storing them directly writes
    // every 128-byte line in eight 16-byte pieces).  The tile is [BM][OUTN] bf16 held as
    // 8-byte units; unit u of row r sits at swz_out(u, r), which spreads the 32 rows one
    // write instruction touches over distinct banks without padding.
    constexpr int OUTN = (EPI == kGemmSwiglu) ? 128 : BN;  // output columns per tile
    constexpr int UPR = OUTN / 4;                            // 8-byte units per row
    static_assert(BM * OUTN * 2 <= STAGES * C::STAGE * 16, "output tile must fit the LDS ring");
    uint2* ot = reinterpret_cast<uint2*>(lds);
    __syncthreads();  // every wave is done reading the ring
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = wm * 64 + j * 32 + fr;
      if constexpr (EPI == kGemmSwiglu) {
#pragma unroll
        for (int i = 0; i < 4; i += 2)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            uint32_t o[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              float v[2];
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                const float gt = bf2f(f2bf(acc[i][j][4 * g + 2 * q + e]));
                const float up = bf2f(f2bf(acc[i + 1][j][4 * g + 2 * q + e]));
                v[e] = gt * (1.0f / (1.0f + expf(-gt))) * up;
              }
              o[q] = pack_bf2(v[0], v[1]);
            }
            const int u = (2 * wn + i / 2) * 8 + 2 * g + fh;
            ot[r * UPR + swz_out(u, r)] = make_uint2(o[0], o[1]);
          }
      } else {
#pragma unroll
        for (int i = 0; i < C::NI; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int u = wn * (C::WTN / 4) + i * 8 + 2 * g + fh;
            ot[r * UPR + swz_out(u, r)] = make_uint2(pack_bf2(acc[i][j][4 * g], acc[i][j][4 * g + 1]),
                                                pack_bf2(acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]));
          }
      }
    }
    __syncthreads();
    tile_copy_out<C::THREADS, BM, UPR, EPI>(p, ot, y, m0, ntile * OUTN, tid, WideOutSwz{});
  }
}

template <int EPI>
__global__ __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_wide_kernel(GemmParams p, int m_tiles) {
  constexpr int BM = C::BM, BK = C::BK, STAGES = C::STAGES;
  static_assert(C::THREADS == 512, "two waves per SIMD");
  __shared__ u32x4_t lds[STAGES * C::STAGE];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wn = wave / C::WM, wm = wave % C::WM;
  // split K: workgroup b takes k-steps [split * KT, (split + 1) * KT) of tile b % tiles and
  // writes its fp32 partial product to partial plane `split` of yf
  const int nsplit = max(1, p.k_splits);
  const int nb = gridDim.x / nsplit, split = blockIdx.x / nb;
  int mtile, ntile;
  tile_of(blockIdx.x - split * nb, nb, m_tiles, mtile, ntile);
  const int m0 = mtile * BM;
  const int KT = p.K / BK / nsplit;
  const int k0 = split * KT * BK;

  // load j of this wave covers tile rows RPL*g .. RPL*g+RPL-1 with g = wave + NW*j;
  // lane i fills LDS slot (row RPL*g + i/CPR, chunk i%CPR) from global chunk (i%CPR) ^ swz(row)
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  __amdgpu_buffer_rsrc_t rsrc[C::LOADS];
  uint32_t voff[C::LOADS];
#pragma unroll
  for (int j = 0; j < C::LOADS; ++j) {
    const bool is_w = j < C::W_LOADS;
    const int g = wv + C::NW * (is_w ? j : j - C::W_LOADS);
    rsrc[j] = is_w ? w_group<EPI, C::BN>(p, ntile, g * C::RPL, k0) : x_group(p, m0, g * C::RPL, k0);
    const int rl = lane / C::CPR, c = (lane % C::CPR) ^ C::swz(g * C::RPL + rl);
    voff[j] = (uint32_t)((rl * p.K + c * 8) * 2);
  }
  f32x16_t acc[C::NI][2];
#pragma unroll
  for (int i = 0; i < C::NI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // fragment addressing: operand lane l supplies tile row base + l%32, k chunk 2*kk + l/32
  const int fr = lane & 31, fh = lane >> 5, fs = C::swz(fr);
  const int a_row = (wn * C::WTN + fr) * C::CPR;
  const int b_row = C::W_CHUNKS + (wm * 64 + fr) * C::CPR;

  // The epilogue's kernel arguments are pulled into SGPRs here: a scalar load still in
  // flight inside the loop would force every LDS wait there to lgkmcnt(0).
  uint16_t* const y = p.y;
  float* const yf = p.yf + (size_t)split * p.M * p.ldy;
  asm volatile("" ::"s"(y), "s"(yf), "s"(p.ldy), "s"(p.M), "s"(p.N));

  issue_stage(lds, rsrc, voff, wv, 0, 0);
  wait_stage();  // stage 0 landed; stage 1 goes to the slot no wave reads yet
  if (STAGES - 1 < KT) issue_stage(lds, rsrc, voff, wv, 1, 1);
  bf16x8_t af[2][C::NI], bfr[2][2];
#pragma unroll
  for (int n = 0; n < C::NI + 2; ++n) read_frag(lds, a_row, b_row, fh ^ fs, n, af[0], bfr[0]);
  int kt = 0;
  for (; kt + STAGES < KT; ++kt)
    k_step<true>(acc, af, bfr, lds, rsrc, voff, wv, a_row, b_row, fh, fs, kt, KT);
  for (; kt < KT; ++kt)
    k_step<false>(acc, af, bfr, lds, rsrc, voff, wv, a_row, b_row, fh, fs, kt, KT);

  wide_epilogue<EPI>(p, acc, lds, y, yf, m0, ntile, wn, wm, lane, tid);
}

// ---------------------------------------------------------------------------
// Ping-pong kernel on v_mfma_f32_16x16x32_bf16, described for its 256 x 256 tile.
//
// The part runs these GEMMs power-limited: the same kernels on all-zero operands run 25-35%
// faster, and on random data a stream of 32x32x16 MFMAs alone (no LDS reads, loads or
// barriers) reached 0.58-0.61 of the nominal peak where the same flops as 16x16x32 MFMAs
// reached 0.61-0.66 (a 16x16x32 MFMA reads and writes a quarter of the accumulators for half
// the flops).  So this kernel runs 16x16x32 MFMAs, and keeps every SIMD's matrix core fed from
// registers:
//
// The two waves that share a SIMD (wave w and w + 4) alternate between a compute phase -- one
// k-step (64 k) of MFMAs from fragments already in registers, 64 (48) back to back -- and a
// memory phase -- the 24 (20) ds_read_b128 of their next k-step's fragments plus their share
// of the direct-to-LDS loads of a later stage.  Group 0 (waves 0-3) owns W rows 0 .. WTN-1 of
// the tile and loads the W half of every stage; group 1 (waves 4-7) owns W rows WTN .. and
// loads the X half; wave 4 g + q owns X rows 64 q .. +63.  Group 1 runs one phase behind group
// 0, and every phase ends at a workgroup barrier:
//   phase 2k+1: group 0 multiplies k-step k; group 1 reads k-step k's fragments (ring slot k%2);
//               every wave waits for its loads of stage k+1 (issued in phase 2k) first
//   phase 2k+2: group 0 reads k-step k+1's fragments (slot (k+1)%2), then issues the W half of
//               stage k+2 into slot k%2; group 1 issues the X half of stage k+2 into slot k%2
//               between its first MFMAs of k-step k
// Slot k%2 is free in phase 2k+2: its last readers (group 1, phase 2k+1) waited for their reads
// before the barrier that ended that phase; a memory phase reads a stage every wave waited for
// before the barrier that started the phase.  Each group runs a loop of its own (s_barrier
// syncs the workgroup wherever each wave executes it), so each role's registers are allocated
// on their own.
//
// MFMA operands: A = 16 W rows, B = 16 X rows, k 32: lane l supplies row l % 16 at k chunk
// 4 ks + l / 16 of the 64-k stage (ks = 0, 1), so D[w][x] puts output row x = l % 16 and output
// columns w = 4 (l / 16) .. +3 in a lane: an 8-byte unit.  LDS chunk slot s of row r holds
// global chunk s ^ swz(r), swz(r) = (r >> 1) & 7: the 16 rows of one chunk a fragment read
// touches fall in 16 distinct 16-byte bank groups (and, with the next chunk's 16, in 32 of a
// 512-byte LDS line).  swz does not depend on a fragment's 16-row block, so a lane's fragment
// offsets are base ^ (ks << 6) plus immediates of 2048 bytes per block.
namespace pp {

// Tile: BN W rows x BM X rows x 64 k per stage.  The two wave groups split the W rows, and the 4
// waves of a group are 4 / WX along W by WX along X.
template <int BN_, int BM_, int NW_ = 3, int WX_ = 4>
struct PC {
  static constexpr int BN = BN_, BM = BM_, BK = 64;
  static constexpr int WX = WX_;               // waves of a group along X
  static constexpr int KS = 2;                 // k32 sub-steps per stage
  static constexpr int WTN = BN / 2 * WX / 4;  // W rows per wave
  static constexpr int WTM = BM / WX;          // X rows per wave
  static constexpr int NA = WTN / 16;          // 16-row W blocks per wave
  static constexpr int NB = WTM / 16;          // 16-row X blocks per wave
  static constexpr int CPR = 8;                // 16-byte chunks per tile row
  static constexpr int W_CHUNKS = BN * CPR;    // one stage's W half
  static constexpr int X_CHUNKS = BM * CPR;    // one stage's X half
  static constexpr int WL = W_CHUNKS / 64 / 4; // W loads per group-0 wave per stage
  static constexpr int XL = X_CHUNKS / 64 / 4; // X loads per group-1 wave per stage
  static constexpr int PL = WL > XL ? WL : XL;
  // The W and X halves have rings of their own: NW W slots (the W rows come from HBM; stage
  // k + NW is issued 2 NW - 2 phases before it is read), and 3 X slots where they fit beside
  // them in the 160 KiB of LDS, else 2.  X slots follow the W slots.
  static constexpr int NW = NW_;
  static constexpr int NX = (NW * W_CHUNKS + 3 * X_CHUNKS) * 16 <= 160 * 1024 ? 3 : 2;
  static constexpr int X_BASE = NW * W_CHUNKS;  // chunk offset of X slot 0
  static constexpr int TOTAL = NW * W_CHUNKS + NX * X_CHUNKS;
  static_assert(WTN % 16 == 0 && WTM % 16 == 0 && BM % 32 == 0 && BN % 32 == 0, "tile shapes");
  static_assert(NW == 3 || NW == 4, "W ring depth");
  static_assert(TOTAL * 16 <= 160 * 1024, "LDS");
  static __device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }
};

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Load j of a wave's stage share (8 tile rows) into LDS chunk base + 256 j (base: the ring slot's
// first chunk plus the wave's first 8-row group).
template <int NL>
__device__ __forceinline__ void issue(u32x4_t* lds, const __amdgpu_buffer_rsrc_t* rs,
                                      uint32_t vo, int base, int kt) {
#pragma unroll
  for (int j = 0; j < NL; ++j)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs[j], (lds_void*)&lds[base + 256 * j], 16, vo,
                                             (uint32_t)(kt * 128), 0, 0);
}

// All fragments of one k-step: the W half at LDS byte offset sa, the X half at sb.
template <class C>
__device__ __forceinline__ void read(const u32x4_t* lds, uint32_t sa, uint32_t sb, uint32_t aA,
                                     uint32_t aB, bf16x8_t (&fa)[C::KS][C::NA],
                                     bf16x8_t (&fb)[C::KS][C::NB]) {
  const char* base = reinterpret_cast<const char*>(lds);
  uint32_t a0 = sa + aA, b0 = sb + aB;
  // (computed here, at the reads: hoisted out of the k loop the offsets of both ring slots
  // would stay live through the MFMAs)
  asm volatile("" : "+v"(a0), "+v"(b0));
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) {
    const char* pa = base + (a0 ^ (uint32_t)(ks << 6));
    const char* pb = base + (b0 ^ (uint32_t)(ks << 6));
#pragma unroll
    for (int i = 0; i < C::NA; ++i) fa[ks][i] = *reinterpret_cast<const bf16x8_t*>(pa + i * 2048);
#pragma unroll
    for (int j = 0; j < C::NB; ++j) fb[ks][j] = *reinterpret_cast<const bf16x8_t*>(pb + j * 2048);
  }
}

// One k-step of MFMAs at raised wave priority; with DMA this wave's loads of stage kt into
// `slot` go out one after each of the first NL MFMAs.
template <class C, int NL, bool DMA>
__device__ __forceinline__ void compute(f32x4_t (&acc)[C::NA][C::NB], const bf16x8_t (&fa)[C::KS][C::NA],
                                        const bf16x8_t (&fb)[C::KS][C::NB], u32x4_t* lds,
                                        const __amdgpu_buffer_rsrc_t* rs, uint32_t vo,
                                        int base, int kt) {
  asm volatile("s_setprio 2" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks)
#pragma unroll
    for (int i = 0; i < C::NA; ++i)
#pragma unroll
      for (int j = 0; j < C::NB; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[ks][i], fb[ks][j], acc[i][j], 0, 0, 0);
        const int n = (ks * C::NA + i) * C::NB + j;
        if (DMA && n < NL)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs[n], (lds_void*)&lds[base + 256 * n], 16, vo,
                                                   (uint32_t)(kt * 128), 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
  asm volatile("s_setprio 0" ::: "memory");
}

// Output staging swizzle (a bijection of a row's units): 8-byte unit u of row r at
// u ^ ((r & 15) << 2) (64 units a row), u ^ ((r & 7) << 2) (32), u ^ ((r & 3) << 2) (16), and for
// 48 the 32-unit form within the first 32 units and the 16-unit form in the last 16; a write
// instruction covers 16 rows x 4 consecutive units.
template <int UPR>
struct OutSwz {
  static_assert(UPR == 64 || UPR == 48 || UPR == 32 || UPR == 16, "units per row");
  __device__ __forceinline__ int operator()(int u, int r) const {
    if constexpr (UPR == 64) return u ^ ((r & 15) << 2);
    else if constexpr (UPR == 32) return u ^ ((r & 7) << 2);
    else if constexpr (UPR == 16) return u ^ ((r & 3) << 2);
    else return u < 32 ? u ^ ((r & 7) << 2) : u ^ ((r & 3) << 2);
  }
};

// Tile b of the nb tiles of p (the LDS ring: at least C::TOTAL chunks).  kGemmF32: k-steps
// split KT .. of the tile's K (KT = K / 64 / k_splits), its fp32 sums to partial plane `split`.
template <int EPI, class C>
__device__ __forceinline__ void pp_tile(const GemmParams& p, int m_tiles, int b, int nb, int split,
                                        u32x4_t* lds) {
  constexpr int BN = C::BN, BM = C::BM;
  constexpr int NA = C::NA, NB = C::NB, WL = C::WL, XL = C::XL, PL = C::PL, KS = C::KS;
  static_assert(EPI != kGemmSwiglu || C::WTN % 64 == 0, "SwiGLU waves hold [32 gate | 32 up] rows");
  static_assert(EPI != kGemmQkvRope || BN == 192, "QKV + RoPE: 192 W rows");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wv >> 2, gw = wv & 3;
  // the wave's output block: W rows wn * WTN .., X rows wm * WTM ..
  const int wn = grp * (4 / C::WX) + gw / C::WX, wm = gw % C::WX;
  int mtile, ntile;
  tile_of(b, nb, m_tiles, mtile, ntile);
  const int m0 = mtile * BM;
  const int KT = EPI == kGemmF32 ? p.K / 64 / p.k_splits : p.K / 64;
  const int k0 = EPI == kGemmF32 ? split * KT * 64 : 0;

  // this wave's share of a stage: 8-row groups gw + 4 j of its half (W or X); lane i fills LDS
  // slot (row 8 g + i / 8, chunk i % 8) from global chunk (i % 8) ^ swz(row), the same for every
  // j (rows 32 apart)
  __amdgpu_buffer_rsrc_t rs[PL];
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    const int g = gw + 4 * j;
    rs[j] = grp == 0 ? w_group<EPI, BN>(p, ntile, min(g, BN / 8 - 1) * 8, k0)
                     : x_group(p, m0, g * 8, k0);
  }
  const int rl = lane / 8;
  const uint32_t vo = (uint32_t)((rl * p.K + ((lane % 8) ^ C::swz(gw * 8 + rl)) * 8) * 2);
  const int dst0 = (grp == 0 ? 0 : C::X_BASE) + gw * 64;  // the wave's first row group, slot 0

  f32x4_t acc[NA][NB];
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // fragment byte offsets within a stage (ks = 0, block 0): lane l reads row base + l % 16 at
  // chunk (l / 16) ^ swz(row)
  const int fr = lane & 15, fq = lane >> 4;
  const uint32_t chunk0 = (uint32_t)((fq ^ C::swz(fr)) * 16);
  const uint32_t aA = (uint32_t)((wn * C::WTN + fr) * C::CPR * 16) + chunk0;
  const uint32_t aB = (uint32_t)((wm * C::WTM + fr) * C::CPR * 16) + chunk0;
  bf16x8_t fa[KS][NA], fb[KS][NB];

  uint16_t* const y = p.y;
  float* const yf = p.yf + (size_t)split * p.M * p.ldy;
  asm volatile("" ::"s"(y), "s"(yf), "s"(p.ldy), "s"(p.M), "s"(p.N));

  // stage k's W half lives in W slot k % NW, its X half in X slot k % NX.  The wait that ends
  // phase 2k+1 leaves in flight only this wave's loads of stages issued after k+1.
  constexpr int NW = C::NW, NX = C::NX;
  constexpr uint32_t WSB = C::W_CHUNKS * 16, XSB = C::X_CHUNKS * 16, XB0 = C::X_BASE * 16;
  if (grp == 0) {
#pragma unroll
    for (int t = 0; t < NW; ++t)
      if (t < KT) issue<WL>(lds, rs, vo, dst0 + t * C::W_CHUNKS, t);
    if (KT >= NW) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NW - 1) * WL) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    // phase 0: fragments of k-step 0
    read<C>(lds, 0, XB0, aA, aB, fa, fb);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    int sw = 0, sx = 0;  // W and X slots of stage k
#pragma unroll 1
    for (int k = 0; k < KT; ++k) {
      const int swn = sw + 1 == NW ? 0 : sw + 1, sxn = sx + 1 == NX ? 0 : sx + 1;
      // phase 2k+1: multiply k-step k
      compute<C, WL, false>(acc, fa, fb, lds, rs, vo, 0, 0);
      // stage k+1 must have landed; stages k+2 .. min(k+NW-1, KT-1) may stay in flight
      if (NW == 4 && k + 3 < KT) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * WL) : "memory");
      else if (k + 2 < KT) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(WL) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      // phase 2k+2: fragments of k-step k+1, then the W half of stage k+NW into W slot sw
      if (k + 1 < KT) read<C>(lds, swn * WSB, XB0 + sxn * XSB, aA, aB, fa, fb);
      if (k + NW < KT) issue<WL>(lds, rs, vo, dst0 + sw * C::W_CHUNKS, k + NW);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      sw = swn;
      sx = sxn;
    }
  } else {
#pragma unroll
    for (int t = 0; t < NX; ++t)
      if (t < KT) issue<XL>(lds, rs, vo, dst0 + t * C::X_CHUNKS, t);
    if (KT >= NX) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NX - 1) * XL) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    int k = 0, sw = 0, sx = 0;
#pragma unroll 1
    for (; k + NX < KT; ++k) {
      // phase 2k+1: fragments of k-step k
      read<C>(lds, sw * WSB, XB0 + sx * XSB, aA, aB, fa, fb);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NX - 2) * XL) : "memory");
      // phase 2k+2: the X half of stage k+NX into X slot sx while multiplying k-step k
      compute<C, XL, true>(acc, fa, fb, lds, rs, vo, dst0 + sx * C::X_CHUNKS, k + NX);
      asm volatile("s_barrier" ::: "memory");
      sw = sw + 1 == NW ? 0 : sw + 1;
      sx = sx + 1 == NX ? 0 : sx + 1;
    }
#pragma unroll 1
    for (; k < KT; ++k) {
      read<C>(lds, sw * WSB, XB0 + sx * XSB, aA, aB, fa, fb);
      if (k + 2 < KT)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NX - 2) * XL) : "memory");
      else
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      compute<C, XL, false>(acc, fa, fb, lds, rs, vo, 0, 0);
      asm volatile("s_barrier" ::: "memory");
      sw = sw + 1 == NW ? 0 : sw + 1;
      sx = sx + 1 == NX ? 0 : sx + 1;
    }
  }

  // ---- epilogue: acc[i][j][r] = D[W row wn*WTN + 16 i + 4 (lane/16) + r][X row wm*WTM + 16 j +
  //      lane%16]; staged in the ring as [BM][OUTN] bf16 (8-byte units), then stored as rows
  if constexpr (EPI == kGemmF32) {
    // a lane's 4 columns of one row; 4 lanes and the next block's 4 make a line
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int m = m0 + wm * C::WTM + 16 * j + fr;
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const int n = ntile * BN + wn * C::WTN + 16 * i + 4 * fq;
        if (m < p.M && n < p.N)
          *reinterpret_cast<f32x4_t*>(yf + (size_t)m * p.ldy + n) = acc[i][j];
      }
    }
    return;
  }
  constexpr int OUTN = (EPI == kGemmSwiglu) ? BN / 2 : BN;
  constexpr int UPR = OUTN / 4;
  static_assert(BM * OUTN * 2 <= C::TOTAL * 16, "output tile must fit the LDS ring");
  const OutSwz<UPR> swz;
  uint2* ot = reinterpret_cast<uint2*>(lds);
  __syncthreads();  // every wave is done reading the ring
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int r = wm * C::WTM + 16 * j + fr;
    if constexpr (EPI == kGemmSwiglu) {
      // W rows of the wave: [32 gate | 32 up] x 2, so block i (gate) pairs with i + 2 (up)
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        if ((i & 2) != 0) continue;
        uint32_t o[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float v[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float gt = bf2f(f2bf(acc[i][j][2 * q + e]));
            const float up = bf2f(f2bf(acc[i + 2][j][2 * q + e]));
            v[e] = gt * (1.0f / (1.0f + expf(-gt))) * up;
          }
          o[q] = pack_bf2(v[0], v[1]);
        }
        const int u = (wn * (C::WTN / 64) + i / 4) * 8 + (i & 1) * 4 + fq;
        ot[r * UPR + swz(u, r)] = make_uint2(o[0], o[1]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const int u = wn * (C::WTN / 4) + 4 * i + fq;
        ot[r * UPR + swz(u, r)] = make_uint2(pack_bf2(acc[i][j][0], acc[i][j][1]),
                                             pack_bf2(acc[i][j][2], acc[i][j][3]));
      }
    }
  }
  __syncthreads();
  if constexpr (EPI == kGemmQkvRope) rope_copy_out<512, BM>(p, ot, m0, ntile, tid, swz);
  else tile_copy_out<512, BM, UPR, EPI>(p, ot, y, m0, ntile * OUTN, tid, swz);
}

template <int EPI, int BN, int BM, int NWR, int WX>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_pp_kernel(GemmParams p, int m_tiles) {
  using C = PC<BN, BM, NWR, WX>;
  __shared__ u32x4_t lds[C::TOTAL];
  const int nb = EPI == kGemmF32 ? gridDim.x / p.k_splits : gridDim.x;
  const int split = EPI == kGemmF32 ? blockIdx.x / nb : 0;
  pp_tile<EPI, C>(p, m_tiles, blockIdx.x - split * nb, nb, split, lds);
}

// Two column ranges of one product in one launch: workgroups 0 .. nb1-1 take 256 x 256 tiles of
// p1, the rest 256 x 128 tiles of p2 (gate/up at S = 2048: three rounds of 256 x 256
// tiles, then the last 2048 columns as 256 x 128 tiles, each starting on a CU as soon as the CU's
// third big tile ends instead of after a kernel boundary).
template <int EPI>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_pp_dual_kernel(GemmParams p1, int m_tiles1, int nb1, GemmParams p2, int m_tiles2) {
  using C1 = PC<256, 256, 3, 2>;
  using C2 = PC<256, 128, 3, 2>;
  __shared__ u32x4_t lds[C1::TOTAL > C2::TOTAL ? C1::TOTAL : C2::TOTAL];
  if ((int)blockIdx.x < nb1)
    pp_tile<EPI, C1>(p1, m_tiles1, blockIdx.x, nb1, 0, lds);
  else
    pp_tile<EPI, C2>(p2, m_tiles2, blockIdx.x - nb1, gridDim.x - nb1, 0, lds);
}

}  // namespace pp

// ---------------------------------------------------------------------------
// Medium-M kernel (17-128 rows: prompts of a few dozen tokens), where a product is bound by its
// weight stream: 64 W rows x XR X rows (XR = 64 or 128) a workgroup, 4 waves each owning 16 W
// rows and all XR X rows (XR / 16 MFMA blocks, v_mfma_f32_16x16x32_bf16), over a K range of
// K / k_splits.  64-k stages (128-byte rows, 8-row direct-to-LDS loads: whole lines) in a ring
// of S slots (4 at XR = 64: 64 KiB, two workgroups a CU; 3 at 128): stage k + S - 1 is issued at
// k-step k, so S - 1 stages are in flight per workgroup.  The weight rows are read once per
// launch and loaded nontemporal (cache policy nt, as the GEMV's); measured 3-5% faster per
// 17-64-token prefill (1-1.5% at 100-128) than the default policy, which the X rows, re-read by
// every tile, keep.
// One barrier per k-step: after it, every wave's loads of stage k have landed and every wave is
// done with slot (k - 1) % S, which takes stage k + S - 1.
// Epilogues: fp32 partial planes (split K, reduced by the split reductions), bf16, residual,
// and SwiGLU over [32 gate | 32 up] W rows (output columns 32 t ..), through an fp32 LDS tile.
// The X rows are re-read by every W tile from L2 (one K range: XR x K / k_splits x 2 bytes).
namespace mid {

using pp::f32x4_t;

template <int XR_, int WR_>
struct MC {
  static constexpr int XR = XR_, WR = WR_;
  static constexpr int NWV = WR / 16;                // waves, 16 W rows each
  static constexpr int NB = XR / 16;                 // X blocks per wave
  static constexpr int W_CHUNKS = WR * 8, X_CHUNKS = XR * 8;
  static constexpr int STAGE = W_CHUNKS + X_CHUNKS;  // 16-byte chunks per stage
  static constexpr int S = XR == 64 ? 4 : 3;         // ring slots
  static constexpr int WL = WR / 8 / NWV, XL = XR / 8 / NWV;  // 8-row loads per wave per stage
  static constexpr int L = WL + XL;
  static constexpr int U = WR / 4;                   // 16-byte units of an fp32 output row
  static_assert(XR == 64 || XR == 128, "X rows per tile");
  static_assert(WR == 64 || WR == 128, "W rows per tile");
  static_assert(S * STAGE * 16 <= 160 * 1024, "LDS");
};

// This wave's loads of stage kt into ring slot `slot`: W groups wv + NWV j, then X groups.
template <class C>
__device__ __forceinline__ void mid_issue(u32x4_t* lds, const __amdgpu_buffer_rsrc_t* rs,
                                          uint32_t vo, int wv, int slot, int kt) {
  const uint32_t koff = (uint32_t)(kt * 128);
#pragma unroll
  for (int j = 0; j < C::WL; ++j) {  // weight rows: nontemporal (aux 2 = nt)
    const int dst = slot * C::STAGE + (wv + C::NWV * j) * 64;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs[j], (lds_void*)&lds[dst], 16, vo, koff, 0, 2);
  }
#pragma unroll
  for (int j = C::WL; j < C::L; ++j) {  // X rows: default policy
    const int dst = slot * C::STAGE + C::W_CHUNKS + (wv + C::NWV * (j - C::WL)) * 64;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs[j], (lds_void*)&lds[dst], 16, vo, koff, 0, 0);
  }
}

// s_waitcnt vmcnt(n * L): n younger stages may stay in flight (n <= 6).
template <int L>
__device__ __forceinline__ void mid_wait(int n) {
  switch (n) {
    case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * L) : "memory"); break;
    case 3: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * L) : "memory"); break;
    case 4: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * L) : "memory"); break;
    case 5: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(5 * L) : "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(6 * L) : "memory"); break;
  }
}

template <int EPI, int XR, int WR>
__global__ __launch_bounds__(WR * 4) void gemm_mid_kernel(GemmParams p, int n_tiles) {
  using C = MC<XR, WR>;
  constexpr int U = C::U;
  constexpr int NB = C::NB, S = C::S;
  static_assert(EPI == kGemmF32 || EPI == kGemmBf16 || EPI == kGemmResid || EPI == kGemmSwiglu,
                "epilogues");
  __shared__ u32x4_t lds[S * C::STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nsplit = max(1, p.k_splits);
  const int split = blockIdx.x / n_tiles, ntile = blockIdx.x - split * n_tiles;
  const int KT = p.K / 64 / nsplit;
  const int k0 = split * KT * 64;

  // loads: W groups g = wv + NWV j of 8 rows, X groups likewise; row 8 g + r has
  // swz = (4 (g & 1) + r / 2) & 7 with g & 1 = wv & 1, so one lane offset serves every group
  __amdgpu_buffer_rsrc_t rs[C::L];
#pragma unroll
  for (int j = 0; j < C::WL; ++j) rs[j] = w_group<EPI, WR>(p, ntile, (wv + C::NWV * j) * 8, k0);
#pragma unroll
  for (int j = 0; j < C::XL; ++j) rs[C::WL + j] = x_group(p, 0, (wv + C::NWV * j) * 8, k0);
  const int rl = lane >> 3;
  const uint32_t vo =
      (uint32_t)((rl * p.K + (((lane & 7) ^ ((4 * (wv & 1) + (rl >> 1)) & 7)) * 8)) * 2);

  // fragments: lane l reads row l % 16 of its block at chunk (l / 16 + 4 ks) ^ ((row >> 1) & 7)
  const int fr = lane & 15, fq = lane >> 4;
  const uint32_t sw0 = (uint32_t)((fq ^ ((fr >> 1) & 7)) * 16);
  const uint32_t aA = (uint32_t)((wv * 16 + fr) * 128) + sw0;
  const uint32_t aB = (uint32_t)(C::W_CHUNKS * 16 + fr * 128) + sw0;

  f32x4_t acc[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int t = 0; t < S - 1; ++t)
    if (t < KT) mid_issue<C>(lds, rs, vo, wv, t, t);
  const char* base = reinterpret_cast<const char*>(lds);
  int slot = 0;
#pragma unroll 1
  for (int k = 0; k < KT; ++k) {
    // stage k has landed (stages k+1 .. min(k+S-2, KT-1) may stay in flight) for every wave
    mid_wait<C::L>(min(S - 2, KT - 1 - k));
    asm volatile("s_barrier" ::: "memory");
    if (k + S - 1 < KT) mid_issue<C>(lds, rs, vo, wv, slot == 0 ? S - 1 : slot - 1, k + S - 1);
    uint32_t ra = (uint32_t)(slot * C::STAGE * 16) + aA, rb = (uint32_t)(slot * C::STAGE * 16) + aB;
    asm volatile("" : "+v"(ra), "+v"(rb));
    bf16x8_t fa[2], fb[2][NB];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      fa[ks] = *reinterpret_cast<const bf16x8_t*>(base + (ra ^ (uint32_t)(ks << 6)));
#pragma unroll
      for (int j = 0; j < NB; ++j)
        fb[ks][j] = *reinterpret_cast<const bf16x8_t*>(base + (rb ^ (uint32_t)(ks << 6)) + j * 2048);
    }
    // all of the step's reads issued before its first MFMA (left alone, the scheduler puts each
    // read just before its use: one LDS round trip per MFMA)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[ks], fb[ks][j], acc[j], 0, 0, 0);
    slot = slot == S - 1 ? 0 : slot + 1;
  }

  // epilogue: acc[j][r] = D[W col 16 wv + 4 (lane / 16) + r][X row 16 j + lane % 16], staged as
  // an fp32 [XR][WR] tile (row m at WR m floats, 16-byte unit u at u ^ (m % U))
  float4* ot = reinterpret_cast<float4*>(lds);
  constexpr int T = 64 * C::NWV;
  const auto at = [&](int m, int u) -> float4& { return ot[m * U + (u ^ (m & (U - 1)))]; };
  __syncthreads();  // every wave is done with the ring (its last wait was vmcnt(0))
#pragma unroll
  for (int j = 0; j < NB; ++j)
    at(16 * j + fr, 4 * wv + fq) = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
  __syncthreads();
  if constexpr (EPI == kGemmF32) {
    float* const yf = p.yf + (size_t)split * p.M * p.ldy;
    for (int it = tid; it < XR * U; it += T) {
      const int m = it / U, u = it % U, n = ntile * WR + 4 * u;
      if (m < p.M && n < p.N) *reinterpret_cast<float4*>(yf + (size_t)m * p.ldy + n) = at(m, u);
    }
  } else if constexpr (EPI == kGemmSwiglu) {
    // W rows [32 gate | 32 up] x (WR / 64): tile columns 64 b .. 64 b + 31 are the gate of output
    // columns ntile WR / 2 + 32 b + c, 64 b + 32 .. the up of the same
    constexpr int CPR = WR / 16;  // 8-column output groups per row
    for (int it = tid; it < XR * CPR; it += T) {
      const int m = it / CPR, c = it % CPR, b = c >> 2, c8 = c & 3;
      const int n = ntile * (WR / 2) + 32 * b + 8 * c8;
      if (m >= p.M || n >= p.N) continue;
      uint32_t o[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float4 g = at(m, 16 * b + 2 * c8 + h);
        const float4 up = at(m, 16 * b + 8 + 2 * c8 + h);
        const float gv[4] = {g.x, g.y, g.z, g.w}, uv[4] = {up.x, up.y, up.z, up.w};
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float gt = bf2f(f2bf(gv[e])), ut = bf2f(f2bf(uv[e]));
          v[e] = gt * (1.0f / (1.0f + expf(-gt))) * ut;
        }
        o[2 * h] = pack_bf2(v[0], v[1]);
        o[2 * h + 1] = pack_bf2(v[2], v[3]);
      }
      *reinterpret_cast<uint4*>(p.y + (size_t)m * p.ldy + n) = make_uint4(o[0], o[1], o[2], o[3]);
    }
  } else {
    constexpr int CPR = WR / 8;  // 8-column groups per row
    for (int it = tid; it < XR * CPR; it += T) {
      const int m = it / CPR, c8 = it % CPR, n = ntile * WR + 8 * c8;
      if (m >= p.M || n >= p.N) continue;
      const float4 a = at(m, 2 * c8), b = at(m, 2 * c8 + 1);
      uint4 o = make_uint4(pack_bf2(a.x, a.y), pack_bf2(a.z, a.w), pack_bf2(b.x, b.y), pack_bf2(b.z, b.w));
      uint16_t* dst = p.y + (size_t)m * p.ldy + n;
      if constexpr (EPI == kGemmResid) {
        // y = bf16(y + bf16(acc)) (residual_add.cu:17-19)
        const uint4 r = *reinterpret_cast<const uint4*>(dst);
        o = make_uint4(pack_bf2(bf_lo(r.x) + bf_lo(o.x), bf_hi(r.x) + bf_hi(o.x)),
                       pack_bf2(bf_lo(r.y) + bf_lo(o.y), bf_hi(r.y) + bf_hi(o.y)),
                       pack_bf2(bf_lo(r.z) + bf_lo(o.z), bf_hi(r.z) + bf_hi(o.z)),
                       pack_bf2(bf_lo(r.w) + bf_lo(o.w), bf_hi(r.w) + bf_hi(o.w)));
      }
      *reinterpret_cast<uint4*>(dst) = o;
    }
  }
}

}  // namespace mid

}  // namespace wide

template <int EPI>
int launch_wide(const GemmParams& p, hipStream_t st) {
  const int m_tiles = (p.M + wide::C::BM - 1) / wide::C::BM;
  const int n_tiles = (EPI == kGemmSwiglu) ? (p.N + 127) / 128 : (p.N + wide::C::BN - 1) / wide::C::BN;
  const long long blocks = (long long)m_tiles * n_tiles * std::max(1, p.k_splits);
  IE_REQUIRE(blocks <= 0x7fffffff, "gemm: too many tiles");
  hipLaunchKernelGGL((wide::gemm_wide_kernel<EPI>), dim3((unsigned)blocks), dim3(wide::C::THREADS),
                     0, st, p, m_tiles);
  IE_CHECK_LAUNCH();
  return IE_OK;
}

template <int EPI, int WBN, int XBM = 256, int NW = 3, int WX = 4>
int launch_pp(const GemmParams& p, hipStream_t st) {
  const int m_tiles = (p.M + XBM - 1) / XBM;
  const int n_tiles = (EPI == kGemmSwiglu) ? (p.N + WBN / 2 - 1) / (WBN / 2) : (p.N + WBN - 1) / WBN;
  const long long blocks = (long long)m_tiles * n_tiles * (EPI == kGemmF32 ? p.k_splits : 1);
  IE_REQUIRE(blocks <= 0x7fffffff && (EPI == kGemmF32 ? p.k_splits >= 1 && p.K / 64 % p.k_splits == 0
                                                      : p.k_splits <= 1),
             "gemm: ping-pong tiles");
  hipLaunchKernelGGL((wide::pp::gemm_pp_kernel<EPI, WBN, XBM, NW, WX>), dim3((unsigned)blocks),
                     dim3(512), 0, st, p, m_tiles);
  IE_CHECK_LAUNCH();
  return IE_OK;
}

template <int EPI>
int launch_pp_dual(const GemmParams& head, const GemmParams& tail, hipStream_t st) {
  const int m1 = (head.M + 255) / 256, m2 = (tail.M + 127) / 128;
  const int n1 = (EPI == kGemmSwiglu) ? (head.N + 127) / 128 : (head.N + 255) / 256;
  const int n2 = (EPI == kGemmSwiglu) ? (tail.N + 127) / 128 : (tail.N + 255) / 256;
  const long long b1 = (long long)m1 * n1, b2 = (long long)m2 * n2;
  IE_REQUIRE(b1 + b2 <= 0x7fffffff && head.k_splits <= 1 && tail.k_splits <= 1,
             "gemm: ping-pong tiles");
  hipLaunchKernelGGL((wide::pp::gemm_pp_dual_kernel<EPI>), dim3((unsigned)(b1 + b2)),
                     dim3(512), 0, st, head, m1, (int)b1, tail, m2);
  IE_CHECK_LAUNCH();
  return IE_OK;
}

template <int EPI>
int launch_e(const GemmParams& p, hipStream_t st) {
  const int m_tiles = (p.M + BM - 1) / BM;
  const int n_tiles = (EPI == kGemmSwiglu) ? (p.N + 63) / 64 : (p.N + BN - 1) / BN;
  const long long blocks = (long long)m_tiles * n_tiles;
  IE_REQUIRE(blocks <= 0x7fffffff, "gemm: too many tiles");
  hipLaunchKernelGGL((gemm_kernel<EPI>), dim3((unsigned)blocks), dim3(256), 0, st, p, m_tiles);
  IE_CHECK_LAUNCH();
  return IE_OK;
}

// ---------------------------------------------------------------------------
// Tile shapes of the ping-pong kernel: W rows x X rows, waves of a group along X, and the time of
// one 64-k step of one tile in us (below).  SwiGLU needs waves of whole [32 gate | 32 up] groups;
// 192 W rows are 96 RoPE pairs (the fused QKV epilogue).
struct TileKind {
  int bn, bm, wx;
  double step;
};
constexpr TileKind kTiles[] = {
    {128, 128, 4, 0.535}, {128, 160, 2, 0.606}, {128, 192, 4, 0.661}, {128, 224, 2, 0.742},
    {128, 256, 4, 0.828}, {256, 160, 2, 0.995}, {256, 192, 2, 1.127}, {256, 224, 2, 1.277},
    {256, 256, 2, 1.431}, {192, 128, 4, 0.738}, {192, 192, 4, 0.921}, {192, 256, 4, 1.135},
};
constexpr int kTileKinds = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kTileBig = 8, kTileRope0 = 9, kTileRopeBig = 11;
constexpr double kStep256x128 = 0.85;  // the dual launch's tail tile

// Kernel of the tiles past 128 rows: 0 = the DMA-ring kernel; 1 = the ping-pong kernel for the
// 256-row X tiles; 2 (default) = the ping-pong kernel; 3 = as 2 with 4 W ring slots (2 X slots) on
// the 192 x 256 tiles.  Outputs are bit-identical across all: the same K splits, and the same MFMA
// order in every accumulator whatever the tile.
int g_gemm_schedule = 2;

// A product's tile shape and K splits by the least modelled time.
struct TilePlan {
  int kind = -1, splits = 1;
  double us = 1e30;
};

// QKV projection as a product of its own or fused: its unsplit tiles are the 192-row ones, so that
// both forms take the same plan (and give the same bits).
bool rope_product(int epi, const GemmParams& p) {
  return epi == kGemmQkvRope || (epi == kGemmBf16 && p.n0 < p.N);
}

// Time of one tile with kt k-steps, `wgs` workgroups in the launch (or of one round of it).
double tile_us(int bn, int bm, double step, double kt, double wgs) {
  const double idle = wgs < 256 ? 1 - wgs / 256 : 0;
  return kt * step * (1 - 0.28 * idle) + 3.95 + 4.18 * bn * bm / 65536;
}

// Model (us), fitted to 78 measured shapes (the four layer products at 130 .. 6000 rows, weights
// from HBM, tile shapes x K splits).  Against 1069 timings of the four products at 16 row counts it is
// 6.7% rms off, and the shape that it picks is 1.4% off the best timed one on average (15% at most
// but for down at 130 rows, 37%):
//   launch 1.4 + rounds x (k-steps x step + 3.95 + 4.18 x tile / 64 Ki)
// a step 28% faster on an empty chip than on a full one; past one round 0.71 of the time goes
// with whole rounds, 0.29 with the tiles; K splits add 3.2 + 0.245 per MB of fp32 partials; the
// weights stream at 3.5 TB/s at best beside the products.  The RMSNorm that follows a layer's residual
// product counts too where it is a launch of its own (unsplit; the split reduction runs it).
// Before, tiles were 256 x 256, 256 x 128 or 192 x 256 (and 128 x 128 with an older kernel), K
// split up to 1024 rows only: 640 rows 201 -> 134 us (gate/up), 117 -> 77 (down), 1200 rows down
// 189 -> 125, 6000 rows down 661 -> 551.
TilePlan plan_tiles(int epi, const GemmParams& p) {
  const bool sw = epi == kGemmSwiglu, rope = rope_product(epi, p);
  const int kt = p.K / 64;
  // SwiGLU: unsplit a tile's W rows are half gate, half up; split it is a plain product of 2N columns
  const int cols = sw ? 2 * p.N : p.N;
  const bool can_split =
      p.split_ws && epi != kGemmF32 && p.N % (sw ? 16 : 8) == 0 && p.ldy % 8 == 0;
  const double plane = (double)p.M * cols * 4;
  const double weights = (double)cols * p.K * 2 / 3.5e6;
  TilePlan best;
  for (int k = 0; k < kTileKinds; ++k) {
    const TileKind& t = kTiles[k];
    // (192 W rows: the fused QKV's; a plain bf16 product of one round may take them too, 2048 x 4096 x
    // 6144 at 85.8 us against 89.3 -- past one round the model is too coarse to tell them apart)
    if (t.bn == 192 && !rope && epi != kGemmBf16) continue;
    const long long m_tiles = (p.M + t.bm - 1) / t.bm;
    for (int s = 1; s <= 16; ++s) {
      const bool split = s > 1;
      const int width = sw && !split ? t.bn / 2 : t.bn;
      const long long tiles = m_tiles * (((split ? cols : p.N) + width - 1) / width);
      if (split ? !can_split || kt % s != 0 || tiles * s > 512 || t.bn == 192 ||
                      s * plane > (double)p.split_ws_bytes
                : (rope && t.bn != 192) || (!rope && t.bn == 192 && tiles > 256) ||
                      (sw && (t.bn / 2 * t.wx / 4) % 64 != 0))
        continue;
      const double wgs = (double)tiles * s;
      const double rounds = wgs <= 256 ? 1 : 0.71 * ((tiles * s + 255) / 256) + 0.29 * wgs / 256;
      double us = std::max(rounds * tile_us(t.bn, t.bm, t.step, (double)kt / s, wgs), weights) + 1.4;
      if (split) us += 3.2 + 0.245e-6 * s * plane;
      else if (p.norm_follows) us += 2 + 0.0021 * p.M;
      if (us < best.us) best = {k, s, us};
    }
  }
  return best;
}

// The plan's product by the schedule's kernel (kGemmF32: p.k_splits partial planes).
template <int EPI>
int launch_kind(int kind, const GemmParams& p, hipStream_t st) {
  if (g_gemm_schedule == 0 || (g_gemm_schedule == 1 && kTiles[kind].bm != 256)) {
    if constexpr (EPI != kGemmQkvRope) return launch_wide<EPI>(p, st);
  }
  constexpr bool sw = EPI == kGemmSwiglu;
  if constexpr (EPI == kGemmBf16 || EPI == kGemmQkvRope) {
    switch (kind) {
      case kTileRope0: return launch_pp<EPI, 192, 128>(p, st);
      case kTileRope0 + 1: return launch_pp<EPI, 192, 192>(p, st);
      case kTileRopeBig:
        return g_gemm_schedule == 3 ? launch_pp<EPI, 192, 256, 4>(p, st) : launch_pp<EPI, 192, 256>(p, st);
    }
  }
  if constexpr (EPI != kGemmQkvRope) {
    switch (kind) {
      case 0: return launch_pp<EPI, 128, 128>(p, st);
      case 1: if constexpr (!sw) return launch_pp<EPI, 128, 160, 3, 2>(p, st); break;
      case 2: return launch_pp<EPI, 128, 192>(p, st);
      case 3: if constexpr (!sw) return launch_pp<EPI, 128, 224, 3, 2>(p, st); break;
      case 4: return launch_pp<EPI, 128, 256>(p, st);
      case 5: return launch_pp<EPI, 256, 160, 3, 2>(p, st);
      case 6: return launch_pp<EPI, 256, 192, 3, 2>(p, st);
      case 7: return launch_pp<EPI, 256, 224, 3, 2>(p, st);
      case kTileBig: return launch_pp<EPI, 256, 256, 3, 2>(p, st);
    }
  }
  set_error("gemm: tile kind %d for epilogue %d", kind, EPI);
  return IE_ERR_INVALID_ARG;
}

// Output columns [c, N) of p as a GEMM of its own (c a multiple of 64, and of 16 past a
// weight split point).
GemmParams column_tail(int epi, const GemmParams& p, int c) {
  GemmParams q = p;
  const size_t off = (size_t)c * p.K;
  q.N = p.N - c;
  if (p.y) q.y = p.y + c;
  if (p.yf) q.yf = p.yf + c;
  if (epi == kGemmSwiglu) {
    q.w0 = p.w0 + off;
    q.w1 = p.w1 + off;
    return q;
  }
  const int e0 = std::min(p.n0, p.N), e1 = std::min(p.n0 + p.n1, p.N);
  if (c < e0) {
    q.w0 = p.w0 + off;
    q.n0 = e0 - c;
  } else if (c < e1) {
    q.w0 = p.w1 + (size_t)(c - e0) * p.K;
    q.n0 = e1 - c;
    q.w1 = p.w2;
    q.n1 = q.N - q.n0;
  } else {
    q.w0 = p.w2 + (size_t)(c - e1) * p.K;
    q.n0 = q.N;
    q.n1 = 0;
  }
  return q;
}

// The columns past the full rounds of 256 x 256 tiles as 256 x 128 tiles of the same launch, when
// that beats the plan (gate/up at S = 2048: 3 rounds, then the last 2048 columns as one round of the
// smaller tiles, in place of a half-empty fourth round): those columns' count, else 0.
int dual_tail(int epi, const GemmParams& p, double plan_us) {
  const int tn = epi == kGemmSwiglu ? 128 : 256, m_tiles = (p.M + 255) / 256;
  const long long tiles = (long long)m_tiles * ((p.N + tn - 1) / tn);
  if (g_gemm_schedule < 2 || tiles <= 256 || tiles % 256 == 0 || 256 % m_tiles != 0) return 0;
  const int head = (int)(tiles / 256 * 256 / m_tiles) * tn;
  if (head >= p.N) return 0;
  const double kt = p.K / 64;
  const long long tail = (long long)((p.M + 127) / 128) * ((p.N - head + tn - 1) / tn);
  const double us = 1.4 + (double)(tiles / 256) * tile_us(256, 256, kTiles[kTileBig].step, kt, 256) +
                    (double)((tail + 255) / 256) * tile_us(256, 128, kStep256x128, kt, 256) +
                    (p.norm_follows ? 2 + 0.0021 * p.M : 0);
  return us < plan_us ? p.N - head : 0;
}

// Sums over the split planes of the 4 partials at each of C offsets, in plane order, four planes'
// loads in flight at a time (one after the other, each plane's load was a memory latency: layers of
// 17-128 rows, whose QKV, O and down products split 2-8 ways, are level to 1.8% faster in turn, 17
// rows 101.0 -> 99.3 us).
template <int C>
__device__ __forceinline__ void split_sum(const float* src, const size_t (&off)[C], size_t plane,
                                          int splits, float4 (&a)[C]) {
  for (int s0 = 0; s0 < splits; s0 += 4) {
    float4 v[4][C];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s0 + u < splits)
#pragma unroll
        for (int c = 0; c < C; ++c)
          v[u][c] = *reinterpret_cast<const float4*>(src + (s0 + u) * plane + off[c]);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s0 + u < splits)
#pragma unroll
        for (int c = 0; c < C; ++c) {
          if (s0 + u == 0)
            a[c] = v[u][c];
          else
            a[c].x += v[u][c].x, a[c].y += v[u][c].y, a[c].z += v[u][c].z, a[c].w += v[u][c].w;
        }
  }
}

__device__ __forceinline__ float silu_mul(float g, float u) {
  g = bf2f(f2bf(g));
  return g * (1.0f / (1.0f + expf(-g))) * bf2f(f2bf(u));
}

// Split K's reduction: y = epilogue(sum of the fp32 partial planes), 8 columns per thread.
// bf16: bf16(sum); residual: bf16(y + bf16(sum)); SwiGLU (planes of 2N columns, gate then up):
// bf16(silu(bf16(g)) * bf16(u)) -- the unsplit epilogues' roundings.
template <int EPI>
__global__ __launch_bounds__(256) void split_reduce_kernel(const float* part, int splits, int M,
                                                           int N, uint16_t* y, int ldy) {
  constexpr int W = EPI == kGemmSwiglu ? 2 : 1;  // plane width in output columns
  const int per_row = N / 8;
  const size_t total = (size_t)M * per_row, plane = (size_t)M * N * W;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total;
       i += (size_t)gridDim.x * blockDim.x) {
    const int m = (int)(i / per_row), n = (int)(i % per_row) * 8;
    const float* src = part + (size_t)m * N * W + n;
    float4 a, b;
    if constexpr (EPI == kGemmSwiglu) {
      float4 v[4];
      split_sum<4>(src, {0, 4, (size_t)N, (size_t)N + 4}, plane, splits, v);
      a = make_float4(silu_mul(v[0].x, v[2].x), silu_mul(v[0].y, v[2].y), silu_mul(v[0].z, v[2].z), silu_mul(v[0].w, v[2].w));
      b = make_float4(silu_mul(v[1].x, v[3].x), silu_mul(v[1].y, v[3].y), silu_mul(v[1].z, v[3].z), silu_mul(v[1].w, v[3].w));
    } else {
      float4 v[2];
      split_sum<2>(src, {0, 4}, plane, splits, v);
      a = v[0], b = v[1];
    }
    uint4 o = make_uint4(pack_bf2(a.x, a.y), pack_bf2(a.z, a.w), pack_bf2(b.x, b.y), pack_bf2(b.z, b.w));
    uint16_t* dst = y + (size_t)m * ldy + n;
    if constexpr (EPI == kGemmResid) {
      const uint4 r = *reinterpret_cast<const uint4*>(dst);
      o = make_uint4(pack_bf2(bf_lo(r.x) + bf_lo(o.x), bf_hi(r.x) + bf_hi(o.x)),
                     pack_bf2(bf_lo(r.y) + bf_lo(o.y), bf_hi(r.y) + bf_hi(o.y)),
                     pack_bf2(bf_lo(r.z) + bf_lo(o.z), bf_hi(r.z) + bf_hi(o.z)),
                     pack_bf2(bf_lo(r.w) + bf_lo(o.w), bf_hi(r.w) + bf_hi(o.w)));
    }
    *reinterpret_cast<uint4*>(dst) = o;
  }
}

// The residual reduction followed by the RMSNorm of the same rows (N = 4096, one 256-thread
// workgroup per row): y = bf16(y + bf16(sum)), then rn_out = bf16(bf16(y * r) * w) with r from
// the fp32 sum of squares of the new y -- each thread owns 16-byte chunks t and t + 256 of the
// row and sums their squares in the same order as rmsnorm_kernel, so both outputs equal the
// reduction followed by that kernel bit for bit, without writing and re-reading y between them.
__global__ __launch_bounds__(256) void split_reduce_norm_kernel(const float* part, int splits,
                                                                int M, uint16_t* y, int ldy,
                                                                const uint16_t* w,
                                                                uint16_t* out) {
  __shared__ float red[4];
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const size_t plane = (size_t)M * kHidden;
  uint4 v[2], wv[2], rv[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    rv[k] = reinterpret_cast<const uint4*>(y + (size_t)m * ldy)[tid + 256 * k];
    wv[k] = reinterpret_cast<const uint4*>(w)[tid + 256 * k];
  }
  float4 sum[4];
  split_sum<4>(part + (size_t)m * kHidden + tid * 8, {0, 4, 2048, 2052}, plane, splits, sum);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int n = (tid + 256 * k) * 8;
    const float4 a = sum[2 * k], b = sum[2 * k + 1];
    const uint4 o = make_uint4(pack_bf2(a.x, a.y), pack_bf2(a.z, a.w), pack_bf2(b.x, b.y),
                               pack_bf2(b.z, b.w));
    uint16_t* dst = y + (size_t)m * ldy + n;
    const uint4 r = rv[k];
    v[k] = make_uint4(pack_bf2(bf_lo(r.x) + bf_lo(o.x), bf_hi(r.x) + bf_hi(o.x)),
                      pack_bf2(bf_lo(r.y) + bf_lo(o.y), bf_hi(r.y) + bf_hi(o.y)),
                      pack_bf2(bf_lo(r.z) + bf_lo(o.z), bf_hi(r.z) + bf_hi(o.z)),
                      pack_bf2(bf_lo(r.w) + bf_lo(o.w), bf_hi(r.w) + bf_hi(o.w)));
    *reinterpret_cast<uint4*>(dst) = v[k];
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t e[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ss = fmaf(bf_lo(e[q]), bf_lo(e[q]), ss);
      ss = fmaf(bf_hi(e[q]), bf_hi(e[q]), ss);
    }
  }
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  const float rr = rsqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)kHidden + kRmsEps);
  uint4* o4 = reinterpret_cast<uint4*>(out + (size_t)m * kHidden);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t e[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
    const uint32_t f[4] = {wv[k].x, wv[k].y, wv[k].z, wv[k].w};
    uint32_t o[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float lo = bf2f(f2bf(bf_lo(e[q]) * rr)) * bf_lo(f[q]);
      const float hi = bf2f(f2bf(bf_hi(e[q]) * rr)) * bf_hi(f[q]);
      o[q] = pack_bf2(lo, hi);
    }
    o4[tid + 256 * k] = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// The QKV reduction with RoPE and the K/V scatter (prefill, kGemmQkvRope): each thread sums 4
// RoPE pairs of one row (dims j..j+3 and j+64..j+67 of one head of [q|k|v]) over the split
// planes in plane order, rounds to bf16 (the bf16 reduction's values), rotates q and k with the
// scatter kernel's arithmetic at position start_pos + m, and stores q to y [M][32][128], k and v
// to the cache (or its pages).
__global__ __launch_bounds__(256) void split_reduce_rope_kernel(const float* part, int splits,
                                                                GemmParams p) {
  constexpr int kQuads = (kQHeads + 2 * kKVHeads) * 16;  // 4-pair groups per row
  const size_t plane = (size_t)p.M * kQKVDim;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < (size_t)p.M * kQuads;
       i += (size_t)gridDim.x * blockDim.x) {
    const int m = (int)(i / kQuads), qd = (int)(i % kQuads);
    const int head = qd >> 4, j = (qd & 15) * 4;
    const float* src = part + (size_t)m * kQKVDim + head * kHeadDim + j;
    const int pos = p.start_pos + m;
    // (V heads take no rotation; their table entries are loaded and unused)
    float cs[4], sn[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      cs[e] = p.rope_cos[(size_t)pos * 64 + j + e];
      sn[e] = p.rope_sin[(size_t)pos * 64 + j + e];
    }
    float4 sum[2];
    split_sum<2>(src, {0, 64}, plane, splits, sum);
    const float4 a = sum[0], b = sum[1];
    const float av[4] = {bf2f(f2bf(a.x)), bf2f(f2bf(a.y)), bf2f(f2bf(a.z)), bf2f(f2bf(a.w))};
    const float bv[4] = {bf2f(f2bf(b.x)), bf2f(f2bf(b.y)), bf2f(f2bf(b.z)), bf2f(f2bf(b.w))};
    float lo[4], hi[4];
    if (head < kQHeads + kKVHeads) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = rope_lo(av[e], bv[e], cs[e], sn[e]);
        hi[e] = rope_hi(av[e], bv[e], cs[e], sn[e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) lo[e] = av[e], hi[e] = bv[e];
    }
    uint16_t* dst;
    if (head < kQHeads) {
      dst = p.y + ((size_t)m * kQHeads + head) * kHeadDim;
    } else {
      const bool is_k = head < kQHeads + kKVHeads;
      const int kvh = head - kQHeads - (is_k ? 0 : kKVHeads);
      uint16_t* const plane_kv = is_k ? p.k_cache : p.v_cache;
      if (p.block_table) {  // paged: row pos % kPagePos of the page holding block pos / kPagePos
        const int page = p.block_table[pos / kPagePos];
        if (page < 0 || page >= p.n_pages) continue;
        dst = plane_kv + (size_t)page * kPageElems + ((size_t)kvh * kPagePos + pos % kPagePos) * kHeadDim;
      } else {
        dst = plane_kv + ((size_t)kvh * kMaxCtx + pos) * kHeadDim;
      }
    }
    *reinterpret_cast<uint2*>(dst + j) = make_uint2(pack_bf2(lo[0], lo[1]), pack_bf2(lo[2], lo[3]));
    *reinterpret_cast<uint2*>(dst + j + 64) = make_uint2(pack_bf2(hi[0], hi[1]), pack_bf2(hi[2], hi[3]));
  }
}

// The reduction of a split product: p.split_ws holds `splits` fp32 planes of M x NP (NP = 2N
// for SwiGLU: gate then up), y = epilogue(sum) -- RoPE and the K/V scatter, residual + RMSNorm
// (p.rn_out), residual, SwiGLU or bf16.
int launch_split_reduce(int epi, const GemmParams& p, int splits, hipStream_t st) {
  const bool sw = epi == kGemmSwiglu, rope = epi == kGemmQkvRope;
  const size_t total = (size_t)p.M * p.N / 8;
  const int blocks = (int)std::min<size_t>((total + 255) / 256, 2048);
  if (sw) {
    hipLaunchKernelGGL(split_reduce_kernel<kGemmSwiglu>, dim3(blocks), dim3(256), 0, st,
                       p.split_ws, splits, p.M, p.N, p.y, p.ldy);
  } else if (rope) {
    const size_t items = (size_t)p.M * (kQHeads + 2 * kKVHeads) * 16;
    hipLaunchKernelGGL(split_reduce_rope_kernel, dim3((unsigned)std::min<size_t>((items + 255) / 256, 2048)),
                       dim3(256), 0, st, p.split_ws, splits, p);
  } else if (epi == kGemmResid && p.rn_out) {
    hipLaunchKernelGGL(split_reduce_norm_kernel, dim3(p.M), dim3(256), 0, st, p.split_ws, splits,
                       p.M, p.y, p.ldy, p.rn_w, p.rn_out);
    if (p.rn_done) *p.rn_done = 1;
  } else if (epi == kGemmResid) {
    hipLaunchKernelGGL(split_reduce_kernel<kGemmResid>, dim3(blocks), dim3(256), 0, st,
                       p.split_ws, splits, p.M, p.N, p.y, p.ldy);
  } else {
    hipLaunchKernelGGL(split_reduce_kernel<kGemmBf16>, dim3(blocks), dim3(256), 0, st,
                       p.split_ws, splits, p.M, p.N, p.y, p.ldy);
  }
  IE_CHECK_LAUNCH();
  return IE_OK;
}

// The tiled product of any M: the plan's tiles, K split into fp32 planes summed by the reduction
// that applies the epilogue, or unsplit.  p's operands 16-byte aligned.
int launch_tiled(int epi, const GemmParams& p, hipStream_t st) {
  const TilePlan plan = plan_tiles(epi, p);
  IE_REQUIRE(plan.kind >= 0, "gemm: no tile shape for epilogue %d", epi);
  if (plan.splits > 1) {
    GemmParams q = p;
    q.yf = p.split_ws;
    if (epi == kGemmSwiglu) {
      q.N = 2 * p.N;  // rows [0, N) of w0 (gate), then [N, 2N) of w1 (up)
      q.n0 = p.N;
      q.n1 = p.N;
    }
    q.ldy = q.N;
    q.k_splits = plan.splits;
    IE_TRY(launch_kind<kGemmF32>(plan.kind, q, st));
    return launch_split_reduce(epi, p, plan.splits, st);
  }
  if (epi == kGemmBf16 || epi == kGemmResid || epi == kGemmSwiglu) {
    const int tail = rope_product(epi, p) ? 0 : dual_tail(epi, p, plan.us);
    if (tail > 0) {
      GemmParams head = p;
      head.N = p.N - tail;
      const GemmParams rest = column_tail(epi, p, head.N);
      switch (epi) {
        case kGemmBf16: return launch_pp_dual<kGemmBf16>(head, rest, st);
        case kGemmResid: return launch_pp_dual<kGemmResid>(head, rest, st);
        default: return launch_pp_dual<kGemmSwiglu>(head, rest, st);
      }
    }
  }
  GemmParams q = p;
  q.k_splits = 1;
  switch (epi) {
    case kGemmBf16: return launch_kind<kGemmBf16>(plan.kind, q, st);
    case kGemmResid: return launch_kind<kGemmResid>(plan.kind, q, st);
    case kGemmF32: return launch_kind<kGemmF32>(plan.kind, q, st);
    case kGemmSwiglu: return launch_kind<kGemmSwiglu>(plan.kind, q, st);
    case kGemmQkvRope: return launch_kind<kGemmQkvRope>(plan.kind, q, st);
  }
  set_error("gemm: bad epilogue %d", epi);
  return IE_ERR_INVALID_ARG;
}

// Direct-to-LDS loads move 16 bytes: the bases (rows are K x 2 bytes apart, K a multiple of 64)
// must be 16-byte aligned; other operands take the register-staged 128 x 128 kernel.
bool operands_aligned(const GemmParams& p) {
  const auto a16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
  return a16(p.x) && a16(p.w0) && a16(p.w1) && a16(p.w2) && a16(p.yf);
}

// Medium M (16 < M <= 128, K a multiple of 64): the 64-W-row streaming kernel, with its fp32
// partials reduced by the split reductions, or (gate/up and products of many tiles) unsplit
// with the epilogue in the kernel.  1: not applicable.
int launch_mid(int epi, const GemmParams& p, hipStream_t st) {
  if (g_gemm_schedule < 2 || p.M <= 16 || p.M > 128 || p.K % 64 != 0 || p.K < 64 ||
      p.N % 8 != 0 || p.ldy % 8 != 0 || epi == kGemmF32)
    return 1;
  const bool sw = epi == kGemmSwiglu, rope = epi == kGemmQkvRope;
  const int kt = p.K / 64;
  const bool x128 = p.M > 64;
  // 65-128 rows: SwiGLU over 64-column tiles (128 W rows, 8 waves: each tile re-reads the X
  // rows from L2 for twice the weight rows), when they alone fill most of the chip (in situ at
  // 100 and 128 rows 2.6% and 3.7% faster per prefill than 32-column tiles; at 64 rows and
  // fewer, level or slower)
  if (sw && x128 && p.N % 64 == 0 && p.N / 64 >= 192) {
    const int n_tiles = p.N / 64;
    GemmParams q = p;
    q.k_splits = 1;
    hipLaunchKernelGGL((wide::mid::gemm_mid_kernel<kGemmSwiglu, 128, 128>), dim3(n_tiles), dim3(512), 0,
                       st, q, n_tiles);
    IE_CHECK_LAUNCH();
    return IE_OK;
  }
  // unsplit: SwiGLU over 32-column tiles, bf16 / residual over 64-column tiles, once the tiles
  // alone fill most of the chip
  if (!rope && !p.rn_out && (sw ? p.N / 32 : (p.N + 63) / 64) >= 192 && (!sw || p.N % 32 == 0)) {
    const int n_tiles = sw ? p.N / 32 : (p.N + 63) / 64;
    GemmParams q = p;
    q.k_splits = 1;
#define IE_MID(E, XR, G) \
  hipLaunchKernelGGL((wide::mid::gemm_mid_kernel<E, XR, 64>), dim3(G), dim3(256), 0, st, q, n_tiles)
    switch (epi) {
      case kGemmSwiglu: if (x128) IE_MID(kGemmSwiglu, 128, n_tiles); else IE_MID(kGemmSwiglu, 64, n_tiles); break;
      case kGemmResid: if (x128) IE_MID(kGemmResid, 128, n_tiles); else IE_MID(kGemmResid, 64, n_tiles); break;
      default: if (x128) IE_MID(kGemmBf16, 128, n_tiles); else IE_MID(kGemmBf16, 64, n_tiles); break;
    }
    IE_CHECK_LAUNCH();
    return IE_OK;
  }
  if (!p.split_ws) return 1;
  // split K over fp32 planes of NP columns (SwiGLU: gate rows then up rows)
  const int NP = sw ? 2 * p.N : p.N;
  const int n_tiles = (NP + 63) / 64;
  const size_t plane = (size_t)p.M * NP * sizeof(float);
  int splits = 1;
  for (int sp = 2; sp <= 16; ++sp)
    if (kt % sp == 0 && (long long)n_tiles * sp <= 256 && (size_t)sp * plane <= (size_t)p.split_ws_bytes)
      splits = sp;
  if (splits < 2 && n_tiles < 128) return 1;
  GemmParams q = p;
  q.yf = p.split_ws;
  q.ldy = NP;
  q.k_splits = splits;
  if (sw) {
    q.N = NP;
    q.n0 = p.N;  // rows [0, N) of w0 (gate), then [N, 2N) of w1 (up)
    q.n1 = p.N;
    q.w2 = p.w1;
  }
  const unsigned blocks = (unsigned)(n_tiles * splits);
  if (x128) IE_MID(kGemmF32, 128, blocks);
  else IE_MID(kGemmF32, 64, blocks);
#undef IE_MID
  IE_CHECK_LAUNCH();
  return launch_split_reduce(epi, p, splits, st);
}

}  // namespace

int launch_gemm(int epi, const GemmParams& p, hipStream_t st) {
  IE_REQUIRE(p.M >= 1 && p.N >= 1 && p.K >= BK, "gemm: bad shape M=%d N=%d K=%d", p.M, p.N, p.K);
  IE_REQUIRE(p.K % BK == 0, "gemm: K=%d must be a multiple of %d", p.K, BK);
  IE_REQUIRE(p.N % 4 == 0, "gemm: N=%d must be a multiple of 4", p.N);
  IE_REQUIRE(p.ldy >= p.N, "gemm: ldy=%d < N=%d", p.ldy, p.N);
  // a 16-row load group must not straddle two weight matrices
  IE_REQUIRE(epi == kGemmSwiglu || ((p.n0 >= p.N || p.n0 % 16 == 0) &&
                                    (p.n0 + p.n1 >= p.N || (p.n0 + p.n1) % 16 == 0)),
             "gemm: weight split points n0=%d n0+n1=%d inside N=%d must be multiples of 16", p.n0,
             p.n0 + p.n1, p.N);
  if (gemm_skinny_fits(p)) return launch_gemm_skinny(epi, p, st);
  if (epi >= kGemmBf16 && epi <= kGemmSwiglu && !p.ss_in && !p.ss_out && p.k_splits <= 1) {
    const int rc = launch_mid(epi, p, st);
    if (rc != 1) return rc;
  }
  if (gemm_skinny_mb_fits(epi, p)) return launch_gemm_skinny_mb(epi, p, st);
  IE_REQUIRE(epi >= kGemmBf16 && epi <= kGemmSwiglu, "gemm: epilogue %d needs M <= 16", epi);
  IE_REQUIRE(!p.ss_in && !p.ss_out, "gemm: the folded RMSNorm needs M <= 16");
  IE_REQUIRE(p.k_splits <= 1, "gemm: k_splits is the launcher's");
  IE_REQUIRE(!p.rn_out || (epi == kGemmResid && p.N == kHidden && p.rn_w),
             "gemm: the fused RMSNorm output follows a residual product of %d columns", kHidden);
  if (!operands_aligned(p)) {
    switch (epi) {
      case kGemmBf16: return launch_e<kGemmBf16>(p, st);
      case kGemmResid: return launch_e<kGemmResid>(p, st);
      case kGemmF32: return launch_e<kGemmF32>(p, st);
      default: return launch_e<kGemmSwiglu>(p, st);
    }
  }
  return launch_tiled(epi, p, st);
}

}  // namespace ie

namespace ie {

int launch_qkv_rope_prefill(const GemmParams& p, hipStream_t st) {
  IE_REQUIRE(p.N == kQKVDim && p.K == kHidden && p.n0 == kHidden && p.n1 == kKVDim && p.y &&
                 p.k_cache && p.v_cache && p.rope_cos && p.rope_sin && !p.d_seq_len &&
                 p.start_pos >= 0,
             "qkv_rope_prefill: the [q|k|v] projection of one sequence");
  if (g_gemm_schedule < 1 || gemm_skinny_fits(p)) return 1;
  {
    const int rc = launch_mid(kGemmQkvRope, p, st);
    if (rc != 1) return rc;
  }
  if (gemm_skinny_mb_fits(kGemmBf16, p)) return 1;
  if (!operands_aligned(p)) return 1;
  return launch_tiled(kGemmQkvRope, p, st);
}

}  // namespace ie

extern "C" int ie_tune_gemm_schedule(int schedule) {
  IE_REQUIRE(schedule >= 0 && schedule <= 3, "tune_gemm_schedule: %d not in [0, 3]", schedule);
  ie::g_gemm_schedule = schedule;
  return IE_OK;
}
