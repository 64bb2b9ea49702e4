// tm_ce_gemm.hip -- gfx950 bf16 MFMA GEMMs of the fused linear + cross-entropy, per chunk of rows
// (torchure/loss/fused_linear_ce.py:38,52,57: bf16 matmuls, fp32 accumulation, bf16 results):
//   logits_ring_kernel   logits = h W^T         (rows x V, K = D), persistent, for dim at least
//                        192 and logits rows a multiple of 8 elements apart; logits_gemm_kernel
//                        otherwise
//   grad_h_gemm_kernel   grad_h = grad_logits W (rows x D, K = V), split over K, reading W as it
//                        is stored (V x D), with
//   splits_reduce_kernel summing the fp32 partials of each element over the splits in a fixed
//                        order (split 0 first) and rounding once to bf16 (RNE), so the result
//                        does not depend on scheduling
//   grad_w_ring_kernel   grad_W = grad_logits^T h (V x D, K = rows), persistent, for rows a
//                        multiple of 128 (>= 256); grad_w_gemm_kernel otherwise
//   gemm_tile_kernel     any of the three where those leave CUs idle: 128 x 128 tiles (256 x 256 for
//                        some grad_h and grad_W), K split where that pays
// A cost model (tile_us, wide_splits, ring_us) chooses.
//
// The others are 256 x 256 output tiles per workgroup. All are on v_mfma_f32_32x32x16_bf16 with fp32
// accumulation: the ring kernels, grad_h_gemm_kernel and gemm_tile_kernel on 8 wave64, two a SIMD
// (each 128 x 64 of a 256 x 256 tile, 128 accumulators), so that one wave's MFMAs run while the
// other waits; the one-tile kernels on 4 wave64 (each 128 x 128, 256 accumulators in the AGPRs).
// Every element sees the same MFMA sequence in the ring, the one-tile and the unsplit small-tile
// kernels. Operands stream
// global -> LDS with direct loads (global_load_lds, 16 bytes a lane) into two stages (64 KB for a
// 256 x 256 tile) of 64-deep K slices. gfx950's LDS has 64 four-byte banks and serves a 16-byte-per-lane read 16
// lanes at a time, so the 16 lanes reading 16 consecutive 128-byte rows must hit 16 different
// 16-byte bank groups: a row's chunk c sits at slot c ^ ((row >> 1) & 7), which gives rows 2j and
// 2j+1 (one even, one odd: the two halves of the banks) the slot pattern c ^ j. (The 32-bank
// pattern c ^ (row & 7) put rows r and r+8 on one bank group and doubled the read time.)
// Workgroup w runs on XCD w % 8; each XCD takes a contiguous range of tiles (or of split-tile
// pairs), so the operand panels its 32 CUs share are read from HBM about once and then served
// from that XCD's L2.
//
// For the reference's default chunk of 1024 rows, grad_h is a long-K GEMM (K = V = 151,936 for
// the Qwen3 head) with a small output (1024 x 1024): 16 tiles for 256 CUs, which the library GEMM
// ran at about 450 TFLOP/s. Splitting K gives every CU a (split, tile) pair.

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <mutex>

#include "torchure_amd.h"
#include "tm_internal.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

template <typename... A>
int gemm_fail(int code, const char* fmt, A... args) {
  return tm_internal_fail(code, fmt, args...);
}

constexpr int kTile = 256;      // output tile edge (rows and columns)
constexpr int kSliceK = 64;     // K depth of one LDS stage (128 bytes of bf16 per row)

// s_waitcnt immediate that waits for vmcnt <= n only (gfx9 encoding: vmcnt bits 3:0 and
// 15:14; expcnt and lgkmcnt at their maxima, so they are not waited for).
constexpr int waitcnt_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

__device__ __forceinline__ uint32_t rne_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  const uint32_t r = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
  return (f != f) ? 0x7FC0u : r;
}

// out[i] = bf16(((P[0][i] + P[1][i]) + P[2][i]) + ...), four elements per thread, eight splits'
// loads in flight (one at a time, a small output's 32 splits took 11 us of latency).
__global__ __launch_bounds__(256) void splits_reduce_kernel(const float* __restrict__ partials,
                                                            uint16_t* __restrict__ out, int64_t n, int splits) {
  const int64_t e = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (e >= n) return;
  f32x4 sum = *(const f32x4*)(partials + e);
  for (int s0 = 1; s0 < splits; s0 += 8) {
    f32x4 p[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < splits) p[u] = *(const f32x4*)(partials + static_cast<int64_t>(s0 + u) * n + e);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (s0 + u >= splits) break;
      sum.x = sum.x + p[u].x;
      sum.y = sum.y + p[u].y;
      sum.z = sum.z + p[u].z;
      sum.w = sum.w + p[u].w;
    }
  }
  u32x2 o;
  o.x = rne_bf16(sum.x) | (rne_bf16(sum.y) << 16);
  o.y = rne_bf16(sum.z) | (rne_bf16(sum.w) << 16);
  *(u32x2*)(out + e) = o;
}

// ------------------------------------------------------------------ logits = hidden @ W^T
//
// fused_linear_ce.py:38 `logits = h @ w.t()` per chunk: C (rows x vocab) = A (rows x dim) times
// B (vocab x dim) transposed, both operands K-contiguous (K = dim), bf16 in and out, fp32
// accumulation. A 256 x 256 output tile per workgroup of 4 wave64 (2 x 2), each wave 128 x 128
// with 256 fp32 accumulators (the AGPRs) on v_mfma_f32_32x32x16_bf16. Operands stream
// global -> LDS (global_load_lds, 16 bytes a lane, 1 KB = 8 rows of a 64-deep K slice per
// instruction) into two 64 KB stages whose 128-byte rows hold their 16-byte chunks at slot
// c ^ ((row >> 1) & 7). Schedule per 64-deep stage (4 K16 steps), in nt_mainloop below:
//   - the next step's 8 fragments (16-byte LDS reads, inline asm) are issued one per two MFMAs
//     of the current step, so the reads run under the MFMAs; sched_barrier pins that order and
//     an `s_waitcnt lgkmcnt(0)` that names the fragments as operands keeps every MFMA behind
//     the wait for its data;
//   - the stage barrier sits at the start of the last K16 step: after it, that step's MFMAs
//     run while the next stage's first fragments are read and the 16 loads of the stage after
//     next are issued into the buffer just finished. No step waits on LDS right after a barrier.
// Operand roles are swapped (the MFMA's first operand is the weight tile), so a lane holds 4
// consecutive output columns of one row; the tile is converted to bf16 (RNE, v_cvt_pk_bf16_f32)
// into LDS rows of 256 B (+16 B pad) and written back in whole rows, 16 bytes a lane: writing
// 8-byte pieces of 32 rows per instruction straight from the accumulators made the L2 take
// 16-byte partial-line writes, twice as many L2 requests as the operand reads, and cost 12%.
// Rows past `rows` and columns past `vocab` load a clamped (valid) row and are not stored.
// Tile order: workgroup w runs on XCD w % 8, which takes a contiguous range of tile positions;
// within it, groups of gm x gn tiles (gm * gn = 32, one per CU of the XCD) run together so that
// their operand panels are read from HBM about once per group and served from that XCD's L2.

constexpr int kLgTile = 256;                                    // output tile edge
constexpr int kLgStage = 2 * kLgTile * kSliceK * 2;             // 64 KB: A and B slices
constexpr int kLgPitch = 272;                                   // output staging row pitch
constexpr int kLgLds = 4 * 128 * kLgPitch > 2 * kLgStage ? 4 * 128 * kLgPitch : 2 * kLgStage;  // 139,264 B

// Tile of position p: n-blocks of gn tile columns; inside each, m-blocks of gm tile rows, a
// block's gm x gn tiles consecutive in p.
__device__ __forceinline__ void lg_tile_of(int p, int tiles_m, int tiles_n, int gm, int gn, int& tm, int& tn) {
  const int per_nb = tiles_m * gn;
  const int nb = p / per_nb, rem = p - nb * per_nb;
  const int gn_eff = min(gn, tiles_n - nb * gn);
  const int mb = rem / (gm * gn_eff), rem2 = rem - mb * gm * gn_eff;
  tm = mb * gm + rem2 / gn_eff;
  tn = nb * gn + rem2 % gn_eff;
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two floats -> packed bf16, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  const bf16x2 h = __builtin_convertvector(f32x2{a, b}, bf16x2);
  return __builtin_bit_cast(uint32_t, h);
}

template <bool kN, bool kN2>
struct LgFlags {
  static constexpr bool kNextV = kN, kNext2V = kN2;
};

// Main loop of logits_gemm_kernel (both operands K-contiguous): acc[n block][m block] of a
// 256 x 256 tile, rows m0.. of A and n0.. of B (`ld` elements apart, rows past M or N clamped to
// the last), over n_it 64-deep K slices from element k0. 4 waves, wave (wm, wn) = 128 x 128.
__device__ __forceinline__ void nt_mainloop(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                            int64_t ld, int m0, int n0, int M, int N, int64_t k0, int n_it,
                                            uint8_t* smem, f32x16 (&acc)[4][4]) {
  const int lane = threadIdx.x & 63;
  // wave-uniform in a scalar register, so each load's LDS destination (M0) is scalar arithmetic
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // Load j of this wave fills LDS rows 8 q .. 8 q + 7 of [A tile; B tile], q = 16 wave + j; the
  // lane loads 16-byte chunk (lane % 8) ^ ((row >> 1) & 7) of row 8 q + lane / 8 into slot lane % 8.
  const uint16_t* src[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int q = wave * 16 + j;
    const int r = (q % 32) * 8 + lane / 8;
    const int c = (lane % 8) ^ ((r >> 1) & 7);
    src[j] = (q < 32 ? A + static_cast<int64_t>(min(m0 + r, M - 1)) * ld
                     : B + static_cast<int64_t>(min(n0 + r, N - 1)) * ld) + k0 + c * 8;
  }
  auto load = [&](int it, int stage, int j) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(src[j] + it * kSliceK),
                                     (void __attribute__((address_space(3)))*)(smem + stage * kLgStage + (wave * 16 + j) * 1024),
                                     16, 0, 0);
  };
  // Fragment reads: lane reads row R0 + lane % 32 (R0 a multiple of 32), chunk 2 kk + lane / 32,
  // at slot (2 kk) ^ tx with tx = (lane / 32) ^ ((lane >> 1) & 7).
  const int tx = (lane >> 5) ^ ((lane >> 1) & 7);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + (lane & 31) * 128;
  uint32_t vk[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) vk[kk] = lds0 + (((2 * kk) ^ tx) * 16);
  const uint32_t offA = wm * 128 * 128, offB = kLgTile * 128 + wn * 128 * 128;

#define TM_RD(dst, base, imm) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "i"(imm))
#define TM_WAIT8(f)                                                                                       \
  asm volatile("s_waitcnt lgkmcnt(0)"                                                                   \
               : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7]))
  // fragment g: g < 4 -> B (n) block g, g >= 4 -> A (m) block g - 4
  bf16x8 f0[8], f1[8];
#pragma unroll
  for (int j = 0; j < 16; ++j) load(0, 0, j);
  if (n_it > 1) {
#pragma unroll
    for (int j = 0; j < 16; ++j) load(1, 1, j);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(16));
  } else {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
  }
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int g = 0; g < 8; ++g) TM_RD(f0[g], vk[0] + (g < 4 ? offB : offA), (g % 4) * 32 * 128);
  TM_WAIT8(f0);
  __builtin_amdgcn_sched_barrier(0);

  auto stage = [&](int i, auto step) {
    constexpr bool kNext = decltype(step)::kNextV, kNext2 = decltype(step)::kNext2V;
    const int s = i & 1;
    const uint32_t soff = s * kLgStage, noff = (s ^ 1) * kLgStage;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      bf16x8* cur = (kk & 1) ? f1 : f0;
      bf16x8* nxt = (kk & 1) ? f0 : f1;
      if (kk == 3 && kNext) {
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // this wave's loads of stage i + 1 are in LDS
        __builtin_amdgcn_s_barrier();               // every wave's; and stage i's reads are done
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        if (kk < 3) {
          TM_RD(nxt[g], vk[kk + 1] + soff + (g < 4 ? offB : offA), (g % 4) * 32 * 128);
        } else if (kNext) {
          TM_RD(nxt[g], vk[0] + noff + (g < 4 ? offB : offA), (g % 4) * 32 * 128);
        }
        if (kk == 3 && kNext2) {
          load(i + 2, s, 2 * g);
          load(i + 2, s, 2 * g + 1);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int idx = 2 * g + h, ii = idx / 4, jj = idx % 4;
          acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[ii], cur[4 + jj], acc[ii][jj], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (kk < 3 || kNext) {
        TM_WAIT8(nxt);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  int i = 0;
  for (; i + 2 < n_it; ++i) stage(i, LgFlags<true, true>{});
  if (i + 1 < n_it) stage(i++, LgFlags<true, false>{});
  if (i < n_it) stage(i, LgFlags<false, false>{});
#undef TM_RD
#undef TM_WAIT8
}

__global__ __launch_bounds__(256) void logits_gemm_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                          uint16_t* __restrict__ C, int M, int N, int64_t ldc, int K,
                                                          int tiles_m, int tiles_n, int gm, int gn) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int T = tiles_m * tiles_n;
  const int t8 = (T + 7) / 8;
  const int p = (blockIdx.x % 8) * t8 + blockIdx.x / 8;  // XCD blockIdx % 8 takes positions [x t8, (x+1) t8)
  if (p >= T) return;
  int tm, tn;
  lg_tile_of(p, tiles_m, tiles_n, gm, gn, tm, tn);
  const int m0 = tm * kLgTile, n0 = tn * kLgTile;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  f32x16 acc[4][4];  // [n block][m block]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};
  nt_mainloop(A, B, K, m0, n0, M, N, 0, K / kSliceK, smem, acc);

  // D[n][m] of a 32 x 32 block: register r of lane l holds n = 8 (r / 4) + 4 (l / 32) + r % 4,
  // m = l % 32. Each wave stages its 128 x 128 bf16 tile in LDS, then writes whole rows.
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_s_barrier();  // every wave is done reading the operand stages
  uint8_t* tile = smem + wave * 128 * kLgPitch;
#pragma unroll
  for (int ii = 0; ii < 4; ++ii)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int mr = jj * 32 + (lane & 31), nc = ii * 32 + 8 * q + 4 * (lane >> 5);
        u32x2 o;
        o.x = pack_bf16x2(acc[ii][jj][4 * q], acc[ii][jj][4 * q + 1]);
        o.y = pack_bf16x2(acc[ii][jj][4 * q + 2], acc[ii][jj][4 * q + 3]);
        *(u32x2*)(tile + mr * kLgPitch + nc * 2) = o;
      }
  __builtin_amdgcn_s_waitcnt(0);  // this wave reads back only its own rows
  const int mb = m0 + wm * 128, nb = n0 + wn * 128;
  const bool vec = (ldc & 7) == 0;
#pragma unroll 4
  for (int it = 0; it < 32; ++it) {
    const int mr = it * 4 + (lane >> 4), ch = lane & 15;
    const int m = mb + mr, n = nb + ch * 8;
    if (m >= M) continue;
    const u32x4 v = *(const u32x4*)(tile + mr * kLgPitch + ch * 16);
    uint16_t* dst = C + m * ldc + n;
    if (vec && n + 8 <= N) {
      __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(dst));  // streamed out: keep L2 for operands
    } else {
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      for (int e = 0; e < 8 && n + e < N; ++e) dst[e] = static_cast<uint16_t>(w[e / 2] >> (16 * (e & 1)));
    }
  }
}

// ------------------------------------------------ logits, persistent: one workgroup per CU
//
// The same product, tiles, fragments and summation order as logits_gemm_kernel (bit-identical
// results), for dim a multiple of 64 and at least 192, rows of the logits a multiple of 8 elements
// apart, operands under 4 GiB (1024 x 768 x 32,001 with rows padded to 32,064: 47 us, against 100
// on logits_gemm_kernel with rows 32,001 apart). With K = dim short (16 slices at dim 1024), a tile's
// fill (its first two stages' loads) and its epilogue (its accumulators converted to bf16 and
// written) were a large share of a tile's time; here both overlap the neighbouring tiles' MFMAs:
//   - workgroup c of XCD x (blockIdx = 8 c + x) runs tile positions x t8 + c, + W, + 2W, ...
//     (W workgroups per XCD), so the 32 tiles an XCD runs at a time are the same groups of
//     tiles as in logits_gemm_kernel;
//   - the operand stages form one ring across tiles: the next tile's stages 0 and 1 are loaded
//     during the current tile's last two stages (the tile after the last is the last again, a
//     harmless reload drained before exit);
//   - 8 waves, two a SIMD: wave (wm, wn) = (w / 4, w % 4) computes rows wm * 128 .. +127 and
//     columns wn * 64 .. +63 of the tile, 4 m blocks x 2 n blocks of 32 x 32 (128 accumulators,
//     in VGPRs); while one wave of a SIMD waits for LDS, its loads, the stage barrier or its
//     stores, the other's MFMAs run (measured on MI355X: 4-12% faster than one wave a SIMD with
//     128 x 128 each, the same bits). Per K16 step a wave reads 6 fragments and issues 8 MFMAs;
//     waves 0-3 load the hidden rows, waves 4-7 the weight rows, 8 loads a stage each;
//   - the finished tile's accumulators leave during the next tile's first K16 step: block
//     (ii, jj) is converted to bf16 (RNE) just before that step's MFMA on it, which restarts
//     its accumulation from zero; the 2 blocks of an m block (32 rows x the wave's 64 columns)
//     go to this wave's 4 KB of LDS past the two stages (128-byte rows, chunk c of row r at slot
//     c ^ ((r >> 1) & 7)) and are written back as 128-byte row pieces, 16 bytes a lane; the
//     last tile's output goes the same way after the loop.
// LDS: two 64 KB stages + 8 x 4 KB = 160 KB, the whole of a CU's. Operand addresses are 32-bit
// byte offsets from the operand's base (scalar), one per load.

constexpr int kRgLds = 2 * kLgStage + 8 * 4096;  // 163,840 B

template <bool kN2, bool kPre, bool kFirst, bool kEpi>
struct RgFlags {
  static constexpr bool kNext2V = kN2, kPreV = kPre, kFirstV = kFirst, kEpiV = kEpi;
};

template <bool kV>
struct RgBool {
  static constexpr bool value = kV;
};

__global__ __launch_bounds__(512) void logits_ring_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                          uint16_t* __restrict__ C, int M, int N, int ldc, int K,
                                                          int tiles_m, int tiles_n, int gm, int gn, int wpx) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int T = tiles_m * tiles_n;
  const int t8 = (T + 7) / 8;
  const int x = blockIdx.x % 8;
  const int pend = min((x + 1) * t8, T);
  int p = x * t8 + static_cast<int>(blockIdx.x / 8);
  if (p >= pend) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int n_it = K / kSliceK;  // >= 3
  int par = 0;                   // the stage that holds the current tile's slice 0

  // Waves 0-3 load the A rows of the tile, waves 4-7 the B rows; load j of wave w fills rows
  // 64 (w % 4) + 8 j + lane / 8 of its operand, the lane's chunk (lane % 8) ^ (lane / 16) ^ (4 (j % 2)).
  const char* opnd = reinterpret_cast<const char*>(wave < 4 ? A : B);
  const int lim = (wave < 4 ? M : N) - 1;
  uint32_t soff[8];
  int lrow = lane / 8;
  uint32_t lc16 = static_cast<uint32_t>(((lane % 8) ^ (lane / 16)) * 16);
  auto set_src = [&](int m0, int n0) {
    asm volatile("" : "+v"(lrow), "+v"(lc16));
    const int r0 = (wave < 4 ? m0 : n0) + (wave % 4) * 64;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      soff[j] = static_cast<uint32_t>(min(r0 + 8 * j + lrow, lim)) * static_cast<uint32_t>(2 * K) +
                (lc16 ^ ((j & 1) * 64));
  };
  auto load = [&](int it, int stage, int j) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(opnd + (soff[j] + it * 128u)),
                                     (void __attribute__((address_space(3)))*)(smem + stage * kLgStage + (wave * 8 + j) * 1024),
                                     16, 0, 0);
  };
  const int tx = (lane >> 5) ^ ((lane >> 1) & 7);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + (lane & 31) * 128;
  uint32_t vk[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) vk[kk] = lds0 + (((2 * kk) ^ tx) * 16);
  const uint32_t offA = wm * 128 * 128, offB = kLgTile * 128 + wn * 64 * 128;

  // Output staging, this wave's 4 KB: row r (of an m block's 32) at 128 r, chunk c at slot
  // c ^ ((r >> 1) & 7). A lane writes row lane % 32, half lane / 32 of chunk c; it reads back chunk
  // lane % 8 of row 8 it + lane / 8.
  const uint32_t ebo = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + 2 * kLgStage + wave * 4096;
  const int wr = lane & 31;
  uint32_t wa = ebo + wr * 128 + (lane >> 5) * 8;
  const uint32_t wsw = static_cast<uint32_t>((wr >> 1) & 7);
  uint32_t ra[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = k * 8 + (lane >> 3);
    ra[k] = ebo + r * 128 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
  }
  uint32_t sl = static_cast<uint32_t>(((lane >> 3) * ldc + (lane & 7) * 8) * 2);  // byte offset of the lane's store

#define TM_RD(dst, base, imm) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "i"(imm))
#define TM_WAIT6(f) \
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]))
  // fragment g: g < 2 -> B (n) block g, g >= 2 -> A (m) block g - 2
  bf16x8 f0[6], f1[6];
  f32x16 acc[2][4];  // [n block][m block]
  int pm0 = 0, pn0 = 0;

  auto epi_block = [&](int ii, int jj, bool mfma, bf16x8* cur) {
    asm volatile("" : "+v"(acc[ii][jj]));
    u32x2 o[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      o[q].x = pack_bf16x2(acc[ii][jj][4 * q], acc[ii][jj][4 * q + 1]);
      o[q].y = pack_bf16x2(acc[ii][jj][4 * q + 2], acc[ii][jj][4 * q + 3]);
    }
    if (mfma) {
      asm volatile("" : "+v"(cur[ii]) : "v"(o[0]), "v"(o[1]), "v"(o[2]), "v"(o[3]));
      acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[ii], cur[2 + jj], f32x16{}, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t a = wa + (((static_cast<uint32_t>(ii * 4 + q)) ^ wsw) << 4);
      asm volatile("ds_write_b64 %0, %1" ::"v"(a), "v"(o[q]) : "memory");
    }
  };
  auto epi_store = [&](int jj) {
    u32x4 v[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) asm volatile("ds_read_b128 %0, %1" : "=v"(v[it]) : "v"(ra[it]));
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
    const int rows_left = M - (pm0 + wm * 128 + jj * 32), cols_left = N - (pn0 + wn * 64);
    char* qb = reinterpret_cast<char*>(C) + (static_cast<int64_t>(pm0 + wm * 128 + jj * 32) * ldc + pn0 + wn * 64) * 2;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      if (it * 8 + (lane >> 3) < rows_left && (lane & 7) * 8 < cols_left)
        __builtin_nontemporal_store(v[it], reinterpret_cast<u32x4*>(qb + (sl + static_cast<uint32_t>(it * 8 * ldc * 2))));
    }
  };

  int tm, tn;
  lg_tile_of(p, tiles_m, tiles_n, gm, gn, tm, tn);
  int m0 = tm * kLgTile, n0 = tn * kLgTile;
  set_src(m0, n0);
#pragma unroll
  for (int j = 0; j < 8; ++j) load(0, 0, j);
#pragma unroll
  for (int j = 0; j < 8; ++j) load(1, 1, j);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(8));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int g = 0; g < 6; ++g) TM_RD(f0[g], vk[0] + (g < 2 ? offB : offA), (g < 2 ? g : g - 2) * 32 * 128);
  TM_WAIT6(f0);
  __builtin_amdgcn_sched_barrier(0);

  int pn = p, m0n = m0, n0n = n0;
  bool has_next = false;
  auto tile = [&](auto epi_first) {
    constexpr bool kEpiFirst = decltype(epi_first)::value;
    asm volatile("" : "+v"(wa), "+v"(ra[0]), "+v"(ra[1]), "+v"(ra[2]), "+v"(ra[3]), "+v"(sl));
    pn = p + wpx;
    has_next = pn < pend;
    int tmn, tnn;
    lg_tile_of(has_next ? pn : p, tiles_m, tiles_n, gm, gn, tmn, tnn);
    m0n = tmn * kLgTile;
    n0n = tnn * kLgTile;

    auto stage = [&](int i, auto step) {
      constexpr bool kNext2 = decltype(step)::kNext2V, kPre = decltype(step)::kPreV;
      constexpr bool kFirst = decltype(step)::kFirstV, kEpi = decltype(step)::kEpiV;
      const int s = (i + par) & 1;
      const uint32_t soff_s = s * kLgStage, noff = (s ^ 1) * kLgStage;
      if (kPre) {
        set_src(m0n, n0n);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        bf16x8* cur = (kk & 1) ? f1 : f0;
        bf16x8* nxt = (kk & 1) ? f0 : f1;
        if (kEpi && kk == 0) {  // first K16 step, with the previous tile's output
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) {
              const int g = jj * 2 + ii;
              if (g < 6) TM_RD(nxt[g], vk[1] + soff_s + (g < 2 ? offB : offA), (g < 2 ? g : g - 2) * 32 * 128);
              epi_block(ii, jj, true, cur);
              __builtin_amdgcn_sched_barrier(0);
            }
            epi_store(jj);
            __builtin_amdgcn_sched_barrier(0);
          }
          TM_WAIT6(nxt);
          __builtin_amdgcn_sched_barrier(0);
          continue;
        }
        if (kk == 3) {
          __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < 8; ++g) {
          if (g < 6) {
            if (kk < 3) {
              TM_RD(nxt[g], vk[kk + 1] + soff_s + (g < 2 ? offB : offA), (g < 2 ? g : g - 2) * 32 * 128);
            } else {
              TM_RD(nxt[g], vk[0] + noff + (g < 2 ? offB : offA), (g < 2 ? g : g - 2) * 32 * 128);
            }
          }
          if (kk == 3 && kNext2) {
            const int it2 = i + 2 >= n_it ? i + 2 - n_it : i + 2;
            load(it2, s, g);
          }
          const int jj = g / 2, ii = g % 2;
          if (kFirst && kk == 0)
            acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[ii], cur[2 + jj], f32x16{}, 0, 0, 0);
          else
            acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[ii], cur[2 + jj], acc[ii][jj], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        TM_WAIT6(nxt);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    stage(0, RgFlags<true, false, true, kEpiFirst>{});
    for (int i = 1; i < n_it - 2; ++i) stage(i, RgFlags<true, false, false, false>{});
    stage(n_it - 2, RgFlags<true, true, false, false>{});
    stage(n_it - 1, RgFlags<true, false, false, false>{});
    par = (par + n_it) & 1;  // an odd number of slices leaves the next tile's slice 0 in the other stage
    pm0 = m0;
    pn0 = n0;
  };
  tile(RgBool<false>{});
  while (has_next) {
    p = pn;
    m0 = m0n;
    n0 = n0n;
    __builtin_amdgcn_sched_barrier(0);
    tile(RgBool<true>{});
  }
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) epi_block(ii, jj, false, f0);
    epi_store(jj);
  }
  __builtin_amdgcn_s_waitcnt(0);
#undef TM_RD
#undef TM_WAIT6
}

// The ring kernel's preconditions: at least 3 K slices (a tile's first stage must not be the one
// that already loads the next tile), whole 8-column store groups in a logits row of ld elements,
// 32-bit operand offsets and store offsets.
bool logits_ring_fits(int64_t rows, int64_t vocab, int64_t dim, int64_t ld) {
  return dim % kSliceK == 0 && dim >= 3 * kSliceK && ld % 8 == 0 && rows * dim * 2 < (int64_t(1) << 32) &&
         vocab * dim * 2 < (int64_t(1) << 32) && 32 * ld * 2 < (int64_t(1) << 31);
}

// ------------------------------------------------- grad_h = grad_logits @ W, K split over workgroups
//
// fused_linear_ce.py:52 `grad_h = grad_logits @ w` per chunk: C (rows x dim) = G (rows x V) times
// W (V x dim), K = V. K is long and the output small (16 tiles for a 1024-row chunk at dim
// 1024), so workgroup (split, tile) computes one 256 x 256 tile over one range of K slices and
// writes its fp32 partial tile (straight from the accumulators, 16 bytes a lane: 4 consecutive
// columns of one row; a split with no K slices writes zeros); splits_reduce_kernel adds the
// partials. Pair p = split x tiles + tile; workgroup w runs on XCD w % 8, which takes pairs
// [x p8, (x+1) p8): the workgroups of an XCD share a split's K range of both operands in its L2.
// A stage holds G's 256 rows x 64 K as 128-byte rows (the logits GEMM's layout and fragment
// reads) and W's 64 K rows x 256 columns as 512-byte rows (grad_W's layout for its K-major
// operand, fragments from two ds_read_b64_tr_b16), so W is read as it is stored: no transposed
// copy. 8 waves, two a SIMD, wave (wm, wn) = (w / 4, w % 4) computing rows wm * 128 .. +127 and
// columns wn * 64 .. +63 (4 x 2 blocks, 128 accumulators; 4 fragment reads, 4 half-fragment
// reads and 8 MFMAs per K16 step; 8 loads a stage a wave: waves 0-3 G, waves 4-7 W). Measured on
// MI355X: as fast as, or up to 6% faster than, the same schedule on W^T (the bits are the same),
// which also needed the transpose (0.13 ms at dim 1024, 0.34 at 2560).
//
// kRagged: rows or dim off a multiple of 256, or a vocabulary off a multiple of 64. Loads past the
// last row, column group or weight row take the last one; G's rows are `ld` elements apart with
// zeros from vocab to the next multiple of 64, so the weight row loaded again in the last K slice
// meets zeros; the stores of rows and columns past the edge are left out.

template <bool kRagged>
__global__ __launch_bounds__(512) void grad_h_gemm_kernel(const uint16_t* __restrict__ G, const uint16_t* __restrict__ W,
                                                          float* __restrict__ partials, int rows, int dim, int64_t ld,
                                                          int vocab, int tiles, int splits, int iters_per_split) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int pairs = tiles * splits;
  const int p8 = (pairs + 7) / 8;
  const int p = (blockIdx.x % 8) * p8 + blockIdx.x / 8;
  if (p >= pairs) return;
  const int s = p / tiles, tile = p - s * tiles;
  const int tiles_n = kRagged ? (dim + kLgTile - 1) / kLgTile : dim / kLgTile;
  const int m0 = (tile / tiles_n) * kLgTile, n0 = (tile % tiles_n) * kLgTile;
  const int total = (vocab + kSliceK - 1) / kSliceK;
  const int it0 = s * iters_per_split;
  const int n_it = max(0, min(iters_per_split, total - it0));
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int64_t k0 = static_cast<int64_t>(it0) * kSliceK;

  // Loads, 8 a wave a stage. Waves 0-3: G rows (m) 64 (w % 4) + 8 j + lane / 8 of the tile, the
  // lane's chunk (lane % 8) ^ ((row >> 1) & 7), into LDS rows 8 (8 w + j) .. of the A half (32 KB).
  // Waves 4-7: W rows (k) 16 (w % 4) + 2 j + lane / 32 of the slice, columns n0 + 8 c with
  // c = (lane % 32) ^ (4 (row & 3)), into the B half (512-byte rows), slot lane % 32.
  const uint16_t* src[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (wave < 4) {
      const int r = (wave % 4) * 64 + 8 * j + lane / 8;
      const int c = (lane % 8) ^ ((r >> 1) & 7);
      src[j] = G + static_cast<int64_t>(min(m0 + r, rows - 1)) * ld + k0 + c * 8;
    } else {
      const int kr = (wave % 4) * 16 + 2 * j + lane / 32;
      const int c = (lane % 32) ^ (4 * (kr & 3));
      src[j] = W + (k0 + kr) * dim + (kRagged ? min(n0 + 8 * c, dim - 8) : n0 + 8 * c);
    }
  }
  const int64_t step = wave < 4 ? kSliceK : static_cast<int64_t>(kSliceK) * dim;  // elements per stage
  // the slice (if it is this split's) with weight rows past the vocabulary
  const int it_last = kRagged && vocab % kSliceK != 0 ? total - 1 - it0 : -1;
  auto load = [&](int it, int stage, int j) {
    const uint16_t* from = src[j] + it * step;
    if (kRagged && it == it_last && wave >= 4) {
      const int64_t past = k0 + it * kSliceK + (wave % 4) * 16 + 2 * j + lane / 32 - (vocab - 1);
      if (past > 0) from -= past * dim;
    }
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)from,
                                     (void __attribute__((address_space(3)))*)(smem + stage * kLgStage + (wave * 8 + j) * 1024),
                                     16, 0, 0);
  };
  // A fragments (m blocks) as nt_mainloop: row R0 + lane % 32, chunk 2 kk + lane / 32
  const int tx = (lane >> 5) ^ ((lane >> 1) & 7);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  const uint32_t la = lds0 + (lane & 31) * 128;
  uint32_t vk[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) vk[kk] = la + (((2 * kk) ^ tx) * 16) + wm * 128 * 128;
  // B half-fragments (n blocks) as grad_W's H operand
  const int s16 = lane & 15, s4 = s16 >> 2;
  const int lcf = ((lane >> 4) & 1) * 2 + ((s16 & 3) >> 1);
  const uint32_t rowb = (8 * (lane >> 5) + s4) * 512 + (s16 & 1) * 8;
  uint32_t bd[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) bd[b] = lds0 + kLgTile * 128 + rowb + (4 * ((2 * wn + b) ^ s4) + lcf) * 16;
#define TM_RD(dst, base, imm) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "i"(imm))
#define TM_TR(dst, base, imm) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "i"(imm))
#define TM_WAIT(a, b)                                                                                 \
  asm volatile("s_waitcnt lgkmcnt(0)"                                                                \
               : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]))
  // per K16 step: A blocks 0-3 (bf16x8); B half-fragments h = 2 b + r (bf16x4), b the n block,
  // r rows +0 / +4
  bf16x8 a0[4], a1[4];
  bf16x4 b0[4], b1[4];
  // g 0..3: A block g; 4..7: B half-fragment g - 4
  auto rd = [&](bf16x8* fa, bf16x4* fb, uint32_t so, int kk, int g) {
    if (g < 4) TM_RD(fa[g], vk[kk] + so, g * 32 * 128);
    else {
      const int h = g - 4, b = h >> 1, r = h & 1;
      TM_TR(fb[h], bd[b] + so, kk * 16 * 512 + r * 4 * 512);
    }
  };
  f32x16 acc[2][4];  // [n block][m block]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};
  if (n_it > 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) load(0, 0, j);
    if (n_it > 1) {
#pragma unroll
      for (int j = 0; j < 8; ++j) load(1, 1, j);
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(8));
    } else {
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    }
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 8; ++g) rd(a0, b0, 0, 0, g);
    TM_WAIT(a0, b0);
    __builtin_amdgcn_sched_barrier(0);
    auto stage = [&](int i, auto step_f) {
      constexpr bool kNext = decltype(step_f)::kNextV, kNext2 = decltype(step_f)::kNext2V;
      const int st = i & 1;
      const uint32_t soff = st * kLgStage, noff = (st ^ 1) * kLgStage;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        bf16x8* ca = (kk & 1) ? a1 : a0;
        bf16x8* na = (kk & 1) ? a0 : a1;
        bf16x4* cb = (kk & 1) ? b1 : b0;
        bf16x4* nb = (kk & 1) ? b0 : b1;
        if (kk == 3 && kNext) {
          __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < 8; ++g) {
          if (kk < 3) rd(na, nb, soff, kk + 1, g);
          else if (kNext) rd(na, nb, noff, 0, g);
          if (kk == 3 && kNext2) load(i + 2, st, g);
          const int jj = g / 2, ii = g % 2;
          const bf16x8 bf = __builtin_shufflevector(cb[2 * ii], cb[2 * ii + 1], 0, 1, 2, 3, 4, 5, 6, 7);
          acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf, ca[jj], acc[ii][jj], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (kk < 3 || kNext) {
          TM_WAIT(na, nb);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    int i = 0;
    for (; i + 2 < n_it; ++i) stage(i, LgFlags<true, true>{});
    if (i + 1 < n_it) stage(i++, LgFlags<true, false>{});
    if (i < n_it) stage(i, LgFlags<false, false>{});
  }
#undef TM_RD
#undef TM_TR
#undef TM_WAIT
  float* P = partials + static_cast<int64_t>(s) * rows * dim;
#pragma unroll
  for (int ii = 0; ii < 2; ++ii)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = m0 + wm * 128 + jj * 32 + (lane & 31);
        const int n = n0 + wn * 64 + ii * 32 + 8 * q + 4 * (lane >> 5);
        const f32x4 v = {acc[ii][jj][4 * q], acc[ii][jj][4 * q + 1], acc[ii][jj][4 * q + 2], acc[ii][jj][4 * q + 3]};
        if (!kRagged || (m < rows && n < dim)) *(f32x4*)(P + static_cast<int64_t>(m) * dim + n) = v;
      }
}

// ------------------------------------------------------- grad_W = grad_logits^T @ hidden
//
// fused_linear_ce.py:57 `gw = grad_logits.t() @ h` per chunk: C (vocab x dim) = G^T H with
// G = grad_logits (rows x vocab) and H = hidden (rows x dim), both stored with the contraction
// (rows) outermost. Same 256 x 256 tiles, 4 waves of 128 x 128, two 64 KB stages and the same
// schedule as logits_gemm_kernel; a stage holds 64 rows x 256 columns of each operand, 512-byte
// LDS rows whose 16-byte chunks sit at slot c ^ (4 (row & 3)). MFMA operands need 8 consecutive
// rows of one column per lane: gfx950's transposing LDS read ds_read_b64_tr_b16 gives, in each
// 16-lane group, lane i element i % 4 of the 8-byte pieces addressed by lanes i/4, i/4 + 4,
// i/4 + 8 and i/4 + 12, so with lane s addressing row s/4 at column 4 (s % 4) lane i receives
// rows 0-3 of column i; two such reads (rows +0 and +4) make a fragment. The slot swizzle puts
// the 4 rows of a read, and the 32 columns two 16-lane groups read together, on 16 different
// 16-byte bank groups. Columns past vocab or dim load a clamped (valid) column and are not stored.
// G's rows are `ldg` elements apart. K rows are contracted, a multiple of 64; kRagged: H has only
// k_rows of them, and G's rows past those are zero (a load of a later H row takes the last one).

constexpr int kGwOp = 64 * 512;       // one operand's stage: 64 rows x 256 bf16
constexpr int kGwStage = 2 * kGwOp;   // 64 KB

template <bool kRagged>
__global__ __launch_bounds__(256) void grad_w_gemm_kernel(const uint16_t* __restrict__ G, const uint16_t* __restrict__ H,
                                                          uint16_t* __restrict__ C, int V, int ldg, int D, int K,
                                                          int k_rows, int tiles_v, int tiles_d, int gm, int gn) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int T = tiles_v * tiles_d;
  const int t8 = (T + 7) / 8;
  const int p = (blockIdx.x % 8) * t8 + blockIdx.x / 8;
  if (p >= T) return;
  int tv, td;
  lg_tile_of(p, tiles_v, tiles_d, gm, gn, tv, td);
  const int v0 = tv * kLgTile, d0 = td * kLgTile;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;  // vocab half, dim half
  const int n_it = K / kSliceK;

  // Load j of this wave, q = 16 wave + j: operand q / 32 (G, then H), rows 2 (q % 32) and
  // 2 (q % 32) + 1 of the stage; slot lane % 32 of row 2 (q % 32) + lane / 32 takes logical chunk
  // (lane % 32) ^ (4 (row & 3)).
  const uint16_t* src[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int q = wave * 16 + j;
    const int kr = 2 * (q % 32) + lane / 32;
    const int c = (lane % 32) ^ (4 * (kr & 3));
    src[j] = q < 32 ? G + static_cast<int64_t>(kr) * ldg + min(v0 + 8 * c, ldg - 8)
                    : H + static_cast<int64_t>(kr) * D + min(d0 + 8 * c, D - 8);
  }
  const int64_t step_g = static_cast<int64_t>(kSliceK) * ldg, step_h = static_cast<int64_t>(kSliceK) * D;
  auto load = [&](int it, int stage, int j) {
    const int q = wave * 16 + j;
    const uint16_t* from = src[j] + it * (q < 32 ? step_g : step_h);
    if (kRagged && q >= 32 && (it + 1) * kSliceK > k_rows) {
      const int64_t past = it * kSliceK + 2 * (q % 32) + lane / 32 - (k_rows - 1);
      if (past > 0) from -= past * D;
    }
    __builtin_amdgcn_global_load_lds(
        (const void __attribute__((address_space(1)))*)from,
        (void __attribute__((address_space(3)))*)(smem + stage * kGwStage + q * 1024), 16, 0, 0);
  };
  // Fragment of 32-column block b at K16 step kk: lane l (s = l % 16) reads row
  // 16 kk + 8 (l / 32) + s / 4 (+4 for the second half) at column 32 b + 16 ((l / 16) % 2) + 4 (s % 4),
  // whose physical chunk is 4 (b ^ (s / 4)) + ((l / 16) % 2) * 2 + (s % 4) / 2 past the wave's 16.
  const int s16 = lane & 15, s4 = s16 >> 2;
  const int lc = ((lane >> 4) & 1) * 2 + ((s16 & 3) >> 1);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  const uint32_t rowb = (8 * (lane >> 5) + s4) * 512 + (s16 & 1) * 8;
  uint32_t bv[4], bd[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    bv[b] = lds0 + rowb + (16 * wm + 4 * (b ^ s4) + lc) * 16;
    bd[b] = lds0 + kGwOp + rowb + (16 * wn + 4 * (b ^ s4) + lc) * 16;
  }

  f32x16 acc[4][4];  // [dim block][vocab block]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};

#define TM_TR(dst, base, imm) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "i"(imm))
#define TM_WAIT16(f)                                                                                        \
  asm volatile("s_waitcnt lgkmcnt(0)"                                                                     \
               : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7]), \
                 "+v"(f[8]), "+v"(f[9]), "+v"(f[10]), "+v"(f[11]), "+v"(f[12]), "+v"(f[13]), "+v"(f[14]),      \
                 "+v"(f[15]))
  // half-fragment h = 2 g + r: g < 4 -> dim block g, g >= 4 -> vocab block g - 4; r: rows +0 / +4
  bf16x4 f0[16], f1[16];
  auto rd = [&](bf16x4* f, uint32_t soff, int kk, int h) {
    const int g = h >> 1, r = h & 1;
    TM_TR(f[h], (g < 4 ? bd[g] : bv[g - 4]) + soff, kk * 16 * 512 + r * 4 * 512);
  };
#pragma unroll
  for (int j = 0; j < 16; ++j) load(0, 0, j);
  if (n_it > 1) {
#pragma unroll
    for (int j = 0; j < 16; ++j) load(1, 1, j);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(16));
  } else {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
  }
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int h = 0; h < 16; ++h) rd(f0, 0, 0, h);
  TM_WAIT16(f0);
  __builtin_amdgcn_sched_barrier(0);

  auto stage = [&](int i, auto step) {
    constexpr bool kNext = decltype(step)::kNextV, kNext2 = decltype(step)::kNext2V;
    const int s = i & 1;
    const uint32_t soff = s * kGwStage, noff = (s ^ 1) * kGwStage;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      bf16x4* cur = (kk & 1) ? f1 : f0;
      bf16x4* nxt = (kk & 1) ? f0 : f1;
      if (kk == 3 && kNext) {
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int q = 0; q < 16; ++q) {  // one half-fragment read, at most one load, one MFMA
        if (kk < 3) rd(nxt, soff, kk + 1, q);
        else if (kNext) rd(nxt, noff, 0, q);
        if (kk == 3 && kNext2) load(i + 2, s, q);
        const int ii = q / 4, jj = q % 4;
        const bf16x8 a = __builtin_shufflevector(cur[2 * ii], cur[2 * ii + 1], 0, 1, 2, 3, 4, 5, 6, 7);
        const bf16x8 b = __builtin_shufflevector(cur[8 + 2 * jj], cur[9 + 2 * jj], 0, 1, 2, 3, 4, 5, 6, 7);
        acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[ii][jj], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (kk < 3 || kNext) {
        TM_WAIT16(nxt);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  int i = 0;
  for (; i + 2 < n_it; ++i) stage(i, LgFlags<true, true>{});
  if (i + 1 < n_it) stage(i++, LgFlags<true, false>{});
  if (i < n_it) stage(i, LgFlags<false, false>{});
#undef TM_TR
#undef TM_WAIT16

  // D[d][v] of a block: lane holds 4 consecutive dim columns of one vocab row (as the logits)
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_s_barrier();
  uint8_t* tile = smem + wave * 128 * kLgPitch;
#pragma unroll
  for (int ii = 0; ii < 4; ++ii)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int vr = jj * 32 + (lane & 31), dc = ii * 32 + 8 * q + 4 * (lane >> 5);
        u32x2 o;
        o.x = pack_bf16x2(acc[ii][jj][4 * q], acc[ii][jj][4 * q + 1]);
        o.y = pack_bf16x2(acc[ii][jj][4 * q + 2], acc[ii][jj][4 * q + 3]);
        *(u32x2*)(tile + vr * kLgPitch + dc * 2) = o;
      }
  __builtin_amdgcn_s_waitcnt(0);
  const int vb = v0 + wm * 128, db = d0 + wn * 128;
#pragma unroll 4
  for (int it = 0; it < 32; ++it) {
    const int vr = it * 4 + (lane >> 4), ch = lane & 15;
    const int v = vb + vr, d = db + ch * 8;
    if (v >= V || d >= D) continue;  // D is a multiple of 8: a group is whole or out
    const u32x4 val = *(const u32x4*)(tile + vr * kLgPitch + ch * 16);
    __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(C + static_cast<int64_t>(v) * D + d));
  }
}

// ------------------------------------------------ grad_W, persistent: one workgroup per CU
//
// grad_w_gemm_kernel's tiles, loads, transposing fragment reads and summation order (bit-identical
// results) in logits_ring_kernel's persistent form: workgroup c of XCD x runs the XCD's tile
// positions c, c + W, ...; the next tile's first two stages load during the current tile's last
// two; 8 waves, two a SIMD, wave (wm, wn) = (w / 4, w % 4) computing vocab rows wm * 128 .. +127
// and dim columns wn * 64 .. +63 (4 vocab x 2 dim blocks; 12 transposing half-fragment reads and
// 8 MFMAs per K16 step; measured on MI355X: 4-10% faster than one wave a SIMD, the same bits);
// the finished tile's accumulators are converted and staged block by block during the next tile's
// first K16 step (32 vocab rows x the wave's 64 dim columns at a time through the wave's 4 KB past
// the stages) and written as 128-byte row pieces of grad_W. For rows (K, with their padding) a
// multiple of 128 and at least 256, dim a multiple of 8, operands under 4 GiB; grad_w_gemm_kernel
// otherwise.

template <bool kRagged>
__global__ __launch_bounds__(512) void grad_w_ring_kernel(const uint16_t* __restrict__ G, const uint16_t* __restrict__ H,
                                                          uint16_t* __restrict__ C, int V, int ldg, int D, int K,
                                                          int k_rows, int tiles_v, int tiles_d, int gm, int gn,
                                                          int wpx) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int T = tiles_v * tiles_d;
  const int t8 = (T + 7) / 8;
  const int x = blockIdx.x % 8;
  const int pend = min((x + 1) * t8, T);
  int p = x * t8 + static_cast<int>(blockIdx.x / 8);
  if (p >= pend) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;  // vocab half, dim quarter
  const int n_it = K / kSliceK;             // even, >= 4

  // Waves 0-3 load G (rows 16 (wave % 4) .. +15 of a stage), waves 4-7 H. Load j: stage rows
  // 16 (wave % 4) + 2 j + lane / 32, slot lane % 32 taking chunk (lane % 32) ^ (4 (row & 3)) =
  // (lane % 32) ^ (4 (lane / 32)) ^ (8 (j % 2)).
  const char* opnd = reinterpret_cast<const char*>(wave < 4 ? G : H);
  const int ld = wave < 4 ? ldg : D;
  const int lim8 = ld - 8;
  const uint32_t step = static_cast<uint32_t>(kSliceK) * static_cast<uint32_t>(ld) * 2u;  // bytes per stage
  uint32_t soff[8];
  uint32_t cap[2] = {0xFFFFFFFFu, 0xFFFFFFFFu};  // kRagged: last H row's offsets, even and odd j
  int lkr = lane >> 5;
  int lc = (lane & 31) ^ (4 * (lane >> 5));
  auto set_src = [&](int v0, int d0) {
    asm volatile("" : "+v"(lkr), "+v"(lc));
    const int col0 = wave < 4 ? v0 : d0;
    const int r0 = (wave % 4) * 16;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int kr = r0 + 2 * j + lkr;
      const int c = lc ^ (8 * (j & 1));
      const uint32_t col = static_cast<uint32_t>(min(col0 + 8 * c, lim8));
      soff[j] = (static_cast<uint32_t>(kr) * static_cast<uint32_t>(ld) + col) * 2u;
      if (kRagged && j < 2 && wave >= 4) cap[j] = (static_cast<uint32_t>(k_rows - 1) * static_cast<uint32_t>(ld) + col) * 2u;
    }
  };
  auto load = [&](int it, int stage, int j) {
    uint32_t off = soff[j] + static_cast<uint32_t>(it) * step;
    if (kRagged) off = min(off, cap[j & 1]);
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(opnd + off),
                                     (void __attribute__((address_space(3)))*)(smem + stage * kGwStage + (wave * 8 + j) * 1024),
                                     16, 0, 0);
  };
  // transposing fragment reads as in grad_w_gemm_kernel, for the wave's 4 vocab and 2 dim blocks
  const int s16 = lane & 15, s4 = s16 >> 2;
  const int lcf = ((lane >> 4) & 1) * 2 + ((s16 & 3) >> 1);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  const uint32_t rowb = (8 * (lane >> 5) + s4) * 512 + (s16 & 1) * 8;
  uint32_t bv[4], bd[2];
#pragma unroll
  for (int b = 0; b < 4; ++b) bv[b] = lds0 + rowb + (16 * wm + 4 * (b ^ s4) + lcf) * 16;
#pragma unroll
  for (int b = 0; b < 2; ++b) bd[b] = lds0 + kGwOp + rowb + (4 * ((2 * wn + b) ^ s4) + lcf) * 16;

  // Output staging, this wave's 4 KB: vocab row r (of a vocab block's 32) at 128 r, chunk c at
  // slot c ^ ((r >> 1) & 7); read back as chunk lane % 8 of row 8 it + lane / 8.
  const uint32_t ebo = lds0 + 2 * kGwStage + wave * 4096;
  const int wr = lane & 31;
  uint32_t wa = ebo + wr * 128 + (lane >> 5) * 8;
  const uint32_t wsw = static_cast<uint32_t>((wr >> 1) & 7);
  uint32_t ra[4];
#pragma unroll
  for (int kq = 0; kq < 4; ++kq) {
    const int r = kq * 8 + (lane >> 3);
    ra[kq] = ebo + r * 128 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
  }
  uint32_t sl = static_cast<uint32_t>(((lane >> 3) * D + (lane & 7) * 8) * 2);

#define TM_TR(dst, base, imm) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "i"(imm))
#define TM_WAIT12(f)                                                                                        \
  asm volatile("s_waitcnt lgkmcnt(0)"                                                                     \
               : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7]), \
                 "+v"(f[8]), "+v"(f[9]), "+v"(f[10]), "+v"(f[11]))
  // half-fragment h = 2 g + r: g < 2 -> dim block g, g >= 2 -> vocab block g - 2; r: rows +0 / +4
  bf16x4 f0[12], f1[12];
  auto rd = [&](bf16x4* f, uint32_t so, int kk, int h) {
    const int g = h >> 1, r = h & 1;
    TM_TR(f[h], (g < 2 ? bd[g] : bv[g - 2]) + so, kk * 16 * 512 + r * 4 * 512);
  };
  f32x16 acc[2][4];  // [dim block][vocab block]
  int pv0 = 0, pd0 = 0;  // origin of the tile whose output is being written

  // block (ii, jj) -> staging (and the next tile's first MFMA on it), as in logits_ring_kernel

  auto epi_block = [&](int ii, int jj, bool mfma, bf16x4* cur) {
    asm volatile("" : "+v"(acc[ii][jj]));
    u32x2 o[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      o[q].x = pack_bf16x2(acc[ii][jj][4 * q], acc[ii][jj][4 * q + 1]);
      o[q].y = pack_bf16x2(acc[ii][jj][4 * q + 2], acc[ii][jj][4 * q + 3]);
    }
    if (mfma) {
      asm volatile("" : "+v"(cur[2 * ii]) : "v"(o[0]), "v"(o[1]), "v"(o[2]), "v"(o[3]));
      const bf16x8 a = __builtin_shufflevector(cur[2 * ii], cur[2 * ii + 1], 0, 1, 2, 3, 4, 5, 6, 7);
      const bf16x8 b = __builtin_shufflevector(cur[4 + 2 * jj], cur[5 + 2 * jj], 0, 1, 2, 3, 4, 5, 6, 7);
      acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, f32x16{}, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t a = wa + (((static_cast<uint32_t>(ii * 4 + q)) ^ wsw) << 4);
      asm volatile("ds_write_b64 %0, %1" ::"v"(a), "v"(o[q]) : "memory");
    }
  };
  // vocab block jj (32 rows x the wave's 64 dim columns) -> grad_W, 16 bytes a lane (D % 8 == 0)
  auto epi_store = [&](int jj) {
    u32x4 v[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) asm volatile("ds_read_b128 %0, %1" : "=v"(v[it]) : "v"(ra[it]));
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
    const int rows_left = V - (pv0 + wm * 128 + jj * 32), cols_left = D - (pd0 + wn * 64);
    char* qb = reinterpret_cast<char*>(C) + (static_cast<int64_t>(pv0 + wm * 128 + jj * 32) * D + pd0 + wn * 64) * 2;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      if (it * 8 + (lane >> 3) < rows_left && (lane & 7) * 8 < cols_left)
        __builtin_nontemporal_store(v[it], reinterpret_cast<u32x4*>(qb + (sl + static_cast<uint32_t>(it * 8 * D * 2))));
    }
  };

  int tv, td;
  lg_tile_of(p, tiles_v, tiles_d, gm, gn, tv, td);
  int v0 = tv * kLgTile, d0 = td * kLgTile;
  set_src(v0, d0);
#pragma unroll
  for (int j = 0; j < 8; ++j) load(0, 0, j);
#pragma unroll
  for (int j = 0; j < 8; ++j) load(1, 1, j);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(8));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int h = 0; h < 12; ++h) rd(f0, 0, 0, h);
  TM_WAIT12(f0);
  __builtin_amdgcn_sched_barrier(0);

  int pn = p, v0n = v0, d0n = d0;
  bool has_next = false;
  // one tile, as in logits_ring_kernel
  auto tile = [&](auto epi_first) {
    constexpr bool kEpiFirst = decltype(epi_first)::value;
    asm volatile("" : "+v"(wa), "+v"(ra[0]), "+v"(ra[1]), "+v"(ra[2]), "+v"(ra[3]), "+v"(sl));
    pn = p + wpx;
    has_next = pn < pend;
    int tvn, tdn;
    lg_tile_of(has_next ? pn : p, tiles_v, tiles_d, gm, gn, tvn, tdn);
    v0n = tvn * kLgTile;
    d0n = tdn * kLgTile;

    auto stage = [&](int i, auto step) {
      constexpr bool kNext2 = decltype(step)::kNext2V, kPre = decltype(step)::kPreV;
      constexpr bool kFirst = decltype(step)::kFirstV, kEpi = decltype(step)::kEpiV;
      const int s = i & 1;
      const uint32_t so = s * kGwStage, noff = (s ^ 1) * kGwStage;
      if (kPre) {
        set_src(v0n, d0n);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        bf16x4* cur = (kk & 1) ? f1 : f0;
        bf16x4* nxt = (kk & 1) ? f0 : f1;
        if (kEpi && kk == 0) {
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) {
              const int bi = jj * 2 + ii;
              rd(nxt, so, 1, bi);
              if (bi < 4) rd(nxt, so, 1, 8 + bi);
              epi_block(ii, jj, true, cur);
              __builtin_amdgcn_sched_barrier(0);
            }
            epi_store(jj);
            __builtin_amdgcn_sched_barrier(0);
          }
          TM_WAIT12(nxt);
          __builtin_amdgcn_sched_barrier(0);
          continue;
        }
        if (kk == 3) {
          __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {  // one MFMA, one or two half-fragment reads, at most one load
          if (kk < 3) {
            rd(nxt, so, kk + 1, q);
            if (q < 4) rd(nxt, so, kk + 1, 8 + q);
          } else {
            rd(nxt, noff, 0, q);
            if (q < 4) rd(nxt, noff, 0, 8 + q);
          }
          if (kk == 3 && kNext2) {
            const int it2 = i + 2 >= n_it ? i + 2 - n_it : i + 2;
            load(it2, s, q);
          }
          const int jj = q / 2, ii = q % 2;
          const bf16x8 a = __builtin_shufflevector(cur[2 * ii], cur[2 * ii + 1], 0, 1, 2, 3, 4, 5, 6, 7);
          const bf16x8 b = __builtin_shufflevector(cur[4 + 2 * jj], cur[5 + 2 * jj], 0, 1, 2, 3, 4, 5, 6, 7);
          if (kFirst && kk == 0)
            acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, f32x16{}, 0, 0, 0);
          else
            acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[ii][jj], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        TM_WAIT12(nxt);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    stage(0, RgFlags<true, false, true, kEpiFirst>{});
    for (int i = 1; i < n_it - 2; ++i) stage(i, RgFlags<true, false, false, false>{});
    stage(n_it - 2, RgFlags<true, true, false, false>{});
    stage(n_it - 1, RgFlags<true, false, false, false>{});
    pv0 = v0;
    pd0 = d0;
  };
  tile(RgBool<false>{});
  while (has_next) {
    p = pn;
    v0 = v0n;
    d0 = d0n;
    __builtin_amdgcn_sched_barrier(0);
    tile(RgBool<true>{});
  }
  // the last tile's output; then the redundant reload of that tile's first stages completes
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) epi_block(ii, jj, false, f0);
    epi_store(jj);
  }
  __builtin_amdgcn_s_waitcnt(0);
#undef TM_TR
#undef TM_WAIT12
}


// k: the contracted rows (grad_logits' rows with their padding), ld: its row stride.
bool grad_w_ring_fits(int64_t k, int64_t ld, int64_t dim) {
  return k % 128 == 0 && k >= 256 && ld % 8 == 0 && dim % 8 == 0 && k * ld * 2 < (int64_t(1) << 32) &&
         k * dim * 2 < (int64_t(1) << 32) && 32 * dim * 2 < (int64_t(1) << 32);
}

// ------------------------------------------------------- the three products on smaller tiles
//
// One kernel for shapes whose 256 x 256 tiles leave CUs idle (fewer tiles than CUs, a nearly empty
// last round, a hidden size that wastes half a tile): C (M x N) = A B over K slices of 64, tiles
// of 64 kMB x 128 kNB, 8 wave64 of (32 kMB) x (32 kNB), wave (wm, wn) = (w / 4, w % 4), with the
// loads, LDS layouts, fragments and schedule of the 256 x 256 kernels:
//   kAK: A is M x K (lda apart), else K x M; kBK: B is N x K, else K x N, of which only kb rows
//   exist (a later row loads the last one against zeros of A).
// Workgroup (split, tile) covers K slices [split * per, ..): with kPartial it writes its fp32 tile
// to `out` + split * M * N for splits_reduce_kernel, else (one split) bf16, 16 bytes a lane after
// v_permlane32_swap joins the two halves of a row's 8 columns.
template <int kMB, int kNB, bool kAK, bool kBK, bool kPartial>
__global__ __launch_bounds__(512) void gemm_tile_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                        void* __restrict__ out, int M, int N, int64_t lda, int64_t ldb,
                                                        int64_t ldc, int slices, int kb, int tiles_m, int tiles_n,
                                                        int gm, int gn, int per) {
  constexpr int kTM = 64 * kMB, kTN = 128 * kNB, kLoads = (kTM + kTN) / 64, kInA = kTM / 8;
  constexpr int kStage = (kTM + kTN) * 128;
  constexpr int kRdA = kAK ? kMB : 2 * kMB, kRdB = kBK ? kNB : 2 * kNB, kRd = kRdA + kRdB, kMf = kMB * kNB;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int T = tiles_m * tiles_n, pairs = T * ((slices + per - 1) / per);
  const int p8 = (pairs + 7) / 8;
  const int p = (blockIdx.x % 8) * p8 + blockIdx.x / 8;
  if (p >= pairs || static_cast<int>(blockIdx.x / 8) >= p8) return;
  const int split = p / T;
  int tm, tn;
  lg_tile_of(p - split * T, tiles_m, tiles_n, gm, gn, tm, tn);
  const int m0 = tm * kTM, n0 = tn * kTN;
  const int it0 = split * per, n_it = min(per, slices - it0);
  const int64_t k0 = static_cast<int64_t>(it0) * kSliceK;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;

  // Load q = kLoads wave + j: 1 KB of A's stage (q < kInA), then of B's. K-contiguous: 8 rows of
  // 128 bytes, chunk c of row r at slot c ^ ((r >> 1) & 7). K-major: whole rows of the tile's
  // columns, chunk c of row k at slot c ^ (4 (k & 3)).
  const uint16_t* src[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int q = wave * kLoads + j;
    if (q < kInA) {
      if constexpr (kAK) {
        const int r = q * 8 + lane / 8;
        src[j] = A + static_cast<int64_t>(min(m0 + r, M - 1)) * lda + k0 + ((lane % 8) ^ ((r >> 1) & 7)) * 8;
      } else {
        constexpr int kCpr = kTM / 8;
        const int kr = q * (64 / kCpr) + lane / kCpr;
        const int c = (lane % kCpr) ^ (4 * (kr & 3));
        src[j] = A + (k0 + kr) * lda + min(static_cast<int64_t>(m0 + 8 * c), lda - 8);
      }
    } else {
      const int qb = q - kInA;
      if constexpr (kBK) {
        const int r = qb * 8 + lane / 8;
        src[j] = B + static_cast<int64_t>(min(n0 + r, N - 1)) * ldb + k0 + ((lane % 8) ^ ((r >> 1) & 7)) * 8;
      } else {
        constexpr int kCpr = kTN / 8;
        const int kr = qb * (64 / kCpr) + lane / kCpr;
        const int c = (lane % kCpr) ^ (4 * (kr & 3));
        src[j] = B + (k0 + kr) * ldb + min(static_cast<int64_t>(n0 + 8 * c), ldb - 8);
      }
    }
  }
  const int64_t step_a = kAK ? kSliceK : kSliceK * lda, step_b = kBK ? kSliceK : kSliceK * ldb;
  auto load = [&](int it, int stage, int j) {
    const int q = wave * kLoads + j;
    const uint16_t* from = src[j] + it * (q < kInA ? step_a : step_b);
    if (!kBK && q >= kInA && k0 + static_cast<int64_t>(it + 1) * kSliceK > kb) {
      constexpr int kCpr = kTN / 8;
      const int64_t past = k0 + static_cast<int64_t>(it) * kSliceK + (q - kInA) * (64 / kCpr) + lane / kCpr - (kb - 1);
      if (past > 0) from -= past * ldb;
    }
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)from,
                                     (void __attribute__((address_space(3)))*)(smem + stage * kStage + q * 1024), 16, 0, 0);
  };
  // Fragment addresses: K-contiguous, row lane % 32 of a block, chunk 2 kk + lane / 32; K-major,
  // two transposing half-fragment reads (rows +0 and +4), as grad_w_gemm_kernel.
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  const int tx = (lane >> 5) ^ ((lane >> 1) & 7);
  uint32_t vk[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) vk[kk] = lds0 + (lane & 31) * 128 + (((2 * kk) ^ tx) * 16);
  const int s16 = lane & 15, s4 = s16 >> 2;
  const int lcf = ((lane >> 4) & 1) * 2 + ((s16 & 3) >> 1);
  uint32_t ba[kMB], bb[kNB];
#pragma unroll
  for (int i = 0; i < kMB; ++i)
    ba[i] = lds0 + (8 * (lane >> 5) + s4) * (kTM * 2) + (s16 & 1) * 8 + (4 * ((wm * kMB + i) ^ s4) + lcf) * 16;
#pragma unroll
  for (int i = 0; i < kNB; ++i)
    bb[i] = lds0 + kInA * 1024 + (8 * (lane >> 5) + s4) * (kTN * 2) + (s16 & 1) * 8 +
            (4 * ((wn * kNB + i) ^ s4) + lcf) * 16;
  const uint32_t offA = wm * kMB * 32 * 128, offB = kInA * 1024 + wn * kNB * 32 * 128;

#define TM_RD(dst, base, imm) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "i"(imm))
#define TM_TR(dst, base, imm) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "i"(imm))
  bf16x8 a8[2][kAK ? kMB : 1], b8[2][kBK ? kNB : 1];
  bf16x4 a4[2][kAK ? 1 : 2 * kMB], b4[2][kBK ? 1 : 2 * kNB];
  // read g of a step (g < kRdA: A's) into set z
  auto rd = [&](int z, uint32_t so, int kk, int g) {
    if (g < kRdA) {
      if constexpr (kAK) TM_RD(a8[z][g], vk[kk] + so + offA, g * 32 * 128);
      else TM_TR(a4[z][g], ba[g >> 1] + so, kk * 16 * kTM * 2 + (g & 1) * 4 * kTM * 2);
    } else {
      const int h = g - kRdA;
      if constexpr (kBK) TM_RD(b8[z][h], vk[kk] + so + offB, h * 32 * 128);
      else TM_TR(b4[z][h], bb[h >> 1] + so, kk * 16 * kTN * 2 + (h & 1) * 4 * kTN * 2);
    }
  };
  // waits for set z's reads; naming every fragment keeps the MFMAs that use them behind the wait
  auto wait = [&](int z) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int g = 0; g < kRdA; ++g) {
      if constexpr (kAK) asm volatile("" : "+v"(a8[z][g]));
      else asm volatile("" : "+v"(a4[z][g]));
    }
#pragma unroll
    for (int g = 0; g < kRdB; ++g) {
      if constexpr (kBK) asm volatile("" : "+v"(b8[z][g]));
      else asm volatile("" : "+v"(b4[z][g]));
    }
  };
  auto afrag = [&](int z, int i) {
    if constexpr (kAK) return a8[z][i];
    else return __builtin_shufflevector(a4[z][2 * i], a4[z][2 * i + 1], 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto bfrag = [&](int z, int i) {
    if constexpr (kBK) return b8[z][i];
    else return __builtin_shufflevector(b4[z][2 * i], b4[z][2 * i + 1], 0, 1, 2, 3, 4, 5, 6, 7);
  };

  f32x16 acc[kNB][kMB];
#pragma unroll
  for (int i = 0; i < kNB; ++i)
#pragma unroll
    for (int j = 0; j < kMB; ++j) acc[i][j] = f32x16{};
#pragma unroll
  for (int j = 0; j < kLoads; ++j) load(0, 0, j);
  if (n_it > 1) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) load(1, 1, j);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(kLoads));
  } else {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
  }
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int g = 0; g < kRd; ++g) rd(0, 0, 0, g);
  wait(0);
  __builtin_amdgcn_sched_barrier(0);
  auto stage = [&](int i, auto step_f) {
    constexpr bool kNext = decltype(step_f)::kNextV, kNext2 = decltype(step_f)::kNext2V;
    const int st = i & 1;
    const uint32_t soff = st * kStage, noff = (st ^ 1) * kStage;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int z = kk & 1;
      if (kk == 3 && kNext) {
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int f = 0; f < kMf; ++f) {  // one MFMA, its share of the next step's reads and of the loads
#pragma unroll
        for (int g = f * kRd / kMf; g < (f + 1) * kRd / kMf; ++g) {
          if (kk < 3) rd(z ^ 1, soff, kk + 1, g);
          else if (kNext) rd(z ^ 1, noff, 0, g);
        }
        if (kk == 3 && kNext2) {
#pragma unroll
          for (int j = f * kLoads / kMf; j < (f + 1) * kLoads / kMf; ++j) load(i + 2, st, j);
        }
        const int jj = f / kNB, ii = f % kNB;
        acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfrag(z, ii), afrag(z, jj), acc[ii][jj], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (kk < 3 || kNext) {
        wait(z ^ 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  int i = 0;
  for (; i + 2 < n_it; ++i) stage(i, LgFlags<true, true>{});
  if (i + 1 < n_it) stage(i++, LgFlags<true, false>{});
  if (i < n_it) stage(i, LgFlags<false, false>{});
#undef TM_RD
#undef TM_TR

  // D[n][m] of a block: register r of lane l holds n = 8 (r / 4) + 4 (l / 32) + r % 4, m = l % 32
#pragma unroll
  for (int jj = 0; jj < kMB; ++jj) {
    const int m = m0 + (wm * kMB + jj) * 32 + (lane & 31);
#pragma unroll
    for (int ii = 0; ii < kNB; ++ii) {
      const int nb = n0 + (wn * kNB + ii) * 32;
      if constexpr (kPartial) {
        float* P = static_cast<float*>(out) + static_cast<int64_t>(split) * M * N;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = nb + 8 * q + 4 * (lane >> 5);
          const f32x4 v = {acc[ii][jj][4 * q], acc[ii][jj][4 * q + 1], acc[ii][jj][4 * q + 2], acc[ii][jj][4 * q + 3]};
          if (m < M && n < N) *(f32x4*)(P + static_cast<int64_t>(m) * N + n) = v;
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; q += 2) {
          uint32_t lo[2], hi[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            lo[e] = pack_bf16x2(acc[ii][jj][4 * q + 2 * e], acc[ii][jj][4 * q + 2 * e + 1]);
            hi[e] = pack_bf16x2(acc[ii][jj][4 * q + 4 + 2 * e], acc[ii][jj][4 * q + 5 + 2 * e]);
            const auto s = __builtin_amdgcn_permlane32_swap(lo[e], hi[e], false, false);
            lo[e] = s[0];
            hi[e] = s[1];
          }
          // lanes below 32: columns 8 q .. 8 q + 7, lanes above: the next 8
          const int n = nb + 8 * q + 8 * (lane >> 5);
          const u32x4 v = {lo[0], lo[1], hi[0], hi[1]};
          if (m < M && n < N)  // rows hold whole groups of 8 (ldc and the last group's end <= ldc)
            *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(out) + m * ldc + n) = v;
        }
      }
    }
  }
}

// Tile groups per XCD round (gm row tiles x gn weight panels, gm gn = 32), chosen from a sweep of
// the logits ring kernel on MI355X (V = 151,936; TFLOP/s of the best against the next best):
//   dim <= 1024: 1 x 32 up to 4 row tiles (1063 against 855 for 4 x 8 at 1024 rows: the hidden
//                chunk sits in every XCD's L2 and a round takes one row of 32 panels), 2 x 16 up
//                to 8, 4 x 8 above;
//   dim <= 2560: 2 x 16 up to 8 row tiles (1048 against 899 for 1 x 32 at 1024 x 2560), 4 x 8
//                above;
//   dim <= 4096: 4 x 8 (1118 against 1008 for 1 x 32 at 1024 x 4096);
//   wider:       8 x 4 from 8 row tiles (1195 against 1125 for 4 x 8 at 8192 x 5120), 4 x 8 below.
// Wider panels (256 x dim) leave fewer in an XCD's 4 MB L2, so rounds share each panel among more
// tiles.
void logits_groups(int64_t tiles_m, int64_t dim, int& gm, int& gn) {
  if (dim <= 1024) gm = tiles_m <= 4 ? 1 : (tiles_m <= 8 ? 2 : 4);
  else if (dim <= 2560) gm = tiles_m <= 8 ? 2 : 4;
  else if (dim <= 4096) gm = 4;
  else gm = tiles_m >= 8 ? 8 : 4;
  gn = 32 / gm;
}

// Which kernel, and how many splits of K: the least estimated time. The model is the launch's
// rounds over the CUs, times K slices a workgroup, times the measured time of a slice, plus a
// tile's epilogue, plus, with splits, the fp32 partials' way out and back and the reduction. Over 78
// products (64-7129 rows, dim 256-2560, vocabulary 1000-152,000) its choice took 0.8% more time than
// the best one on average, over 3% more in 5 of them, at most 16%. The rounds are those of a
// whole MI355X's 256 CUs: on a partition with fewer the choice is as valid but may not be the fastest.
constexpr double kUsSlice256 = 1.42;       // a 64-deep K slice of a 256 x 256 tile, one workgroup a CU
constexpr double kUsSlice128 = 0.62;       // of a 128 x 128 tile, one workgroup a CU: latency
constexpr double kUsSlice128Pair = 0.95;   // the same with two a CU
constexpr double kUsLaunch = 3.0, kUsEpilogue = 1.5, kUsReduce = 2.5, kBytesPerUs = 4.5e6;
constexpr int64_t kMaxPartialBytes = int64_t(2) << 30;

struct TilePlan {
  bool wide;       // 256 x 256 tiles, else 128 x 128
  int64_t splits;  // of K, every one with at least one slice
  double us;
};

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

double tile_us(bool wide, int64_t M, int64_t N, int64_t slices, int64_t splits) {
  const int64_t edge = wide ? 256 : 128, per = ceil_div(slices, splits);
  const int64_t wgs = ceil_div(M, edge) * ceil_div(N, edge) * splits;
  double us = kUsLaunch;
  if (wide) us += ceil_div(wgs, 256) * (per * kUsSlice256 + 2 * kUsEpilogue);
  else if (wgs <= 256) us += per * kUsSlice128 + kUsEpilogue;
  else us += ceil_div(wgs, 512) * (per * kUsSlice128Pair + kUsEpilogue);
  if (splits > 1) us += kUsReduce + static_cast<double>(splits * M * N) * 8.0 / kBytesPerUs;
  return us;
}

// The small tiles' best number of splits, up to `most`. They have to be 5% ahead of the others: a
// workgroup's partials leave under the next round's products, which the model does not see, and
// wide tiles gain more from that (1024 x 768 x 32,001: 66 us against 69, both estimated at 70).
constexpr double kLead = 1.05;

TilePlan best_tiles(bool wide, int64_t M, int64_t N, int64_t slices, int64_t least, int64_t most) {
  const double lead = wide ? 1.0 : kLead;
  TilePlan best = {wide, 0, 0.0};
  for (int64_t s = least; s <= most && s <= slices; ++s) {
    if (ceil_div(slices, ceil_div(slices, s)) != s) continue;  // some split would be empty
    if (s > 1 && s * M * N * 4 > kMaxPartialBytes) break;
    const double us = lead * tile_us(wide, M, N, slices, s);
    if (best.splits == 0 || us < best.us) best = {wide, s, us};
  }
  return best;
}

// Splits of grad_h on 256 x 256 tiles: whole rounds of workgroups at 1.7 us a K slice and 8 us to
// store a partial tile, and the reduction at about 5 TB/s. S = 16 for a 1024-row chunk of the
// Qwen3-0.6B head (dim 1024: 16 tiles, 256 workgroups), 4 for 4096 rows and 2 for 8192 rows.
int64_t wide_splits(int64_t rows, int64_t vocab, int64_t dim) {
  const int64_t tiles = ceil_div(rows, kTile) * ceil_div(dim, kTile), iters = ceil_div(vocab, kSliceK);
  int64_t best = 1;
  double best_us = 0.0;
  for (int64_t s = 1; s <= 256; ++s) {
    const double us = static_cast<double>(ceil_div(tiles * s, 256)) * (1.7 * static_cast<double>(ceil_div(iters, s)) + 8.0) +
                      static_cast<double>(s) * static_cast<double>(rows * dim) * 4.0 / 5e6;
    if (s == 1 || us < best_us) {
      best = s;
      best_us = us;
    }
  }
  return best;
}

TilePlan grad_h_plan(int64_t rows, int64_t vocab, int64_t dim) {
  const int64_t slices = ceil_div(vocab, kSliceK);
  TilePlan plan = {true, wide_splits(rows, vocab, dim), 0.0};
  plan.us = tile_us(true, rows, dim, slices, plan.splits);
  const TilePlan small = best_tiles(false, rows, dim, slices, 1, plan.splits);
  return small.splits > 0 && small.us < plan.us ? small : plan;
}

// The persistent kernels' time: whole rounds of 256 x 256 tiles, the epilogue under the next
// tile's products.
double ring_us(int64_t M, int64_t N, int64_t slices) {
  return kUsLaunch + 2.0 + ceil_div(ceil_div(M, kLgTile) * ceil_div(N, kLgTile), 256) * slices * kUsSlice256;
}

// grad_W on the tile kernel (splits > 0), or on the 256 x 256 kernels (0). Without a workspace
// there are no splits.
TilePlan grad_w_plan(int64_t pad_rows, int64_t vocab, int64_t dim, bool workspace) {
  const int64_t slices = pad_rows / kSliceK;
  TilePlan p = best_tiles(false, vocab, dim, slices, 1, workspace ? 256 : 1);
  const TilePlan wide = best_tiles(true, vocab, dim, slices, 2, workspace ? 256 : 1);
  if (wide.splits > 0 && wide.us < p.us) p = wide;
  return p.us < ring_us(vocab, dim, slices) ? p : TilePlan{true, 0, 0.0};
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The GEMM kernels' dynamic LDS (128-160 KB) exceeds the 64 KB default:
// the attribute is set once per device and kernel, with that device current, before the first
// launch there. The device's CU count (for the ring kernels' workgroups per XCD) is read then.
constexpr int kMaxDevices = 64;
std::mutex g_lds_mu;
bool g_lds_set[15][kMaxDevices] = {};
int g_cus[kMaxDevices] = {};

enum Kernel {
  kGradH, kLogits, kGradW, kLogitsRing, kGradWRing, kGradHRagged, kGradWRagged, kGradWRingRagged,
  kTileLogits, kTileGradH, kTileGradHSplit, kTileGradHWide, kTileGradW, kTileGradWSplit, kTileGradWSplitWide,
};
constexpr int kTileLds128 = 2 * 256 * 128, kTileLds256 = 2 * 512 * 128;

// `cus`, when given, receives the device's CU count.
hipError_t allow_lds(hipStream_t stream, Kernel which, int* cus = nullptr) {
  int dev = -1;
  hipError_t e = stream ? hipStreamGetDevice(stream, &dev) : hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_lds_mu);
  if (g_lds_set[which][dev]) {
    if (cus) *cus = g_cus[dev];
    return hipSuccess;
  }
  int cur = -1;
  e = hipGetDevice(&cur);
  if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
  struct Entry {
    const void* fn;
    int bytes;
  };
  const Entry entries[15] = {
      {reinterpret_cast<const void*>(grad_h_gemm_kernel<false>), 2 * kLgStage},
      {reinterpret_cast<const void*>(logits_gemm_kernel), kLgLds},
      {reinterpret_cast<const void*>(grad_w_gemm_kernel<false>), kLgLds},
      {reinterpret_cast<const void*>(logits_ring_kernel), kRgLds},
      {reinterpret_cast<const void*>(grad_w_ring_kernel<false>), kRgLds},
      {reinterpret_cast<const void*>(grad_h_gemm_kernel<true>), 2 * kLgStage},
      {reinterpret_cast<const void*>(grad_w_gemm_kernel<true>), kLgLds},
      {reinterpret_cast<const void*>(grad_w_ring_kernel<true>), kRgLds},
      {reinterpret_cast<const void*>(gemm_tile_kernel<2, 1, true, true, false>), kTileLds128},
      {reinterpret_cast<const void*>(gemm_tile_kernel<2, 1, true, false, false>), kTileLds128},
      {reinterpret_cast<const void*>(gemm_tile_kernel<2, 1, true, false, true>), kTileLds128},
      {reinterpret_cast<const void*>(gemm_tile_kernel<4, 2, true, false, false>), kTileLds256},
      {reinterpret_cast<const void*>(gemm_tile_kernel<2, 1, false, false, false>), kTileLds128},
      {reinterpret_cast<const void*>(gemm_tile_kernel<2, 1, false, false, true>), kTileLds128},
      {reinterpret_cast<const void*>(gemm_tile_kernel<4, 2, false, false, true>), kTileLds256},
  };
  if (e == hipSuccess)
    e = hipFuncSetAttribute(entries[which].fn, hipFuncAttributeMaxDynamicSharedMemorySize, entries[which].bytes);
  if (e == hipSuccess && g_cus[dev] == 0) e = hipDeviceGetAttribute(&g_cus[dev], hipDeviceAttributeMultiprocessorCount, dev);
  if (cur >= 0 && cur != dev) {
    const hipError_t back = hipSetDevice(cur);
    if (e == hipSuccess) e = back;
  }
  if (e == hipSuccess) {
    g_lds_set[which][dev] = true;
    if (cus) *cus = g_cus[dev];
  }
  return e;
}

// One gemm_tile_kernel launch: M x N outputs of `slices` K slices in `splits` parts.
template <int kMB, int kNB, bool kAK, bool kBK, bool kPartial>
int tile_launch(Kernel which, const uint16_t* A, const uint16_t* B, void* out, int64_t M, int64_t N, int64_t lda,
                int64_t ldb, int64_t ldc, int64_t slices, int64_t kb, int64_t gm, int64_t gn, int64_t splits,
                hipStream_t s, const char* who) {
  const hipError_t lds = allow_lds(s, which);
  if (lds != hipSuccess) return gemm_fail(TM_ELAUNCH, "%s: LDS attribute: %s", who, hipGetErrorString(lds));
  const int64_t tm = ceil_div(M, 64 * kMB), tn = ceil_div(N, 128 * kNB);
  hipLaunchKernelGGL((gemm_tile_kernel<kMB, kNB, kAK, kBK, kPartial>),
                     dim3(static_cast<uint32_t>((tm * tn * splits + 7) / 8 * 8)), dim3(512),
                     (64 * kMB + 128 * kNB) * 256, s, A, B, out, static_cast<int>(M), static_cast<int>(N), lda, ldb, ldc,
                     static_cast<int>(slices), static_cast<int>(kb), static_cast<int>(tm), static_cast<int>(tn),
                     static_cast<int>(gm), static_cast<int>(gn), static_cast<int>(ceil_div(slices, splits)));
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gemm_fail(TM_ELAUNCH, "%s: launch failed: %s", who, hipGetErrorString(e));
  return TM_OK;
}

int reduce_launch(const float* partials, uint16_t* out, int64_t n, int64_t splits, hipStream_t s, const char* who) {
  hipLaunchKernelGGL(splits_reduce_kernel, dim3(static_cast<uint32_t>((n / 4 + 255) / 256)), dim3(256), 0, s, partials,
                     out, n, static_cast<int>(splits));
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gemm_fail(TM_ELAUNCH, "%s: reduction failed: %s", who, hipGetErrorString(e));
  return TM_OK;
}

// small_tiles: the tile kernel where the model finds it faster (the same bits).
int logits_launch(uint16_t* d_logits, int64_t ld, const uint16_t* d_hidden, const uint16_t* d_weight, int64_t rows,
                  int64_t vocab, int64_t dim, bool small_tiles, void* stream) {
  if (rows <= 0 || vocab <= 0 || dim <= 0 || dim % kSliceK)
    return gemm_fail(TM_EINVAL, "tm_ce_logits_bf16: rows %lld and vocab %lld must be positive, dim %lld a positive "
                     "multiple of %d", (long long)rows, (long long)vocab, (long long)dim, kSliceK);
  if (ld < vocab || ld > 0x7FFFFFFF)
    return gemm_fail(TM_EINVAL, "tm_ce_logits_bf16: logits rows %lld elements apart, vocab %lld", (long long)ld,
                     (long long)vocab);
  const int64_t tiles_m = (rows + kLgTile - 1) / kLgTile, tiles_n = (vocab + kLgTile - 1) / kLgTile;
  if (rows > 0x7FFFFFFF || vocab > 0x7FFFFFFF || dim > 0x7FFFFFFF || tiles_m * tiles_n > 0x7FFFFFF0)
    return gemm_fail(TM_EINVAL, "tm_ce_logits_bf16: %lld x %lld x %lld is too large", (long long)rows,
                     (long long)vocab, (long long)dim);
  if (!d_logits || !d_hidden || !d_weight) return gemm_fail(TM_EINVAL, "tm_ce_logits_bf16: null pointer");
  if (!aligned16(d_logits) || !aligned16(d_hidden) || !aligned16(d_weight))
    return gemm_fail(TM_EINVAL, "tm_ce_logits_bf16: pointers must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t slices = dim / kSliceK;
  if (small_tiles && ld % 8 == 0 && kLead * tile_us(false, rows, vocab, slices, 1) < ring_us(rows, vocab, slices)) {
    const int64_t t128 = ceil_div(rows, 128), gm128 = t128 < 4 ? t128 : 4;
    return tile_launch<2, 1, true, true, false>(kTileLogits, d_hidden, d_weight, d_logits, rows, vocab, dim, dim, ld,
                                                slices, vocab, gm128, 32 / gm128, 1, s, "tm_ce_logits_bf16");
  }
  int gm, gn;
  logits_groups(tiles_m, dim, gm, gn);
  if (logits_ring_fits(rows, vocab, dim, ld)) {
    int cus = 0;
    const hipError_t lds = allow_lds(s, kLogitsRing, &cus);
    if (lds != hipSuccess)
      return gemm_fail(TM_ELAUNCH, "tm_ce_logits_bf16: LDS attribute: %s", hipGetErrorString(lds));
    const int wpx = cus >= 16 ? cus / 8 : 1;  // one workgroup per CU of each XCD
    hipLaunchKernelGGL(logits_ring_kernel, dim3(static_cast<uint32_t>(8 * wpx)), dim3(512), kRgLds, s, d_hidden,
                       d_weight, d_logits, static_cast<int>(rows), static_cast<int>(vocab), static_cast<int>(ld),
                       static_cast<int>(dim), static_cast<int>(tiles_m), static_cast<int>(tiles_n), gm, gn, wpx);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return gemm_fail(TM_ELAUNCH, "logits_ring_kernel: launch failed: %s", hipGetErrorString(e));
    return TM_OK;
  }
  const hipError_t lds = allow_lds(s, kLogits);
  if (lds != hipSuccess)
    return gemm_fail(TM_ELAUNCH, "tm_ce_logits_bf16: LDS attribute: %s", hipGetErrorString(lds));
  const int64_t grid = (tiles_m * tiles_n + 7) / 8 * 8;
  hipLaunchKernelGGL(logits_gemm_kernel, dim3(static_cast<uint32_t>(grid)), dim3(256), kLgLds, s, d_hidden, d_weight,
                     d_logits, static_cast<int>(rows), static_cast<int>(vocab), ld, static_cast<int>(dim),
                     static_cast<int>(tiles_m), static_cast<int>(tiles_n), gm, gn);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gemm_fail(TM_ELAUNCH, "logits_gemm_kernel: launch failed: %s", hipGetErrorString(e));
  return TM_OK;
}

// tiles: the tile kernel where the model finds it faster, with splits of K (other bits) if the
// workspace holds them.
int grad_w_launch(uint16_t* d_grad_w, const uint16_t* d_grad_logits, int64_t ld, int64_t pad_rows,
                  const uint16_t* d_hidden, int64_t rows, int64_t vocab, int64_t dim, void* d_ws, size_t ws_bytes,
                  bool tiles, void* stream) {
  if (rows <= 0 || vocab <= 0 || dim <= 0 || dim % 8 || ld % 8 || ld < vocab || pad_rows % kSliceK || pad_rows < rows ||
      pad_rows - rows >= 2 * kTile)
    return gemm_fail(TM_EINVAL, "tm_ce_grad_w_bf16: rows %lld and vocab %lld must be positive, dim %lld a positive "
                     "multiple of 8, grad_logits rows (%lld with padding, a multiple of %d) %lld elements apart, a "
                     "multiple of 8", (long long)rows, (long long)vocab, (long long)dim, (long long)pad_rows, kSliceK,
                     (long long)ld);
  const int64_t tiles_v = (vocab + kLgTile - 1) / kLgTile, tiles_d = (dim + kLgTile - 1) / kLgTile;
  if (pad_rows > 0x7FFFFFFF || ld > 0x7FFFFFFF || dim > 0x7FFFFFFF || tiles_v * tiles_d > 0x7FFFFFF0)
    return gemm_fail(TM_EINVAL, "tm_ce_grad_w_bf16: %lld x %lld x %lld is too large", (long long)rows,
                     (long long)vocab, (long long)dim);
  if (!d_grad_w || !d_grad_logits || !d_hidden) return gemm_fail(TM_EINVAL, "tm_ce_grad_w_bf16: null pointer");
  if (!aligned16(d_grad_w) || !aligned16(d_grad_logits) || !aligned16(d_hidden))
    return gemm_fail(TM_EINVAL, "tm_ce_grad_w_bf16: pointers must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  TilePlan plan = {true, 0, 0.0};
  if (tiles) {
    plan = grad_w_plan(pad_rows, vocab, dim, d_ws != nullptr);
    if (plan.splits > 1 && ws_bytes < static_cast<size_t>(plan.splits) * vocab * dim * sizeof(float))
      return gemm_fail(TM_EINVAL, "tm_ce_grad_w_bf16: workspace of %zu bytes, %zu needed", ws_bytes,
                       static_cast<size_t>(plan.splits) * vocab * dim * sizeof(float));
    if (plan.splits > 1 && !aligned16(d_ws))
      return gemm_fail(TM_EINVAL, "tm_ce_grad_w_bf16: pointers must be 16-byte aligned");
  }
  if (plan.splits > 0) {
    const char* who = "tm_ce_grad_w_bf16";
    const int64_t slices = pad_rows / kSliceK, tn = ceil_div(dim, plan.wide ? 256 : 128);
    const int64_t pn = tn < 8 ? tn : 8, pm = 32 / pn;
    if (plan.splits == 1)
      return tile_launch<2, 1, false, false, false>(kTileGradW, d_grad_logits, d_hidden, d_grad_w, vocab, dim, ld, dim,
                                                    dim, slices, rows, pm, pn, 1, s, who);
    const int rc =
        plan.wide ? tile_launch<4, 2, false, false, true>(kTileGradWSplitWide, d_grad_logits, d_hidden, d_ws, vocab, dim,
                                                          ld, dim, dim, slices, rows, pm, pn, plan.splits, s, who)
                  : tile_launch<2, 1, false, false, true>(kTileGradWSplit, d_grad_logits, d_hidden, d_ws, vocab, dim, ld,
                                                          dim, dim, slices, rows, pm, pn, plan.splits, s, who);
    return rc ? rc : reduce_launch(static_cast<const float*>(d_ws), d_grad_w, vocab * dim, plan.splits, s, who);
  }
  const int gn = static_cast<int>(tiles_d < 4 ? tiles_d : 4), gm = 32 / gn;  // a round of 32: 8 x 4
  const bool ragged = rows != pad_rows, ring = grad_w_ring_fits(pad_rows, ld, dim);
  int cus = 0;
  const hipError_t lds = allow_lds(s, ring ? (ragged ? kGradWRingRagged : kGradWRing) : (ragged ? kGradWRagged : kGradW), &cus);
  if (lds != hipSuccess)
    return gemm_fail(TM_ELAUNCH, "tm_ce_grad_w_bf16: LDS attribute: %s", hipGetErrorString(lds));
  const int V = static_cast<int>(vocab), L = static_cast<int>(ld), D = static_cast<int>(dim),
            K = static_cast<int>(pad_rows), R = static_cast<int>(rows), tv = static_cast<int>(tiles_v),
            td = static_cast<int>(tiles_d);
  if (ring) {
    const int wpx = cus >= 16 ? cus / 8 : 1;
    const dim3 grid(static_cast<uint32_t>(8 * wpx));
    if (ragged)
      hipLaunchKernelGGL(grad_w_ring_kernel<true>, grid, dim3(512), kRgLds, s, d_grad_logits, d_hidden, d_grad_w, V, L, D,
                         K, R, tv, td, gm, gn, wpx);
    else
      hipLaunchKernelGGL(grad_w_ring_kernel<false>, grid, dim3(512), kRgLds, s, d_grad_logits, d_hidden, d_grad_w, V, L,
                         D, K, R, tv, td, gm, gn, wpx);
  } else {
    const dim3 grid(static_cast<uint32_t>((tiles_v * tiles_d + 7) / 8 * 8));
    if (ragged)
      hipLaunchKernelGGL(grad_w_gemm_kernel<true>, grid, dim3(256), kLgLds, s, d_grad_logits, d_hidden, d_grad_w, V, L, D,
                         K, R, tv, td, gm, gn);
    else
      hipLaunchKernelGGL(grad_w_gemm_kernel<false>, grid, dim3(256), kLgLds, s, d_grad_logits, d_hidden, d_grad_w, V, L,
                         D, K, R, tv, td, gm, gn);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gemm_fail(TM_ELAUNCH, "grad_w kernel: launch failed: %s", hipGetErrorString(e));
  return TM_OK;
}

}  // namespace

extern "C" {

size_t tm_ce_grad_h_workspace_bytes(int64_t rows, int64_t vocab, int64_t dim) {
  if (rows % kTile || dim % kTile || vocab % kSliceK) return 0;
  return tm_ce_grad_h_ld_workspace_bytes(rows, vocab, dim);
}

int tm_ce_grad_h_bf16(uint16_t* d_grad_h, const uint16_t* d_grad_logits, const uint16_t* d_w, int64_t rows,
                      int64_t vocab, int64_t dim, void* d_ws, size_t ws_bytes, void* stream) {
  if (rows <= 0 || dim <= 0 || vocab <= 0 || rows % kTile || dim % kTile || vocab % kSliceK)
    return gemm_fail(TM_EINVAL,
                     "tm_ce_grad_h_bf16: rows %lld and dim %lld must be positive multiples of %d, vocab %lld "
                     "of %d", (long long)rows, (long long)dim, kTile, (long long)vocab, kSliceK);
  return tm_ce_grad_h_ld_bf16(d_grad_h, d_grad_logits, vocab, d_w, rows, vocab, dim, d_ws, ws_bytes, stream);
}

size_t tm_ce_grad_h_ld_workspace_bytes(int64_t rows, int64_t vocab, int64_t dim) {
  if (rows <= 0 || dim <= 0 || vocab <= 0 || dim % 8) return 0;
  // enough for either tile size: the small tiles take no more splits than the wide ones would
  return static_cast<size_t>(wide_splits(rows, vocab, dim)) * rows * dim * sizeof(float);
}

int tm_ce_grad_h_ld_bf16(uint16_t* d_grad_h, const uint16_t* d_grad_logits, int64_t ld, const uint16_t* d_w,
                         int64_t rows, int64_t vocab, int64_t dim, void* d_ws, size_t ws_bytes, void* stream) {
  if (rows <= 0 || dim <= 0 || vocab <= 0 || dim % 8 || ld % 8 || ld < (vocab + kSliceK - 1) / kSliceK * kSliceK)
    return gemm_fail(TM_EINVAL,
                     "tm_ce_grad_h_bf16: rows %lld and vocab %lld must be positive, dim %lld a positive multiple of 8, "
                     "grad_logits rows %lld elements apart a multiple of 8 and hold whole groups of %d", (long long)rows,
                     (long long)vocab, (long long)dim, (long long)ld, kSliceK);
  if (rows > (1 << 20) || dim > (1 << 16) || vocab > 0x7FFFFF00)
    return gemm_fail(TM_EINVAL, "tm_ce_grad_h_bf16: rows %lld, dim %lld or vocab %lld too large", (long long)rows,
                     (long long)dim, (long long)vocab);
  if (!d_grad_h || !d_grad_logits || !d_w || !d_ws)
    return gemm_fail(TM_EINVAL, "tm_ce_grad_h_bf16: null pointer");
  if (!aligned16(d_grad_h) || !aligned16(d_grad_logits) || !aligned16(d_w) || !aligned16(d_ws))
    return gemm_fail(TM_EINVAL, "tm_ce_grad_h_bf16: pointers must be 16-byte aligned");
  const size_t need = tm_ce_grad_h_ld_workspace_bytes(rows, vocab, dim);
  if (ws_bytes < need)
    return gemm_fail(TM_EINVAL, "tm_ce_grad_h_bf16: workspace of %zu bytes, %zu needed", ws_bytes, need);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const char* who = "tm_ce_grad_h_bf16";
  const TilePlan plan = grad_h_plan(rows, vocab, dim);
  const int64_t splits = plan.splits, slices = ceil_div(vocab, kSliceK);
  float* partials = static_cast<float*>(d_ws);
  if (!plan.wide || splits == 1) {
    const int64_t gm = ceil_div(rows, plan.wide ? 256 : 128) < 8 ? ceil_div(rows, plan.wide ? 256 : 128) : 8;
    if (splits == 1)
      return plan.wide ? tile_launch<4, 2, true, false, false>(kTileGradHWide, d_grad_logits, d_w, d_grad_h, rows, dim,
                                                               ld, dim, dim, slices, vocab, gm, 4, 1, s, who)
                       : tile_launch<2, 1, true, false, false>(kTileGradH, d_grad_logits, d_w, d_grad_h, rows, dim, ld,
                                                               dim, dim, slices, vocab, gm, 4, 1, s, who);
    const int rc = tile_launch<2, 1, true, false, true>(kTileGradHSplit, d_grad_logits, d_w, partials, rows, dim, ld, dim,
                                                        dim, slices, vocab, gm, 4, splits, s, who);
    return rc ? rc : reduce_launch(partials, d_grad_h, rows * dim, splits, s, who);
  }
  const int64_t tiles = ceil_div(rows, kTile) * ceil_div(dim, kTile), per = ceil_div(slices, splits);
  const bool ragged = rows % kTile != 0 || dim % kTile != 0 || vocab % kSliceK != 0;
  const hipError_t lds = allow_lds(s, ragged ? kGradHRagged : kGradH);
  if (lds != hipSuccess)
    return gemm_fail(TM_ELAUNCH, "tm_ce_grad_h_bf16: LDS attribute: %s", hipGetErrorString(lds));
  const dim3 grid(static_cast<uint32_t>((tiles * splits + 7) / 8 * 8));
  if (ragged)
    hipLaunchKernelGGL(grad_h_gemm_kernel<true>, grid, dim3(512), 2 * kLgStage, s, d_grad_logits, d_w, partials,
                       static_cast<int>(rows), static_cast<int>(dim), ld, static_cast<int>(vocab),
                       static_cast<int>(tiles), static_cast<int>(splits), static_cast<int>(per));
  else
    hipLaunchKernelGGL(grad_h_gemm_kernel<false>, grid, dim3(512), 2 * kLgStage, s, d_grad_logits, d_w, partials,
                       static_cast<int>(rows), static_cast<int>(dim), ld, static_cast<int>(vocab),
                       static_cast<int>(tiles), static_cast<int>(splits), static_cast<int>(per));
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gemm_fail(TM_ELAUNCH, "grad_h_gemm_kernel: launch failed: %s", hipGetErrorString(e));
  return reduce_launch(partials, d_grad_h, rows * dim, splits, s, who);
}

int tm_ce_logits_bf16(uint16_t* d_logits, const uint16_t* d_hidden, const uint16_t* d_weight, int64_t rows,
                      int64_t vocab, int64_t dim, void* stream) {
  return logits_launch(d_logits, vocab, d_hidden, d_weight, rows, vocab, dim, false, stream);
}

int tm_ce_logits_ld_bf16(uint16_t* d_logits, int64_t ld, const uint16_t* d_hidden, const uint16_t* d_weight,
                         int64_t rows, int64_t vocab, int64_t dim, void* stream) {
  return logits_launch(d_logits, ld, d_hidden, d_weight, rows, vocab, dim, true, stream);
}

int tm_ce_grad_w_bf16(uint16_t* d_grad_w, const uint16_t* d_grad_logits, const uint16_t* d_hidden, int64_t rows,
                      int64_t vocab, int64_t dim, void* stream) {
  if (rows <= 0 || vocab <= 0 || dim <= 0 || rows % kSliceK || vocab % 8 || dim % 8)
    return gemm_fail(TM_EINVAL, "tm_ce_grad_w_bf16: rows %lld must be a positive multiple of %d, vocab %lld and dim "
                     "%lld positive multiples of 8", (long long)rows, kSliceK, (long long)vocab, (long long)dim);
  return grad_w_launch(d_grad_w, d_grad_logits, vocab, rows, d_hidden, rows, vocab, dim, nullptr, 0, false, stream);
}

size_t tm_ce_grad_w_ld_workspace_bytes(int64_t pad_rows, int64_t vocab, int64_t dim) {
  if (pad_rows <= 0 || vocab <= 0 || dim <= 0 || pad_rows % kSliceK) return 0;
  const TilePlan plan = grad_w_plan(pad_rows, vocab, dim, true);
  return plan.splits > 1 ? static_cast<size_t>(plan.splits) * vocab * dim * sizeof(float) : 0;
}

int tm_ce_grad_w_ld_bf16(uint16_t* d_grad_w, const uint16_t* d_grad_logits, int64_t ld, int64_t pad_rows,
                         const uint16_t* d_hidden, int64_t rows, int64_t vocab, int64_t dim, void* d_ws,
                         size_t ws_bytes, void* stream) {
  return grad_w_launch(d_grad_w, d_grad_logits, ld, pad_rows, d_hidden, rows, vocab, dim, d_ws, ws_bytes, true, stream);
}

}  // extern "C"
