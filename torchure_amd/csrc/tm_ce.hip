// tm_ce.hip -- gfx950 kernels of the chunked fused linear + cross-entropy.
//
// The reference (torchure/loss/fused_linear_ce.py:31-59) computes, per chunk of rows,
//   logits = h @ W^T (bf16 GEMM), lse = logsumexp(float(logits)), loss = lse - target,
//   grad_logits = bf16(softmax - onehot) on valid rows (0 on ignored rows),
//   grad_h = grad_logits @ W, grad_W += grad_logits^T @ h,
// and scales both grads by grad_out / n_valid in backward (:94-127).
// The GEMMs are in tm_ce_gemm.hip. These kernels do the rest:
//   ce_rows_kernel        one workgroup per row: row max, sum of exp, target logit,
//                         per-row loss, then softmax - onehot written back over the
//                         logits as bf16 (RNE). A row of up to kRegCols vectors per
//                         thread (1 to 16 waves by the vocabulary) stays in registers
//                         (one HBM read, one write); longer
//                         rows use an online (max, sum-of-exp) read, then a second
//                         read for the write pass. exp is the hardware base-2 exp
//                         (full-range exp2f wherever a result would be denormal), and
//                         the bf16 rounding is the hardware RNE convert.
//   ce_loss_kernel        one workgroup: fixed-order sum of the per-row losses and of
//                         the valid-row count -> loss_sum, n_valid, mean loss.
//   ce_grads_kernel       the chunks' bf16 grad_W added into the fp32 grad_W, and backward's
//                         scaling: grad_W *= g / n_valid, grad_h (bf16) *= bf16(g / n_valid) or
//                         its fp32 widening times g / n_valid, in one launch.

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include <type_traits>

#include "torchure_amd.h"
#include "tm_internal.h"

#pragma clang fp contract(off)

namespace {

constexpr int kRowThreadsMax = 1024;    // 16 wave64 on a row of the largest vocabularies kept in registers
constexpr int kRowThreadsStream = 256;  // threads per row on the streaming path (longer rows)
constexpr int kStreamUnroll = 4;  // vectors per thread loaded together on the streaming path
constexpr int kRegCols = 20;  // most 8-element vectors per thread kept in registers (V <= 163,840)
constexpr int kMaxWaves = kRowThreadsMax / 64;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename... A>
int ce_fail(int code, const char* fmt, A... args) {
  return tm_internal_fail(code, fmt, args...);
}

__device__ __forceinline__ float lo16(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi16(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ uint32_t rne16(float f) {
  const uint32_t u = __float_as_uint(f);
  const uint32_t r = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
  return (f != f) ? 0x7FC0u : r;
}

constexpr float kLog2e = 1.4426950408889634f;

// The exponent (x - c) * log2(e) of exp(x - c). With kFold it is one fma against the
// precomputed cl = c * log2(e); cl carries an absolute rounding error of half an ulp of
// |c| * log2(e), which for |c| <= kFoldMax is at most 3.8e-6 (a relative error below
// 2.6e-6 in the result, far under half a bf16 ulp). Rows with larger |c| take the two-step
// form, exact at x = c and accurate at any magnitude.
constexpr float kFoldMax = 64.0f;

template <bool kFold>
__device__ __forceinline__ float tlog2(float x, float c, float cl) {
  return kFold ? fmaf(x, kLog2e, -cl) : (x - c) * kLog2e;
}

// exp(x - c) through the base-2 exponential: exp2((x - c) * log2(e)), full range
// (denormal results included).
__device__ __forceinline__ float exp_shift(float x, float c) { return exp2f((x - c) * kLog2e); }

// The bare v_exp_f32: identical to exp2f for results >= 2^-126, flushes smaller ones.
__device__ __forceinline__ float exp2_hw(float t) { return __builtin_amdgcn_exp2f(t); }

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two floats -> packed bf16 (round to nearest even) in one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  const bf16x2 h = __builtin_convertvector(f32x2{a, b}, bf16x2);
  return __builtin_bit_cast(uint32_t, h);
}

// (max, sum of exp(x - max)) pairs combine associatively.
__device__ __forceinline__ void ms_merge(float& m, float& s, float m2, float s2) {
  if (m2 == -INFINITY) return;
  if (m2 > m) {
    s = s * exp_shift(m, m2) + s2;
    m = m2;
  } else if (m2 == m) {
    s = s + s2;
  } else {
    s = s + s2 * exp_shift(m2, m);
  }
}

__device__ __forceinline__ void ms_add(float& m, float& s, float x) {
  if (x == -INFINITY) return;  // exp(-inf - m) = 0 contributes nothing
  if (x > m) {
    s = s * exp_shift(m, x) + 1.0f;
    m = x;
  } else {
    s = s + exp_shift(x, m);
  }
}

// Block-wide (max, sumexp) in a fixed order; every thread receives the result.
template <int kCeThreads>
__device__ __forceinline__ void block_ms(float& m, float& s) {
  constexpr int kCeWaves = kCeThreads / 64;
  __shared__ float lm[kMaxWaves], ls[kMaxWaves];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float m2 = __shfl_xor(m, off, 64);
    const float s2 = __shfl_xor(s, off, 64);
    ms_merge(m, s, m2, s2);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    lm[wave] = m;
    ls[wave] = s;
  }
  __syncthreads();
  m = lm[0];
  s = ls[0];
  for (int w = 1; w < kCeWaves; ++w) ms_merge(m, s, lm[w], ls[w]);
  __syncthreads();
}

// (m, s) and (m2, s2) combined against the larger maximum (0 where both are -inf): unlike
// ms_merge, a NaN sum under a maximum of -inf (a part of the row that is all NaN) is kept.
__device__ __forceinline__ void ms_join(float& m, float& s, float m2, float s2) {
  const float top = fmaxf(m, m2);
  const float ref = top == -INFINITY ? 0.0f : top;
  s = s * exp_shift(m, ref) + s2 * exp_shift(m2, ref);
  m = top;
}

// Block-wide (max, sum of exp) and maximum of b (a negated minimum) in one fixed-order
// reduction; every thread receives the results.
template <int kCeThreads>
__device__ __forceinline__ void block_join(float& m, float& s, float& b) {
  constexpr int kCeWaves = kCeThreads / 64;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float m2 = __shfl_xor(m, off, 64), s2 = __shfl_xor(s, off, 64);
    ms_join(m, s, m2, s2);
    b = fmaxf(b, __shfl_xor(b, off, 64));
  }
  if constexpr (kCeWaves > 1) {
    __shared__ float lm[kMaxWaves], ls[kMaxWaves], lb[kMaxWaves];
    if ((threadIdx.x & 63) == 0) {
      lm[threadIdx.x >> 6] = m;
      ls[threadIdx.x >> 6] = s;
      lb[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    // every wave reduces the waves' results itself, in lanes (a serial walk over 16 of them took
    // a chain of 32 exponentials)
    const int w = threadIdx.x & (kCeWaves - 1);
    m = lm[w];
    s = ls[w];
    b = lb[w];
#pragma unroll
    for (int off = kCeWaves / 2; off > 0; off >>= 1) {
      const float m2 = __shfl_xor(m, off, 64), s2 = __shfl_xor(s, off, 64);
      ms_join(m, s, m2, s2);
      b = fmaxf(b, __shfl_xor(b, off, 64));
    }
  }
}

// logits: rows x vocab bf16 (row-major, row stride ld elements), overwritten with
// grad_logits (kGrad; without it the logits are only read). labels: int64 per row.
// row_loss: fp32 per row (0 for ignored rows). Columns vocab .. width - 1, and rows from n_rows
// on, are padding that the gradient pass sets to zero for the GEMMs (width = vocab: no padding).
//
// kCols > 0: the row stays in registers, kCols vectors of 8 a thread (kCols * kCeThreads * 8 >=
// vocab); kCols = 0: a row too long for them. Bound: HBM, at 4 bytes an element (2 without the
// gradient), once enough rows are in flight. A workgroup goes through load, reduce, exponentials
// and stores in series, so a CU needs other rows to load while one reduces: the fewest waves
// whose registers hold the row (row_shape) leave room for 16 rows a CU up to a vocabulary of
// 10,240, 4 at 32,768 and one from 81,921 up, where a row fills the register file. A fixed
// 1024 threads of 20 vectors had one row a CU at every vocabulary, and reloaded the last vector
// in place of the missing ones. Measured on MI355X, logits not in cache, fixed / this shape:
//   8192 x 4096: 253 / 26 us (5.2 TB/s); 4096 x 32,768: 188 / 109 us; 4096 x 81,920: 304 / 249 us;
//   8192 x 151,936: 965 / 965 us (5.2 TB/s), 1024 rows of it 143 / 131 us; loss only 475 / 364 us
//   (6.8 TB/s: with 12 vectors held instead of the row, two rows a CU).
template <int kCols, int kCeThreads, bool kGrad>
__global__ __launch_bounds__(kCeThreads, kGrad ? 4 : 8) void ce_rows_kernel(uint16_t* __restrict__ logits,
                                                             int64_t ld,
                                                             const int64_t* __restrict__ labels,
                                                             int64_t vocab, int64_t ignore_index,
                                                             float* __restrict__ row_loss, int64_t n_rows,
                                                             int64_t width) {
  const int64_t r = blockIdx.x;
  uint16_t* row = logits + r * ld;
  if (kGrad && r >= n_rows) {  // a padding row, 16-byte aligned and whole vectors
    for (int64_t v = threadIdx.x; v < width / 8; v += kCeThreads)
      __builtin_nontemporal_store(u32x4{0u, 0u, 0u, 0u}, reinterpret_cast<u32x4*>(row + v * 8));
    return;
  }
  const int64_t label = labels[r];
  const bool valid = label != ignore_index;
  const int64_t nvec = vocab >> 3;  // full 8-element vectors (16 B)
  const bool vec = ((reinterpret_cast<uint64_t>(row) & 15u) == 0);
  const int64_t vend = vec ? nvec * 8 : 0;

  constexpr bool kInRegs = kCols > 0;
  constexpr int kBatch = 4;                                       // vectors a thread takes together
  constexpr int kHeld = kGrad ? kCols : (kCols < 12 ? kCols : 12);  // vectors a thread holds
  u32x4 keep[kInRegs ? kHeld : 1];
  float lse;
  float row_min = -INFINITY;  // known only on the register path
  if constexpr (kInRegs) {
    // Each thread keeps a running (max, sum of exp) over batches of kBatch vectors, so a batch
    // is reduced while the later ones are still loading. With the gradient the whole row stays
    // in registers, every load issued before any is used; the loss alone needs each batch once
    // and holds three. Compile-time indices keep `keep` in VGPRs. A thread past the row's last
    // vector loads that vector again, a real element of the row, which leaves the max and min as
    // they are; the sum and the stores below skip those slots. The loss-only pass reads the row
    // non-temporally (3-22% faster than temporal loads from 1024 to 8192 rows of the Qwen3
    // vocabulary, same bits); the gradient pass, which rewrites the row, measured no better with
    // them at 2048 rows and beyond.
    float m = -INFINITY, s = 0.0f;
    float nmin = -INFINITY;  // -(row minimum), for the gradient pass
    if (vec && nvec > 0) {
      auto load = [&](int k) {
        const int64_t v = threadIdx.x + static_cast<int64_t>(k) * kCeThreads;
        const u32x4* src = reinterpret_cast<const u32x4*>(row + (v < nvec ? v : nvec - 1) * 8);
        keep[k % kHeld] = kGrad ? *src : __builtin_nontemporal_load(src);
      };
#pragma unroll
      for (int k = 0; k < kHeld; ++k) load(k);
      __builtin_amdgcn_sched_barrier(0);  // keep the scheduler from starting the max before the last load
#pragma unroll
      for (int k0 = 0; k0 < kCols; k0 += kBatch) {
        float top = m;
#pragma unroll
        for (int k = k0; k < k0 + kBatch; ++k) {
          const u32x4 w = keep[k % kHeld];
          top = fmaxf(top, fmaxf(fmaxf(fmaxf(lo16(w.x), hi16(w.x)), fmaxf(lo16(w.y), hi16(w.y))),
                                 fmaxf(fmaxf(lo16(w.z), hi16(w.z)), fmaxf(lo16(w.w), hi16(w.w)))));
          if (kGrad)
            nmin = fmaxf(nmin, -fminf(fminf(fminf(lo16(w.x), hi16(w.x)), fminf(lo16(w.y), hi16(w.y))),
                                      fminf(fminf(lo16(w.z), hi16(w.z)), fminf(lo16(w.w), hi16(w.w)))));
        }
        // the compiler must finish the minimum here and unpack the vectors again for each use: put
        // off, or kept unpacked, the row's elements take twice the registers and spill
        asm volatile("" : "+v"(nmin));
        auto opaque = [&] {
#pragma unroll
          for (int k = k0; k < k0 + kBatch; ++k)
            asm volatile("" : "+v"(keep[k % kHeld]));
        };
        opaque();
        const float ref = top == -INFINITY ? 0.0f : top;
        // terms below 2^-126 (flushed by the bare exp) cannot move a sum that is >= 1
        s = s * exp2_hw(tlog2<false>(m, ref, 0.0f));
        m = top;
#pragma unroll
        for (int k = k0; k < k0 + kBatch; ++k) {
          if (threadIdx.x + static_cast<int64_t>(k) * kCeThreads < nvec) {
            const u32x4 w = keep[k % kHeld];
            auto e = [&](float x) { return exp2_hw(tlog2<false>(x, ref, 0.0f)); };
            s += ((e(lo16(w.x)) + e(hi16(w.x))) + (e(lo16(w.y)) + e(hi16(w.y)))) +
                 ((e(lo16(w.z)) + e(hi16(w.z))) + (e(lo16(w.w)) + e(hi16(w.w))));
          }
        }
        opaque();
        __builtin_amdgcn_sched_barrier(0);  // and one batch's exponentials at a time
        if (!kGrad) {
#pragma unroll
          for (int k = k0 + kHeld; k < k0 + kHeld + kBatch && k < kCols; ++k) load(k);
        }
      }
    }
    if (vend < vocab) {  // the last few elements, or a row that is not 16-byte aligned
      float top = m;
      for (int64_t i = vend + threadIdx.x; i < vocab; i += kCeThreads) {
        const float x = __uint_as_float(static_cast<uint32_t>(row[i]) << 16);
        top = fmaxf(top, x);
        nmin = fmaxf(nmin, -x);
      }
      const float ref = top == -INFINITY ? 0.0f : top;
      s = s * exp_shift(m, ref);
      m = top;
      for (int64_t i = vend + threadIdx.x; i < vocab; i += kCeThreads)
        s += exp_shift(__uint_as_float(static_cast<uint32_t>(row[i]) << 16), ref);
    }
    block_join<kCeThreads>(m, s, nmin);
    row_min = -nmin;
    lse = m + logf(s);
  } else {
    // Row too long for registers: one online (max, sum-of-exp) read, one write pass.
    float m = -INFINITY, s = 0.0f;
    if (vec) {
      // 8 independent (max, sum) pairs per thread (one per vector lane) for ILP
      float mm[8], ss[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        mm[j] = -INFINITY;
        ss[j] = 0.0f;
      }
      auto add8 = [&](const u32x4 w) {
        ms_add(mm[0], ss[0], lo16(w.x)); ms_add(mm[1], ss[1], hi16(w.x));
        ms_add(mm[2], ss[2], lo16(w.y)); ms_add(mm[3], ss[3], hi16(w.y));
        ms_add(mm[4], ss[4], lo16(w.z)); ms_add(mm[5], ss[5], hi16(w.z));
        ms_add(mm[6], ss[6], lo16(w.w)); ms_add(mm[7], ss[7], hi16(w.w));
      };
      // kStreamUnroll loads in flight before they are used, same element order per lane
      int64_t v = threadIdx.x;
      for (; v + (kStreamUnroll - 1) * kCeThreads < nvec; v += kStreamUnroll * kCeThreads) {
        u32x4 w[kStreamUnroll];
#pragma unroll
        for (int u = 0; u < kStreamUnroll; ++u)
          w[u] = *reinterpret_cast<const u32x4*>(row + (v + u * kCeThreads) * 8);
#pragma unroll
        for (int u = 0; u < kStreamUnroll; ++u) add8(w[u]);
      }
      for (; v < nvec; v += kCeThreads) add8(*reinterpret_cast<const u32x4*>(row + v * 8));
#pragma unroll
      for (int j = 0; j < 8; ++j) ms_merge(m, s, mm[j], ss[j]);
    }
    for (int64_t i = vend + threadIdx.x; i < vocab; i += kCeThreads)
      ms_add(m, s, __uint_as_float(static_cast<uint32_t>(row[i]) << 16));
    block_ms<kCeThreads>(m, s);
    lse = m + logf(s);
  }

  // every thread has the same lse; the target logit is read before any write
  const float target = (valid && label >= 0 && label < vocab)
                           ? __uint_as_float(static_cast<uint32_t>(row[label]) << 16)
                           : 0.0f;
  __syncthreads();
  // A label outside [0, vocab) that is not ignore_index makes the reference's gather fail
  // (a device-side assert); here the row's loss is NaN, so the mean loss shows it without a
  // host synchronisation. Its gradient row is the plain softmax.
  const bool in_range = label >= 0 && label < vocab;
  if (threadIdx.x == 0) row_loss[r] = !valid ? 0.0f : (in_range ? lse - target : __builtin_nanf(""));
  if constexpr (!kGrad) return;  // loss only: no gradient pass (no barrier follows)

  // grad = exp(x - lse) on valid rows (0 on ignored rows), minus 1 at the label.
  auto g_of = [&](float x, int64_t idx) -> float {
    if (!valid) return 0.0f;
    float p = exp_shift(x, lse);
    if (idx == label) p = p - 1.0f;
    return p;
  };
  const int64_t label_vec = (valid && label >= 0) ? (label >> 3) : -1;
  const float cl = lse * kLog2e;
  const bool fold = fabsf(lse) <= kFoldMax;
  // both exponent forms are monotonic in x, so the smallest exponent of the row is the row
  // minimum's: if it is >= -126 no result of the row is denormal and every vector takes the
  // bare exp (row_min is -inf on the streaming path, which then checks per vector)
  const bool row_fast = (fold ? tlog2<true>(row_min, lse, cl) : tlog2<false>(row_min, lse, cl)) >= -126.0f;
  auto put8 = [&](const u32x4 w, int64_t v, auto fold_tag) {
    constexpr bool F = decltype(fold_tag)::value;
    const int64_t b = v * 8;
    u32x4 o;
    if (!valid) {
      o = u32x4{0u, 0u, 0u, 0u};
    } else {
      float t[8] = {tlog2<F>(lo16(w.x), lse, cl), tlog2<F>(hi16(w.x), lse, cl),
                    tlog2<F>(lo16(w.y), lse, cl), tlog2<F>(hi16(w.y), lse, cl),
                    tlog2<F>(lo16(w.z), lse, cl), tlog2<F>(hi16(w.z), lse, cl),
                    tlog2<F>(lo16(w.w), lse, cl), tlog2<F>(hi16(w.w), lse, cl)};
      float p[8];
      bool fast = row_fast;
      if (!fast) {
        const float tmin = fminf(fminf(fminf(t[0], t[1]), fminf(t[2], t[3])),
                                 fminf(fminf(t[4], t[5]), fminf(t[6], t[7])));
        fast = tmin >= -126.0f;
      }
      if (fast) {
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = exp2_hw(t[j]);
      } else {  // some result is a denormal: the full-range exp2
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = exp2f(t[j]);
      }
      if (v == label_vec) p[label & 7] = p[label & 7] - 1.0f;
      o.x = pack_bf16x2(p[0], p[1]);
      o.y = pack_bf16x2(p[2], p[3]);
      o.z = pack_bf16x2(p[4], p[5]);
      o.w = pack_bf16x2(p[6], p[7]);
    }
    // non-temporal: the GEMMs that read grad_logits next find none of it in cache anyway
    // (0.3-2.5 GB); 0-7% faster than temporal stores from 8192 down to 1024 rows
    __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(row + b));
  };
  auto write_row = [&](auto fold_tag) {
    if constexpr (kInRegs && kGrad) {
#pragma unroll
      for (int k = 0; k < kCols; ++k) {
        const int64_t v = threadIdx.x + static_cast<int64_t>(k) * kCeThreads;
        u32x4 w = keep[k];
        asm volatile("" : "+v"(w));  // unpacked here, not before the branches
        if (v < nvec) put8(w, v, fold_tag);
      }
    } else {
      int64_t v = threadIdx.x;
      for (; v + (kStreamUnroll - 1) * kCeThreads < nvec; v += kStreamUnroll * kCeThreads) {
        u32x4 w[kStreamUnroll];
#pragma unroll
        for (int u = 0; u < kStreamUnroll; ++u)
          w[u] = *reinterpret_cast<const u32x4*>(row + (v + u * kCeThreads) * 8);
#pragma unroll
        for (int u = 0; u < kStreamUnroll; ++u) put8(w[u], v + u * kCeThreads, fold_tag);
      }
      for (; v < nvec; v += kCeThreads) put8(*reinterpret_cast<const u32x4*>(row + v * 8), v, fold_tag);
    }
  };
  if (vec) {
    if (fold) write_row(std::true_type{});
    else write_row(std::false_type{});
  }
  for (int64_t i = vend + threadIdx.x; i < vocab; i += kCeThreads)
    row[i] = static_cast<uint16_t>(rne16(g_of(__uint_as_float(static_cast<uint32_t>(row[i]) << 16), i)));
  for (int64_t i = vocab + threadIdx.x; i < width; i += kCeThreads) row[i] = 0;
}

// x joined to (max, sum of exp(x - max)), with the full-precision expf, for fp32 outputs.
__device__ __forceinline__ void ms_add_f(float& m, float& s, float x) {
  if (x == -INFINITY) return;
  if (x > m) {
    s = s * expf(m - x) + 1.0f;
    m = x;
  } else {
    s = s + (x == m ? 1.0f : expf(x - m));  // equal: exp(0), also where both are +inf
  }
}

// What the sum's exponents are taken against: the maximum, 0 where that is infinite, as
// torch.logsumexp does: a +inf logit makes lse +inf, not NaN, however many there are (ms_add_f counts
// them).
__device__ __forceinline__ float finite_ref(float top) { return fabsf(top) == INFINITY ? 0.0f : top; }

// What a sum under the maximum m is multiplied by when the maximum becomes top (>= m).
__device__ __forceinline__ float raised(float m, float top) { return m == top ? 1.0f : expf(m - top); }

// fp32 logits: hidden states and weight in fp32 outside autocast, where the reference's
// products are fp32 GEMMs (fused_linear_ce.py:38,52,57 with w = weight.to(hidden.dtype) at
// :65) and its chunk math runs on fp32 logits (:39-51): lse = max + log(sum), then (kGrad) the
// gradient in place, exp(x - lse) on valid rows (0 on ignored rows) minus 1 at the label, with
// the reference's rounding steps: the fp32 difference x - lse, then a full-precision exp.
// One workgroup of kCeThreads per row. kCols > 0: the row stays in registers, kCols vectors of 4
// a thread, all loaded before the first is used and reduced by batches, so it is read once.
// kCols = 0: longer rows, read by batches and again for the gradient, and rows off 16 bytes,
// element by element. Bound: HBM, 8 bytes an element (4 for the loss alone). Against 256 threads
// that read every row twice with an online (max, sum): 1024 x 20,008 52 -> 40 us (4.1 TB/s), the
// loss alone 30 -> 19; 4096 x 4096 36 -> 27; 256 x 151,936 (too long) 230 -> 96; 1024 x 20,001
// (off 16 bytes) 90 -> 59.
template <int kCols, int kCeThreads, bool kGrad>
__global__ __launch_bounds__(kCeThreads, 4) void ce_rows_f32_kernel(float* __restrict__ logits, int64_t ld,
                                                                    const int64_t* __restrict__ labels,
                                                                    int64_t vocab, int64_t ignore_index,
                                                                    float* __restrict__ row_loss) {
  const int64_t r = blockIdx.x;
  float* row = logits + r * ld;
  const int64_t label = labels[r];
  const bool valid = label != ignore_index;
  const int64_t nvec = vocab >> 2;  // full 4-element vectors (16 B)
  const bool vec = ((reinterpret_cast<uint64_t>(row) & 15u) == 0);
  const int64_t vend = vec ? nvec * 4 : 0;
  constexpr int kBatch = kCols > 0 && kCols < 4 ? kCols : 4;
  f32x4 keep[kCols > 0 ? kCols : kBatch];
  float m = -INFINITY, s = 0.0f;
  auto load = [&](int64_t v) {  // past the end: the last vector again, skipped in add
    return *reinterpret_cast<const f32x4*>(row + (v < nvec ? v : nvec - 1) * 4);
  };
  auto add = [&](const f32x4* w, int64_t v0) {  // kBatch vectors, the first one v0
    float top = m;
#pragma unroll
    for (int k = 0; k < kBatch; ++k) top = fmaxf(top, fmaxf(fmaxf(w[k].x, w[k].y), fmaxf(w[k].z, w[k].w)));
    const float ref = finite_ref(top);
    s = s * raised(m, top);
    m = top;
#pragma unroll
    for (int k = 0; k < kBatch; ++k)
      if (v0 + k * kCeThreads < nvec)
        s += (expf(w[k].x - ref) + expf(w[k].y - ref)) + (expf(w[k].z - ref) + expf(w[k].w - ref));
  };
  if (vec && nvec > 0) {
    if constexpr (kCols > 0) {
#pragma unroll
      for (int k = 0; k < kCols; ++k) keep[k] = load(threadIdx.x + static_cast<int64_t>(k) * kCeThreads);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < kCols; k += kBatch) {
        add(keep + k, threadIdx.x + static_cast<int64_t>(k) * kCeThreads);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      for (int64_t v = threadIdx.x; v < nvec; v += kBatch * kCeThreads) {
#pragma unroll
        for (int k = 0; k < kBatch; ++k) keep[k] = load(v + k * kCeThreads);
        add(keep, v);
      }
    }
  }
  for (int64_t i = vend + threadIdx.x; i < vocab; i += kCeThreads) ms_add_f(m, s, row[i]);
  // The workgroup's (max, sum) in a fixed order, in every thread: the maximum first, so that a
  // thread's sum is rescaled once a level (4096 x 1024: 15.8 us merging pairs step by step, 11.4 so).
  constexpr int kCeWaves = kCeThreads / 64;
  auto join = [&](int lanes) {
    float top = m;
#pragma unroll
    for (int off = lanes / 2; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off, 64));
    s = s * raised(m, top);
    m = top;
#pragma unroll
    for (int off = lanes / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  };
  join(64);
  __shared__ float lm[kCeWaves], ls[kCeWaves];
  if ((threadIdx.x & 63) == 0) {
    lm[threadIdx.x >> 6] = m;
    ls[threadIdx.x >> 6] = s;
  }
  __syncthreads();
  m = lm[threadIdx.x & (kCeWaves - 1)];
  s = ls[threadIdx.x & (kCeWaves - 1)];
  join(kCeWaves);
  const float lse = m + logf(s);
  const bool in_range = label >= 0 && label < vocab;
  const float target = (valid && in_range) ? row[label] : 0.0f;
  __syncthreads();  // the target is read before any write
  if (threadIdx.x == 0) row_loss[r] = !valid ? 0.0f : (in_range ? lse - target : __builtin_nanf(""));
  if constexpr (!kGrad) return;
  auto g_of = [&](float x, int64_t idx) -> float {
    if (!valid) return 0.0f;
    const float p = expf(x - lse);
    return idx == label ? p - 1.0f : p;
  };
  auto put = [&](const f32x4 x, int64_t v) {
    const int64_t b = v * 4;
    const f32x4 g = {g_of(x.x, b), g_of(x.y, b + 1), g_of(x.z, b + 2), g_of(x.w, b + 3)};
    *reinterpret_cast<f32x4*>(row + b) = g;  // read next by the products
  };
  if (vec) {
    if constexpr (kCols > 0) {
#pragma unroll
      for (int k = 0; k < kCols; ++k) {
        const int64_t v = threadIdx.x + static_cast<int64_t>(k) * kCeThreads;
        if (v < nvec) put(keep[k], v);
      }
    } else {
      for (int64_t v = threadIdx.x; v < nvec; v += kCeThreads) put(*reinterpret_cast<const f32x4*>(row + v * 4), v);
    }
  }
  for (int64_t i = vend + threadIdx.x; i < vocab; i += kCeThreads) row[i] = g_of(row[i], i);
}

// Fixed-order sums over rows: loss_sum, n_valid (count of label != ignore), mean. One workgroup,
// whose time is the latency of its loads: 1024 threads with 4 rows of each in flight (8192 rows:
// 10 us, against 16 with 256 threads and one row at a time).
constexpr int kLossThreads = 1024, kLossUnroll = 4;
__global__ __launch_bounds__(kLossThreads) void ce_loss_kernel(const float* __restrict__ row_loss,
                                                               const int64_t* __restrict__ labels, int64_t rows,
                                                               int64_t ignore_index, float* __restrict__ out2,
                                                               float* __restrict__ mean) {
  __shared__ double sl[kLossThreads / 64];
  __shared__ long long sn[kLossThreads / 64];
  double acc = 0.0;
  long long cnt = 0;
  for (int64_t i0 = threadIdx.x; i0 < rows; i0 += kLossThreads * kLossUnroll) {
    float x[kLossUnroll];
    int64_t l[kLossUnroll];
#pragma unroll
    for (int u = 0; u < kLossUnroll; ++u) {
      const int64_t i = i0 + u * kLossThreads;
      x[u] = i < rows ? row_loss[i] : 0.0f;
      l[u] = i < rows ? labels[i] : ignore_index;
    }
#pragma unroll
    for (int u = 0; u < kLossUnroll; ++u) {
      acc += static_cast<double>(x[u]);
      cnt += l[u] != ignore_index;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    acc += __shfl_xor(acc, off, 64);
    cnt += __shfl_xor(cnt, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    sl[threadIdx.x >> 6] = acc;
    sn[threadIdx.x >> 6] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double total = 0.0;
    long long n = 0;
    for (int w = 0; w < kLossThreads / 64; ++w) {
      total += sl[w];
      n += sn[w];
    }
    const float loss_sum = static_cast<float>(total);
    const float n_valid = static_cast<float>(n < 1 ? 1 : n);  // clamp_min(1)
    out2[0] = loss_sum;
    out2[1] = n_valid;
    *mean = loss_sum / n_valid;
  }
}

// grad_W hand-over (fused_linear_ce.py:80-81 for each chunk in order, and :126 with kScale):
// acc = ((((kAccumulate ? acc : +0) + float(c[0])) + float(c[1])) + ...) [* g / n_valid] over
// n chunks (1 to kMaxFold) in one pass. The reference adds each chunk into a zero-filled
// buffer (+0 + x also maps -0 to +0), so every element sees its fp32 operations in its order:
// the bits of one `+=` per chunk, then `mul_`, for one read and one write of the accumulator
// per n chunks. One wave per 256-element slice and one group of 4 per lane: each load or store
// instruction of the wave is one contiguous span (1 KiB of the fp32 accumulator, 512 B of each
// bf16 chunk), non-temporal, as in the optimizer's update. The slice that holds the end of a
// length not a multiple of 4, and every slice when a pointer is not aligned for the vectors,
// goes element by element.
constexpr int kMaxFold = 8;
struct FoldChunks {
  const uint16_t* p[kMaxFold];
};
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

#define CE_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ T ld_nt(const T* p) {
  return __builtin_nontemporal_load((const CE_GLOBAL T*)p);
}
template <typename T>
__device__ __forceinline__ void st_nt(T* p, T v) {
  __builtin_nontemporal_store(v, (CE_GLOBAL T*)p);
}

// grad_h's part of backward, over the slices after grad_W's in the same launch (one launch less,
// and vectors where the scaling went 2 bytes at a time: 15 us for 8192 x 1024). 512 elements a
// wave, two groups of 4 a lane, both loaded before either is stored (8192 x 1024: under 6 us).
// fused_linear_ce.py:117-126: bf16 grad_h *= bf16(g / n_valid), the scale cast to the grad's
// dtype, then a bf16 multiply. fp32 hidden states under autocast (:68,80,120; wide): the
// reference's fp32 buffer holds the widened bf16 GEMM result (-0 kept) and is scaled in fp32.
// Without autocast (single): grad_h is fp32 and scaled in place.
struct GradH {
  const uint16_t* src;
  void* dst;  // src itself (bf16), or fp32 when wide or single
  int64_t n;
  bool wide, single;
};
constexpr int kGradHSlice = 512;

__device__ __forceinline__ void grad_h_slice(const GradH& gh, int64_t start, float scale) {
  const float scale_b = __uint_as_float(rne16(scale) << 16);
  const bool vec = (reinterpret_cast<uint64_t>(gh.src) & 7u) == 0 &&
                   (reinterpret_cast<uint64_t>(gh.dst) & (gh.wide ? 15u : 7u)) == 0;
  const int64_t end = start + kGradHSlice < gh.n ? start + kGradHSlice : gh.n;
  int64_t done = start;
  if (gh.single) {
    float* g = static_cast<float*>(gh.dst);
    for (int64_t i = start + threadIdx.x; i < end; i += 64) g[i] = g[i] * scale;
    return;
  }
  if (vec) {
    done = start + ((end - start) & ~int64_t(3));
    const int64_t e0 = start + static_cast<int64_t>(threadIdx.x) * 4, e1 = e0 + 256;
    u32x2 w[2] = {};
    if (e0 < done) w[0] = ld_nt(reinterpret_cast<const u32x2*>(gh.src + e0));
    if (e1 < done) w[1] = ld_nt(reinterpret_cast<const u32x2*>(gh.src + e1));
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t e = u == 0 ? e0 : e1;
      if (e >= done) continue;
      const f32x4 x = {lo16(w[u].x), hi16(w[u].x), lo16(w[u].y), hi16(w[u].y)};
      if (gh.wide) {
        st_nt(reinterpret_cast<f32x4*>(static_cast<float*>(gh.dst) + e),
              f32x4{x.x * scale, x.y * scale, x.z * scale, x.w * scale});
      } else {
        u32x2 o;
        o.x = rne16(x.x * scale_b) | (rne16(x.y * scale_b) << 16);
        o.y = rne16(x.z * scale_b) | (rne16(x.w * scale_b) << 16);
        st_nt(reinterpret_cast<u32x2*>(static_cast<uint16_t*>(gh.dst) + e), o);
      }
    }
  }
  for (int64_t i = done + threadIdx.x; i < end; i += 64) {
    const float x = __uint_as_float(static_cast<uint32_t>(gh.src[i]) << 16);
    if (gh.wide) static_cast<float*>(gh.dst)[i] = x * scale;
    else static_cast<uint16_t*>(gh.dst)[i] = static_cast<uint16_t>(rne16(x * scale_b));
  }
}

// Slices [0, fold_slices) are grad_W's; the later ones grad_h's (kScale only).
template <bool kAccumulate, bool kScale>
__global__ __launch_bounds__(64) void ce_grads_kernel(float* __restrict__ acc, FoldChunks ch, int n, int64_t nw,
                                                      int64_t fold_slices, int64_t first_slice, GradH gh,
                                                      const float* __restrict__ grad_out,
                                                      const float* __restrict__ n_valid) {
  const float scale = kScale ? *grad_out / *n_valid : 1.0f;
  const int64_t slice = first_slice + blockIdx.x;
  if (kScale && slice >= fold_slices) {
    grad_h_slice(gh, (slice - fold_slices) * kGradHSlice, scale);
    return;
  }
  uint64_t misaligned = reinterpret_cast<uint64_t>(acc) & 15u;
#pragma unroll
  for (int c = 0; c < kMaxFold; ++c)
    if (c < n) misaligned |= reinterpret_cast<uint64_t>(ch.p[c]) & 7u;
  const int64_t e = slice * 256 + static_cast<int64_t>(threadIdx.x) * 4;
  if (misaligned == 0 && e + 4 <= nw) {
    u32x2 w[kMaxFold];
#pragma unroll
    for (int c = 0; c < kMaxFold; ++c)
      if (c < n) w[c] = ld_nt(reinterpret_cast<const u32x2*>(ch.p[c] + e));
    f32x4 a = kAccumulate ? ld_nt(reinterpret_cast<const f32x4*>(acc + e)) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < kMaxFold; ++c) {
      if (c < n) {
        a.x = a.x + lo16(w[c].x); a.y = a.y + hi16(w[c].x);
        a.z = a.z + lo16(w[c].y); a.w = a.w + hi16(w[c].y);
      }
    }
    if (kScale) {
      a.x = a.x * scale; a.y = a.y * scale; a.z = a.z * scale; a.w = a.w * scale;
    }
    st_nt(reinterpret_cast<f32x4*>(acc + e), a);
    return;
  }
  const int64_t end = e + 4 < nw ? e + 4 : nw;
  for (int64_t i = e; i < end; ++i) {
    float x = kAccumulate ? acc[i] : 0.0f;
#pragma unroll
    for (int c = 0; c < kMaxFold; ++c)
      if (c < n) x = x + __uint_as_float(static_cast<uint32_t>(ch.p[c][i]) << 16);
    if (kScale) x = x * scale;
    acc[i] = x;
  }
}

// bf16 = RNE(fp32), NaN -> 0x7FC0, over two arrays in one launch: the hidden states and the weight
// that autocast casts for the products. 512 elements a wave, two groups of 4 a lane, both loaded
// before either is stored. Bound: HBM, 6 bytes an element; 138 us for 151,936 x 1024 (6.7 TB/s,
// against 148 for the library's cast, which also took a launch for each array).
struct CastPart {
  uint16_t* dst;
  const float* src;
  int64_t n;
};
constexpr int kCastSlice = 512;

__global__ __launch_bounds__(64) void ce_cast_kernel(CastPart a, CastPart b, int64_t slices_a, int64_t first_slice) {
  int64_t slice = first_slice + blockIdx.x;
  const CastPart p = slice < slices_a ? a : b;
  if (slice >= slices_a) slice -= slices_a;
  const int64_t start = slice * kCastSlice;
  const int64_t end = start + kCastSlice < p.n ? start + kCastSlice : p.n;
  int64_t done = start;
  if (((reinterpret_cast<uint64_t>(p.src) & 15u) | (reinterpret_cast<uint64_t>(p.dst) & 7u)) == 0) {
    done = start + ((end - start) & ~int64_t(3));
    const int64_t e0 = start + static_cast<int64_t>(threadIdx.x) * 4, e1 = e0 + 256;
    f32x4 x[2] = {};
    if (e0 < done) x[0] = ld_nt(reinterpret_cast<const f32x4*>(p.src + e0));
    if (e1 < done) x[1] = ld_nt(reinterpret_cast<const f32x4*>(p.src + e1));
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t e = u == 0 ? e0 : e1;
      if (e >= done) continue;
      u32x2 o;
      o.x = rne16(x[u].x) | (rne16(x[u].y) << 16);
      o.y = rne16(x[u].z) | (rne16(x[u].w) << 16);
      *reinterpret_cast<u32x2*>(p.dst + e) = o;  // read next by the GEMMs
    }
  }
  for (int64_t i = done + threadIdx.x; i < end; i += 64) p.dst[i] = static_cast<uint16_t>(rne16(p.src[i]));
}

int ce_check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ce_fail(TM_ELAUNCH, "%s: launch failed: %s", what, hipGetErrorString(e));
  return TM_OK;
}

// Threads a row and vectors a thread of the register path: the fewest waves whose threads hold
// the row in at most kRegCols vectors each, then the smallest count compiled that covers it.
// cols = 0: the row is too long for registers (streaming path).
struct RowShape {
  int threads, cols;
};

RowShape row_shape(int64_t vocab, bool aligned) {
  const int64_t nvec = vocab >> 3;
  // rows off 16 bytes go element by element (but for the aligned one in eight): as many threads
  // as a row takes (87 us against 114 for 1024 rows of 32,001 with 256 threads a row)
  for (int threads = aligned ? 64 : kRowThreadsMax; threads <= kRowThreadsMax; threads *= 2) {
    if (nvec > static_cast<int64_t>(threads) * kRegCols) continue;
    const int need = static_cast<int>((nvec + threads - 1) / threads);
    const int least = threads == 64 ? 4 : 12;
    return {threads, need <= least ? least : (need + 3) / 4 * 4};
  }
  return {kRowThreadsStream, 0};
}

struct RowArgs {
  uint16_t* logits;
  int64_t ld;
  const int64_t* labels;
  int64_t vocab, ignore_index;
  float* row_loss;
  uint32_t blocks;
  int64_t rows, width;
  hipStream_t stream;
};

template <int kCols, int kThreads, bool kGrad>
void row_launch(const RowArgs& a) {
  hipLaunchKernelGGL((ce_rows_kernel<kCols, kThreads, kGrad>), dim3(a.blocks), dim3(kThreads), 0, a.stream, a.logits,
                     a.ld, a.labels, a.vocab, a.ignore_index, a.row_loss, a.rows, a.width);
}

// More than one wave a row means more than kRegCols / 2 vectors a thread.
template <int kThreads, bool kGrad>
void row_launch_cols(int cols, const RowArgs& a) {
  if constexpr (kThreads == 64) {
    if (cols == 4) return row_launch<4, kThreads, kGrad>(a);
    if (cols == 8) return row_launch<8, kThreads, kGrad>(a);
  }
  if (cols == 12) return row_launch<12, kThreads, kGrad>(a);
  if (cols == 16) return row_launch<16, kThreads, kGrad>(a);
  row_launch<20, kThreads, kGrad>(a);
}

// One block per row. The kernel (register or streaming path, and its shape) depends only on the
// vocabulary, so the loss-only pass runs the same arithmetic as the gradient pass and gives the
// same bits.
template <bool kGrad>
int ce_rows_launch(uint16_t* d_logits, int64_t ld, const int64_t* d_labels, int64_t rows, int64_t pad_rows,
                   int64_t vocab, int64_t width, int64_t ignore_index, float* d_row_loss, void* stream,
                   const char* who) {
  if (rows < 0 || vocab <= 0 || ld < vocab)
    return ce_fail(TM_EINVAL, "%s: bad sizes rows=%lld vocab=%lld ld=%lld", who, (long long)rows,
                   (long long)vocab, (long long)ld);
  if (rows == 0) return TM_OK;  // pad_rows is 0 too, or the caller's check has refused it
  if (!d_logits || !d_labels || !d_row_loss) return ce_fail(TM_EINVAL, "%s: null pointer", who);
  const RowShape shape = row_shape(vocab, ld % 8 == 0 && (reinterpret_cast<uintptr_t>(d_logits) & 15u) == 0);
  // a launch holds fewer than 2^32 work-items: longer row lists (small vocabularies in one
  // chunk) go in several launches
  const int64_t max_rows = 0xFFFFFFFFll / shape.threads;
  for (int64_t r0 = 0; r0 < pad_rows; r0 += max_rows) {
    const RowArgs a = {d_logits + r0 * ld, ld, d_labels + r0, vocab, ignore_index, d_row_loss + r0,
                       static_cast<uint32_t>(pad_rows - r0 < max_rows ? pad_rows - r0 : max_rows), rows - r0, width,
                       static_cast<hipStream_t>(stream)};
    if (shape.cols == 0) row_launch<0, kRowThreadsStream, kGrad>(a);
    else if (shape.threads == 64) row_launch_cols<64, kGrad>(shape.cols, a);
    else if (shape.threads == 128) row_launch_cols<128, kGrad>(shape.cols, a);
    else if (shape.threads == 256) row_launch_cols<256, kGrad>(shape.cols, a);
    else if (shape.threads == 512) row_launch_cols<512, kGrad>(shape.cols, a);
    else row_launch_cols<1024, kGrad>(shape.cols, a);
    if (int rc = ce_check_launch(who)) return rc;
  }
  return TM_OK;
}

template <int kCols, int kThreads, bool kGrad>
void row_f32_launch(float* logits, int64_t ld, const int64_t* labels, int64_t vocab, int64_t ignore_index,
                    float* row_loss, uint32_t rows, hipStream_t s) {
  hipLaunchKernelGGL((ce_rows_f32_kernel<kCols, kThreads, kGrad>), dim3(rows), dim3(kThreads), 0, s, logits, ld, labels,
                     vocab, ignore_index, row_loss);
}

template <bool kGrad>
int ce_rows_f32_launch(float* d_logits, int64_t ld, const int64_t* d_labels, int64_t rows, int64_t vocab,
                       int64_t ignore_index, float* d_row_loss, void* stream, const char* who) {
  if (rows < 0 || vocab <= 0 || ld < vocab)
    return ce_fail(TM_EINVAL, "%s: bad sizes rows=%lld vocab=%lld ld=%lld", who, (long long)rows,
                   (long long)vocab, (long long)ld);
  if (rows == 0) return TM_OK;
  if (!d_logits || !d_labels || !d_row_loss) return ce_fail(TM_EINVAL, "%s: null pointer", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  // As many threads as a row takes at 20 vectors each, from 256 on: an fp32 chunk's 1024 rows are
  // too few for one wave a row (1024 x 5120: 16.8 us with 64 threads, 14.6 with 256).
  const bool aligned = ld % 4 == 0 && (reinterpret_cast<uintptr_t>(d_logits) & 15u) == 0;
  const int64_t nvec = vocab >> 2;
  const int threads = aligned && nvec <= 256 * kRegCols ? 256 : aligned && nvec <= 512 * kRegCols ? 512 : 1024;
  const int64_t need = (nvec + threads - 1) / threads;
  const int64_t cols = !aligned || need > kRegCols ? 0 : threads > 256 ? (need <= 12 ? 12 : kRegCols)
                   : need <= 2 ? (need > 0 ? need : 1) : need <= 12 ? (need + 3) / 4 * 4 : kRegCols;
  const int64_t max_rows = 0xFFFFFFFFll / threads;  // a launch holds fewer than 2^32 work-items
  for (int64_t r0 = 0; r0 < rows; r0 += max_rows) {
    const uint32_t nr = static_cast<uint32_t>(rows - r0 < max_rows ? rows - r0 : max_rows);
    float* lg = d_logits + r0 * ld;
    const int64_t* lab = d_labels + r0;
    float* loss = d_row_loss + r0;
    if (cols == 0) row_f32_launch<0, 1024, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (threads == 256 && cols == 1) row_f32_launch<1, 256, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (threads == 256 && cols == 2) row_f32_launch<2, 256, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (threads == 256 && cols == 8) row_f32_launch<8, 256, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (threads == 256 && cols == 4) row_f32_launch<4, 256, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (threads == 256 && cols == 12) row_f32_launch<12, 256, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (threads == 256) row_f32_launch<kRegCols, 256, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (threads == 512 && cols == 12) row_f32_launch<12, 512, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (threads == 512) row_f32_launch<kRegCols, 512, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else if (cols == 12) row_f32_launch<12, 1024, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    else row_f32_launch<kRegCols, 1024, kGrad>(lg, ld, lab, vocab, ignore_index, loss, nr, s);
    if (int rc = ce_check_launch(who)) return rc;
  }
  return TM_OK;
}

// One ce_grads_kernel pass: grad_W's nw elements (one 64-thread workgroup per 256-element slice),
// then grad_h's (512-element slices, only with a scale), over as many launches as the 2^32
// work-item limit of a launch requires.
int grads_launch(float* d_grad_w, const FoldChunks& ch, int n_chunks, int64_t nw, int accumulate, const GradH& gh,
                 const float* d_grad_out, const float* d_n_valid, void* stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool scale = d_grad_out != nullptr;
  const int64_t fold = (nw + 255) / 256, slices = fold + (gh.n + kGradHSlice - 1) / kGradHSlice;
  constexpr int64_t kMaxSlicesPerLaunch = int64_t(1) << 25;  // 2^31 work-items
  for (int64_t first = 0; first < slices; first += kMaxSlicesPerLaunch) {
    const int64_t count = slices - first < kMaxSlicesPerLaunch ? slices - first : kMaxSlicesPerLaunch;
    const dim3 grid(static_cast<uint32_t>(count)), block(64);
    if (accumulate && scale)
      hipLaunchKernelGGL((ce_grads_kernel<true, true>), grid, block, 0, s, d_grad_w, ch, n_chunks, nw, fold, first, gh,
                         d_grad_out, d_n_valid);
    else if (accumulate)
      hipLaunchKernelGGL((ce_grads_kernel<true, false>), grid, block, 0, s, d_grad_w, ch, n_chunks, nw, fold, first, gh,
                         d_grad_out, d_n_valid);
    else if (scale)
      hipLaunchKernelGGL((ce_grads_kernel<false, true>), grid, block, 0, s, d_grad_w, ch, n_chunks, nw, fold, first, gh,
                         d_grad_out, d_n_valid);
    else
      hipLaunchKernelGGL((ce_grads_kernel<false, false>), grid, block, 0, s, d_grad_w, ch, n_chunks, nw, fold, first,
                         gh, d_grad_out, d_n_valid);
    const int rc = ce_check_launch("ce_grads_kernel");
    if (rc != TM_OK) return rc;
  }
  return TM_OK;
}

template <bool kTwo>
int ce_grad_w_launch(float* d_grad_w, const uint16_t* d_chunk, const uint16_t* d_chunk2, int64_t nw,
                     int accumulate, const float* d_grad_out, const float* d_n_valid, void* stream,
                     const char* who) {
  if (nw < 0) return ce_fail(TM_EINVAL, "%s: negative size", who);
  if (nw == 0) return TM_OK;
  if (!d_grad_w || !d_chunk || (kTwo && !d_chunk2) || (d_grad_out != nullptr) != (d_n_valid != nullptr))
    return ce_fail(TM_EINVAL, "%s: null pointer", who);
  FoldChunks ch = {};
  ch.p[0] = d_chunk;
  if (kTwo) ch.p[1] = d_chunk2;
  return grads_launch(d_grad_w, ch, kTwo ? 2 : 1, nw, accumulate, GradH{}, d_grad_out, d_n_valid, stream);
}

int fold_chunks(const uint16_t* const* h_chunks, int n_chunks, FoldChunks& ch, const char* who) {
  for (int c = 0; c < n_chunks; ++c) {
    if (!h_chunks || !h_chunks[c]) return ce_fail(TM_EINVAL, "%s: null chunk %d", who, c);
    ch.p[c] = h_chunks[c];
  }
  return TM_OK;
}

}  // namespace

extern "C" {

int tm_ce_rows_bf16(uint16_t* d_logits, int64_t ld, const int64_t* d_labels, int64_t rows,
                    int64_t vocab, int64_t ignore_index, float* d_row_loss, void* stream) {
  return ce_rows_launch<true>(d_logits, ld, d_labels, rows, rows, vocab, vocab, ignore_index, d_row_loss, stream,
                              "tm_ce_rows_bf16");
}

int tm_ce_rows_padded_bf16(uint16_t* d_logits, int64_t ld, const int64_t* d_labels, int64_t rows, int64_t pad_rows,
                           int64_t vocab, int64_t ignore_index, float* d_row_loss, void* stream) {
  if (rows < 1 || pad_rows < rows || ld % 8 || (reinterpret_cast<uintptr_t>(d_logits) & 15u))
    return ce_fail(TM_EINVAL, "tm_ce_rows_padded_bf16: rows %lld of %lld, 16-byte aligned rows wanted (ld %lld)",
                   (long long)rows, (long long)pad_rows, (long long)ld);
  return ce_rows_launch<true>(d_logits, ld, d_labels, rows, pad_rows, vocab, ld, ignore_index, d_row_loss, stream,
                              "tm_ce_rows_padded_bf16");
}

int tm_ce_rows_loss_bf16(const uint16_t* d_logits, int64_t ld, const int64_t* d_labels, int64_t rows,
                         int64_t vocab, int64_t ignore_index, float* d_row_loss, void* stream) {
  // the kGrad=false kernels only read the logits
  return ce_rows_launch<false>(const_cast<uint16_t*>(d_logits), ld, d_labels, rows, rows, vocab, vocab, ignore_index,
                               d_row_loss, stream, "tm_ce_rows_loss_bf16");
}

int tm_ce_rows_f32(float* d_logits, int64_t ld, const int64_t* d_labels, int64_t rows, int64_t vocab,
                   int64_t ignore_index, float* d_row_loss, void* stream) {
  return ce_rows_f32_launch<true>(d_logits, ld, d_labels, rows, vocab, ignore_index, d_row_loss, stream,
                                  "tm_ce_rows_f32");
}

int tm_ce_rows_loss_f32(const float* d_logits, int64_t ld, const int64_t* d_labels, int64_t rows, int64_t vocab,
                        int64_t ignore_index, float* d_row_loss, void* stream) {
  return ce_rows_f32_launch<false>(const_cast<float*>(d_logits), ld, d_labels, rows, vocab, ignore_index,
                                   d_row_loss, stream, "tm_ce_rows_loss_f32");
}

int tm_ce_loss(const float* d_row_loss, const int64_t* d_labels, int64_t rows, int64_t ignore_index,
               float* d_out3, void* stream) {
  return tm_ce_mean_loss(d_row_loss, d_labels, rows, ignore_index, d_out3, d_out3 ? d_out3 + 2 : nullptr, stream);
}

int tm_ce_mean_loss(const float* d_row_loss, const int64_t* d_labels, int64_t rows, int64_t ignore_index,
                    float* d_out2, float* d_loss, void* stream) {
  if (rows < 0) return ce_fail(TM_EINVAL, "tm_ce_loss: negative rows");
  if (!d_out2 || !d_loss || (rows > 0 && (!d_row_loss || !d_labels)))
    return ce_fail(TM_EINVAL, "tm_ce_loss: null pointer");
  hipLaunchKernelGGL(ce_loss_kernel, dim3(1), dim3(kLossThreads), 0, static_cast<hipStream_t>(stream),
                     d_row_loss, d_labels, rows, ignore_index, d_out2, d_loss);
  return ce_check_launch("ce_loss_kernel");
}

int tm_ce_finish(float* d_grad_w, const uint16_t* const* h_chunks, int n_chunks, int64_t nw, int accumulate,
                 const uint16_t* d_grad_h, void* d_grad_h_out, int64_t nh, int wide, const float* d_grad_out,
                 const float* d_n_valid, void* stream) {
  const char* who = "tm_ce_finish";
  if (nh < 0 || nw < 0 || n_chunks < 0 || n_chunks > kMaxFold)
    return ce_fail(TM_EINVAL, "%s: %d chunks (0 to %d) of %lld elements, grad_h of %lld", who, n_chunks, kMaxFold,
                   (long long)nw, (long long)nh);
  if (wide < 0 || wide > 2 || (wide == 2 && static_cast<const void*>(d_grad_h) != d_grad_h_out))
    return ce_fail(TM_EINVAL, "%s: grad_h kind %d (2 is in place)", who, wide);
  if ((nh > 0 && (!d_grad_h || !d_grad_h_out)) || (nw > 0 && !d_grad_w) || !d_grad_out || !d_n_valid)
    return ce_fail(TM_EINVAL, "%s: null pointer", who);
  FoldChunks ch = {};
  if (nw > 0)
    if (int rc = fold_chunks(h_chunks, n_chunks, ch, who)) return rc;
  return grads_launch(d_grad_w, ch, nw > 0 ? n_chunks : 0, nw, accumulate, GradH{d_grad_h, d_grad_h_out, nh, wide == 1, wide == 2},
                      d_grad_out, d_n_valid, stream);
}

int tm_ce_scale_grads(uint16_t* d_grad_h, int64_t nh, float* d_grad_w, int64_t nw,
                      const float* d_grad_out, const float* d_n_valid, void* stream) {
  if (nh < 0 || nw < 0) return ce_fail(TM_EINVAL, "tm_ce_scale_grads: negative size");
  if ((nh > 0 && !d_grad_h) || (nw > 0 && !d_grad_w) || !d_grad_out || !d_n_valid)
    return ce_fail(TM_EINVAL, "tm_ce_scale_grads: null pointer");
  return tm_ce_finish(d_grad_w, nullptr, 0, nw, 1, d_grad_h, d_grad_h, nh, 0, d_grad_out, d_n_valid, stream);
}

int tm_ce_cast2(uint16_t* d_dst0, const float* d_src0, int64_t n0, uint16_t* d_dst1, const float* d_src1, int64_t n1,
                void* stream) {
  if (n0 < 0 || n1 < 0) return ce_fail(TM_EINVAL, "tm_ce_cast2: negative size");
  if ((n0 > 0 && (!d_dst0 || !d_src0)) || (n1 > 0 && (!d_dst1 || !d_src1)))
    return ce_fail(TM_EINVAL, "tm_ce_cast2: null pointer");
  const int64_t s0 = (n0 + kCastSlice - 1) / kCastSlice, slices = s0 + (n1 + kCastSlice - 1) / kCastSlice;
  constexpr int64_t kMaxSlicesPerLaunch = int64_t(1) << 25;  // 2^31 work-items
  for (int64_t first = 0; first < slices; first += kMaxSlicesPerLaunch) {
    const int64_t count = slices - first < kMaxSlicesPerLaunch ? slices - first : kMaxSlicesPerLaunch;
    hipLaunchKernelGGL(ce_cast_kernel, dim3(static_cast<uint32_t>(count)), dim3(64), 0,
                       static_cast<hipStream_t>(stream), CastPart{d_dst0, d_src0, n0}, CastPart{d_dst1, d_src1, n1}, s0,
                       first);
    if (int rc = ce_check_launch("ce_cast_kernel")) return rc;
  }
  return TM_OK;
}

int tm_ce_grad_w(float* d_grad_w, const uint16_t* d_chunk, int64_t nw, int accumulate,
                 const float* d_grad_out, const float* d_n_valid, void* stream) {
  return ce_grad_w_launch<false>(d_grad_w, d_chunk, nullptr, nw, accumulate, d_grad_out, d_n_valid, stream,
                                 "tm_ce_grad_w");
}

int tm_ce_grad_w2(float* d_grad_w, const uint16_t* d_chunk, const uint16_t* d_chunk2, int64_t nw,
                  int accumulate, const float* d_grad_out, const float* d_n_valid, void* stream) {
  return ce_grad_w_launch<true>(d_grad_w, d_chunk, d_chunk2, nw, accumulate, d_grad_out, d_n_valid, stream,
                                "tm_ce_grad_w2");
}

int tm_ce_grad_w_fold(float* d_grad_w, const uint16_t* const* h_chunks, int n_chunks, int64_t nw, int accumulate,
                      const float* d_grad_out, const float* d_n_valid, void* stream) {
  const char* who = "tm_ce_grad_w_fold";
  if (nw < 0 || n_chunks < 1 || n_chunks > kMaxFold)
    return ce_fail(TM_EINVAL, "%s: %d chunks (1 to %d) of %lld elements", who, n_chunks, kMaxFold, (long long)nw);
  if (!h_chunks || !d_grad_w || (d_grad_out != nullptr) != (d_n_valid != nullptr))
    return ce_fail(TM_EINVAL, "%s: null pointer", who);
  FoldChunks ch = {};
  if (int rc = fold_chunks(h_chunks, n_chunks, ch, who)) return rc;
  if (nw == 0) return TM_OK;
  return grads_launch(d_grad_w, ch, n_chunks, nw, accumulate, GradH{}, d_grad_out, d_n_valid, stream);
}

int tm_ce_widen_scale(float* d_dst, const uint16_t* d_src, int64_t n, const float* d_grad_out,
                      const float* d_n_valid, void* stream) {
  if (n < 0) return ce_fail(TM_EINVAL, "tm_ce_widen_scale: negative size");
  if (n == 0) return TM_OK;
  if (!d_dst || !d_src || !d_grad_out || !d_n_valid) return ce_fail(TM_EINVAL, "tm_ce_widen_scale: null pointer");
  return tm_ce_finish(nullptr, nullptr, 0, 0, 0, d_src, d_dst, n, 1, d_grad_out, d_n_valid, stream);
}

}  // extern "C"
