// Row reductions on gfx950: softmax, RMSNorm, LayerNorm.
//
// Reference semantics: test/python/triton/test_softmax.py:41-69 (max-subtract,
// exp in fp32, sum, divide), test_rms_norm.py:34-60 (x / sqrt(mean(x^2)+eps)
// * g), test_layer_norm.py:39-79 (mean, biased variance, rstd, affine, mean and
// rstd written per row), as lowered on the HVX path by
// lib/Conversion/LinalgToLLVM/VectorRowReducePass.cpp:10-31 (vector fold +
// rotate butterfly) and SplitReduceGenericPass.cpp:62-93.
//
// Design: a row is loaded ONCE into registers with 128-bit loads (consecutive
// lanes read consecutive 16-byte chunks), reduced across each wave with DPP +
// readlane and across the S waves that share the row through LDS, and written
// back from registers: one HBM read and one HBM write per element.  S grows
// with the row: one wave up to 128 vectors of 16 bytes, then 2, 4, 8 and 16
// waves, so that a lane holds few vectors, its chain of arithmetic stays
// short and a call of few rows still fills CUs.  Rows beyond 16 waves x 16
// vectors a lane (131072 f16, 65536 f32 columns) are streamed by 16 waves,
// re-reading the row per pass.  Rows need no alignment: gfx950 takes 16-byte
// accesses at any element address, and only a row's last partial vector is
// read and written element by element.
#include <type_traits>

#include "device_util.h"
#include "hxm_internal.h"

namespace hxm {

enum RowOp { kSoftmax = 0, kRmsNorm = 1, kLayerNorm = 2 };

// Waves of a workgroup whose rows take S waves each.
constexpr int row_waves(int S) { return S < 4 ? 4 : S; }

template <typename T>
struct RowVec {
  static constexpr int N = 16 / sizeof(T);  // elements per 16-byte vector
};

// exp(x) for x <= 0 via the hardware exp2 (v_exp_f32): exp(x) = 2^(x*log2 e).
__device__ __forceinline__ float exp_f32(float x) {
  return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}

struct RowArgs {
  const void* x;
  int64_t ldx;
  void* y;
  int64_t ldy;
  const void* gamma;
  const void* beta;
  float* mean_out;
  float* rstd_out;
  int64_t rows;
  int64_t cols;
  float eps;
};

// One 16-byte vector of a row in its storage type.
template <typename T>
using RawVec = T __attribute__((ext_vector_type(RowVec<T>::N)));

// The same vector at any element address (a row may start anywhere).
template <typename T>
using AnyVec = T __attribute__((ext_vector_type(RowVec<T>::N), aligned(sizeof(T))));

// Row loads are plain (cacheable) and row stores nontemporal.  On a stream
// that reads and writes HBM at once this pairing ran fastest of the four
// (64 MiB copy, one box: plain loads + nontemporal stores 20.2 us,
// nontemporal both 22.2-22.6, nontemporal loads + plain stores 22.5, plain
// both 24.6); RMSNorm 22.1 -> 20.8 us and softmax 22.9 -> 20.9 us at
// 8192 x 4096 f16 with nontemporal loads replaced.  A read-only stream is the
// other way round (the GEMV's weights stay nontemporal).
template <typename T>
__device__ __forceinline__ RawVec<T> load_any(const T* p) {
  return *reinterpret_cast<const AnyVec<T>*>(p);
}
template <typename T>
__device__ __forceinline__ void store_any(T* p, RawVec<T> v) {
  __builtin_nontemporal_store(static_cast<AnyVec<T>>(v), reinterpret_cast<AnyVec<T>*>(p));
}

// The row's last, partial vector (elements [c0, cols), at least one): element
// by element, the rest of the vector set to `fill`.
template <typename T>
__device__ __forceinline__ RawVec<T> load_tail(const T* __restrict__ row, int64_t c0, int64_t cols,
                                               T fill) {
  constexpr int N = RowVec<T>::N;
  const int rem = static_cast<int>(cols - c0);
  RawVec<T> v;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const T e = row[c0 + min(j, rem - 1)];
    v[j] = j < rem ? e : fill;
  }
  return v;
}
template <typename T>
__device__ __forceinline__ void store_tail(T* __restrict__ row, int64_t c0, int64_t cols,
                                           RawVec<T> v) {
#pragma unroll
  for (int j = 0; j < RowVec<T>::N; ++j)
    if (c0 + j < cols) row[c0 + j] = v[j];
}

// The S wave totals of a row combined pairwise (the rounding of S sequential
// adds of near-equal totals showed in f32 LayerNorm means).
template <int S, typename Op>
__device__ __forceinline__ float wave_totals(const float* t, Op op) {
  float v[S];
#pragma unroll
  for (int k = 0; k < S; ++k) v[k] = t[k];
#pragma unroll
  for (int w = 1; w < S; w *= 2)
#pragma unroll
    for (int k = 0; k + w < S; k += 2 * w) v[k] = op(v[k], v[k + w]);
  return v[0];
}

// Makes the compiler treat the row registers as rewritten, so that each pass
// widens the stored values again instead of keeping fp32 copies of the
// whole row alive across passes (which would double the register count).
template <typename T, int VPL>
__device__ __forceinline__ void fresh(RawVec<T> (&v)[VPL]) {
#pragma unroll
  for (int i = 0; i < VPL; ++i) asm volatile("" : "+v"(v[i]));
}

// Register-resident kernel: S waves share a row, wave w of the row holding its
// vectors w, w + S, ... of every 64-lane slot (VPL slots a lane) in the storage
// type (f16/bf16 rows take half the registers of fp32 copies, so more waves
// fit per SIMD and more bytes are in flight).  Values are widened to fp32 as
// each pass reads them.
//
// FULL (chosen on the host): the row fills every slot, cols == S * VPL * 64 * N,
// and no padding logic is compiled.  Measured with one wave per row, LayerNorm
// f16 at 4096 columns: 107 VGPRs with it, 62 without; 25.7 against 25.2 us.
// Otherwise the host picks the smallest VPL that holds the row, so that the
// row's last, partial vector lies in one of the slots [TAIL0, VPL).
//
// S > 1: the wave totals meet in LDS behind a barrier.  Each wave's chain of
// arithmetic after its loads is S times shorter, and that chain is what the
// last rows of the grid add after the last bytes land.  Measured (8192 x 4096
// f16, one box, two alternating passes each): S = 1 against S = 2, RMSNorm
// 20.74 -> 20.20 us, LayerNorm 21.77 -> 20.70 us, softmax 20.86 -> 20.88 us;
// S = 2 against S = 4 (one row per workgroup), softmax 20.87 -> 19.96 us,
// RMSNorm 19.97 -> 19.84 us, LayerNorm 20.8 -> 20.94 us (its two dependent
// reductions each cross the LDS).
//
// L < 64: a row is as short as one 16-lane row of the wave and a wave holds
// 64 / L of them, so short rows do not leave most lanes idle.
template <typename T, int OP, int VPL, int S, bool FULL, int L = 64>
__global__ __launch_bounds__(row_waves(S) * 64) void row_kernel(RowArgs a) {
  static_assert(L == 64 || (L == 16 && S == 1), "short rows: 16 lanes of one wave");
  constexpr int N = RowVec<T>::N;
  constexpr int WAVES = row_waves(S);
  constexpr int TAIL0 = VPL <= 4 ? VPL - 1 : VPL / 2;
  const int lane = threadIdx.x % L;  // within the row
  const int wv = threadIdx.x >> 6;
  const int half = wv % S;  // this wave's share of the row
  // Softmax takes its row groups XCD-contiguously: workgroups are dispatched
  // round-robin over the 8 XCDs, so ordinal b (on XCD x = b % 8) takes group
  // x * (G / 8) + min(x, G % 8) + b / 8 of the G in the grid (a bijection),
  // and each XCD streams one contiguous eighth of the rows.  Measured at
  // 8192 x 4096 f16 (three alternating passes, one box): softmax 20.01-20.02
  // against 20.16-20.22 us; RMSNorm 19.90-19.97 against 19.89-19.91 and
  // LayerNorm 20.98-21.01 against 20.88-20.93, so those keep the plain order.
  int blk = blockIdx.x;
  if constexpr (OP == kSoftmax) {
    const int G = gridDim.x, x = blk & 7;
    blk = x * (G >> 3) + min(x, G & 7) + (blk >> 3);
  }
  const int64_t r = static_cast<int64_t>(blk) * (WAVES * (64 / L) / S) +
                    (L == 64 ? wv / S : static_cast<int>(threadIdx.x) / L);
  if constexpr (S == 1 && L == 64) {
    if (r >= a.rows) return;  // whole wave leaves; no barriers below
  }
  // Otherwise lanes past the last row stay for the reductions, read row 0 and
  // store nothing.
  const bool valid = r < a.rows;
  const int64_t rv = valid ? r : 0;
  const T* __restrict__ xr = static_cast<const T*>(a.x) + rv * a.ldx;
  T* __restrict__ yr = static_cast<T*>(a.y) + rv * a.ldy;
  // Row total: the wave's, then (S > 1) the S waves' in a fixed order, so
  // every wave of the row holds the same value.  Each slot serves one
  // reduction of the kernel, so no slot is rewritten after the barrier.
  __shared__ float red[2][WAVES];
  auto row_reduce = [&](float x, auto op, int slot) {
    if constexpr (L == 16) return row16_reduce(x, op);
    x = wave_reduce(x, op);
    if constexpr (S > 1) {
      if (lane == 0) red[slot][wv] = x;
      __syncthreads();
      x = wave_totals<S>(red[slot] + (wv / S) * S, op);
    }
    return x;
  };
  const int64_t cols = a.cols;
  const T* __restrict__ g = static_cast<const T*>(a.gamma);
  const T* __restrict__ b = static_cast<const T*>(a.beta);
  auto col0 = [&](int i) { return ((static_cast<int64_t>(i) * S + half) * L + lane) * N; };
  // Slot i holds row elements only (uniform; every slot before TAIL0 does).
  auto whole = [&](int i) { return FULL || i < TAIL0 || (i + 1) * (S * L * N) <= cols; };
  // Vector i of a row or of gamma / beta.  A lane past the row (or on its
  // partial vector) loads column 0 instead, a valid address, and takes the
  // fill, so that no branch splits the wave's loads and all of them are in
  // flight together.
  auto load_at = [&](const T* __restrict__ p, int i, T fill) -> RawVec<T> {
    if constexpr (FULL) return load_any(p + col0(i));
    if (i < TAIL0) return load_any(p + col0(i));
    const int64_t c = col0(i);
    RawVec<T> v = RawVec<T>(fill);
    if (cols >= N) {  // uniform
      const bool in = c + N <= cols;
      const RawVec<T> t = load_any(p + (in ? c : 0));
      v = in ? t : v;
    }
    if (c < cols && c + N > cols) v = load_tail(p, c, cols, fill);
    return v;
  };
  auto store_at = [&](int i, RawVec<T> v) {
    if (!valid) return;
    const int64_t c = col0(i);
    if (FULL || i < TAIL0 || c + N <= cols) store_any(yr + c, v);
    else if (c < cols) store_tail(yr, c, cols, v);
  };

  const T fill = static_cast<T>(OP == kSoftmax ? -__builtin_huge_valf() : 0.0f);
  RawVec<T> v[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) v[i] = load_at(xr, i, fill);
  // gamma / beta vector i, read in the output pass (cache hits: every row
  // shares them), so no registers hold them while the row is in flight.
  auto gamma_at = [&](int i) { return g ? load_at(g, i, T(0)) : RawVec<T>(T(1)); };
  auto beta_at = [&](int i) { return b ? load_at(b, i, T(0)) : RawVec<T>(T(0)); };

  if constexpr (OP == kSoftmax) {
    // The row maximum is exact in the storage type, so f16 rows take it with
    // packed f16 max (two lanes per instruction) before widening once.
    float m;
    if constexpr (std::is_same<T, _Float16>::value) {
      RawVec<T> mv = v[0];
#pragma unroll
      for (int i = 1; i < VPL; ++i) mv = __builtin_elementwise_max(mv, v[i]);
      m = tof(mv[0]);
#pragma unroll
      for (int j = 1; j < N; ++j) m = fmaxf(m, tof(mv[j]));
    } else {
      m = -__builtin_huge_valf();
#pragma unroll
      for (int i = 0; i < VPL; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) m = fmaxf(m, tof(v[i][j]));
    }
    m = row_reduce(m, OpMax(), 0);
    fresh(v);
    // exp(x - m) = 2^(x*log2(e) - m*log2(e)): one (mixed-precision) fma per
    // element feeds the hardware exp2, once per element.  Each numerator is
    // rounded to the storage type in place of its input, and the fp32 sum
    // adds those rounded numerators: the reference's kernel computes
    // num = exp(z).to(x.dtype), denom = sum(num) in fp32, y = num / denom
    // (test/python/triton/test_softmax.py:64-66).  The row stays in the
    // registers it arrived in.
    // The output pass is one mixed-precision fma per element, x * inv +
    // (-0), with `nzero` hidden from the optimizer so it stays an fma (it
    // rounds exactly like the product).  Padded -inf columns give 0.
    // Measured (8192 x 4096 f16, one box): 23.2 us, against 23.4 us with
    // two exponentials per element (eight waves per SIMD either way).
    //
    // The fma's addend is m*log2(e) rounded once, off by up to half an ulp:
    // one factor for the whole row, which the division takes out again, as
    // long as it is near 1 -- always for f16, for f32 and bf16 below 2^22
    // (half an ulp is at most 1/4 there).  In a row of a larger maximum (a
    // wholly masked one) the numerators would over- or underflow, or the
    // addend itself would, so it has m taken off in place first: in f32 as
    // x - m, in bf16 rounded again, which changes no numerator (neighbouring
    // values are 2^14 or more apart there, so a difference is 0 or its
    // numerator is).  A branch no ordinary row takes (8192 x 4096 bf16 19.96 us
    // with it, 19.84 without; subtracting in every row 32 x 131072 12.7 -> 13.6).
    constexpr float kLog2e = 1.4426950408889634f;
    if constexpr (!std::is_same<T, _Float16>::value) {
      if (!(fabsf(m) < 4194304.0f)) {
#pragma unroll
        for (int i = 0; i < VPL; ++i)
#pragma unroll
          for (int j = 0; j < N; ++j) v[i][j] = fromf<T>(tof(v[i][j]) - m);
        m = 0.0f;
      }
    }
    const float mb = -m * kLog2e;
    float nzero = -0.0f;
    asm volatile("" : "+v"(nzero));
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      RawVec<T> e;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const float ej = __builtin_amdgcn_exp2f(fmaf(tof(v[i][j]), kLog2e, mb));
        e[j] = fromf<T>(ej);
        s += tof(e[j]);
      }
      // The numerators exist in the storage type here, one vector at a
      // time: otherwise the compiler sinks the roundings into the output
      // pass and keeps every fp32 exponential live (80 instead of 45 VGPRs).
      asm volatile("" : "+v"(e));
      v[i] = e;
    }
    s = row_reduce(s, OpSum(), 1);
    const float inv = 1.0f / s;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      RawVec<T> o;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        // The pin keeps every element on the same two roundings (fp32, then
        // the storage type): left free, the backend fuses some of them into
        // a single-rounding v_fma_mixlo_f16 and not others.
        float p = fmaf(tof(v[i][j]), inv, nzero);
        asm volatile("" : "+v"(p));
        o[j] = fromf<T>(p);
      }
      store_at(i, o);
    }
  } else if constexpr (OP == kRmsNorm) {
    // Every pass is written as fmas whose f16 operands gfx950 takes straight
    // into v_fma_mix_f32 (no separate widening).  `nzero` (-0) is hidden from
    // the optimizer so x*y + (-0) stays an fma: it rounds exactly like x*y,
    // the sign of zero included.  For f16 rows the backend folds the output
    // fma and the conversion into one v_fma_mix{lo,hi}_f16, which rounds
    // once to f16 instead of to fp32 and then to f16 (the two differ only
    // next to an f16 rounding midpoint, inside the tolerance; LayerNorm's
    // output is the same).  Measured (8192 x 4096 f16): 22.23 against
    // 22.30 us with widen-then-multiply, at the copy rate of its bytes.
    float nzero = -0.0f;
    asm volatile("" : "+v"(nzero));
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < VPL; ++i)
#pragma unroll
      for (int j = 0; j < N; ++j) ss = fmaf(tof(v[i][j]), tof(v[i][j]), ss);
    ss = row_reduce(ss, OpSum(), 0);
    fresh(v);
    const float rstd = 1.0f / sqrtf(ss / static_cast<float>(cols) + a.eps);
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const RawVec<T> gi = gamma_at(i);
      RawVec<T> o;
#pragma unroll
      for (int j = 0; j < N; ++j)
        o[j] = fromf<T>(fmaf(fmaf(tof(v[i][j]), rstd, nzero), tof(gi[j]), nzero));
      store_at(i, o);
    }
  } else {  // kLayerNorm
    // The row is widened into mixed-precision fmas as in RMSNorm: the sum as
    // fma(x, 1, s), the centred values as fma(x, 1, -mean) (x - mean,
    // rounded once), with `one` hidden from the optimizer so x*1 stays an
    // fma.  The output is fma((x - mean) * rstd, gamma, beta) from the same
    // centred value: it differs from separately rounded steps in the last
    // fp32 bit only.  (A form that folded the mean into one fma,
    // fma(fma(x, rstd, -mean*rstd), gamma, beta), saved an operation per
    // element but lost the cancellation: a constant row gave beta plus the
    // rounding error of mean*rstd instead of beta.)
    float one = 1.0f;
    asm volatile("" : "+v"(one));
    // A scheduling barrier closes each vector of every pass: the passes
    // then run vector by vector as written (measured 25.05 against 25.2 us).
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
#pragma unroll
      for (int j = 0; j < N; ++j) s = fmaf(tof(v[i][j]), one, s);
      __builtin_amdgcn_sched_barrier(0);
    }
    const float mean = row_reduce(s, OpSum(), 0) / static_cast<float>(cols);
    const float nmean = -mean;
    fresh(v);
    // Padding slots (columns >= cols, loaded as 0) must not add mean^2: only
    // slots that are not whole take the per-element test.
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      if (whole(i)) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const float d = fmaf(tof(v[i][j]), one, nmean);
          q = fmaf(d, d, q);
        }
      } else {
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const float d = (col0(i) + j < cols) ? fmaf(tof(v[i][j]), one, nmean) : 0.0f;
          q = fmaf(d, d, q);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const float var = row_reduce(q, OpSum(), 1) / static_cast<float>(cols);
    fresh(v);
    const float rstd = 1.0f / sqrtf(var + a.eps);
    if (lane == 0 && half == 0 && valid) {
      if (a.mean_out) a.mean_out[r] = mean;
      if (a.rstd_out) a.rstd_out[r] = rstd;
    }
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const RawVec<T> gi = gamma_at(i), bi = beta_at(i);
      RawVec<T> o;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const float d = fmaf(tof(v[i][j]), one, nmean);
        o[j] = fromf<T>(fmaf(d * rstd, tof(gi[j]), tof(bi[j])));
      }
      store_at(i, o);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Streaming kernel for rows longer than the register budget: S waves share a
// row and re-read it per pass (softmax 3: max, sum of rounded numerators,
// output; RMSNorm 2, LayerNorm 3).
//
// f32 LayerNorm above 4096 columns keeps one wave per row (registers to 8192
// columns, then this kernel with S = 1): the mean of a long row is the
// difference of near-equal sums, and its fp32 rounding in another order (a few
// 1e-6 of a mean near zero at 1e5 columns) would show in the mean and rstd
// that callers keep for the backward pass.  (Compensated or 64-bit partial sums
// over more waves would be nearer the true mean; not built.)  Eight loads in
// flight: 175 x 50688 229 -> 88 us, 4096 x 8192 (registers) 75.7 -> 47.3.
template <typename T, int OP, int S>
__global__ __launch_bounds__(S * 64) void row_kernel_stream(RowArgs a) {
  constexpr int N = RowVec<T>::N;
  const int64_t r = blockIdx.x;
  const T* __restrict__ xr = static_cast<const T*>(a.x) + r * a.ldx;
  T* __restrict__ yr = static_cast<T*>(a.y) + r * a.ldy;
  const int64_t cols = a.cols;
  const T* __restrict__ g = static_cast<const T*>(a.gamma);
  const T* __restrict__ b = static_cast<const T*>(a.beta);
  __shared__ float red[2][S];
  auto row_reduce = [&](float x, auto op, int slot) {
    x = wave_reduce(x, op);
    if constexpr (S == 1) return x;
    if ((threadIdx.x & 63) == 0) red[slot][threadIdx.x >> 6] = x;
    __syncthreads();
    return wave_totals<S>(red[slot], op);
  };
  // f(c0, vector, elements of it inside the row) over this thread's vectors.
  auto each = [&](T fill, auto f) {
    const int64_t nfull = cols / N;
    int64_t i = threadIdx.x;
    for (; i + 7 * S * 64 < nfull; i += 8 * S * 64) {  // eight loads in flight
      RawVec<T> v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = load_any(xr + (i + u * S * 64) * N);
#pragma unroll
      for (int u = 0; u < 8; ++u) f((i + u * S * 64) * N, v[u], N);
    }
    for (; i < nfull; i += S * 64) f(i * N, load_any(xr + i * N), N);
    const int rem = static_cast<int>(cols - nfull * N);
    if (rem && static_cast<int64_t>(threadIdx.x) == nfull % (S * 64))
      f(nfull * N, load_tail(xr, nfull * N, cols, fill), rem);
  };
  auto store = [&](int64_t c0, RawVec<T> v, int n) {
    if (n == N) store_any(yr + c0, v);
    else store_tail(yr, c0, cols, v);
  };
  auto param = [&](const T* p, int64_t c0, int n, T none) -> RawVec<T> {
    if (!p) return RawVec<T>(none);
    return n == N ? load_any(p + c0) : load_tail(p, c0, cols, none);
  };

  if constexpr (OP == kSoftmax) {
    // The row max, then the fp32 sum of the numerators rounded to the
    // storage type (the reference's arithmetic, as in row_kernel): an online
    // max/sum would rescale sums of unrounded numerators instead.
    float m = -__builtin_huge_valf();
    each(static_cast<T>(-__builtin_huge_valf()), [&](int64_t, RawVec<T> v, int) {
#pragma unroll
      for (int j = 0; j < N; ++j) m = fmaxf(m, tof(v[j]));
    });
    m = row_reduce(m, OpMax(), 0);
    float s = 0.0f;
    each(static_cast<T>(-__builtin_huge_valf()), [&](int64_t, RawVec<T> v, int n) {
#pragma unroll
      for (int j = 0; j < N; ++j) s += j < n ? tof(fromf<T>(exp_f32(tof(v[j]) - m))) : 0.0f;
    });
    s = row_reduce(s, OpSum(), 1);
    const float scale = 1.0f / s;
    each(T(0), [&](int64_t c0, RawVec<T> v, int n) {
      RawVec<T> o;
#pragma unroll
      for (int j = 0; j < N; ++j) o[j] = fromf<T>(tof(fromf<T>(exp_f32(tof(v[j]) - m))) * scale);
      store(c0, o, n);
    });
  } else if constexpr (OP == kRmsNorm) {
    float ss = 0.0f;
    each(T(0), [&](int64_t, RawVec<T> v, int) {
#pragma unroll
      for (int j = 0; j < N; ++j) ss += tof(v[j]) * tof(v[j]);
    });
    ss = row_reduce(ss, OpSum(), 0);
    const float scale = 1.0f / sqrtf(ss / static_cast<float>(cols) + a.eps);
    each(T(0), [&](int64_t c0, RawVec<T> v, int n) {
      const RawVec<T> gv = param(g, c0, n, T(1));
      RawVec<T> o;
#pragma unroll
      for (int j = 0; j < N; ++j) o[j] = fromf<T>((tof(v[j]) * scale) * tof(gv[j]));
      store(c0, o, n);
    });
  } else {
    float s = 0.0f;
    each(T(0), [&](int64_t, RawVec<T> v, int) {
#pragma unroll
      for (int j = 0; j < N; ++j) s += tof(v[j]);
    });
    const float mean = row_reduce(s, OpSum(), 0) / static_cast<float>(cols);
    float q = 0.0f;
    each(T(0), [&](int64_t, RawVec<T> v, int n) {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const float d = j < n ? tof(v[j]) - mean : 0.0f;
        q += d * d;
      }
    });
    const float var = row_reduce(q, OpSum(), 1) / static_cast<float>(cols);
    const float rstd = 1.0f / sqrtf(var + a.eps);
    if (threadIdx.x == 0) {
      if (a.mean_out) a.mean_out[r] = mean;
      if (a.rstd_out) a.rstd_out[r] = rstd;
    }
    each(T(0), [&](int64_t c0, RawVec<T> v, int n) {
      const RawVec<T> gv = param(g, c0, n, T(1)), bv = param(b, c0, n, T(0));
      RawVec<T> o;
#pragma unroll
      for (int j = 0; j < N; ++j)
        o[j] = fromf<T>((tof(v[j]) - mean) * rstd * tof(gv[j]) + tof(bv[j]));
      store(c0, o, n);
    });
  }
}

namespace {

// Waves per row (S) and 16-byte vectors per lane (VPL) by the row's vectors:
// the fewest slots that hold the row, three or four a lane before the next S
// (one wave up to 256 vectors, where the whole chip's rows are short enough:
// 8192 x 2048 f16 8.6 us with one wave a row, 10.1 with two).  Rows below 64
// vectors share a wave four at a time once there are enough of them to fill
// the chip that way (20000 x 300 f16 softmax 8.3 -> 5.8 us, 60000 x 64 14.9 ->
// 5.0; 100 x 300 2.5 -> 2.7).  Before, every row had one wave, unaligned rows
// were read element by element and rows above 1024 vectors re-read per pass
// (softmax / RMSNorm / LayerNorm, one box, HIP graph): f16 2047 x 5003 30.9 /
// 38.8 / 48.7 -> 8.3 / 8.4 / 9.7 us, 85 x 16857 85.0 / 77.6 / 122.2 -> 5.8 /
// 5.0 / 6.5, 2048 x 16384 50.2 / 42.1 / 66.0 -> 22.2 / 20.1 / 20.7, f32 4096 x
// 8192 75.9 / 57.6 / 75.3 -> 39.4 / 38.9 / 47.3, 175 x 50688 207.7 / 153.4 /
// 229.3 -> 14.4 / 13.4 / 88.
constexpr int64_t kShortRowsMin = 2048;
template <typename T, int OP>
hxm_status launch_rows_t(const RowArgs& a, hipStream_t stream) {
  constexpr int N = RowVec<T>::N;
  const int64_t nv = (a.cols + N - 1) / N;
  hxm_status st = HXM_OK;
  // Rows one call may hold: four to a 256-thread workgroup (the full rows of
  // 512 vectors: their own one or two) within the launch limit.  Wider
  // workgroups launch in as many pieces as that takes.
  auto launch = [&](auto kernel, int threads, int per_group, int per_group_limit) {
    if ((st = check_grid("row kernel", (a.rows + per_group_limit - 1) / per_group_limit, 256)) !=
        HXM_OK)
      return;
    const int64_t piece = (0xffffffffLL / threads) * per_group;
    for (int64_t r = 0; r < a.rows; r += piece) {
      RowArgs p = a;
      p.x = static_cast<const T*>(a.x) + r * a.ldx;
      p.y = static_cast<T*>(a.y) + r * a.ldy;
      if (a.mean_out) p.mean_out = a.mean_out + r;
      if (a.rstd_out) p.rstd_out = a.rstd_out + r;
      p.rows = a.rows - r < piece ? a.rows - r : piece;
      const int64_t groups = (p.rows + per_group - 1) / per_group;
      kernel<<<dim3(static_cast<unsigned>(groups)), dim3(threads), 0, stream>>>(p);
    }
  };
  auto run = [&](auto VC, auto SC, auto LC) {
    constexpr int V = decltype(VC)::value, S = decltype(SC)::value, L = decltype(LC)::value;
    constexpr int per_group = row_waves(S) * (64 / L) / S;
    if (a.cols == static_cast<int64_t>(V) * S * L * N)
      launch(row_kernel<T, OP, V, S, true, L>, 64 * row_waves(S), per_group,
             nv == 512 ? per_group : 4);
    else
      launch(row_kernel<T, OP, V, S, false, L>, 64 * row_waves(S), per_group, 4);
  };
#define HXM_ROWS_L(V, S, L)                                                        \
  run(std::integral_constant<int, V>{}, std::integral_constant<int, S>{}, \
      std::integral_constant<int, L>{})
#define HXM_ROWS(V, S) HXM_ROWS_L(V, S, 64)
  const bool shared = a.rows >= kShortRowsMin;
  if (shared && nv <= 16) HXM_ROWS_L(1, 1, 16);
  else if (shared && nv <= 32) HXM_ROWS_L(2, 1, 16);
  else if (shared && nv <= 48) HXM_ROWS_L(3, 1, 16);
  else if (shared && nv < 64) HXM_ROWS_L(4, 1, 16);
  else if (nv <= 64) HXM_ROWS(1, 1);
  else if (nv <= 128) HXM_ROWS(2, 1);
  else if (nv <= 192) HXM_ROWS(3, 1);
  else if (nv <= 256) HXM_ROWS(4, 1);
  else if (OP == kLayerNorm && nv <= 384) HXM_ROWS(3, 2);
  else if (OP == kLayerNorm && nv <= 512) HXM_ROWS(4, 2);
  else if (nv <= 512) HXM_ROWS(2, 4);
  else if (nv <= 768) HXM_ROWS(3, 4);
  else if (nv <= 1024) HXM_ROWS(4, 4);
  else if (OP == kLayerNorm && sizeof(T) == 4 && nv <= 1536) HXM_ROWS(24, 1);
  else if (OP == kLayerNorm && sizeof(T) == 4 && nv <= 2048) HXM_ROWS(32, 1);
  else if (OP == kLayerNorm && sizeof(T) == 4) launch(row_kernel_stream<T, OP, 1>, 64, 1, 4);
  else if (nv <= 1536) HXM_ROWS(3, 8);
  else if (nv <= 2048) HXM_ROWS(4, 8);
  else if (nv <= 3072) HXM_ROWS(3, 16);
  else if (nv <= 4096) HXM_ROWS(4, 16);
  else if (nv <= 8192) HXM_ROWS(8, 16);
  else if (nv <= 16384) HXM_ROWS(16, 16);
  else launch(row_kernel_stream<T, OP, 16>, 1024, 1, 4);
#undef HXM_ROWS
#undef HXM_ROWS_L
  if (st != HXM_OK) return st;
  return check_launch("row kernel");
}

template <int OP>
hxm_status launch_rows(const RowArgs& a, int32_t dtype, hipStream_t stream) {
  switch (dtype) {
    case HXM_F16: return launch_rows_t<_Float16, OP>(a, stream);
    case HXM_BF16: return launch_rows_t<__bf16, OP>(a, stream);
    default: return launch_rows_t<float, OP>(a, stream);
  }
}

hxm_status validate_rows(const char* op, const void* x, int64_t ldx,
                         const void* y, int64_t ldy, int64_t rows,
                         int64_t cols, int32_t dtype) {
  if (dtype != HXM_F16 && dtype != HXM_BF16 && dtype != HXM_F32)
    return fail(HXM_UNSUPPORTED_DTYPE,
                "unsupported-dtype: %s takes f16, bf16 or f32 (got %d)", op,
                dtype);
  if (rows < 0 || cols < 1)
    return fail(HXM_INVALID_ARG, "invalid-argument: %s rows=%lld cols=%lld",
                op, (long long)rows, (long long)cols);
  if (rows > 0 && (!x || !y))
    return fail(HXM_INVALID_ARG, "invalid-argument: %s null x or y", op);
  if (ldx < cols || ldy < cols)
    return fail(HXM_INVALID_ARG,
                "invalid-argument: %s ldx=%lld ldy=%lld < cols=%lld", op,
                (long long)ldx, (long long)ldy, (long long)cols);
  if (rows > (int64_t(1) << 33))
    return fail(HXM_UNSUPPORTED_SHAPE, "tile-alignment: %s rows=%lld too many",
                op, (long long)rows);
  return HXM_OK;
}

}  // namespace
}  // namespace hxm

using namespace hxm;

extern "C" {

hxm_status hxm_softmax_rows(const void* x, int64_t ldx, void* y, int64_t ldy,
                            int64_t rows, int64_t cols, int32_t dtype,
                            void* stream) {
  hxm_status st = validate_rows("softmax", x, ldx, y, ldy, rows, cols, dtype);
  if (st != HXM_OK) return st;
  if ((st = require_device(nullptr)) != HXM_OK) return st;
  if (rows == 0) return ok();
  RowArgs a{x, ldx, y, ldy, nullptr, nullptr, nullptr, nullptr, rows, cols, 0.0f};
  return launch_rows<kSoftmax>(a, dtype, as_stream(stream));
}

hxm_status hxm_rmsnorm_rows(const void* x, int64_t ldx, const void* gamma,
                            void* y, int64_t ldy, int64_t rows, int64_t cols,
                            float eps, int32_t dtype, void* stream) {
  hxm_status st = validate_rows("rmsnorm", x, ldx, y, ldy, rows, cols, dtype);
  if (st != HXM_OK) return st;
  if (!(eps >= 0.0f))
    return fail(HXM_INVALID_ARG, "invalid-argument: rmsnorm eps must be >= 0");
  if ((st = require_device(nullptr)) != HXM_OK) return st;
  if (rows == 0) return ok();
  RowArgs a{x, ldx, y, ldy, gamma, nullptr, nullptr, nullptr, rows, cols, eps};
  return launch_rows<kRmsNorm>(a, dtype, as_stream(stream));
}

hxm_status hxm_layernorm_rows(const void* x, int64_t ldx, const void* gamma,
                              const void* beta, void* y, int64_t ldy,
                              float* mean_out, float* rstd_out, int64_t rows,
                              int64_t cols, float eps, int32_t dtype,
                              void* stream) {
  hxm_status st = validate_rows("layernorm", x, ldx, y, ldy, rows, cols, dtype);
  if (st != HXM_OK) return st;
  if (!(eps >= 0.0f))
    return fail(HXM_INVALID_ARG, "invalid-argument: layernorm eps must be >= 0");
  if ((st = require_device(nullptr)) != HXM_OK) return st;
  if (rows == 0) return ok();
  RowArgs a{x, ldx, y, ldy, gamma, beta, mean_out, rstd_out, rows, cols, eps};
  return launch_rows<kLayerNorm>(a, dtype, as_stream(stream));
}

}  // extern "C"
