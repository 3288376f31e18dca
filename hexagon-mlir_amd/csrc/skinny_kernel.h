#pragma once
// Skinny MFMA matmuls on gfx950: up to 64 rows of A per workgroup (a GEMM or
// matmul has at most kSkinnyRowsMax; the plain-layout GEMV any number, 16 at a
// time) against the [N, K] image of B, or B as it is [K, N].
//
// What bounds such a call is the weight stream: each weight byte meets at
// most 64 rows, far below the matrix cores' ratio.  The LDS-staged tiles
// spend it badly: a 256x256 tile leaves most CUs without a workgroup (86 of
// 256 CUs for the 22016 gate/up rows, 32 for a 4096-row down projection) and
// each walks all of K alone.  Here a workgroup owns 16 * CB channels and its
// NW waves split K:
//   * a wave takes SL bytes of K of every row at a time (U such slabs in one
//     batch, the next batch's loads in flight while this one is multiplied),
//     the waves of the workgroup consecutive batches; every weight byte is
//     read by one wave of the grid;
//   * consecutive lanes read consecutive 16-byte chunks of a row, so each load
//     covers whole 128-byte lines, and the slab is turned into MFMA fragments
//     (lane = row) through LDS, in an area of the wave's own: no barrier in
//     the K loop.  Loading fragments straight from memory touches a different
//     row with every lane of a quad, four lines per clock instead of one:
//     one row of A, gate/up 22016 x 4096 20.8 us that way, 18.4 us through
//     LDS in 64-byte slabs and 14.1 us in 128-byte slabs; 4096 x 11008 13.0,
//     11.8 and 9.6 us (one box; a plain read of the same bytes 13.9 and 7.9);
//   * W is the first operand of v_mfma_*_16x16x* (rows = channels), A the
//     second (columns = rows of A): the CB channel groups share each A
//     fragment and the 16-row blocks of A each converted weight fragment;
//   * buffer loads: rows past M or N and 16-byte chunks past K take an offset
//     beyond the resource, which returns zeros without a memory access, so
//     every load is unconditional and the waits the compiler places are exact;
//   * at the end the NW partial tiles are added in wave order through LDS (a
//     fixed order) and the epilogue runs on the sums.
// Gate/up + SwiGLU and down projection (hidden 4096, intermediate 11008),
// against the 256-row tiles: 1 row 65.8 -> 14.1 and 94.7 -> 9.6 us, 16 rows
// 66.2 -> 19.2 and 94.8 -> 13.3, 32 rows 66.6 -> 25.0 and 95.1 -> 19.3, 57
// rows 67.5 -> 40.7 and 96.5 -> 30.4 (one box; from 33 rows on a K split of the
// 64x128 tile can be the shorter one, 27.0 and 18.0 there: default_w8_config).
#include <type_traits>

#include "gemm_kernel.h"

namespace hxm {

// Operand kinds.
enum SkinnyKind { kSkW8 = 0, kSkF16 = 1, kSkBF16 = 2, kSkI8 = 3 };

struct SkinnyArgs {
  const uint8_t* A;  // [M, K] rows of lda_bytes
  const uint8_t* B;  // [N, K] rows of ldb_bytes
  void* C;
  int64_t lda_bytes, ldb_bytes, ldc;  // ldc in elements
  int M, N;
  int KB;            // K bytes of a B row, a multiple of 16
  int n_out;         // kEpiSwiglu: output columns (N is the image's rows)
  int out_dtype;     // kEpiFloat: HXM_F16 / HXM_BF16 / HXM_F32
  int accumulate;    // kEpiI32, kEpiFloat
  const float* row_scale;
  const float* col_scale;    // kEpiGemv: f16
  const _Float16* residual;  // kEpiW8Res
  int64_t ldr;
};

// Offset added to a lane's chunk past K (or row past the end).  Both
// operands' spans are below it: 64 rows of at most 2^23 bytes (the entries
// admit operands whose 256 rows lie within 2 GiB).
constexpr uint32_t kSkOob = 0x40000000u;

// KN (f16, bf16 and int8): B is the plain [K, N] operand instead, in any
// alignment.  A slab is then SL bytes of A's K as rows of 16 * CB channels, and
// the words of neighbouring K rows are put together into fragments as they
// leave LDS (kn_fragment), so the call needs no transposed copy of B: packing
// one reads, writes and reads again what this reads once.
template <int KIND, int MR, int CB, int NW, int SL, int U, int EPI, bool KN = false>
__global__ __launch_bounds__(NW * 64) void skinny_kernel(SkinnyArgs g) {
  constexpr bool W8 = KIND == kSkW8;
  constexpr int XL = W8 ? 2 : 1;       // A bytes per weight byte
  constexpr bool SW = EPI == kEpiSwiglu;
  static_assert(!SW || CB % 2 == 0, "gate and up groups come in pairs");
  constexpr int MT = (MR + 15) / 16;   // 16-row blocks of A
  constexpr int JS = SL / 64;          // 64-byte pieces of a slab: one weight fragment each
  // Staging: rows of a slab read by consecutive lanes, 16 bytes each, kept in
  // LDS with 16 bytes of padding per row.
  constexpr int WL = SL / 16, WN = 16 / (64 / WL);            // lanes per W row, loads per group
  constexpr int AL = SL * XL / 16;                            // lanes per A row
  constexpr int AN = (MR * AL + 63) / 64;                     // A loads per slab
  constexpr int kWRow = SL + 16, kARow = SL * XL + 16;
  constexpr int kARows = AN * 64 / AL;                        // staged A rows (>= MR)
  constexpr int EB = KIND == kSkF16 || KIND == kSkBF16 ? 2 : 1;
  constexpr int kKnRows = SL / EB, kKnBytes = 16 * CB * EB;   // KN: slab rows, bytes of each
  constexpr int kKnPitch = kKnBytes + 4, RL = kKnBytes / 16;  // lanes per row
  static_assert(!KN || (!W8 && (EPI == kEpiFloat || EPI == kEpiI32 || EPI == kEpiDequant) &&
                        (kKnPitch * kKnRows) % 16 == 0), "[K, N] operands");
  constexpr int WL_N = KN ? kKnRows * RL / 64 : CB * WN;      // weight loads per slab
  constexpr int kSlab = (KN ? kKnRows * kKnPitch : CB * 16 * kWRow) + kARows * kARow;
  using acc_t = typename std::conditional<KIND == kSkI8, v4i32, v4f32>::type;
  constexpr int MC = MT * CB <= 4 ? MT : (4 / CB > 0 ? 4 / CB : 1);  // row blocks per reduction round
  constexpr int TC = MC * CB;                                        // tiles per round
  static_assert(MT % MC == 0, "reduction rounds");
  constexpr int kRed = NW * TC * 64 * 16, kStg = NW * U * kSlab;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kRed > kStg ? kRed : kStg];
  acc_t(*part)[TC][64] = reinterpret_cast<acc_t(*)[TC][64]>(lds);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  // Channel blocks go to workgroups XCD-contiguously (workgroups are
  // dispatched round-robin over the 8 XCDs), so that each XCD streams one
  // contiguous eighth of the weights.
  const int G = gridDim.x, b = blockIdx.x, xcd = b & 7;
  const int blk = xcd * (G >> 3) + min(xcd, G & 7) + (b >> 3);
  const int m_base = blockIdx.y * MR;
  const int rows = min(MR, g.M - m_base);

  // First B row of channel group c.  SwiGLU: rows [128q, 128q + 64) of the
  // image are gate channels and the next 64 the same up channels; group c of
  // the CB/2 gate groups is paired with group c + CB/2, 64 rows further.
  auto b_row0 = [&](int c) {
    if constexpr (SW) {
      const int grp = blk * (CB / 2) + c % (CB / 2);  // 16-channel output group
      return (grp >> 2) * 128 + (grp & 3) * 16 + (c / (CB / 2)) * 64;
    } else {
      return (blk * CB + c) * 16;
    }
  };
  __amdgpu_buffer_rsrc_t wr[KN ? 1 : CB];
  if constexpr (!KN)
#pragma unroll
  for (int c = 0; c < CB; ++c) {
    const int row0 = b_row0(c);
    const int left = min(16, g.N - row0);
    const int64_t bytes = left > 0 ? (left - 1) * g.ldb_bytes + g.KB : 0;
    wr[c] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(g.B) + (left > 0 ? row0 : 0) * g.ldb_bytes, static_cast<short>(0),
        static_cast<int>(bytes), 0x00020000);
  }
  const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(g.A) + m_base * g.lda_bytes, static_cast<short>(0),
      static_cast<int>((rows - 1) * g.lda_bytes + g.KB * XL), 0x00020000);
  // A row past N or M lies past its resource by itself.
  const int wr_ = lane / WL, wc = (lane % WL) * 16;
  const int ar_ = lane / AL, ac = (lane % AL) * 16;
  uint32_t woff[WN], aoff[AN];
#pragma unroll
  for (int t = 0; t < WN; ++t)
    woff[t] = static_cast<uint32_t>((t * (64 / WL) + wr_) * g.ldb_bytes + wc);
#pragma unroll
  for (int t = 0; t < AN; ++t) {
    const int row = t * (64 / AL) + ar_;
    aoff[t] = row < rows ? static_cast<uint32_t>(row * g.lda_bytes + ac) : kSkOob;
  }

  acc_t acc[MT][CB];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[t][c] = acc_t{};

  struct Batch {
    v4i32 w[U][WL_N], a[U][AN];
  };
  // KN: the lane's chunk of a row -- the row's last one is the last 16 bytes
  // of B's row, shifted down -- and the K rows it takes.
  const int kn_n = blk * (16 * CB) + (lane % RL) * (16 / EB);
  const int kn_at = min(kn_n, g.N - 16 / EB), kn_out = min(kn_n - kn_at, 16 / EB);
  const int kn_k = lane / RL, K = g.KB / EB;
  const int slabs = (g.KB + SL - 1) / SL;
  auto load = [&](Batch& q, int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k0 = (s0 * U + u) * SL;
      const uint32_t wk = k0 + (k0 + wc < g.KB ? 0u : kSkOob);
      const uint32_t ak = k0 * XL + (k0 * XL + ac < g.KB * XL ? 0u : kSkOob);
      if constexpr (KN) {
        // Rows past K load row K - 1 (they are zeroed on the way to LDS).
#pragma unroll
        for (int t = 0; t < WL_N; ++t) {
          const int k = min(k0 / EB + t * (64 / RL) + kn_k, K - 1);
          typedef v4i32 any __attribute__((aligned(1)));
          q.w[u][t] = *reinterpret_cast<const any*>(g.B + k * g.ldb_bytes + kn_at * EB);
        }
      } else {
#pragma unroll
        for (int c = 0; c < CB; ++c)  // nontemporal: the weights are streamed once
#pragma unroll
          for (int t = 0; t < WN; ++t)
            q.w[u][c * WN + t] = __builtin_bit_cast(
                v4i32, __builtin_amdgcn_raw_buffer_load_b128(wr[c], woff[t] + wk, 0, 2));
      }
#pragma unroll
      for (int t = 0; t < AN; ++t)
        q.a[u][t] = __builtin_bit_cast(
            v4i32, __builtin_amdgcn_raw_buffer_load_b128(ar, aoff[t] + ak, 0, 0));
    }
  };
  uint8_t* const area = lds + wave * (U * kSlab);
  auto multiply = [&](const Batch& q, int s0) {
    asm volatile("" ::: "memory");  // the previous slab's reads come first
#pragma unroll
    for (int u = 0; u < U; ++u) {
      uint8_t* const as = area + u * kSlab;
      uint8_t* const ws = as + kARows * kARow;
      if constexpr (KN) {
#pragma unroll
        for (int t = 0; t < WL_N; ++t) {
          const int row = t * (64 / RL) + kn_k;
          const bool in = (s0 * U + u) * kKnRows + row < K;
          unsigned __int128 v = __builtin_bit_cast(unsigned __int128, q.w[u][t]);
          v = in && kn_out < 16 / EB ? v >> (kn_out * 8 * EB) : 0;
          const v4u32_t o = __builtin_bit_cast(v4u32_t, v);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            *reinterpret_cast<uint32_t*>(ws + row * kKnPitch + (lane % RL) * 16 + e * 4) = o[e];
        }
      } else {
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
          for (int t = 0; t < WN; ++t)
            *reinterpret_cast<v4i32*>(ws + (c * 16 + t * (64 / WL) + wr_) * kWRow + wc) =
                q.w[u][c * WN + t];
      }
#pragma unroll
      for (int t = 0; t < AN; ++t)
        *reinterpret_cast<v4i32*>(as + (t * (64 / AL) + ar_) * kARow + ac) = q.a[u][t];
    }
    // One wave's LDS operations complete in order; this keeps the compiler's.
    asm volatile("" ::: "memory");
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint8_t* const as = area + u * kSlab;
      const uint8_t* const ws = as + kARows * kARow;
#pragma unroll
      for (int j = 0; j < JS; ++j) {
        v4i32 af[MT][XL];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int h = 0; h < XL; ++h)
            af[t][h] = *reinterpret_cast<const v4i32*>(
                as + (MR < 16 ? r16 % kARows : t * 16 + r16) * kARow + ((j * 4 + kq) * XL + h) * 16);
#pragma unroll
        for (int c = 0; c < CB; ++c) {
          v4i32 w;
          if constexpr (KN)
            w = kn_fragment<EB>(ws, kKnPitch, (j * 4 + kq) * (16 / EB), (c * 16 + r16) * EB);
          else
            w = *reinterpret_cast<const v4i32*>(ws + (c * 16 + r16) * kWRow + (j * 4 + kq) * 16);
          if constexpr (W8) {
            const v8f16 wa = i8x8_to_f16<b_offset_binary(EPI)>(static_cast<uint32_t>(w[0]),
                                                               static_cast<uint32_t>(w[1]));
            const v8f16 wb = i8x8_to_f16<b_offset_binary(EPI)>(static_cast<uint32_t>(w[2]),
                                                               static_cast<uint32_t>(w[3]));
#pragma unroll
            for (int t = 0; t < MT; ++t) {
              acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  wa, __builtin_bit_cast(v8f16, af[t][0]), acc[t][c], 0, 0, 0);
              acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  wb, __builtin_bit_cast(v8f16, af[t][1]), acc[t][c], 0, 0, 0);
            }
          } else {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
              if constexpr (KIND == kSkF16)
                acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(v8f16, w), __builtin_bit_cast(v8f16, af[t][0]), acc[t][c],
                    0, 0, 0);
              else if constexpr (KIND == kSkBF16)
                acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(v8bf16, w), __builtin_bit_cast(v8bf16, af[t][0]), acc[t][c],
                    0, 0, 0);
              else
                acc[t][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, af[t][0], acc[t][c], 0, 0, 0);
            }
          }
        }
      }
    }
  };
  // Two batches of U slabs in flight alternately; loads past K fetch nothing.
  Batch q0, q1;
  const int end = (slabs + U - 1) / U;
  load(q0, wave);
  for (int s = wave; s < end; s += 2 * NW) {
    load(q1, s + NW);
    multiply(q0, s);
    load(q0, s + 2 * NW);
    if (s + NW < end) multiply(q1, s + NW);
  }
  __syncthreads();  // the sums reuse the staging areas

  // Sum of the NW partial tiles and the epilogue, TC tiles a round.  Lane l of
  // a tile holds D[channel 4 * (l / 16) + v][row l % 16].
#pragma unroll
  for (int t0 = 0; t0 < MT; t0 += MC) {
    if (t0 > 0) __syncthreads();  // the previous round's sums are read
#pragma unroll
    for (int t = 0; t < MC; ++t)
#pragma unroll
      for (int c = 0; c < CB; ++c) part[wave][t * CB + c][lane] = acc[t0 + t][c];
    __syncthreads();
    constexpr int OT = SW ? TC / 2 : TC;  // output tiles of the round
    for (int i = threadIdx.x; i < OT * 64; i += NW * 64) {
      const int ot = i >> 6, l = i & 63;
      const int t = SW ? ot / (CB / 2) : ot / CB, c = SW ? ot % (CB / 2) : ot % CB;
      auto total = [&](int cc) {
        acc_t s = part[0][t * CB + cc][l];
#pragma unroll
        for (int w = 1; w < NW; ++w) s += part[w][t * CB + cc][l];
        return s;
      };
      const int m = m_base + (t0 + t) * 16 + (l & 15);
      const int ch = 4 * (l >> 4);
      const int n = SW ? (blk * (CB / 2) + c) * 16 + ch : b_row0(c) + ch;
      const int n_end = SW ? g.n_out : g.N;
      if (m >= g.M || n >= n_end) continue;
      const acc_t a = total(c);
      const int64_t off = static_cast<int64_t>(m) * g.ldc + n;
      if constexpr (EPI == kEpiI32) {
        int32_t* p = static_cast<int32_t*>(g.C) + off;
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (n + v < n_end)
            p[v] = static_cast<int32_t>(static_cast<uint32_t>(a[v]) +
                                        (g.accumulate ? static_cast<uint32_t>(p[v]) : 0u));
      } else if constexpr (EPI == kEpiFloat) {
        auto put = [&](auto* p) {
          using O = typename std::remove_reference<decltype(*p)>::type;
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (n + v < n_end)
              p[v] = static_cast<O>(g.accumulate ? a[v] + static_cast<float>(p[v]) : a[v]);
        };
        if (g.out_dtype == HXM_F32) put(static_cast<float*>(g.C) + off);
        else if (g.out_dtype == HXM_F16) put(static_cast<_Float16*>(g.C) + off);
        else put(static_cast<__bf16*>(g.C) + off);
      } else {
        // f16 outputs in the tile kernels' spellings: fp32 products and sums,
        // each rounded once (the pins keep the backend from fusing them into
        // the conversion).
        v4f16_t h;
        acc_t up = a;
        if constexpr (SW) up = total(c + CB / 2);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int nv = n + v < n_end ? n + v : n;
          if constexpr (SW) {
            const float gv = a[v] * g.col_scale[b_row0(c) + ch + nv - n];
            const float uv = up[v] * g.col_scale[b_row0(c + CB / 2) + ch + nv - n];
            const float ex = __builtin_amdgcn_exp2f(-gv * 1.4426950408889634f);
            h[v] = static_cast<_Float16>(gv * __builtin_amdgcn_rcpf(1.0f + ex) * uv);
          } else {
            float p = static_cast<float>(a[v]);
            if constexpr (EPI == kEpiDequant) p *= g.row_scale[m];
            if constexpr (EPI == kEpiGemv)
              p *= static_cast<float>(reinterpret_cast<const _Float16*>(g.col_scale)[nv]);
            else
              p *= g.col_scale[nv];
            asm volatile("" : "+v"(p));
            if constexpr (EPI == kEpiW8Res) {
              p = p + static_cast<float>(g.residual[static_cast<int64_t>(m) * g.ldr + nv]);
              asm volatile("" : "+v"(p));
            }
            h[v] = static_cast<_Float16>(p);
          }
        }
        _Float16* p = static_cast<_Float16*>(g.C) + off;
        if (n + 4 <= n_end && (reinterpret_cast<uintptr_t>(p) & 7) == 0) {
          *reinterpret_cast<v4f16_t*>(p) = h;
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (n + v < n_end) p[v] = h[v];
        }
      }
    }
  }
}

}  // namespace hxm
