// K split of the W8A16 GEMMs: the 128x128 and 64x128 tiles with workgroup row z taking one
// slice of K into an fp32 partial plane, and the pass that adds the planes.
//
// A call of few tiles is bound by the walk over K of each: at 57 rows the
// 128x128 tile's down projection (hidden 4096, intermediate 11008) is 32 tiles
// of 172 stages, 67 us on an eighth of the chip (and 27 us for the skinny
// kernel, which stages x once per 16 channels).  Sliced 8 ways every CU has a
// workgroup: 18.3 us with the planes' write and read (S * M * N * 4 bytes each)
// and the second launch.  512 x 1024 x 4096: 27.5 us unsplit, 14.5 in 6 slices;
// 256 rows of hidden 11008, intermediate 2048, gate/up: 71.6, 32.6 in 4.
//
// Up to 64 rows the 64x128 tile takes the place of the 128x128 one: half the x
// rows staged and half the MFMA work.  57 rows, 4096 -> 11008 gate/up in 2
// slices 34.2, 27.0 us; the down projection in 8 slices 19.4, 18.0.
#include "gemm_kernel.h"

namespace hxm {

template <int I, int EPI>
static constexpr gemm_fn part_kernel() {
  constexpr ConfigKey k = kW8Keys[kW8PartEntry + I];
  return gemm_kernel<_Float16, k.bm, k.bn, k.bkb, k.st, k.wm, k.wn, EPI>;
}
extern const gemm_fn kW8PartFns[kW8PartEntries][2] = {
    {part_kernel<0, kEpiW8Part>(), part_kernel<0, kEpiSwPart>()},
    {part_kernel<1, kEpiW8Part>(), part_kernel<1, kEpiSwPart>()}};

// One thread: four consecutive output columns of a row.  Plane rows are ldp
// floats, a multiple of four; SwiGLU reads the gate channels and, 64 image rows
// on, the up channels.  The epilogues are the tile kernels' (fp32 products and
// sums, each rounded once).
template <int EPI>
__global__ __launch_bounds__(256) void w8_reduce_kernel(GemmArgs g, const float* __restrict__ planes,
                                                        int S, int64_t plane, int64_t ldp, int quads) {
  const int n_end = EPI == kEpiSwiglu ? g.n_out : g.N;
  const unsigned t = blockIdx.x * 256 + threadIdx.x;
  const unsigned mu = t / static_cast<unsigned>(quads);
  if (mu >= static_cast<unsigned>(g.M)) return;
  const int64_t m = mu;
  const int n = static_cast<int>(t - mu * quads) * 4;
  const int col = EPI == kEpiSwiglu ? (n >> 6) * 128 + (n & 63) : n;
  const float* p = planes + m * ldp + col;
  auto total = [&](const float* q) {
    // Four loads in flight; the sum goes in plane order.
    v4f32 s = *reinterpret_cast<const v4f32*>(q);
    int z = 1;
    for (; z + 4 <= S; z += 4) {
      v4f32 w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = *reinterpret_cast<const v4f32*>(q + (z + i) * plane);
#pragma unroll
      for (int i = 0; i < 4; ++i) s += w[i];
    }
    for (; z < S; ++z) s += *reinterpret_cast<const v4f32*>(q + z * plane);
    return s;
  };
  const v4f32 a = total(p);
  v4f32 up = a;
  if constexpr (EPI == kEpiSwiglu) up = total(p + 64);
  _Float16* c = static_cast<_Float16*>(g.C) + m * g.ldc + n;
  v4f16_t h;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int e = n + v < n_end ? v : 0;
    if constexpr (EPI == kEpiSwiglu) {
      const float gv = a[v] * g.col_scale[col + e];
      const float uv = up[v] * g.col_scale[col + 64 + e];
      const float ex = __builtin_amdgcn_exp2f(-gv * 1.4426950408889634f);
      h[v] = static_cast<_Float16>(gv * __builtin_amdgcn_rcpf(1.0f + ex) * uv);
    } else {
      float r = a[v] * g.col_scale[n + e];
      asm volatile("" : "+v"(r));
      if constexpr (EPI == kEpiW8Res) {
        r = r + static_cast<float>(g.residual[m * g.ldr + n + e]);
        asm volatile("" : "+v"(r));
      }
      h[v] = static_cast<_Float16>(r);
    }
  }
  if (n + 4 <= n_end && (reinterpret_cast<uintptr_t>(c) & 7) == 0) {
    *reinterpret_cast<v4f16_t*>(c) = h;
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (n + v < n_end) c[v] = h[v];
  }
}

hxm_status launch_w8_reduce(int epi, const GemmArgs& g, const float* planes, int S, int64_t ldp,
                            hipStream_t stream) {
  const int quads = ((epi == kEpiSwiglu ? g.n_out : g.N) + 3) / 4;
  const int64_t blocks = (static_cast<int64_t>(g.M) * quads + 255) / 256;
  hxm_status st = check_grid("w8a16 split reduce", blocks, 256);
  if (st != HXM_OK) return st;
  const int64_t plane = static_cast<int64_t>(g.M) * ldp;
  auto run = [&](auto kernel) {
    kernel<<<dim3(static_cast<unsigned>(blocks)), 256, 0, stream>>>(g, planes, S, plane, ldp, quads);
  };
  if (epi == kEpiSwiglu) run(w8_reduce_kernel<kEpiSwiglu>);
  else if (epi == kEpiW8Res) run(w8_reduce_kernel<kEpiW8Res>);
  else run(w8_reduce_kernel<kEpiW8>);
  return check_launch("w8a16 split reduce");
}

}  // namespace hxm
