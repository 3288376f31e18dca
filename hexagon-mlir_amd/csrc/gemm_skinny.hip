// Launch rules of the skinny W8A16 matmuls (skinny_kernel.h): the default of
// hxm_gemm_w8a16, _residual and _swiglu at 1 to kSkinnyRowsMax rows.
#include "skinny_kernel.h"

namespace hxm {

namespace {

struct SkinnyShape {
  int rows, groups, threads, lds;  // rows of A and 16-channel groups per workgroup
  void (*fn)(SkinnyArgs);
};

template <int MR, int CB, int NW, int SL, int U, int EPI>
constexpr SkinnyShape w8_shape() {
  constexpr int slab = CB * 16 * (SL + 16) +
                       ((MR * SL * 2 / 16 + 63) / 64) * 64 / (SL * 2 / 16) * (SL * 2 + 16);
  constexpr int mt = (MR + 15) / 16, mc = mt * CB <= 4 ? mt : (4 / CB > 0 ? 4 / CB : 1);
  constexpr int red = NW * mc * CB * 64 * 16, stg = NW * U * slab;
  return SkinnyShape{MR, EPI == kEpiSwiglu ? CB / 2 : CB, NW * 64, red > stg ? red : stg,
                     skinny_kernel<kSkW8, MR, CB, NW, SL, U, EPI>};
}

// The workgroup for M rows.  A rows are covered by the smallest of 4, 16, 32
// and 64: rows past M cost no memory, but their LDS reads and MFMAs do run.
// 128-byte slabs except at 64 rows, where a slab's A rows (16 KiB a wave)
// would leave one wave per SIMD (gate/up 51.4 us against 40.7, down 35.5
// against 30.4).  Gate/up takes 16 + 16 channels, the others 16: more
// channels per workgroup share the A slabs but leave CUs idle (down, 16 rows:
// 32 channels 22.0 us against 16.2 in 64-byte slabs).  Four waves instead of
// eight from 32 rows up for gate/up, whose 688 workgroups fill the chip by
// themselves.
template <int EPI>
SkinnyShape w8_shape_for(int64_t M) {
  if constexpr (EPI == kEpiSwiglu) {
    if (M <= 4) return w8_shape<4, 2, 8, 128, 1, EPI>();
    if (M <= 16) return w8_shape<16, 2, 8, 128, 1, EPI>();
    if (M <= 32) return w8_shape<32, 2, 4, 128, 1, EPI>();
    return w8_shape<64, 2, 4, 64, 1, EPI>();
  } else {
    if (M <= 4) return w8_shape<4, 1, 8, 128, 2, EPI>();
    if (M <= 16) return w8_shape<16, 1, 8, 128, 1, EPI>();
    if (M <= 32) return w8_shape<32, 1, 8, 128, 1, EPI>();
    return w8_shape<64, 1, 8, 64, 1, EPI>();
  }
}

SkinnyShape w8_shape_of(int epi, int64_t M) {
  return epi == kEpiSwiglu  ? w8_shape_for<kEpiSwiglu>(M)
         : epi == kEpiW8Res ? w8_shape_for<kEpiW8Res>(M)
                            : w8_shape_for<kEpiW8>(M);
}

int64_t groups_of(const SkinnyShape& s, int64_t n_out) {
  return ((n_out + 15) / 16 + s.groups - 1) / s.groups;
}

}  // namespace

hxm_gemm_config skinny_config() { return hxm_gemm_config{16, 16, 64, 1, 8, 0, 1}; }

bool is_skinny_config(const hxm_gemm_config& c) {
  const hxm_gemm_config s = skinny_config();
  return c.bm == s.bm && c.bn == s.bn && c.bk == s.bk && c.waves_m == s.waves_m &&
         c.waves_n == s.waves_n && c.stages == s.stages && c.split_k <= 1;
}

bool skinny_fits(int64_t M, int64_t N, int64_t K) {
  return M > 0 && N > 0 && K > 0 && M <= kSkinnyRowsMax && grid_fits((N + 15) / 16, 512);
}

void skinny_plan_w8(int epi, int64_t M, int64_t n_out, hxm_plan* p) {
  const SkinnyShape s = w8_shape_of(epi, M);
  p->config = skinny_config();
  p->threads = s.threads;
  p->tiles = groups_of(s, n_out) * ((M + s.rows - 1) / s.rows);
  p->lds_bytes = s.lds;
}

hxm_status launch_skinny_w8(int epi, const GemmArgs& g, hipStream_t stream) {
  SkinnyArgs a{};
  a.A = g.A;
  a.B = g.B;
  a.C = g.C;
  a.lda_bytes = g.lda_bytes;
  a.ldb_bytes = g.ldb_bytes;
  a.ldc = g.ldc;
  a.M = g.M;
  a.N = g.N;
  a.KB = g.K_bytes / 2;
  a.n_out = g.n_out;
  a.col_scale = g.col_scale;
  a.residual = g.residual;
  a.ldr = g.ldr;
  const SkinnyShape s = w8_shape_of(epi, g.M);
  const dim3 grid(static_cast<unsigned>(groups_of(s, g.n_out)),
                  static_cast<unsigned>((g.M + s.rows - 1) / s.rows));
  hipLaunchKernelGGL(s.fn, grid, dim3(s.threads), 0, stream, a);
  return check_launch("skinny w8a16 gemm");
}

}  // namespace hxm
