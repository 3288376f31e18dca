// Launch rules of the skinny matmuls (skinny_kernel.h): the default of the
// W8A16 GEMMs, of hxm_gemm_i8 / _dequant and of hxm_matmul at 1 to
// kSkinnyRowsMax rows, and of hxm_gemv_w8a16 on plain [N, K] weights at any M > 1
// (in blocks of 16 rows, one grid row each).
#include "skinny_kernel.h"

namespace hxm {

namespace {

struct SkinnyShape {
  int rows, groups, threads, lds;  // rows of A and 16-channel output groups per workgroup
  void (*fn)(SkinnyArgs);
};

template <int KIND, int MR, int CB, int NW, int SL, int U, int EPI, bool KN = false>
constexpr SkinnyShape shape() {
  constexpr int al = SL * (KIND == kSkW8 ? 2 : 1) / 16;  // lanes per A row of a slab
  constexpr int eb = KIND == kSkF16 || KIND == kSkBF16 ? 2 : 1;
  constexpr int slab = (KN ? SL / eb * (16 * CB * eb + 4) : CB * 16 * (SL + 16)) + (MR * al + 63) / 64 * 64 / al * (al * 16 + 16);
  constexpr int mt = (MR + 15) / 16, mc = mt * CB <= 4 ? mt : (4 / CB > 0 ? 4 / CB : 1);
  constexpr int red = NW * mc * CB * 64 * 16, stg = NW * U * slab;
  return SkinnyShape{MR, EPI == kEpiSwiglu ? CB / 2 : CB, NW * 64, red > stg ? red : stg,
                     skinny_kernel<KIND, MR, CB, NW, SL, U, EPI, KN>};
}

// The workgroup for M rows.  A rows are covered by the smallest of 4, 16, 32
// and 64: rows past M cost no memory, but their LDS reads and MFMAs do run.
// 128-byte slabs except for f16 x int8 at 64 rows, where a slab's A rows
// (16 KiB a wave) would leave one wave per SIMD (gate/up 51.4 us against
// 40.7, down 35.5 against 30.4).  Gate/up takes 16 + 16 channels, the others
// 16: more channels per workgroup share the A slabs but leave CUs idle (down,
// 16 rows: 32 channels 22.0 us against 16.2 in 64-byte slabs).  Four waves
// instead of eight from 32 rows up for gate/up, whose 688 workgroups fill the
// chip by themselves.
template <int KIND, int EPI>
SkinnyShape shape_for(int64_t M) {
  if constexpr (EPI == kEpiSwiglu) {
    if (M <= 4) return shape<KIND, 4, 2, 8, 128, 1, EPI>();
    if (M <= 16) return shape<KIND, 16, 2, 8, 128, 1, EPI>();
    if (M <= 32) return shape<KIND, 32, 2, 4, 128, 1, EPI>();
    return shape<KIND, 64, 2, 4, 64, 1, EPI>();
  } else {
    if (M <= 4) return shape<KIND, 4, 1, 8, 128, 2, EPI>();
    if (M <= 16 || EPI == kEpiGemv) return shape<KIND, 16, 1, 8, 128, 1, EPI>();
    if constexpr (EPI != kEpiGemv) {
      if (M <= 32) return shape<KIND, 32, 1, 8, 128, 1, EPI>();
      return shape<KIND, 64, 1, 8, KIND == kSkW8 ? 64 : 128, 1, EPI>();
    }
  }
}

SkinnyShape shape_of(int32_t table, int epi, int64_t M) {
  switch (epi) {
    case kEpiSwiglu: return shape_for<kSkW8, kEpiSwiglu>(M);
    case kEpiW8Res: return shape_for<kSkW8, kEpiW8Res>(M);
    case kEpiW8: return shape_for<kSkW8, kEpiW8>(M);
    case kEpiGemv: return shape_for<kSkW8, kEpiGemv>(M);
    case kEpiI32: return shape_for<kSkI8, kEpiI32>(M);
    case kEpiDequant: return shape_for<kSkI8, kEpiDequant>(M);
    default:
      return table == HXM_BF16 ? shape_for<kSkBF16, kEpiFloat>(M) : shape_for<kSkF16, kEpiFloat>(M);
  }
}

// A [K, N] B: 32 channels per workgroup (64 or 32 bytes of each row; with 16 a
// row piece would be a quarter of a line or less), one batch ahead.
template <int KIND, int EPI>
SkinnyShape kn_shape_for(int64_t M) {
  if (M <= 4) return shape<KIND, 4, 2, 8, 128, 1, EPI, true>();
  if (M <= 16) return shape<KIND, 16, 2, 8, 128, 1, EPI, true>();
  if (M <= 32) return shape<KIND, 32, 2, 8, 128, 1, EPI, true>();
  return shape<KIND, 64, 2, 8, 128, 1, EPI, true>();
}

SkinnyShape kn_shape_of(int32_t table, int epi, int64_t M) {
  if (epi == kEpiI32) return kn_shape_for<kSkI8, kEpiI32>(M);
  if (epi == kEpiDequant) return kn_shape_for<kSkI8, kEpiDequant>(M);
  return table == HXM_BF16 ? kn_shape_for<kSkBF16, kEpiFloat>(M)
                           : kn_shape_for<kSkF16, kEpiFloat>(M);
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

// Up to 32 rows the skinny kernel streams the weights faster than any tile.
// Above, a workgroup of 16 channels x 64 rows pays for its own A slabs, and the
// line is drawn by how many of them the chip must run (f16, N x K, M: skinny /
// best tile us, HIP graph, one box): 4096 x 4096, 64: 13.2 / 14.4 (256
// workgroups); 1024 x 4096, 256: 11.2 / 14.0 (256); 2048 x 4096, 192: 19.3 /
// 14.4 (384); below 2 KiB of K the tiles' fixed time is the shorter one (4096 x
// 512, 64: 4.4 / 4.1). int8 alike; the f16 x int8 calls are default_w8_config's.
bool skinny_default(int32_t table, int epi, int64_t M, int64_t n_out, int64_t K) {
  if (!skinny_fits(M, n_out, K)) return false;
  const int64_t kb = K * dtype_bytes(table);
  if (M <= 32) return kb >= 256;
  return kb >= 2048 && skinny_groups(table, epi, M, n_out) <= 256;
}

// Workgroups of a call.
int64_t skinny_groups(int32_t table, int epi, int64_t M, int64_t n_out) {
  const SkinnyShape s = shape_of(table, epi, M);
  return groups_of(s, n_out) * ((M + s.rows - 1) / s.rows);
}

void skinny_plan(int32_t table, int epi, int64_t M, int64_t n_out, bool kn, hxm_plan* p) {
  const SkinnyShape s = kn ? kn_shape_of(table, epi, M) : shape_of(table, epi, M);
  p->config = skinny_config();
  p->threads = s.threads;
  p->tiles = groups_of(s, n_out) * ((M + s.rows - 1) / s.rows);
  p->lds_bytes = s.lds;
}

// Reading B once instead of packing it first (read, write, read): f16 direct /
// pack and skinny / pack and best tile (us, HIP graph, one box), 16 rows: 512 x
// 512 3.3 / 4.6 / 6.3, 2048 x 2048 5.7 / 11.4 / 14.5, 4096 x 4096 11.5 / 19.6 /
// 25.6; int8 4096 x 4096 7.9 / 16.7 / 19.7.  Few workgroups with a long K are
// the exception, which the pack spreads over the chip: 512 x 4096 8.7 / 7.5,
// 64 x 8192 14.6 / 11.8.
bool skinny_takes_kn(int64_t N, int64_t K, int64_t elem_bytes) {
  return N * elem_bytes >= 16 && !((N + 31) / 32 <= 16 && K * elem_bytes >= 8192);
}

hxm_status launch_skinny(int32_t table, int epi, const GemmArgs& g, bool kn, hipStream_t stream) {
  SkinnyArgs a{};
  a.A = g.A;
  a.B = g.B;
  a.C = g.C;
  a.lda_bytes = g.lda_bytes;
  a.ldb_bytes = g.ldb_bytes;
  a.ldc = g.ldc;
  a.M = g.M;
  a.N = g.N;
  a.KB = table == kSkinnyW8 ? g.K_bytes / 2 : g.K_bytes;
  a.n_out = g.n_out;
  a.out_dtype = g.out_dtype;
  a.accumulate = g.accumulate;
  a.row_scale = g.row_scale;
  a.col_scale = g.col_scale;
  a.residual = g.residual;
  a.ldr = g.ldr;
  const SkinnyShape s = kn ? kn_shape_of(table, epi, g.M) : shape_of(table, epi, g.M);
  const dim3 grid(static_cast<unsigned>(groups_of(s, epi == kEpiSwiglu ? g.n_out : g.N)),
                  static_cast<unsigned>((g.M + s.rows - 1) / s.rows));
  hipLaunchKernelGGL(s.fn, grid, dim3(s.threads), 0, stream, a);
  return check_launch("skinny gemm");
}

}  // namespace hxm
