// Operand packs of the matmuls: the [K, N] -> [N, K] weight image (one-time
// prepack, or per call for a plain row-major B) and the f32 -> fp16 operand
// images (the reference's hmx_pack_act_f32 / hmx_pack_weight_f32,
// HMXAPI.h:107-137, which quantise in the pack; its host prepack spells the
// conversion as x + 0.0f -- -0 becomes +0 -- then IEEE round to nearest even,
// hmx_weight_prepack.py:196-207).
//
// All of them stream their operand once, so HBM bounds them.  The transpose
// works on tiles of 128 bytes of K by 128 bytes of N: whole 128-byte lines are
// read (16 bytes a lane) and written (8 lanes to a line), and the tile is
// turned by reading 4-byte words of neighbouring K rows from LDS and swapping
// their bytes with v_perm.  Against 32 x 32 element tiles that moved one element
// a lane (HIP graph, one box): int8 4096 x 4096 21.1 -> 6.4 us, 11008 x 4096
// 51.0 -> 15.4, 4112 x 1500 9.6 -> 4.4, f16 4096 x 4096 22.3 -> 11.6 (5.8 TB/s);
// a call of a few tiles is one tile's latency, f16 256 x 256 2.6 -> 2.5, int8
// 2.5 -> 3.2.  Both f32 operand packs are one launch: f32 1000-cube matmul
// 19.9 -> 16.8, 128-cube 7.3 -> 5.1, 4096-cube 175 -> 146.
#include <algorithm>
#include <type_traits>

#include "device_util.h"
#include "hxm_internal.h"

namespace hxm {

namespace {

__device__ __forceinline__ _Float16 f32_operand_to_f16(float x) {
  return static_cast<_Float16>(x + 0.0f);
}
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}

// 16-byte accesses at any element address (a [K, N] operand may start and
// stride anywhere).
template <typename T, int N>
using AnyVec = T __attribute__((ext_vector_type(N), aligned(sizeof(T))));

// Elements [c0, c0 + 16 / sizeof(T)) of a row, those at or past `cols` zero.
// LONG (cols >= 16 / sizeof(T), chosen once per kernel): always one load, the
// row's last 16 bytes shifted down for its partial chunk, so that a thread's
// loads are unconditional and all in flight together (a branch around each
// made 1000 x 1000 int8 6.4 us).  Shorter rows are read element by element.
template <typename T, bool LONG>
__device__ __forceinline__ v4u32_t load16(const T* __restrict__ row, int64_t c0, int64_t cols) {
  constexpr int E = 16 / sizeof(T);
  if constexpr (LONG) {
    const int64_t at = c0 < cols - E ? c0 : cols - E;
    const int past = static_cast<int>(c0 - at < E ? c0 - at : E);  // elements to shift out
    const unsigned __int128 v = __builtin_bit_cast(
        unsigned __int128, *reinterpret_cast<const AnyVec<T, E>*>(row + at));
    constexpr int kBits = 8 * sizeof(T);
    return __builtin_bit_cast(v4u32_t, past < E ? v >> (past * kBits) : 0);
  } else {
    typedef T vt __attribute__((ext_vector_type(E)));
    vt v = {};
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (c0 + e < cols) v[e] = row[c0 + e];
    return __builtin_bit_cast(v4u32_t, v);
  }
}

// 16 bytes of D from a row of S: a copy, or eight f32 quantised to fp16.
template <typename S, typename D, bool LONG>
__device__ __forceinline__ v4u32_t load_chunk(const S* __restrict__ row, int64_t c0, int64_t cols) {
  if constexpr (sizeof(S) == sizeof(D)) {
    return load16<S, LONG>(row, c0, cols);
  } else {
    const v4f32 a = __builtin_bit_cast(v4f32, load16<S, LONG>(row, c0, cols));
    const v4f32 b = __builtin_bit_cast(v4f32, load16<S, LONG>(row, c0 + 4, cols));
    v8f16 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = f32_operand_to_f16(a[e]);
      v[e + 4] = f32_operand_to_f16(b[e]);
    }
    return __builtin_bit_cast(v4u32_t, v);
  }
}

// One tile of [K, N] S (row stride ld) -> [N, ldd] D, image columns [K, kp) zero.
template <typename S, typename D>
__device__ __forceinline__ void transpose_tile(const S* __restrict__ src, int64_t ld,
                                               D* __restrict__ dst, int64_t ldd, int64_t K,
                                               int64_t N, int64_t kp, int64_t k0, int64_t n0) {
  constexpr int EB = sizeof(D), TE = 128 / EB, E = 16 / EB, Q = 4 / EB;
  constexpr int kPitch = 33;  // words per LDS row: 128 bytes and one word
  __shared__ uint32_t tile[TE * kPitch];
  v4u32_t v[TE / 32];
  auto load = [&](auto LONG) {
#pragma unroll
    for (int i = 0; i < TE / 32; ++i) {
      const int64_t k = k0 + i * 32 + (threadIdx.x >> 3), n = n0 + (threadIdx.x & 7) * E;
      v[i] = load_chunk<S, D, decltype(LONG)::value>(src + (k < K ? k : K - 1) * ld, n, N);
    }
#pragma unroll
    for (int i = 0; i < TE / 32; ++i)
      if (k0 + i * 32 + (threadIdx.x >> 3) >= K) v[i] = v4u32_t{0, 0, 0, 0};
  };
  if (N >= 16 / static_cast<int>(sizeof(S))) load(std::true_type{});  // uniform
  else load(std::false_type{});
#pragma unroll
  for (int i = 0; i < TE / 32; ++i)
#pragma unroll
    for (int w = 0; w < 4; ++w)
      tile[(i * 32 + (threadIdx.x >> 3)) * kPitch + (threadIdx.x & 7) * 4 + w] = v[i][w];
  __syncthreads();
  // Thread (c, q): K elements [E * c, +E) of the Q image rows Q * q.
  const int c = threadIdx.x & 7, q = threadIdx.x >> 3;
  uint32_t d[E];
#pragma unroll
  for (int e = 0; e < E; ++e) d[e] = tile[(c * E + e) * kPitch + q];
  v4u32_t o[Q];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if constexpr (EB == 1) {
      const uint32_t *x = d + 4 * w;
      const uint32_t a = perm(x[1], x[0], 0x05010400u), b = perm(x[3], x[2], 0x05010400u);
      const uint32_t e = perm(x[1], x[0], 0x07030602u), f = perm(x[3], x[2], 0x07030602u);
      o[0][w] = perm(b, a, 0x05040100u);
      o[1][w] = perm(b, a, 0x07060302u);
      o[2][w] = perm(f, e, 0x05040100u);
      o[3][w] = perm(f, e, 0x07060302u);
    } else {
      o[0][w] = perm(d[2 * w + 1], d[2 * w], 0x05040100u);
      o[1][w] = perm(d[2 * w + 1], d[2 * w], 0x07060302u);
    }
  }
  const int64_t k = k0 + c * E;
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    const int64_t n = n0 + q * Q + j;
    if (n >= N || k >= kp) continue;
    D* p = dst + n * ldd + k;
    typedef D vd __attribute__((ext_vector_type(E)));
    if (k + E <= kp) {
      *reinterpret_cast<AnyVec<D, E>*>(p) = __builtin_bit_cast(vd, o[j]);
    } else {  // the row's last, partial chunk in pieces of 8, 4, 2 and 1 bytes
      unsigned __int128 v = __builtin_bit_cast(unsigned __int128, o[j]);
      const int bytes = static_cast<int>(kp - k) * EB;
      auto piece = [&](auto* zero) {
        using P = typename std::remove_reference<decltype(*zero)>::type;
        if constexpr (sizeof(P) >= EB) {
          if (bytes & sizeof(P)) {
            typedef P anyP __attribute__((aligned(EB)));
            *reinterpret_cast<anyP*>(p) = static_cast<P>(v);
            v >>= 8 * sizeof(P);
            p += sizeof(P) / EB;
          }
        }
      };
      piece(static_cast<uint64_t*>(nullptr));
      piece(static_cast<uint32_t*>(nullptr));
      piece(static_cast<uint16_t*>(nullptr));
      piece(static_cast<uint8_t*>(nullptr));
    }
  }
}

template <typename S, typename D>
__global__ __launch_bounds__(256) void transpose_kernel(const S* __restrict__ src, int64_t ld,
                                                        D* __restrict__ dst, int64_t ldd, int64_t K,
                                                        int64_t N) {
  constexpr int TE = 128 / sizeof(D);
  transpose_tile<S, D>(src, ld, dst, ldd, K, N, K, static_cast<int64_t>(blockIdx.y) * TE,
                       static_cast<int64_t>(blockIdx.x) * TE);
}

// Row-major [rows, cols] f32 (row stride ld) -> [rows, kp] f16, one 16-byte
// unit of the image at a time.  IDX: 32-bit where the units allow it (the row
// is a division).
template <typename IDX>
__device__ __forceinline__ void pack_rows(const float* __restrict__ src, int64_t ld,
                                          _Float16* __restrict__ dst, int64_t rows, int64_t cols,
                                          int64_t kp, int64_t block, int64_t blocks) {
  const IDX per = static_cast<IDX>(kp / 8), units = static_cast<IDX>(rows) * per;
  const IDX step = static_cast<IDX>(blocks) * 256;
  for (IDX u = static_cast<IDX>(block) * 256 + threadIdx.x; u < units; u += step) {
    const IDX r = u / per, c = (u - r * per) * 8;
    const float* row = src + static_cast<int64_t>(r) * ld;
    const v4u32_t v = cols >= 4 ? load_chunk<float, _Float16, true>(row, c, cols)
                                : load_chunk<float, _Float16, false>(row, c, cols);
    *reinterpret_cast<v4u32_t*>(dst + static_cast<int64_t>(u) * 8) = v;
  }
}

// Both operands of an f32 matmul in one launch: workgroups [0, a_blocks) pack
// A's rows, the rest B -- [K, N] by transpose tiles (KN), or the rows of an
// [N, K] B.
template <typename IDX, bool KN>
__global__ __launch_bounds__(256) void pack_f32_kernel(const float* __restrict__ A, int64_t lda,
                                                       _Float16* __restrict__ ai, int64_t M,
                                                       const float* __restrict__ B, int64_t ldb,
                                                       _Float16* __restrict__ bi, int64_t N,
                                                       int64_t K, int64_t kp, int a_blocks,
                                                       int n_tiles) {
  const int b = blockIdx.x;
  if (b < a_blocks) {
    pack_rows<IDX>(A, lda, ai, M, K, kp, b, a_blocks);
  } else if constexpr (KN) {
    const int t = b - a_blocks;
    transpose_tile<float, _Float16>(B, ldb, bi, kp, K, N, kp, static_cast<int64_t>(t / n_tiles) * 64,
                                    static_cast<int64_t>(t % n_tiles) * 64);
  } else {
    pack_rows<IDX>(B, ldb, bi, N, K, kp, b - a_blocks, gridDim.x - a_blocks);
  }
}

}  // namespace

namespace {
template <typename S, typename D>
hxm_status launch_transpose(const void* src, int64_t ld, void* dst, int64_t ldo, int64_t K, int64_t N,
                            hipStream_t stream, const char* what) {
  // The entries' launch limit is that of 32-wide tiles: K at most 65535 * 32.
  hxm_status st = check_grid(what, (N + 31) / 32, 256, (K + 31) / 32);
  if (st != HXM_OK) return st;
  constexpr int64_t te = 128 / sizeof(D);
  const dim3 grid(static_cast<unsigned>((N + te - 1) / te), static_cast<unsigned>((K + te - 1) / te));
  transpose_kernel<S, D><<<grid, 256, 0, stream>>>(static_cast<const S*>(src), ld,
                                                   static_cast<D*>(dst), ldo, K, N);
  return check_launch(what);
}
}  // namespace

hxm_status pack_kn_image(const void* B, int64_t ldb, void* out, int64_t ldo, int64_t K, int64_t N,
                         int64_t eb, hipStream_t stream, const char* what) {
  return eb == 1 ? launch_transpose<uint8_t, uint8_t>(B, ldb, out, ldo, K, N, stream, what)
                 : launch_transpose<uint16_t, uint16_t>(B, ldb, out, ldo, K, N, stream, what);
}

hxm_status pack_kn_f32_image(const float* B, int64_t ldb, _Float16* out, int64_t ldo, int64_t K,
                             int64_t N, hipStream_t stream) {
  return launch_transpose<float, _Float16>(B, ldb, out, ldo, K, N, stream, "f32 weight image");
}

hxm_status pack_f32_operands(const float* A, int64_t lda, _Float16* ai, int64_t M, const float* B,
                             int64_t ldb, _Float16* bi, int64_t N, int64_t K, int64_t kp, bool kn,
                             hipStream_t stream) {
  hxm_status st = HXM_OK;
  if (kn && (st = check_grid("f32 weight pack", (N + 31) / 32, 256, (kp + 31) / 32)) != HXM_OK)
    return st;
  auto blocks = [](int64_t units) {
    return std::min<int64_t>((units + 255) / 256, 65536);
  };
  const int64_t ua = M * (kp / 8), ub = N * (kp / 8);
  const int64_t na = M > 0 ? blocks(ua) : 0, nt = (N + 63) / 64;
  const int64_t nb = kn ? nt * ((kp + 63) / 64) : blocks(ub);
  if ((st = check_grid("f32 operand pack", na + nb, 256)) != HXM_OK) return st;
  const dim3 grid(static_cast<unsigned>(na + nb));
  // 32-bit units leave room for a grid stride past the end.
  const bool narrow = std::max(ua, ub) < (int64_t(1) << 31);
  auto launch = [&](auto kernel) {
    kernel<<<grid, 256, 0, stream>>>(A, lda, ai, M, B, ldb, bi, N, K, kp, static_cast<int>(na),
                                     static_cast<int>(nt));
  };
  if (kn) narrow ? launch(pack_f32_kernel<uint32_t, true>) : launch(pack_f32_kernel<uint64_t, true>);
  else narrow ? launch(pack_f32_kernel<uint32_t, false>) : launch(pack_f32_kernel<uint64_t, false>);
  return check_launch("f32 operand pack");
}

}  // namespace hxm
