// Internal helpers shared by the HIP translation units of libhxm: status and
// reason reporting, dtype sizes, launch checks and the library-owned
// per-stream workspace.  Nothing here is part of the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/hxm.h"
#include "host_logic.h"

namespace hxm {

// Records `reason` as this thread's last error and returns `st`.  Reasons
// start with the manifest vocabulary word ("tile-alignment", ...) so that a
// caller can switch on the prefix.
hxm_status fail(hxm_status st, const char* fmt, ...)
    __attribute__((format(printf, 2, 3)));
// Clears the thread's last error and returns HXM_OK.
hxm_status ok();

inline int64_t dtype_bytes(int32_t dt) {
  switch (dt) {
    case HXM_F16:
    case HXM_BF16: return 2;
    case HXM_F32:
    case HXM_I32: return 4;
    case HXM_I8: return 1;
    default: return 0;
  }
}

inline bool aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}


// Refuses a launch that grid_fits rejects ("tile-alignment"); HXM_OK otherwise.
hxm_status check_grid(const char* what, int64_t groups_x, int threads, int64_t groups_y = 1);

// Checks the launch that was just enqueued.
hxm_status check_launch(const char* what);

// Current device's gfx950 check (cached per device).  Returns HXM_OK or
// HXM_NO_DEVICE with a reason.
hxm_status require_device(int* device_out);

// Library-owned scratch for one (device, stream, slot), grown on demand and
// kept until hxm_release_cache().  Calls on the same stream are ordered, so
// one buffer per stream never races with itself.  Slot 0 holds per-call
// operand packs and the tuner's reference output; slot 1 the split-K
// partial planes, so the two never overwrite or reallocate each other.
constexpr int kWsMain = 0, kWsSplitK = 1, kWsStreamK = 2;
// Largest split-K partial-plane buffer (S * M * N int32) a call may ask for;
// the buffer stays allocated until hxm_release_cache().
constexpr int64_t kSplitKPlaneBytesMax = int64_t(256) << 20;
// Slot 2 holds the W8A16 stream-K partial tiles and arrival counters.
// *grown (when given) says whether the buffer was (re)allocated by this call.
// True while `stream` captures a graph, or when that cannot be read (the null
// stream during another stream's global-mode capture).
bool stream_capturing(hipStream_t stream);
hxm_status stream_workspace(hipStream_t stream, size_t bytes, void** out, int slot = kWsMain,
                            bool* grown = nullptr);
// CUs of the current device (cached per device; 0 when it cannot be read).
int device_cu_count();

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// The legality lattice of a GEMM config (search.hip): front-end block
// limit, min-rows, MFMA edge and wave grid, LDS budget (0 = 160 KiB) for
// a_bytes / b_bytes per element of A and B; HXM_REASON_OK or the first rule
// it breaks.  Whether the config was compiled is not part of it.
int32_t gpu_lattice(const hxm_gemm_config& c, int64_t a_bytes, int64_t b_bytes,
                    int64_t lds_budget);

// Frees the resident weight images of device `dev` (resident.hip).
hxm_status release_images(int dev);

// The direct-load small-output GEMM (gemm_small.hip): f16 / bf16 A [M, K]
// and B as the [N, K] image, one wave per 16x16 output tile, no LDS.  The
// default of hxm_matmul for outputs of at most kSmallTilesMax 16x16 tiles
// and K <= kSmallKMax; a caller names it with small_gemm_config().
constexpr int64_t kSmallTilesMax = 512;
constexpr int64_t kSmallKMax = 256;
hxm_gemm_config small_gemm_config();
bool is_small_gemm_config(const hxm_gemm_config& c);
bool small_gemm_fits(int64_t M, int64_t N, int64_t K, int32_t ab_dtype);
int64_t small_gemm_lds(int64_t K, bool kn);
hxm_status launch_small_gemm(int32_t ab_dtype, const void* A, int64_t lda, const uint8_t* B,
                             int64_t ldb_bytes, bool kn, void* C, int64_t ldc, int64_t M,
                             int64_t N, int64_t K, int32_t out_dtype, int32_t accumulate,
                             hipStream_t stream);
// kn: B is the plain [K, N] operand, in any alignment, of rows of 16 bytes or more.
inline bool small_takes_kn(int64_t N) { return N >= 8; }

// Operand packs (pack.hip).  [K, N] (elements of eb = 1 or 2 bytes, row stride
// ldb) -> the [N, K] image of row stride ldo; the same from f32 to fp16; and the
// fp16 images of both operands of an f32 matmul ([M, kp] and [N, kp], kp = K
// rounded up to 8, zero past K) in one launch.
hxm_status pack_kn_image(const void* B, int64_t ldb, void* out, int64_t ldo, int64_t K, int64_t N,
                         int64_t eb, hipStream_t stream, const char* what);
hxm_status pack_kn_f32_image(const float* B, int64_t ldb, _Float16* out, int64_t ldo, int64_t K,
                             int64_t N, hipStream_t stream);
hxm_status pack_f32_operands(const float* A, int64_t lda, _Float16* ai, int64_t M, const float* B,
                             int64_t ldb, _Float16* bi, int64_t N, int64_t K, int64_t kp, bool kn,
                             hipStream_t stream);

// The skinny matmul (gemm_skinny.hip): takes 1 to kSkinnyRowsMax rows and is
// the default where skinny_default says so (table: the operand dtype, or
// kSkinnyW8 for f16 A and int8 B; epi: gemm_kernel.h's Epilogue); a caller names
// it with skinny_config().
constexpr int64_t kSkinnyRowsMax = 256;
constexpr int32_t kSkinnyW8 = 0;
bool skinny_default(int32_t table, int epi, int64_t M, int64_t n_out, int64_t K);
int64_t skinny_groups(int32_t table, int epi, int64_t M, int64_t n_out);
hxm_gemm_config skinny_config();
bool is_skinny_config(const hxm_gemm_config& c);
bool skinny_fits(int64_t M, int64_t N, int64_t K);

}  // namespace hxm

#define HXM_HIP_TRY(expr)                                                    \
  do {                                                                       \
    hipError_t _e = (expr);                                                  \
    if (_e != hipSuccess)                                                    \
      return ::hxm::fail(HXM_HIP_ERROR, "hip-error: %s failed: %s", #expr,   \
                         hipGetErrorString(_e));                             \
  } while (0)
