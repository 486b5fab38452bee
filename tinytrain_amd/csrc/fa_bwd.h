// Declarations shared by the backward translation units: the dK/dV pass's per-head view,
// the kernel templates (fa_bwd.hip defines the dQ kernels; the dK/dV kernels, batched and
// packed variable-length, exist only as the D = 64 and D = 128 specializations in
// fa_bwd_dkdv64.hip and fa_bwd_dkdv128.hip, hand-scheduled stage streams), the staged-tile
// helpers of those passes and the dynamic-LDS opt-in.
#pragma once

#include <atomic>

#include "fa_common.h"

namespace ttfa {

// One KV head's rows (k, v, dk, dv: T rows of D) for one sequence, and the G query heads
// that read it: query head g's q / dout rows at q + g * head_stride (elements), its lse /
// delta values at lse + g * row_stride.
struct DkvHead {
  const bf16 *k, *v;
  bf16 *dk, *dv;
  const bf16 *q, *dout;
  const float *lse, *delta;
  int64_t head_stride, row_stride;
  int G, T;
};

// LDS byte address of a pointer into the workgroup's shared memory.
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
  return (uint32_t)(uintptr_t)(const TTFA_LDS void *)p;
}

// Split dK/dV pass: the G * (n_ktiles - kt) stages of key tile kt are dealt to n =
// ceil(count / stages) pieces, evenly; the pieces of a unit (one KV head of one batch) are
// numbered key tile by key tile.
struct DkvPiece {
  int kt, n, it0, it1;  // key tile, its piece count, this piece's stages
};

// Walks the key tiles of a unit in order with each one's piece count, without a division per
// tile (a scalar division costs about 40 instructions, and a long sequence has hundreds of
// tiles): spare is what the tile's pieces could hold beyond its list.
struct DkvTiles {
  int G, stages, kt = 0, n, spare;
  __host__ __device__ __forceinline__ DkvTiles(int n_ktiles, int G_, int stages_)
      : G(G_), stages(stages_) {
    n = (G * n_ktiles + stages - 1) / stages;
    spare = n * stages - G * n_ktiles;
  }
  __host__ __device__ __forceinline__ void next() {  // while kt < n_ktiles
    ++kt;
    spare += G;
    while (spare >= stages) {
      spare -= stages;
      --n;
    }
  }
};

__device__ __forceinline__ DkvPiece dkv_piece(int piece, int n_ktiles, int G, int stages) {
  if (stages >= G * n_ktiles) return {piece, 1, 0, G * (n_ktiles - piece)};
  DkvTiles t(n_ktiles, G, stages);
  while (piece >= t.n) {  // the grid holds exactly the unit's pieces, so kt stays < n_ktiles
    piece -= t.n;
    t.next();
  }
  const int count = G * (n_ktiles - t.kt);
  return {t.kt, t.n, (int)((int64_t)count * piece / t.n), (int)((int64_t)count * (piece + 1) / t.n)};
}

// Pieces of a unit before key tile kt, and kt's own count.
struct DkvSlot {
  int first, n;
};

__device__ __forceinline__ DkvSlot dkv_slot(int kt, int n_ktiles, int G, int stages) {
  DkvTiles t(n_ktiles, G, stages);
  int first = 0;
  while (t.kt < kt) {
    first += t.n;
    t.next();
  }
  return {first, t.n};
}

// fp32 partial sums of one piece: the four waves' accumulators as they lie in registers,
// [wave][dK | dV][column block][a][lane] of 4 floats (register 4a + e of the block), so
// stores and the reducing reads are whole 1 KB rows.
template <int D>
struct DkvPart {
  static constexpr int DB = D / 32;
  static constexpr int FLOATS = 4 * 2 * DB * 4 * 64 * 4;
  static __device__ __forceinline__ int at(int wave, int which, int db, int a, int lane) {
    return ((((wave * 2 + which) * DB + db) * 4 + a) * 64 + lane) * 4;
  }
};

template <int D>
__device__ __forceinline__ void store_part(const f32x16 (&dk)[D / 32], const f32x16 (&dv)[D / 32],
                                           float *part, int wave, int lane) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      *reinterpret_cast<f32x4 *>(part + DkvPart<D>::at(wave, 0, db, a, lane)) =
          f32x4{dk[db][4 * a], dk[db][4 * a + 1], dk[db][4 * a + 2], dk[db][4 * a + 3]};
      *reinterpret_cast<f32x4 *>(part + DkvPart<D>::at(wave, 1, db, a, lane)) =
          f32x4{dv[db][4 * a], dv[db][4 * a + 1], dv[db][4 * a + 2], dv[db][4 * a + 3]};
    }
}

template <int D>
__global__ void fa_bwd_dq_bf16_kernel(const bf16 *__restrict__ Q, const bf16 *__restrict__ K,
                                      const bf16 *__restrict__ V, const bf16 *__restrict__ O,
                                      const bf16 *__restrict__ dO, const float *__restrict__ LSE,
                                      float *__restrict__ Delta, bf16 *__restrict__ dQ, int B,
                                      int Hq, int Hkv, int T, float scale_log2, float scale);
// D = 128 dQ pass over 256-row tiles, 64 rows per wave (fa_bwd_dq128.hip): for launches
// whose 256-row pairs fill the resident workgroup slots and whose T exceeds 1792.
__global__ void fa_bwd_dq_wide_bf16_kernel(const bf16 *__restrict__ Q, const bf16 *__restrict__ K,
                                           const bf16 *__restrict__ V, const bf16 *__restrict__ O,
                                           const bf16 *__restrict__ dO,
                                           const float *__restrict__ LSE, float *__restrict__ Delta,
                                           bf16 *__restrict__ dQ, int B, int Hq, int Hkv, int T,
                                           float scale_log2, float scale, int paired);
template <int D>
__global__ void fa_bwd_dkdv_bf16_kernel(const bf16 *__restrict__ Q, const bf16 *__restrict__ K,
                                        const bf16 *__restrict__ V, const bf16 *__restrict__ dO,
                                        const float *__restrict__ LSE,
                                        const float *__restrict__ Delta, bf16 *__restrict__ dK,
                                        bf16 *__restrict__ dV, int B, int Hq, int Hkv, int T,
                                        float scale_log2, float scale, int paired);
template <int D>
__global__ void fa_bwd_dkdv_varlen_bf16_kernel(
    const bf16 *__restrict__ Q, const bf16 *__restrict__ K, const bf16 *__restrict__ V,
    const bf16 *__restrict__ dO, const float *__restrict__ LSE, const float *__restrict__ Delta,
    bf16 *__restrict__ dK, bf16 *__restrict__ dV, const int *__restrict__ cu_seqlens, int n_seq,
    int total, int max_seqlen, int Hq, int Hkv, float scale_log2, float scale);
template <int D>
__global__ void fa_bwd_dkdv_split_bf16_kernel(
    const bf16 *__restrict__ Q, const bf16 *__restrict__ K, const bf16 *__restrict__ V,
    const bf16 *__restrict__ dO, const float *__restrict__ LSE, const float *__restrict__ Delta,
    bf16 *__restrict__ dK, bf16 *__restrict__ dV, float *__restrict__ part, int n_units, int Hq,
    int Hkv, int T, int stages, float scale_log2, float scale);
template <>
__global__ void fa_bwd_dkdv_split_bf16_kernel<64>(
    const bf16 *__restrict__ Q, const bf16 *__restrict__ K, const bf16 *__restrict__ V,
    const bf16 *__restrict__ dO, const float *__restrict__ LSE, const float *__restrict__ Delta,
    bf16 *__restrict__ dK, bf16 *__restrict__ dV, float *__restrict__ part, int n_units, int Hq,
    int Hkv, int T, int stages, float scale_log2, float scale);
template <>
__global__ void fa_bwd_dkdv_split_bf16_kernel<128>(
    const bf16 *__restrict__ Q, const bf16 *__restrict__ K, const bf16 *__restrict__ V,
    const bf16 *__restrict__ dO, const float *__restrict__ LSE, const float *__restrict__ Delta,
    bf16 *__restrict__ dK, bf16 *__restrict__ dV, float *__restrict__ part, int n_units, int Hq,
    int Hkv, int T, int stages, float scale_log2, float scale);
template <>
__global__ void fa_bwd_dkdv_bf16_kernel<64>(const bf16 *__restrict__ Q, const bf16 *__restrict__ K,
                                            const bf16 *__restrict__ V, const bf16 *__restrict__ dO,
                                            const float *__restrict__ LSE,
                                            const float *__restrict__ Delta, bf16 *__restrict__ dK,
                                            bf16 *__restrict__ dV, int B, int Hq, int Hkv, int T,
                                            float scale_log2, float scale, int paired);
template <>
__global__ void fa_bwd_dkdv_bf16_kernel<128>(const bf16 *__restrict__ Q, const bf16 *__restrict__ K,
                                             const bf16 *__restrict__ V, const bf16 *__restrict__ dO,
                                             const float *__restrict__ LSE,
                                             const float *__restrict__ Delta, bf16 *__restrict__ dK,
                                             bf16 *__restrict__ dV, int B, int Hq, int Hkv, int T,
                                             float scale_log2, float scale, int paired);
template <>
__global__ void fa_bwd_dkdv_varlen_bf16_kernel<64>(
    const bf16 *__restrict__ Q, const bf16 *__restrict__ K, const bf16 *__restrict__ V,
    const bf16 *__restrict__ dO, const float *__restrict__ LSE, const float *__restrict__ Delta,
    bf16 *__restrict__ dK, bf16 *__restrict__ dV, const int *__restrict__ cu_seqlens, int n_seq,
    int total, int max_seqlen, int Hq, int Hkv, float scale_log2, float scale);
template <>
__global__ void fa_bwd_dkdv_varlen_bf16_kernel<128>(
    const bf16 *__restrict__ Q, const bf16 *__restrict__ K, const bf16 *__restrict__ V,
    const bf16 *__restrict__ dO, const float *__restrict__ LSE, const float *__restrict__ Delta,
    bf16 *__restrict__ dK, bf16 *__restrict__ dV, const int *__restrict__ cu_seqlens, int n_seq,
    int total, int max_seqlen, int Hq, int Hkv, float scale_log2, float scale);
// LDS bytes of the dK/dV passes (batched and packed varlen): two 128-row stages of Q and dO
// tiles plus their -LSE/scale and -Delta rows.
constexpr int kDkv64LdsBytes = 2 * (2 * 128 * 64 * 2 + 2 * 128 * 4);
constexpr int kDkv128LdsBytes = 2 * (2 * 128 * 128 * 2 + 2 * 128 * 4);
// D = 128 dQ pass: two 128-key stages of K and V tiles (workgroups of 256 query rows).
constexpr int kDq128LdsBytes = 2 * 2 * 128 * 128 * 2;

// Raises KERN's dynamic-LDS limit (needed above 64 KiB) once per device: later launches,
// including launches under stream capture, make no attribute call.
template <auto KERN>
static hipError_t allow_lds(size_t bytes) {
  static std::atomic<uint64_t> done{0};  // bit d: set on device d
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = dev >= 0 && dev < 64 ? uint64_t{1} << dev : 0;
  if (bit && (done.load(std::memory_order_acquire) & bit)) return hipSuccess;
  e = hipFuncSetAttribute(reinterpret_cast<const void *>(KERN),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
  return e;
}

}  // namespace ttfa
