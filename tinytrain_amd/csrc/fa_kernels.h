// Host-side launchers of the attention kernels (one per kernel family and dtype).
// Arguments are validated by the C ABI layer (ttfa_api.hip) before these run.
#pragma once

#include <hip/hip_runtime.h>

namespace ttfa {

hipError_t launch_fwd_bf16(const void *q, const void *k, const void *v, void *o, float *lse,
                           int B, int Hq, int Hkv, int T, int D, float scale, hipStream_t stream);

// Which bf16 D = 128 kernels a shape runs: the 256-row forward / dQ pass (64 rows per wave)
// or the 128-row ones.  A fixed rule on the shape alone (never on the device's occupancy),
// so a shape's output bits are the same on every device: the wide kernels differ from the
// 128-row ones by rounding.
constexpr int kWideSlots = 256;  // one 256-row workgroup per CU on the 256 CUs of an MI355X
bool fwd128_uses_wide(int B, int Hq, int T);
bool dq128_uses_wide(int B, int Hq, int T);
hipError_t launch_bwd_dq_bf16(const void *q, const void *k, const void *v, const void *o,
                              const void *dout, const float *lse, float *delta, void *dq,
                              int B, int Hq, int Hkv, int T, int D, float scale,
                              hipStream_t stream);
hipError_t launch_bwd_dkdv_bf16(const void *q, const void *k, const void *v, const void *dout,
                                const float *lse, const float *delta, void *dk, void *dv,
                                int B, int Hq, int Hkv, int T, int D, float scale,
                                hipStream_t stream);

// How the dK/dV pass of a batched bf16 shape is split over workgroups (stages == 0: it is
// not, one workgroup per key tile), and its launch with the fp32 partials of
// dkdv_part_floats() floats.
struct DkdvSplit {
  int stages;       // 128-row stages per piece, at most
  int pieces;       // pieces per (batch, KV head)
  int split_tiles;  // key tiles 0 .. split_tiles - 1 have several pieces
};
DkdvSplit dkdv_split(int B, int Hq, int Hkv, int T, int D);
int64_t dkdv_part_floats(const DkdvSplit &s, int B, int Hkv, int D);
hipError_t launch_bwd_dkdv_split_bf16(const void *q, const void *k, const void *v,
                                      const void *dout, const float *lse, const float *delta,
                                      void *dk, void *dv, float *part, const DkdvSplit &s, int B,
                                      int Hq, int Hkv, int T, int D, float scale,
                                      hipStream_t stream);

// Packed variable-length sequences, bf16: q/o [Hq, total, D], k/v [Hkv, total, D],
// lse/delta [Hq, total]; cu_seqlens [n_seq + 1] int32 on the device.
hipError_t launch_fwd_varlen_bf16(const void *q, const void *k, const void *v, void *o,
                                  float *lse, const int *cu_seqlens, int n_seq, int total,
                                  int max_seqlen, int Hq, int Hkv, int D, float scale,
                                  hipStream_t stream);
hipError_t launch_bwd_varlen_bf16(const void *q, const void *k, const void *v, const void *o,
                                  const void *dout, const float *lse, float *delta, void *dq,
                                  void *dk, void *dv, const int *cu_seqlens, int n_seq,
                                  int total, int max_seqlen, int Hq, int Hkv, int D, float scale,
                                  hipStream_t stream);

// KV-cache decode: q/o [B, Hq, Tq, D], caches [B, Hkv, Lmax, D], lse [B, Hq, Tq],
// cache_seqlens [B] int32 on the device; workspace of B * Hq * Tq * n_chunks * (D + 2) floats.
struct DecodeSplit {
  int n_waves;   // waves per workgroup
  int n_chunks;  // workgroups per (batch, KV head) at most, one partial per query row each
  int log2_min;  // a workgroup takes 2^log2_min 32-key blocks before the next one gets any
};
DecodeSplit decode_split(int B, int Hkv, int Lmax, int D);
hipError_t launch_decode_bf16(const void *q, const void *k_cache, const void *v_cache,
                              const int *cache_seqlens, void *o, float *lse, float *workspace,
                              int B, int Hq, int Hkv, int Tq, int Lmax, int D, float scale,
                              hipStream_t stream);

hipError_t launch_fwd_f32(const void *q, const void *k, const void *v, void *o, float *lse,
                          int B, int Hq, int Hkv, int T, int D, float scale, hipStream_t stream);
hipError_t launch_bwd_dq_f32(const void *q, const void *k, const void *v, const void *o,
                             const void *dout, const float *lse, float *delta, void *dq,
                             int B, int Hq, int Hkv, int T, int D, float scale,
                             hipStream_t stream);
hipError_t launch_bwd_dkdv_f32(const void *q, const void *k, const void *v, const void *dout,
                               const float *lse, const float *delta, void *dk, void *dv,
                               int B, int Hq, int Hkv, int T, int D, float scale,
                               hipStream_t stream);
// Both fp32 backward passes as one launch.  Without a split (s.stages == 0; part unused) its
// results are, bitwise, those of dq then dkdv; with one (`stages` = 16-row items here) a
// second launch adds the partials of the split key blocks.
DkdvSplit dkdv_split_f32(int B, int Hq, int Hkv, int T, int D);
int64_t dkdv_part_floats_f32(const DkdvSplit &s, int B, int Hkv, int D);
hipError_t launch_bwd_f32(const void *q, const void *k, const void *v, const void *o,
                          const void *dout, const float *lse, float *delta, void *dq, void *dk,
                          void *dv, float *part, const DkdvSplit &s, int B, int Hq, int Hkv, int T,
                          int D, float scale, hipStream_t stream);

}  // namespace ttfa
