// KV-cache decode attention (bf16 in / fp32 accumulate), gfx950: Tq new query rows per
// (batch, head) against a cache of L_b keys, split over the cache length.
//
// The reference has no decode kernel: generate.py:7-20 recomputes the whole prefix for
// every token, and its roadmap lists a KV-cache inference engine (README.md:158).  What
// is computed is the reference's causal attention (model.py:94-98) restricted to the
// last Tq rows: query i of the new tokens sits at position L_b - Tq + i and sees keys
// 0 .. L_b - Tq + i of the cache, O = softmax(q k^T * scale) v, LSE = m + ln(l).
//
// Work split (split-K, "flash decoding"): a unit is one (batch, KV head).  Its 32-key blocks
// in use (its own cache length, not the capacity) are dealt to as many of its n_chunks
// workgroups as have 2^log2_min of them each, in turn over all of their waves; the others
// leave an empty partial.  So a long cache among short ones still has every chunk, and a short
// one few.  The split depends on the call's shape and on the cache's own length alone, never
// on the other caches, so neighbours do not change a row's bits.
// Workgroups are numbered chunk-major, each chunk's units turned (chunk_turn): consecutive ids
// go to the XCDs in turn, and with a multiple of eight units every chunk of a unit would
// share an XCD (16 caches, every other one 400 of 8000 keys, Hkv 4, D 64: 24.7 -> 17.0 us).
// All G query heads of the KV head and all Tq rows form the R = G * Tq <= 32 query columns of
// one 32x32 MFMA tile (columns past R repeat valid ones and are not stored), so the K and V
// bytes are read once for the whole group.
//
// Data path: a wave has one LDS stage, into which a block's K and V rows are loaded directly,
// whole rows in order (16 bytes per lane, 1 KB per instruction).  The next block's K is
// requested as soon as this one's is in registers, before the scores, its V after the last V
// read, so a wave keeps about one block in flight (it waits on its own vmcnt only; no
// workgroup barriers).  Two stages and the whole next block ahead took twice the LDS, one
// workgroup per CU at D = 128, for the same time (16 x 4096 keys, 8 heads, four chunks: 54.0
// us with one stage, 55.1 with two).  K fragments loaded straight into the MFMA operand
// registers, 32 bytes from each of 32 rows per instruction, read 8% slower at 32 x 4096 keys.
// Per block: S^T = K Q^T, online softmax in the exp2 domain (lazy rescale as in the forward
// kernel), O^T += V^T P^T.  The waves' partials (unnormalised O, running max m in log2 units,
// sum l) are merged through LDS, in wave order.  In a call of one chunk the workgroup writes its
// unit's O and LSE; otherwise each writes one fp32 partial per query row (an empty one where the
// unit's cache leaves it no blocks), and a second kernel merges all chunks with the log-sum-exp
// rule.
//
// What bounds it: the cache bytes from HBM (a plain read kernel reaches 6.8-7.1 TB/s on
// MI355X), for small caches the launches, and for one long cache among short ones the rate of
// the CUs that read it (40-60 GB/s each).
// Back-to-back us per call: with one range of keys per wave, four partials per workgroup and
// always two launches; with as many chunks as gave 256 workgroups, all used whatever the
// length (which left a long cache to one or two CUs); now:
//   B 32, Hkv 8, D 128, 4096 keys each                  99.7   92.5   98.0
//     lengths 410..4096 of 4096                         69.0   57.4   59.8
//     one of 4096, the others up to 500                 28.5   36.9   30.5
//   B 16, Hkv 8, D 128, one of 16384, the others short  45.0   68.1   41.6
//   B 64, Hkv 12, D 64, lengths 200..2000 of 2000       49.5   44.8   43.0
//   B 1, Hkv 8, D 128, 16384 keys                       17.0   17.0   16.9
//   B 1, Hkv 2, D 128, 512 keys                         11.6    9.1    9.1  (one launch)
#include "fa_bwd.h"  // allow_lds
#include "fa_common.h"
#include "fa_kernels.h"

namespace ttfa {

namespace {

constexpr float kDecodeSlack = 8.0f;
constexpr int kDecBlock = 32;  // keys per block
constexpr int kDecMaxSplits = 512;  // partials per query row, at most

template <int D>
struct DecShape {
  static constexpr int KK = D / 16, DB = D / 32, CH = D / 8;
  static constexpr int LOADS = kDecBlock * CH / 64;       // 1 KB DMA blocks per K (V) block
  static constexpr int WAVE_LDS = 2 * kDecBlock * D;      // bf16 elements, [K|V]
};

// s_waitcnt vmcnt(N) (gfx9 encoding: vmcnt bits 3:0 and 15:14; expcnt, lgkmcnt at max)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | 0x0F70 | ((N >> 4) << 14));
}

// One 32-key block of one wave: S^T = K Q^T, mask, online softmax, O^T += V^T P^T.
template <int D, bool MASK, class NextK, class WaitV>
__device__ __forceinline__ void decode_block(const bf16 *Kt, const bf16 *Vt,
                                             const bf16x8 (&qf)[D / 16], f32x16 (&oacc)[D / 32],
                                             float &m_t, float &l_part, float scale_log2, int k0,
                                             int pos, int L, int lane, NextK next_k, WaitV wait_v) {
  using P = DecShape<D>;
  const int lg = lane >> 5;
  bf16x8 kf[P::KK];
#pragma unroll
  for (int kk = 0; kk < P::KK; ++kk) kf[kk] = lds_read_row8<D, 1>(Kt, lane & 31, 2 * kk + lg);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the K rows are in registers
  __builtin_amdgcn_sched_barrier(0);
  next_k();
  __builtin_amdgcn_sched_barrier(0);
  f32x16 s = mfma32(kf[0], qf[0], f32x16{});
#pragma unroll
  for (int kk = 1; kk < P::KK; ++kk) s = mfma32(kf[kk], qf[kk], s);
  if (MASK) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = k0 + 8 * (r >> 2) + 4 * lg + (r & 3);
      if (key > pos || key >= L) s[r] = -INFINITY;
    }
  }
  const float mx = xhalf_max(max16(s, -INFINITY)) * scale_log2;
  if (__builtin_amdgcn_ballot_w64(mx > m_t + kDecodeSlack)) {
    const float m_new = fmax2(m_t, mx);
    // 0 when m_t is still -inf; 1 for a column that stays all-masked (m_new = -inf; its
    // sums are still 0), where exp2(-inf - -inf) would be NaN
    const float alpha = m_new == -INFINITY ? 1.f : exp2f_fast(m_t - m_new);
    m_t = m_new;
    l_part *= alpha;
#pragma unroll
    for (int db = 0; db < P::DB; ++db) oacc[db] *= alpha;
  }
  // A column none of whose keys so far is visible keeps m = -inf; its p are all 0.
  const float m_use = m_t == -INFINITY ? 0.f : m_t;
  bf16x8 pb[2];
  float rs = 0.f;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    float p[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = exp2f_fast(__builtin_fmaf(s[8 * m + e], scale_log2, -m_use));
      rs += p[e];
    }
    pb[m] = pack8(f32x16{p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7]}, 0);
  }
  l_part += rs;
  __builtin_amdgcn_sched_barrier(0);
  wait_v();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    bf16x8 vf[P::DB];
#pragma unroll
    for (int db = 0; db < P::DB; ++db) vf[db] = lds_read_trT<D>(Vt, 16 * m, 32 * db, lane);
#pragma unroll
    for (int db = 0; db < P::DB; ++db) oacc[db] = mfma32(vf[db], pb[m], oacc[db]);
  }
}

// Workgroups of a unit that have work: its nb blocks, 2^log2_min each at least (a power of two:
// a quotient would stand between the length's load and the first block's).
__device__ __forceinline__ int used_chunks(int nb, int n_chunks, int log2_min) {
  return max(min((nb + (1 << log2_min) - 1) >> log2_min, n_chunks), 1);
}

// Places by which chunk `chunk` turns its units (n_units >= 8).  Consecutive workgroups go to the
// XCDs in turn, and those of an XCD to its 32 CUs: 37 = 4 * 8 + 5 moves a unit's chunks to
// other XCDs and other CUs.  Fewer units have more chunks, whose own numbers do that.
__device__ __forceinline__ int chunk_turn(int chunk, int n_units) {
  int turn = chunk * (n_units >= 64 ? 37 : 5);
  if (n_units < 32) turn &= 7;
  while (turn >= n_units) turn -= n_units;  // at most five times
  return turn;
}

}  // namespace

// Grid: (B * Hkv units, n_chunks), workgroups of NW waves.  Partial rows are indexed
// (b * Hq + h) * Tq + i, each with n_chunks slots.
// SPLIT: several chunks; a call of one has no part in that logic (a branch on the length before
// the other loads cost 0.6 of 5.6 us with a short cache).
template <int D, int NW, bool SPLIT>
__global__ __launch_bounds__(64 * NW) void fa_decode_bf16_kernel(
    const bf16 *__restrict__ Q, const bf16 *__restrict__ Kc, const bf16 *__restrict__ Vc,
    const int *__restrict__ cache_seqlens, bf16 *__restrict__ O, float *__restrict__ LSE,
    float *__restrict__ part_o, float *__restrict__ part_ml, int B, int Hq, int Hkv, int Tq,
    int Lmax, int n_chunks, int log2_min, float scale_log2) {
  using P = DecShape<D>;
  constexpr int KK = P::KK, DB = P::DB, CH = P::CH;
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];
  bf16 (*lds)[P::WAVE_LDS] = reinterpret_cast<bf16 (*)[P::WAVE_LDS]>(smem);
  __shared__ float wm[NW][32], wsum[NW][32];
  const int chunk = SPLIT ? blockIdx.y : 0;
  int bhk = blockIdx.x;
  // B * Hkv is the grid's width; reading gridDim instead would put 256 bytes of hidden
  // arguments on every launch (1 us of a short call).
  if (const int n_units = B * Hkv; SPLIT && n_units >= 8) {
    bhk -= chunk_turn(chunk, n_units);
    if (bhk < 0) bhk += n_units;
  }
  const int b = bhk / Hkv, hk = bhk - b * Hkv;
  const int G = Hq / Hkv, R = G * Tq;
  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int lq = lane & 31, lg = lane >> 5;
  const int L = min(max(cache_seqlens[b], 0), Lmax);

  // this lane's query column
  const int col = lq % R, g = col / Tq, i = col - g * Tq;
  const int h = hk * G + g;
  const int pos = L - Tq + i;  // last visible key of this column
  const int64_t qrow = ((int64_t)b * Hq + h) * Tq + i;

  // The unit's blocks in use, in turn over all waves of its workgroups.
  const int nb = (L + kDecBlock - 1) / kDecBlock;
  const int used = SPLIT ? used_chunks(nb, n_chunks, log2_min) : 1, step = used * NW;
  const int blk0 = chunk < used ? chunk * NW + wave : nb;
  bf16 *wl = lds[wave];

  f32x16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) oacc[db] = f32x16{};
  float m_t = -INFINITY, l_part = 0.f;

  if (blk0 < nb) {
    const int64_t kvbase = ((int64_t)b * Hkv + hk) * Lmax * D;
    uint32_t koff[P::LOADS], voff[P::LOADS];  // this lane's byte offsets within a 32-row block
#pragma unroll
    for (int j = 0; j < P::LOADS; ++j) {
      const int e = 64 * j + lane, row = e / CH, pc = e % CH;
      koff[j] = (uint32_t)(row * D + swz_l<D, 1>(row, pc) * 8) * 2;
      voff[j] = (uint32_t)(row * D + swz<D>(row, pc) * 8) * 2;
    }
    auto load = [&](const bf16 *src, const uint32_t (&off)[P::LOADS], bf16 *dst, int k0) {
      const auto rs = make_rsrc(src + kvbase + (int64_t)k0 * D, (uint32_t)(L - k0) * D * 2);
#pragma unroll
      for (int j = 0; j < P::LOADS; ++j) buf_load16_lds(rs, off[j], dst + 64 * j * 8);
    };
    bf16 *Kt = wl, *Vt = wl + kDecBlock * D;
    bf16x8 qf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      qf[kk] = *reinterpret_cast<const bf16x8 *>(Q + qrow * D + 16 * kk + 8 * lg);

    load(Kc, koff, Kt, blk0 * kDecBlock);
    load(Vc, voff, Vt, blk0 * kDecBlock);
    const int first_masked = L - Tq;  // keys past this need the mask for some column
#pragma unroll 1
    for (int blk = blk0; blk < nb; blk += step) {
      const int k0 = blk * kDecBlock, kn = k0 + step * kDecBlock;
      const bool more = blk + step < nb;
      wait_vmcnt<P::LOADS>();  // this block's K is in; its V may be in flight
      __builtin_amdgcn_sched_barrier(0);
      auto next_k = [&] {
        if (more) load(Kc, koff, Kt, kn);
      };
      auto wait_v = [&] {
        if (more) wait_vmcnt<P::LOADS>();  // the next K may be in flight, this V is in
        else wait_vmcnt<0>();
      };
      if (k0 + kDecBlock - 1 > first_masked)
        decode_block<D, true>(Kt, Vt, qf, oacc, m_t, l_part, scale_log2, k0, pos, L, lane, next_k, wait_v);
      else
        decode_block<D, false>(Kt, Vt, qf, oacc, m_t, l_part, scale_log2, k0, pos, L, lane, next_k, wait_v);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the V rows are read
      __builtin_amdgcn_sched_barrier(0);
      if (more) load(Vc, voff, Vt, kn);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  if (SPLIT && chunk >= used) {  // an empty partial, whose O the merge does not read
    if (threadIdx.x < R)
      *reinterpret_cast<f32x2 *>(part_ml + (qrow * n_chunks + chunk) * 2) = f32x2{-INFINITY, 0.f};
    return;
  }

  // Merge of the workgroup's waves: every wave scales its partial to the workgroup's running
  // max and stages it as fp32 rows in its own stage (its blocks are consumed, its loads have
  // landed; 32 columns of D floats fill the stage), then the threads add the waves in
  // order.
  const float l = xhalf_sum(l_part);
  if (lg == 0) {
    // A wave without visible keys (l exactly 0) weighs nothing.  A NaN sum is no empty one: its
    // max may still be -inf (no score compares greater), and then the sum is relative to 0.
    wm[wave][lq] = l == 0.f ? -INFINITY : m_t == -INFINITY ? 0.f : m_t;
    wsum[wave][lq] = l;
  }
  __syncthreads();
  float M = wm[0][lq];
#pragma unroll
  for (int w = 1; w < NW; ++w) M = fmax2(M, wm[w][lq]);
  const float mw = wm[wave][lq], alpha = mw == -INFINITY ? 0.f : exp2f_fast(mw - M);
  float *wf = reinterpret_cast<float *>(wl);
  if (lq < R) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int a = 0; a < 4; ++a)
        *reinterpret_cast<f32x4 *>(wf + lq * D + (((8 * db + 2 * a + lg) ^ (lq & 7)) << 2)) =
            alpha != 0.f ? f32x4{oacc[db][4 * a] * alpha, oacc[db][4 * a + 1] * alpha,
                                 oacc[db][4 * a + 2] * alpha, oacc[db][4 * a + 3] * alpha}
                         : f32x4{};
  }
  __syncthreads();
  for (int e = threadIdx.x; e < R * (D / 4); e += 64 * NW) {
    const int c = e / (D / 4), ch = e % (D / 4);
    f32x4 t{};
    float mx = wm[0][c], ls = 0.f;
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = fmax2(mx, wm[w][c]);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float *src = reinterpret_cast<const float *>(lds[w]) + c * D;
      t += *reinterpret_cast<const f32x4 *>(src + ((ch ^ (c & 7)) << 2));
      ls += wm[w][c] == -INFINITY ? 0.f : wsum[w][c] * exp2f_fast(wm[w][c] - mx);
    }
    const int cg = c / Tq;
    const int64_t row = ((int64_t)b * Hq + hk * G + cg) * Tq + (c - cg * Tq);
    if (!SPLIT) {
      const float inv = ls == 0.f ? 0.f : 1.f / ls;  // NaN sums reach O and LSE
      *reinterpret_cast<bf16x4 *>(O + row * D + 4 * ch) =
          pack4(t[0] * inv, t[1] * inv, t[2] * inv, t[3] * inv);
      if (ch == 0) LSE[row] = ls == 0.f ? -INFINITY : (mx + __log2f(ls)) * kLn2;
    } else {
      const int64_t slot = row * n_chunks + chunk;
      *reinterpret_cast<f32x4 *>(part_o + slot * D + 4 * ch) = t;
      if (ch == 0) *reinterpret_cast<f32x2 *>(part_ml + slot * 2) = f32x2{mx, ls};
    }
  }
}

// Merge the partials of every query row whose unit used several workgroups: M = max m over partials with l != 0,
// O = sum o_s 2^(m_s - M) / sum l_s 2^(m_s - M), LSE = (M + log2 sum) ln 2; a row with no
// visible key (every l exactly 0) gets O = 0, LSE = -inf, and a NaN sum makes both NaN.  One 256-thread workgroup per row: thread t sums
// float4 column t % (D/4) over the partials s = t / (D/4) (mod 256 / (D/4)).  The threads
// reduce M and the weights (kept in LDS), then the partials are weighted (a partial without
// keys holds zeros and weight 0) and the groups added in a fixed order, so the result does
// not depend on timing.
template <int D>
__global__ __launch_bounds__(256) void fa_decode_combine_kernel(
    const float *__restrict__ part_o, const float *__restrict__ part_ml, bf16 *__restrict__ O,
    float *__restrict__ LSE, int n_splits) {
  constexpr int C4 = D / 4, SG = 256 / C4;
  __shared__ float wts[kDecMaxSplits];
  __shared__ float red[8];
  __shared__ f32x4 accs[SG][C4];
  const int row = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const float *ml = part_ml + (int64_t)row * n_splits * 2;
  const int c = tid % C4, sg = tid / C4;
  const f32x4 *po = reinterpret_cast<const f32x4 *>(part_o + (int64_t)row * n_splits * D) + c;
  const f32x2 v0 = tid < n_splits ? *reinterpret_cast<const f32x2 *>(ml + 2 * tid) : f32x2{0.f, 0.f};
  float M = v0[1] != 0.f ? v0[0] : -INFINITY;
  for (int s = tid + 256; s < n_splits; s += 256) {
    const f32x2 v = *reinterpret_cast<const f32x2 *>(ml + 2 * s);
    if (v[1] != 0.f) M = fmax2(M, v[0]);
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) M = fmax2(M, __shfl_xor(M, m));
  if (lane == 0) red[wave] = M;
  __syncthreads();
  M = fmax2(fmax2(red[0], red[1]), fmax2(red[2], red[3]));
  float lsum = 0.f;
  for (int s = tid; s < n_splits; s += 256) {
    const f32x2 v = s == tid ? v0 : *reinterpret_cast<const f32x2 *>(ml + 2 * s);
    const float w = v[1] != 0.f ? exp2f_fast(v[0] - M) : 0.f;
    wts[s] = w;
    lsum = __builtin_fmaf(v[1], w, lsum);
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) lsum += __shfl_xor(lsum, m);
  if (lane == 0) red[4 + wave] = lsum;
  __syncthreads();  // wts and the sums are visible
  lsum = (red[4] + red[5]) + (red[6] + red[7]);
  f32x4 acc{};
#pragma unroll 4
  for (int s = sg; s < n_splits; s += SG) {
    const float w = wts[s];
    const f32x4 x = w != 0.f ? po[(int64_t)s * C4] : f32x4{};  // an unused chunk wrote no O
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = w != 0.f ? __builtin_fmaf(x[e], w, acc[e]) : acc[e];
  }
  accs[sg][c] = acc;
  __syncthreads();
  if (tid < C4) {
    f32x4 t = accs[0][tid];
#pragma unroll
    for (int g = 1; g < SG; ++g) t += accs[g][tid];
    const float inv = lsum == 0.f ? 0.f : 1.f / lsum;
    bf16 *out = O + (int64_t)row * D + 4 * tid;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = (bf16)(t[e] * inv);
  }
  if (tid == 0) LSE[row] = lsum == 0.f ? -INFINITY : (M + __log2f(lsum)) * kLn2;
}

// Workgroups per unit, waves per workgroup, and the blocks a workgroup takes at least.
//  * Caches of up to 16 blocks (512 keys) run as one chunk, in one launch: 9.1 us at 512 keys,
//    D 128, B 1, against 11.0 in two launches for 700.
//  * Otherwise as many chunks as stay within 512 workgroups, the slots of a device whose CUs hold
//    two (a few more ran as a second, nearly empty round: 9 x 12 units, 1168 keys, D 64: 540
//    14.5 us, 432 12.1), or one more where that leaves more than a fifth of the slots empty (16 x 12,
//    10267 keys of uneven caches, D 64: 384 workgroups 65.7, 576 57.0; 24 x 8, 3000, D 128: 39.8,
//    36.5, but all full 61.4, 66.5); from one chunk to two only for 2048 keys or more (36 x 8,
//    3352: 109.4 with one, 100.3 with two; 33 x 8, 1043: 40.1, 40.4, and of uneven caches 20.6,
//    23.5).  Half as many (256 at D 128) read full caches 1-7% faster and leave a long cache among
//    short ones to half as many CUs, of 40-60 GB/s each.
//  * One cache has no others beside it: at D = 128 it takes 256 workgroups (8 heads, 16384
//    keys: 16.7 us; 512: 17.5).
//  * D = 128: four waves where a chunk has 24 blocks or more, else two, which merge sooner (26 x 2,
//    4818 keys, 17 blocks a chunk: 29.9 against 33.7; with 32 blocks, 16 x 8, 4096 keys, four read one
//    long cache in 17.2 against 23.4, full ones in 52.7 against 51.0).  D = 64: four, and eight
//    in a call of one chunk of 48 blocks or more (64 x 12, 2000 keys: 69.4 against 72.7; 512 x 12,
//    512: 142 against 133).
//  * A chunk's least is its share of a full cache, so that short caches cost one workgroup each; with
//    up to 32 units, which leave the device idle, a block for every wave (1 x 8, D 128, 1600 of
//    16384 keys: 8.7 us against 10.7).
DecodeSplit decode_split(int B, int Hkv, int Lmax, int D) {
  const int64_t units = (int64_t)B * Hkv;
  const int64_t blocks = ((int64_t)Lmax + kDecBlock - 1) / kDecBlock;
  if (blocks <= 16) return {4, 1, 0};
  const int64_t slots = B == 1 && D == 128 ? 256 : 512;
  int64_t n = slots / units;
  if (n < 1) n = 1;
  if (n * units < slots * 4 / 5 && (n > 1 || blocks >= 64)) ++n;
  const bool one = n == 1;
  int n_waves = D == 64 ? (one && blocks >= 48 ? 8 : 4) : one || blocks / n >= 24 ? 4 : 2;
  const int64_t most = (blocks + n_waves - 1) / n_waves;
  n = n > most ? most : n > kDecMaxSplits ? kDecMaxSplits : n;
  const int64_t least = units <= 32 ? n_waves : (blocks + n - 1) / n;
  int log2_min = 0;
  while (least >> (log2_min + 1)) ++log2_min;
  return {n_waves, (int)n, log2_min};
}

template <int D, int NW, bool SPLIT>
static hipError_t launch_decode(const void *q, const void *k_cache, const void *v_cache,
                                const int *cache_seqlens, void *o, float *lse, float *part_o,
                                float *part_ml, int B, int Hq, int Hkv, int Tq, int Lmax,
                                int n_chunks, int log2_min, float scale_log2,
                                hipStream_t stream) {
  constexpr size_t lds = NW * DecShape<D>::WAVE_LDS * sizeof(bf16);
  // the kernel's static arrays come on top of the dynamic stages
  if (lds + 2 * NW * 32 * sizeof(float) > 65536) {
    hipError_t e = allow_lds<fa_decode_bf16_kernel<D, NW, SPLIT>>(lds);
    if (e != hipSuccess) return e;
  }
  const dim3 grid((unsigned)((int64_t)B * Hkv), (unsigned)n_chunks), block(64 * NW);
  fa_decode_bf16_kernel<D, NW, SPLIT><<<grid, block, lds, stream>>>(
      (const bf16 *)q, (const bf16 *)k_cache, (const bf16 *)v_cache, cache_seqlens, (bf16 *)o,
      lse, part_o, part_ml, B, Hq, Hkv, Tq, Lmax, n_chunks, log2_min, scale_log2);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !SPLIT) return e;
  const int rows = B * Hq * Tq;
  fa_decode_combine_kernel<D><<<dim3((unsigned)rows), dim3(256), 0, stream>>>(
      part_o, part_ml, (bf16 *)o, lse, n_chunks);
  return hipGetLastError();
}

hipError_t launch_decode_bf16(const void *q, const void *k_cache, const void *v_cache,
                              const int *cache_seqlens, void *o, float *lse, float *workspace,
                              int B, int Hq, int Hkv, int Tq, int Lmax, int D, float scale,
                              hipStream_t stream) {
  const DecodeSplit sp = decode_split(B, Hkv, Lmax, D);
  float *part_o = workspace;
  float *part_ml = workspace + (int64_t)B * Hq * Tq * sp.n_chunks * D;
  auto go = [&](auto launch) {
    return launch(q, k_cache, v_cache, cache_seqlens, o, lse, part_o, part_ml, B, Hq, Hkv, Tq,
                  Lmax, sp.n_chunks, sp.log2_min, scale * kLog2e, stream);
  };
  if (sp.n_chunks == 1) {
    if (D == 64) return sp.n_waves == 8 ? go(launch_decode<64, 8, false>) : go(launch_decode<64, 4, false>);
    return go(launch_decode<128, 4, false>);
  }
  if (D == 64) return go(launch_decode<64, 4, true>);
  return sp.n_waves == 2 ? go(launch_decode<128, 2, true>) : go(launch_decode<128, 4, true>);
}

}  // namespace ttfa
