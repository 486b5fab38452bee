// Causal GQA attention forward/backward in fp32 (the reference's fp32 configuration,
// which must agree with the fp32 eager path to 1e-5) on the fp32 matrix cores.
//
// Same contract as the bf16 kernels (kernels/flash_attn.py:12-217): O, natural-log
// LSE, Delta = rowsum(O*dO), dQ, and dK/dV reduced over the query-head group without
// atomics.  The reference feeds fp32 through the same tiled dot products as bf16
// (kernels/flash_attn.py:49,60); here every product is v_mfma_f32_16x16x4_f32 (fp32
// operands, fp32 accumulate) and the exponentials are the accurate expf / logf.
//
// Work split: 16-row blocks.  A workgroup owns one 16-row query block (forward, dQ) or
// one 16-key block (dK/dV); its waves (eight or four, see below) take the
// block's partner blocks round-robin (the key blocks at or below the diagonal, or the
// query blocks at or above it over the head group), each with its own partial result,
// and the partials are merged through LDS in wave order, so results do not depend on
// timing.
//
// Data path: every 16-row block of Q, K, V, O or dO crosses global memory once per use,
// in fully coalesced 16-byte loads (consecutive lanes read consecutive 16 bytes), into
// registers one block ahead of its use; at its turn the wave writes it to a
// wave-private LDS tile and reads the MFMA operands back from there.  (Loading the
// operands straight from global memory makes every load instruction touch 16 rows,
// which saturates the per-CU load pipeline long before HBM or L2.)  The LDS writes come
// first and the next block's loads go into the same registers: loads issued before the
// writes need a second set and a move per register, which cost the forward 21.4 -> 23.3 us
// at 2x8/2x500 and 105.8 -> 114.7 at 2x16/8x900 (D = 128, eight waves).
//
// MFMA 16x16x4 lane layout (lane = 16 j + n): A supplies A[n][j], B supplies B[j][n],
// and register r of the result is D[4 j + r][n].  A contraction over D features uses
// feature (D / 4) j + kk at k-step kk, so each lane's operand is one contiguous quarter
// of a row ("row fragment").  A contraction over a block's 16 rows uses row 4 j + r at
// k-step r, which is exactly what the lane holds of a previous product: a product's
// result feeds the next one as its B operand with no data movement; the other operand
// is a column of a block ("column fragment").
#include "fa_bwd.h"  // dkv_piece
#include "fa_common.h"
#include "fa_kernels.h"

namespace ttfa {

namespace {

constexpr int kF32Rows = 16;  // rows per block

// Waves per workgroup.  Forward: eight at D = 64, eight or four at D = 128
// (f32_fwd_eight_waves).  Backward: eight at D = 64, four at D = 128, whose 340 operand
// registers do not leave room for two waves per SIMD (with K and V re-read from LDS tiles
// eight fit, spilling 24: 67.2 us against 68.2 at 2x8/2x500, but 27.5 against 21.4 at
// 4x6/2x130).
template <int D>
constexpr int f32_waves() {
  return D == 64 ? 8 : 4;
}

// One LDS tile: a 16-row block, rows padded to D + 4 floats.
template <int D>
constexpr int tile_floats() {
  return kF32Rows * (D + 4);
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Sum / max over the four lanes n, n + 16, n + 32, n + 48 (the lane groups j).
__device__ __forceinline__ float group_sum(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}
__device__ __forceinline__ float group_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}

// A 16-row block in registers: load i of lane l holds floats [4 (64 i + l), + 4) of the
// row-major block (rows past the last valid row, last, repeat it).
template <int D>
struct BlockRegs {
  f32x4 v[D / 16];
};

template <int D>
__device__ __forceinline__ void load_block(BlockRegs<D> &b, const float *__restrict__ base,
                                           int row0, int last, int lane) {
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    const int e = 64 * i + lane, row = e / (D / 4), c4 = e % (D / 4);
    b.v[i] = *reinterpret_cast<const f32x4 *>(base + (int64_t)min(row0 + row, last) * D + 4 * c4);
  }
}

template <int D>
__device__ __forceinline__ void store_block(float *tile, const BlockRegs<D> &b, int lane) {
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    const int e = 64 * i + lane, row = e / (D / 4), c4 = e % (D / 4);
    *reinterpret_cast<f32x4 *>(tile + row * (D + 4) + 4 * c4) = b.v[i];
  }
}

// Row fragment of tile row n: features (D/4) j .. (D/4) j + D/4 - 1.
template <int D>
__device__ __forceinline__ void read_rowfrag(float (&f)[D / 4], const float *tile, int j, int n) {
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    const f32x4 x = *reinterpret_cast<const f32x4 *>(tile + n * (D + 4) + (D / 4) * j + 4 * i);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * i + e] = x[e];
  }
}

// Column fragment: f[4 db + r] = tile[4 j + r][16 db + n].
template <int D>
__device__ __forceinline__ void read_colfrag(float (&f)[D / 4], const float *tile, int j, int n) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int db = 0; db < D / 16; ++db) f[4 * db + r] = tile[(4 * j + r) * (D + 4) + 16 * db + n];
}

// acc[m][n] = sum over D of a[m][:] b[n][:]: A and B both row fragments.
template <int D>
__device__ __forceinline__ f32x4 dot_block(const float (&a)[D / 4], const float (&b)[D / 4]) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < D / 4; ++kk) acc = mfma4(a[kk], b[kk], acc);
  return acc;
}

// acc[db] (features 16 db + 4 j + r', column n) += sum over the block's rows of
// col[row][feature] * w[row][n]; w is a product result (register r = row 4 j + r).
template <int D>
__device__ __forceinline__ void accum_cols(f32x4 (&acc)[D / 16], const float (&col)[D / 4],
                                           const f32x4 &w) {
#pragma unroll
  for (int db = 0; db < D / 16; ++db)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[db] = mfma4(col[4 * db + r], w[r], acc[db]);
}

// Write a wave's partial (lane: features 16 db + 4 j + r of row n) into a tile.
template <int D>
__device__ __forceinline__ void put_partial(float *tile, const f32x4 (&acc)[D / 16], int j,
                                            int n) {
#pragma unroll
  for (int db = 0; db < D / 16; ++db)
    *reinterpret_cast<f32x4 *>(tile + n * (D + 4) + 16 * db + 4 * j) = acc[db];
}

// The merge gives each thread of the workgroup a chunk of CH consecutive features of
// one row: 16 rows x D features over 64 NW threads.
template <int D, int NW>
struct Merge {
  static constexpr int CH = D / (4 * NW);
  int row, c0;
  __device__ Merge() : row(threadIdx.x / (4 * NW)), c0((threadIdx.x % (4 * NW)) * CH) {}
};

template <int CH>
__device__ __forceinline__ void store_chunk(float *dst, const float (&x)[CH], float mul) {
  if constexpr (CH == 2) {
    *reinterpret_cast<f32x2 *>(dst) = f32x2{x[0] * mul, x[1] * mul};
  } else {
#pragma unroll
    for (int e = 0; e < CH; e += 4)
      *reinterpret_cast<f32x4 *>(dst + e) =
          f32x4{x[e] * mul, x[e + 1] * mul, x[e + 2] * mul, x[e + 3] * mul};
  }
}

// Workgroup -> (head bh, block) with the longest blocks first: the forward and dQ
// blocks grow with their index, the dK/dV blocks shrink.
__device__ __forceinline__ void block_of(int bid, int n_bh, int n_blk, bool long_is_low,
                                         int &bh, int &blk) {
  const int rank = bid / n_bh;
  bh = bid - rank * n_bh;
  blk = long_is_low ? rank : n_blk - 1 - rank;
}

// LDS of a workgroup: TPW tiles per wave, wave w's at w * TPW tiles.  A wave's merge
// partials go into its own first tiles, after its last block, so no barrier separates
// the loop from the partial writes.
template <int D, int TPW>
__device__ __forceinline__ float *wave_tiles(float *lds, int wave) {
  return lds + wave * TPW * tile_floats<D>();
}

}  // namespace

template <int D, int NW>
__global__ __launch_bounds__(64 * NW) void fa_fwd_f32_kernel(const float *__restrict__ Q,
                                                             const float *__restrict__ K,
                                                             const float *__restrict__ V,
                                                             float *__restrict__ O,
                                                             float *__restrict__ LSE, int Hq,
                                                             int Hkv, int T, int n_bh,
                                                             float scale) {
  constexpr int TPW = 2;
  __shared__ __attribute__((aligned(16))) float lds[NW * TPW * tile_floats<D>()];
  __shared__ float pm[NW][kF32Rows], pl[NW][kF32Rows];
  const int n_blk = (T + kF32Rows - 1) / kF32Rows;
  int bh, qb;
  block_of(blockIdx.x, n_bh, n_blk, false, bh, qb);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane >> 4, n = lane & 15;
  const int G = Hq / Hkv;
  const int64_t kvh = (int64_t)(bh / Hq) * Hkv + (bh % Hq) / G;
  const float *Kh = K + kvh * T * D, *Vh = V + kvh * T * D;
  const int q0 = qb * kF32Rows, last = T - 1;
  float *tk = wave_tiles<D, TPW>(lds, wave), *tv = tk + tile_floats<D>();

  struct Blk {
    BlockRegs<D> k, v;
  };
  Blk nxt;
  int kb = wave;
  if (kb <= qb) {
    load_block<D>(nxt.k, Kh, kb * kF32Rows, last, lane);
    load_block<D>(nxt.v, Vh, kb * kF32Rows, last, lane);
  }
  float qf[D / 4];
  {
    BlockRegs<D> qr;
    load_block<D>(qr, Q + (int64_t)bh * T * D, q0, last, lane);
    store_block<D>(tk, qr, lane);
    read_rowfrag<D>(qf, tk, j, n);
  }

  float m = -INFINITY, lsum = 0.f;
  f32x4 acc[D / 16];
#pragma unroll
  for (int db = 0; db < D / 16; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (; kb <= qb; kb += NW) {
    store_block<D>(tk, nxt.k, lane);
    store_block<D>(tv, nxt.v, lane);
    if (kb + NW <= qb) {  // in flight during this block's products
      load_block<D>(nxt.k, Kh, (kb + NW) * kF32Rows, last, lane);
      load_block<D>(nxt.v, Vh, (kb + NW) * kF32Rows, last, lane);
    }
    float kf[D / 4];
    read_rowfrag<D>(kf, tk, j, n);
    // S^T block: register r = score of key 16 kb + 4 j + r for query q0 + n.
    const f32x4 st = dot_block<D>(kf, qf);
    f32x4 s;
    float bm = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = st[r] * scale;
      if (kb == qb && 4 * j + r > n) s[r] = -INFINITY;  // key after the query
      bm = fmaxf(bm, s[r]);
    }
    const float m_new = fmaxf(m, group_max(bm));  // finite: key 16 kb precedes every query
    const float alpha = expf(m - m_new);
    f32x4 p;
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = expf(s[r] - m_new);
    lsum = lsum * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
    m = m_new;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) acc[db] *= alpha;
    float vc[D / 4];
    read_colfrag<D>(vc, tv, j, n);
    accum_cols<D>(acc, vc, p);
  }
  lsum = group_sum(lsum);

  put_partial<D>(tk, acc, j, n);
  if (j == 0) {
    pm[wave][n] = m;
    pl[wave][n] = lsum;
  }
  __syncthreads();
  // Merge, waves in order.
  using M = Merge<D, NW>;
  const M mg;
  const int row = mg.row, q = q0 + row;
  if (q >= T) return;
  float mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < NW; ++w) mx = fmaxf(mx, pm[w][row]);
  float L = 0.f, out[M::CH];
#pragma unroll
  for (int e = 0; e < M::CH; ++e) out[e] = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float cw = pm[w][row] == -INFINITY ? 0.f : expf(pm[w][row] - mx);
    L += cw * pl[w][row];
    const float *src = wave_tiles<D, TPW>(lds, w) + row * (D + 4) + mg.c0;
#pragma unroll
    for (int e = 0; e < M::CH; ++e) out[e] += cw * src[e];
  }
  store_chunk<M::CH>(O + ((int64_t)bh * T + q) * D + mg.c0, out, 1.f / L);
  if (mg.c0 == 0) LSE[(int64_t)bh * T + q] = mx + logf(L);
}

// Arguments of the backward passes.
struct F32Bwd {
  const float *Q, *K, *V, *O, *dO, *LSE;
  float *Delta, *dQ, *dK, *dV;
  int Hq, Hkv, T;
  float scale;
};

// Delta and dQ of query block qb of head bh (LDS: NW * 2 tiles).
template <int D>
__device__ __forceinline__ void dq_block(float *lds, const F32Bwd &a, int bh, int qb) {
  constexpr int NW = f32_waves<D>(), TPW = 2;
  const int Hq = a.Hq, Hkv = a.Hkv, T = a.T;
  const float scale = a.scale;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane >> 4, n = lane & 15;
  const int G = Hq / Hkv;
  const int64_t kvh = (int64_t)(bh / Hq) * Hkv + (bh % Hq) / G;
  const float *Kh = a.K + kvh * T * D, *Vh = a.V + kvh * T * D;
  const int q0 = qb * kF32Rows, last = T - 1;
  float *tk = wave_tiles<D, TPW>(lds, wave), *tv = tk + tile_floats<D>();

  struct Blk {
    BlockRegs<D> k, v;
  };
  Blk nxt;
  int kb = wave;
  if (kb <= qb) {
    load_block<D>(nxt.k, Kh, kb * kF32Rows, last, lane);
    load_block<D>(nxt.v, Vh, kb * kF32Rows, last, lane);
  }
  const int64_t hb = (int64_t)bh * T;
  float qf[D / 4], dof[D / 4], delta;
  {
    BlockRegs<D> qr, dor, orr;
    load_block<D>(qr, a.Q + hb * D, q0, last, lane);
    load_block<D>(dor, a.dO + hb * D, q0, last, lane);
    load_block<D>(orr, a.O + hb * D, q0, last, lane);
    store_block<D>(tk, qr, lane);
    store_block<D>(tv, dor, lane);
    read_rowfrag<D>(qf, tk, j, n);
    read_rowfrag<D>(dof, tv, j, n);
    float of[D / 4];
    store_block<D>(tk, orr, lane);
    read_rowfrag<D>(of, tk, j, n);
    float d = 0.f;
#pragma unroll
    for (int i = 0; i < D / 4; ++i) d = __builtin_fmaf(of[i], dof[i], d);
    delta = group_sum(d);
  }
  const int64_t qrow = hb + min(q0 + n, last);
  const float lse = a.LSE[qrow];
  if (wave == 0 && j == 0 && q0 + n < T) a.Delta[qrow] = delta;

  f32x4 acc[D / 16];
#pragma unroll
  for (int db = 0; db < D / 16; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (; kb <= qb; kb += NW) {
    store_block<D>(tk, nxt.k, lane);
    store_block<D>(tv, nxt.v, lane);
    if (kb + NW <= qb) {  // in flight during this block's products
      load_block<D>(nxt.k, Kh, (kb + NW) * kF32Rows, last, lane);
      load_block<D>(nxt.v, Vh, (kb + NW) * kF32Rows, last, lane);
    }
    float kf[D / 4], vf[D / 4];
    read_rowfrag<D>(kf, tk, j, n);
    read_rowfrag<D>(vf, tv, j, n);
    const f32x4 st = dot_block<D>(kf, qf);   // S^T: key 16 kb + 4 j + r, query q0 + n
    const f32x4 dpt = dot_block<D>(vf, dof);  // dP^T, same layout
    f32x4 ds;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float p = (kb == qb && 4 * j + r > n) ? 0.f : expf(st[r] * scale - lse);
      ds[r] = p * (dpt[r] - delta);
    }
    float kc[D / 4];
    read_colfrag<D>(kc, tk, j, n);
    accum_cols<D>(acc, kc, ds);  // dQ^T += K^T dS^T
  }

  put_partial<D>(tk, acc, j, n);
  __syncthreads();
  using M = Merge<D, NW>;
  const M mg;
  const int q = q0 + mg.row;
  if (q >= T) return;
  float out[M::CH];
#pragma unroll
  for (int e = 0; e < M::CH; ++e) out[e] = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float *src = wave_tiles<D, TPW>(lds, w) + mg.row * (D + 4) + mg.c0;
#pragma unroll
    for (int e = 0; e < M::CH; ++e) out[e] += src[e];
  }
  store_chunk<M::CH>(a.dQ + (hb + q) * D + mg.c0, out, scale);
}

// dK and dV of key block kb of KV head bhk (LDS: NW * 2 tiles).  OWN_DELTA:
// form each query row's Delta from O and dO (the same sums, in the same order, as
// dq_block) instead of reading it, so this pass need not wait for the dQ pass.
// PART: only items [i0, i1), with the unscaled sums to part ([dK | dV] row-major tiles)
// unless it is null.
template <int D, bool OWN_DELTA, bool PART = false>
__device__ __forceinline__ void dkdv_block(float *lds, const F32Bwd &a, int bhk, int kb, int i0 = 0,
                                           int i1 = 0, float *part = nullptr) {
  constexpr int NW = f32_waves<D>(), TPW = 2;
  const int Hq = a.Hq, Hkv = a.Hkv, T = a.T;
  const float scale = a.scale;
  const int n_blk = (T + kF32Rows - 1) / kF32Rows;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane >> 4, n = lane & 15;
  const int G = Hq / Hkv;
  const int b = bhk / Hkv, hk = bhk - b * Hkv;
  const int k0 = kb * kF32Rows, last = T - 1;
  float *tq = wave_tiles<D, TPW>(lds, wave), *tdo = tq + tile_floats<D>();

  // Items: (query head g of the group, query block qb >= kb), g-major; wave w takes the
  // items w, w + NW, ...
  const int per_g = n_blk - kb, n_items = PART ? i1 : G * per_g;
  struct Item {
    BlockRegs<D> q, dout;
    BlockRegs<OWN_DELTA ? D : 16> o;
    float lse[4], delta[4];
  };
  auto load_item = [&](Item &it, int i) {
    const int g = i / per_g, qb = kb + (i - g * per_g);
    const int64_t qh = (int64_t)b * Hq + hk * G + g;
    const int q0 = qb * kF32Rows;
    load_block<D>(it.q, a.Q + qh * T * D, q0, last, lane);
    load_block<D>(it.dout, a.dO + qh * T * D, q0, last, lane);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t x = qh * T + min(q0 + 4 * j + r, last);
      it.lse[r] = a.LSE[x];
      if constexpr (!OWN_DELTA) it.delta[r] = a.Delta[x];
    }
  };
  auto load_o = [&](Item &it, int i) {
    const int g = i / per_g, qb = kb + (i - g * per_g);
    const int64_t qh = (int64_t)b * Hq + hk * G + g;
    if constexpr (OWN_DELTA) load_block<D>(it.o, a.O + qh * T * D, qb * kF32Rows, last, lane);
  };
  Item nxt;
  int i = (PART ? i0 : 0) + wave;
  if (i < n_items) {
    load_item(nxt, i);
    load_o(nxt, i);
  }

  // K^T, V^T as B operands: row fragments of key k0 + n.
  float kf[D / 4], vf[D / 4];
  {
    BlockRegs<D> kr, vr;
    const int64_t hb = (int64_t)bhk * T * D;
    load_block<D>(kr, a.K + hb, k0, last, lane);
    load_block<D>(vr, a.V + hb, k0, last, lane);
    store_block<D>(tq, kr, lane);
    store_block<D>(tdo, vr, lane);
    read_rowfrag<D>(kf, tq, j, n);
    read_rowfrag<D>(vf, tdo, j, n);
  }

  f32x4 dk[D / 16], dv[D / 16];
#pragma unroll
  for (int db = 0; db < D / 16; ++db) dk[db] = dv[db] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (; i < n_items; i += NW) {
    const int g = i / per_g, qb = kb + (i - g * per_g), q0 = qb * kF32Rows;
    float delta[4], lse[4];
    store_block<D>(tdo, nxt.dout, lane);
    float qa[D / 4], doa[D / 4], oa[OWN_DELTA ? D / 4 : 1];
    read_rowfrag<D>(doa, tdo, j, n);
    if constexpr (OWN_DELTA) {
      // O passes through the Q tile, as in dq_block: a third tile per wave and O held with
      // the other prefetches cost 69.1 us against 66.9 at 2x8/2x500 D = 128, 81.3 against 78.9
      // at 2x12/4x700 D = 64.
      store_block<D>(tq, nxt.o, lane);
      read_rowfrag<D>(oa, tq, j, n);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) lse[r] = nxt.lse[r];
    if constexpr (!OWN_DELTA) {
#pragma unroll
      for (int r = 0; r < 4; ++r) delta[r] = nxt.delta[r];
    }
    store_block<D>(tq, nxt.q, lane);
    if (i + NW < n_items) load_item(nxt, i + NW);  // in flight during this item's products
    read_rowfrag<D>(qa, tq, j, n);
    // S and dP: register r = query q0 + 4 j + r, key k0 + n.
    const f32x4 s = dot_block<D>(qa, kf);
    const f32x4 dp = dot_block<D>(doa, vf);
    if constexpr (OWN_DELTA) {
      // Delta of row q0 + n in every lane of column n, then row q0 + 4 j + r from lane 4 j + r.
      // Formed here, beside the products, not before them, where it lengthened every item's
      // chain: 1x8/2x100 D = 64 14.30 -> 13.85 us, 2x2/2x437 14.96 -> 14.35, 2x12/4x700 79.5 -> 78.5.
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < D / 4; ++e) d = __builtin_fmaf(oa[e], doa[e], d);
      d = group_sum(d);
#pragma unroll
      for (int r = 0; r < 4; ++r) delta[r] = __shfl(d, 4 * j + r);
    }
    f32x4 p, ds;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int q = q0 + 4 * j + r;
      const bool keep = q < T && (qb != kb || n <= 4 * j + r);
      p[r] = keep ? expf(s[r] * scale - lse[r]) : 0.f;
      ds[r] = p[r] * (dp[r] - delta[r]);
    }
    // O of the next item only now: its registers were the fragments' until here.
    if (i + NW < n_items) load_o(nxt, i + NW);
    float col[D / 4];
    read_colfrag<D>(col, tdo, j, n);
    accum_cols<D>(dv, col, p);   // dV^T += dO^T P
    read_colfrag<D>(col, tq, j, n);
    accum_cols<D>(dk, col, ds);  // dK^T += Q^T dS
  }

  put_partial<D>(tq, dk, j, n);
  put_partial<D>(tdo, dv, j, n);
  __syncthreads();
  using M = Merge<D, NW>;
  const M mg;
  const int key = k0 + mg.row;
  if (key >= T) return;
  float ok[M::CH], ov[M::CH];
#pragma unroll
  for (int e = 0; e < M::CH; ++e) ok[e] = ov[e] = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float *src = wave_tiles<D, TPW>(lds, w) + mg.row * (D + 4) + mg.c0;
#pragma unroll
    for (int e = 0; e < M::CH; ++e) {
      ok[e] += src[e];
      ov[e] += src[tile_floats<D>() + e];
    }
  }
  if (PART && part) {
    float *dst = part + mg.row * D + mg.c0;
    store_chunk<M::CH>(dst, ok, 1.f);
    store_chunk<M::CH>(dst + kF32Rows * D, ov, 1.f);
    return;
  }
  const int64_t o = ((int64_t)bhk * T + key) * D + mg.c0;
  store_chunk<M::CH>(a.dK + o, ok, scale);
  store_chunk<M::CH>(a.dV + o, ov, 1.f);
}

template <int D>
__global__ __launch_bounds__(64 * f32_waves<D>()) void fa_bwd_dq_f32_kernel(F32Bwd a,
                                                                             int n_bh) {
  __shared__ __attribute__((aligned(16))) float lds[f32_waves<D>() * 2 * tile_floats<D>()];
  int bh, qb;
  block_of(blockIdx.x, n_bh, (a.T + kF32Rows - 1) / kF32Rows, false, bh, qb);
  dq_block<D>(lds, a, bh, qb);
}

template <int D>
__global__ __launch_bounds__(64 * f32_waves<D>()) void fa_bwd_dkdv_f32_kernel(F32Bwd a,
                                                                               int n_bhk) {
  __shared__ __attribute__((aligned(16))) float lds[f32_waves<D>() * 2 * tile_floats<D>()];
  int bhk, kb;
  block_of(blockIdx.x, n_bhk, (a.T + kF32Rows - 1) / kF32Rows, true, bhk, kb);
  dkdv_block<D, false>(lds, a, bhk, kb);
}

// Floats of one piece's partial: a 16-key tile of dK, then one of dV.
template <int D>
constexpr int kF32PartFloats = 2 * kF32Rows * D;

// Both backward passes in one launch: the dK/dV workgroups form Delta themselves, so they
// run beside the dQ workgroups instead of after them.  All dK/dV workgroups come first, the
// longest key blocks leading, then the dQ blocks, longest first.  (Interleaved rank by rank,
// the period of the workgroup ids put all dK/dV work of an XCD on the same few CUs: 161 us
// against 82 at 2x12/4x700, D = 64, and 118 against 91 at 4x12/4x500.)
//
// The items of a key block may be dealt to several pieces (dkdv_split_f32): a key block with
// one piece (all of them where items is the longest list) writes dK and dV; the others write
// partial sums, which fa_bwd_f32_reduce_kernel adds in piece order.
template <int D>
__global__ __launch_bounds__(64 * f32_waves<D>()) void fa_bwd_f32_kernel(
    F32Bwd a, float *__restrict__ part, int n_bh, int n_bhk, int n_pieces, int items) {
  __shared__ __attribute__((aligned(16))) float lds[f32_waves<D>() * 2 * tile_floats<D>()];
  const int n_blk = (a.T + kF32Rows - 1) / kF32Rows;
  const int bid = blockIdx.x, n_dkdv = n_pieces * n_bhk;
  if (bid < n_dkdv) {
    const int piece = bid / n_bhk, unit = bid - piece * n_bhk;
    const DkvPiece pc = dkv_piece(piece, n_blk, a.Hq / a.Hkv, items);
    dkdv_block<D, true, true>(lds, a, unit, pc.kt, pc.it0, pc.it1,
                              pc.n == 1 ? nullptr : part + (int64_t)bid * kF32PartFloats<D>);
  } else {
    const int rank = (bid - n_dkdv) / n_bh, bh = bid - n_dkdv - rank * n_bh;
    dq_block<D>(lds, a, bh, n_blk - 1 - rank);
  }
}

// dK and dV of the key blocks with several pieces: one workgroup per (key block, unit), a
// float4 per thread and step, the pieces added in order.
template <int D>
__global__ __launch_bounds__(256) void fa_bwd_f32_reduce_kernel(const float *__restrict__ part,
                                                                float *__restrict__ dK,
                                                                float *__restrict__ dV,
                                                                int n_bhk, int G, int T,
                                                                int items, float scale) {
  const int n_blk = (T + kF32Rows - 1) / kF32Rows;
  const int kb = blockIdx.x / n_bhk, unit = blockIdx.x - kb * n_bhk;
  const DkvSlot slot = dkv_slot(kb, n_blk, G, items);
  const int64_t stride = (int64_t)n_bhk * kF32PartFloats<D>;
  const float *src = part + ((int64_t)slot.first * n_bhk + unit) * kF32PartFloats<D>;
#pragma unroll
  for (int e = threadIdx.x * 4; e < kF32PartFloats<D>; e += 1024) {
    f32x4 x = *reinterpret_cast<const f32x4 *>(src + e);
#pragma unroll 4
    for (int p = 1; p < slot.n; ++p) x += *reinterpret_cast<const f32x4 *>(src + p * stride + e);
    const bool is_v = e >= kF32Rows * D;
    const int r = is_v ? e - kF32Rows * D : e, key = kb * kF32Rows + r / D;
    if (key < T)
      *reinterpret_cast<f32x4 *>((is_v ? dV : dK) + ((int64_t)unit * T + key) * D + r % D) =
          is_v ? x : x * scale;
  }
}

static unsigned blocks_grid(int n_bh, int T) {
  return (unsigned)((int64_t)n_bh * ((T + kF32Rows - 1) / kF32Rows));
}

static dim3 f32_block(int D) { return dim3(64 * (D == 64 ? f32_waves<64>() : f32_waves<128>())); }

static F32Bwd bwd_args(const void *q, const void *k, const void *v, const void *o,
                       const void *dout, const float *lse, float *delta, void *dq, void *dk,
                       void *dv, int Hq, int Hkv, int T, float scale) {
  return F32Bwd{(const float *)q, (const float *)k, (const float *)v, (const float *)o,
                (const float *)dout, lse, delta, (float *)dq, (float *)dk, (float *)dv,
                Hq, Hkv, T, scale};
}

// D = 128 forward: eight waves per workgroup, one workgroup per CU (135 KB of LDS), or four and
// two.  Eight halve a row block's serial chain of key blocks, so they win while the launch is
// about one round of the 256 CUs, or long rows make the chain what counts; beyond that they
// halve the row blocks in flight, and rows of up to four key blocks leave half of them idle.
// Measured, us, eight against four waves (n row blocks, T):
//   T 100: n 252 7.3 / 7.6, 280 9.8 / 8.1      T 64: n 256 6.0 / 5.6, 512 10.4 / 7.5
//   T 200: n 260 10.0 / 11.2, 312 11.4 / 11.2, 468 14.2 / 12.6
//   T 280: n 504 16.2 / 16.8, 576 20.2 / 16.9  T 500: n 512 20.9 / 24.0, 576 26.4 / 24.6
//   T 1000: n 504 32.9 / 42.7, 1134 72.4 / 68.4
//   T 2000: n 500 56.9 / 78.5, 1000 107.9 / 114.3, 1500 159 / 155
// and up to twice as far apart as n grows (T 64, n 3000: 64.3 / 37.2; T 128, n 4096: 45.7 / 30.7).
static bool f32_fwd_eight_waves(int64_t n, int T) {
  return T > 64 && n <= (T <= 128 ? 256 : T <= 256 ? 304 : T <= 1024 ? 512 : 1024);
}

hipError_t launch_fwd_f32(const void *q, const void *k, const void *v, void *o, float *lse,
                          int B, int Hq, int Hkv, int T, int D, float scale, hipStream_t stream) {
  auto go = [&](auto kern, int waves) {
    kern<<<dim3(blocks_grid(B * Hq, T)), dim3(64 * waves), 0, stream>>>(
        (const float *)q, (const float *)k, (const float *)v, (float *)o, lse, Hq, Hkv, T, B * Hq,
        scale);
    return hipGetLastError();
  };
  if (D == 64) return go(fa_fwd_f32_kernel<64, 8>, 8);
  return f32_fwd_eight_waves(blocks_grid(B * Hq, T), T) ? go(fa_fwd_f32_kernel<128, 8>, 8)
                                                        : go(fa_fwd_f32_kernel<128, 4>, 4);
}

hipError_t launch_bwd_dq_f32(const void *q, const void *k, const void *v, const void *o,
                             const void *dout, const float *lse, float *delta, void *dq,
                             int B, int Hq, int Hkv, int T, int D, float scale,
                             hipStream_t stream) {
  const F32Bwd a = bwd_args(q, k, v, o, dout, lse, delta, dq, nullptr, nullptr, Hq, Hkv, T, scale);
  const dim3 grid(blocks_grid(B * Hq, T)), block = f32_block(D);
  if (D == 64)
    fa_bwd_dq_f32_kernel<64><<<grid, block, 0, stream>>>(a, B * Hq);
  else
    fa_bwd_dq_f32_kernel<128><<<grid, block, 0, stream>>>(a, B * Hq);
  return hipGetLastError();
}

hipError_t launch_bwd_dkdv_f32(const void *q, const void *k, const void *v, const void *dout,
                               const float *lse, const float *delta, void *dk, void *dv,
                               int B, int Hq, int Hkv, int T, int D, float scale,
                               hipStream_t stream) {
  const F32Bwd a = bwd_args(q, k, v, nullptr, dout, lse, const_cast<float *>(delta), nullptr,
                            dk, dv, Hq, Hkv, T, scale);
  const dim3 grid(blocks_grid(B * Hkv, T)), block = f32_block(D);
  if (D == 64)
    fa_bwd_dkdv_f32_kernel<64><<<grid, block, 0, stream>>>(a, B * Hkv);
  else
    fa_bwd_dkdv_f32_kernel<128><<<grid, block, 0, stream>>>(a, B * Hkv);
  return hipGetLastError();
}

// Items per piece of a key block's list, or no split.  A key block of a KV head with many
// query heads carries G * n_blk items (about 1.9 us per round of its waves), far more than
// an even share of the launch for each of the 256 resident workgroups; pieces of one such
// share bring the longest list down to it.  Measured, whole backward, one piece per key
// block -> split: 2x8/2x500 D 128 109 -> 67 us, 1x8/2x1000 D 128 208 -> 114, 1x6/2x500 D 128
// 83 -> 37, 4x6/2x130 D 128 28 -> 21, 1x8/2x1000 D 64 101 -> 60; half a share per piece was
// slower (73, 117, 45, 21.5, 63).  It has to save four rounds of the waves, or the reducing
// launch costs more (1x8/8x333 D 128, 3.25 rounds: 24.7 -> 27.6).
DkdvSplit dkdv_split_f32(int B, int Hq, int Hkv, int T, int D) {
  const DkdvSplit none{0, 0, 0};
  const int n = (T + kF32Rows - 1) / kF32Rows, G = Hq / Hkv;
  const int waves = D == 64 ? f32_waves<64>() : f32_waves<128>();
  const int64_t units = (int64_t)B * Hkv, longest = (int64_t)G * n;
  if (longest > (1 << 24) || units * longest > (1 << 28)) return none;
  // all the work of the launch in dK/dV items: a dQ block pair is 3/4 of one
  const int64_t total = units * G * ((int64_t)n * (n + 1) / 2) * 7 / 4;
  int64_t items = (total / 256 + waves - 1) / waves * waves;
  if (items < 2 * waves) items = 2 * waves;
  if (longest - items < 4 * waves) return none;
  DkdvSplit s{(int)items, 0, 0};
  for (DkvTiles t(n, G, s.stages); t.kt < n; t.next()) {
    s.pieces += t.n;
    s.split_tiles += t.n > 1;
  }
  return s;
}

int64_t dkdv_part_floats_f32(const DkdvSplit &s, int B, int Hkv, int D) {
  return (int64_t)s.pieces * B * Hkv * (D == 64 ? kF32PartFloats<64> : kF32PartFloats<128>);
}

template <int D>
static hipError_t launch_bwd_f32_kernels(const F32Bwd &a, float *part, DkdvSplit s, int B,
                                         hipStream_t stream) {
  const int n_bh = B * a.Hq, n_bhk = B * a.Hkv, G = a.Hq / a.Hkv;
  if (s.stages == 0) {  // one piece per key block
    s.pieces = (a.T + kF32Rows - 1) / kF32Rows;
    s.stages = G * s.pieces;
  }
  const unsigned grid = (unsigned)(s.pieces * n_bhk) + blocks_grid(n_bh, a.T);
  fa_bwd_f32_kernel<D><<<dim3(grid), f32_block(D), 0, stream>>>(a, part, n_bh, n_bhk, s.pieces,
                                                                s.stages);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || s.split_tiles == 0) return e;
  fa_bwd_f32_reduce_kernel<D><<<dim3((unsigned)(s.split_tiles * n_bhk)), dim3(256), 0, stream>>>(
      part, a.dK, a.dV, n_bhk, G, a.T, s.stages, a.scale);
  return hipGetLastError();
}

hipError_t launch_bwd_f32(const void *q, const void *k, const void *v, const void *o,
                          const void *dout, const float *lse, float *delta, void *dq, void *dk,
                          void *dv, float *part, const DkdvSplit &s, int B, int Hq, int Hkv, int T,
                          int D, float scale, hipStream_t stream) {
  const F32Bwd a = bwd_args(q, k, v, o, dout, lse, delta, dq, dk, dv, Hq, Hkv, T, scale);
  return D == 64 ? launch_bwd_f32_kernels<64>(a, part, s, B, stream)
                 : launch_bwd_f32_kernels<128>(a, part, s, B, stream);
}

}  // namespace ttfa
