// sg_kv_prep.h -- device bodies shared by the QK-norm/RoPE split kernel,
// the V^T split kernel and the kernel that does both in one launch.
#pragma once
#include "sg_device.h"
#include "sg_kernels.h"

namespace sgd {

constexpr int kKvThreads = 256;  // threads per workgroup of every kernel using these bodies
constexpr int kKvRows = 32;      // (token, head) rows per workgroup of the QK split: 8 lanes each
constexpr int kVtRowStride = 256 + 4;  // fp32 LDS row stride of the V tile

// Attention operands in MFMA fragment order.  K and V are held per kv head and
// 32-key tile (a sequence's tiles are consecutive, its last one padded) as
// 32 KB of 1-KB pieces, each the 64 lanes' 16-byte fragments of one MFMA
// operand half in lane order, so a fragment load -- from global memory or from
// a linear LDS copy -- is 1 KB of contiguous memory for the wave.  (Row-major K
// and dim-major V^T made a fragment load touch 16 rows a power of two apart,
// i.e. a few of the L2's channels.)  Lane = 16 g + ln:
//   K piece (16-key subtile st, k-step ks, hi / lo): key 16 st + ln, dims
//     32 ks + 8 g .. + 7, of 8 * x (kAttnQKScale), split hi / lo;
//   V piece (16-dim group mt, hi / lo): dim 16 mt + ln, keys vt_key(8 g) .. of
//     the tile, zero past the sequence's end (K's pad keys' scores
//     are masked);
//   Q (pre-split for small launches): like K, one set of tiles per query head,
//     a 16-row chunk of a sequence being one subtile.
constexpr int kFragTile = 16384;  // halves per tile: 32 keys x 256 dims, hi and lo
__host__ __device__ constexpr int kfrag_piece(int st, int ks, int lo) { return ((st * 8 + ks) * 2 + lo) * 512; }
__host__ __device__ constexpr int vfrag_piece(int mt, int lo) { return (mt * 2 + lo) * 512; }

// Key order inside a V piece.  Lane group g of an attention wave holds the
// S^T entries of keys 4g..4g+3 (first 16-key subtile) and 16+4g..16+4g+3
// (second); as the B operand of a 32-key MFMA step its slots are positions
// 8g..8g+7, so position p holds key:
__device__ __forceinline__ int vt_key(int p) { return ((p & 4) << 2) | ((p & 24) >> 1) | (p & 3); }

// hi/lo of x * kAttnQKScale for dims 4 d4 .. + 3 of one key (index row_key in
// the padded key numbering) into K's (or Q's) fragments.  kf: this head's tiles.
__device__ __forceinline__ void store_kfrag4(_Float16* __restrict__ kf, int row_key, int d4, const f32x4_t& x) {
  half4_t hv, lv;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const hl16 sp = split_f16(x[u] * sgk::kAttnQKScale);
    hv[u] = sp.hi;
    lv[u] = sp.lo;
  }
  const int key = row_key & 31, ks = d4 >> 3, g = (d4 & 7) >> 1;
  _Float16* p = kf + (int64_t)(row_key >> 5) * kFragTile + kfrag_piece(key >> 4, ks, 0) + (16 * g + (key & 15)) * 8 +
                4 * (d4 & 1);
  *reinterpret_cast<half4_t*>(p) = hv;
  *reinterpret_cast<half4_t*>(p + 512) = lv;
}

// One 8-lane group per (token, head): g = token * (H + HKV) + head (query
// heads first).  RMSNorm with attn_q_norm/attn_k_norm (model_int8.go:374-440),
// then the cached NeoX rotation of pairs (i, i+128) at the token's position
// (rope_cache.go:85-104): x0' = x0*c - x1*s, x1' = x0*s + x1*c, every product
// rounded; then hi/lo fp16 of x * kAttnQKScale in fragment order at the row's
// place (row_key).  Lane j holds float4 slots
// 4j.. of every 32-element chunk, so element e and its partner e + 128 sit in
// the same lane and slot.  tile: this wave's 8 x 40-float LDS tile.
__device__ __forceinline__ void qk_split_group(int64_t g, int j, int r, float* tile, const float* __restrict__ q,
                                               int ldq, const float* __restrict__ k, int ldk,
                                               const float* __restrict__ qw, const float* __restrict__ kw, int H,
                                               int HKV, int T, const int32_t* __restrict__ row_pos,
                                               const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                               float eps, _Float16* __restrict__ qf,
                                               const int32_t* __restrict__ row_key, _Float16* __restrict__ kf,
                                               int n_tiles) {
  constexpr int NC = 8, HALF = 128;
  const int per = H + HKV;
  if (g >= (int64_t)T * per) return;  // whole 8-lane groups
  const int t = (int)(g / per), hh = (int)(g % per);
  const float* src = hh < H ? q + (int64_t)t * ldq + hh * 256 : k + (int64_t)t * ldk + (hh - H) * 256;
  // The row's place with its values: one round trip.
  const int pos = row_pos[t], rk = row_key[t];
  f32x4_t x[NC];
  // The fp32 Q/K row's last read: non-temporal, leaving L2 to re-read operands.
#pragma unroll
  for (int c = 0; c < NC; c++)
    x[c] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(src + 32 * c + 4 * j));
  const float* wn = hh < H ? qw : kw;
  if (wn) sg_rmsnorm8_f4<NC>(x, wn, tile, r, j, eps);
  const float* cr = cos_t + (int64_t)pos * HALF + 4 * j;
  const float* sr = sin_t + (int64_t)pos * HALF + 4 * j;
#pragma unroll
  for (int c = 0; c < NC / 2; c++) {
    const f32x4_t cv = *reinterpret_cast<const f32x4_t*>(cr + 32 * c);
    const f32x4_t sv = *reinterpret_cast<const f32x4_t*>(sr + 32 * c);
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const float v0 = x[c][u], v1 = x[c + NC / 2][u];
      const float a = v0 * cv[u], b = v1 * sv[u], cc = v0 * sv[u], dd = v1 * cv[u];
      x[c][u] = a - b;
      x[c + NC / 2][u] = cc + dd;
    }
  }
  _Float16* dst = (hh < H ? qf + (int64_t)hh * n_tiles * kFragTile : kf + (int64_t)(hh - H) * n_tiles * kFragTile);
#pragma unroll
  for (int c = 0; c < NC; c++) store_kfrag4(dst, rk, 8 * c + j, x[c]);
}

// One 32-key tile of V [T][ldv] fp32 (kv head kvh at column 256*kvh) -> V's
// fragments vf [HKV][n_tiles] tiles (sequence s from tile voff[s] / 32 on),
// zeros past S.  The 32 x 256 fp32 tile is loaded with coalesced float4 rows
// into LDS (tv: [32][kVtRowStride]); a thread then owns one fragment (dim,
// 8-key chunk), reads its 8 keys down the LDS column and stores the hi and lo
// halves as 16-byte writes, 1 KB contiguous per wave.  Every thread of the
// workgroup must call this (it holds a barrier).
__device__ __forceinline__ void v_split_tile(sg_item t, int kvh, float (*tv)[kVtRowStride], const float* __restrict__ v,
                                             int ldv, const int32_t* __restrict__ seq_off,
                                             const int32_t* __restrict__ voff, _Float16* __restrict__ vf,
                                             int n_tiles) {
  constexpr int kHD = 256;
  const int r0 = seq_off[t.seq], S = seq_off[t.seq + 1] - r0, k0 = t.c0;
  const int tid = threadIdx.x;
#pragma unroll
  for (int u = 0; u < 8; u++) {  // 32 keys x 64 float4
    const int idx = tid + kKvThreads * u;
    const int key = idx >> 6, d4 = idx & 63;
    f32x4_t x = {0, 0, 0, 0};
    if (k0 + key < S)  // the fp32 V row's last read: non-temporal
      x = __builtin_nontemporal_load(
          reinterpret_cast<const f32x4_t*>(v + (int64_t)(r0 + k0 + key) * ldv + kvh * kHD + 4 * d4));
    *reinterpret_cast<f32x4_t*>(&tv[key][4 * d4]) = x;
  }
  __syncthreads();
  _Float16* vd = vf + ((int64_t)kvh * n_tiles + (voff[t.seq] + k0) / 32) * kFragTile;
  const int ln = tid & 15, c = (tid >> 4) & 3;
#pragma unroll
  for (int u = 0; u < 4; u++) {  // 16 dim groups x 4 chunks of 8 key positions x 16 dims
    const int mt = (tid >> 6) + 4 * u, dim = 16 * mt + ln;
    uint32_t hw[4], lw[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
      uint32_t hb[2], lb[2];
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int p = 8 * c + 2 * m + e;  // position in the tile row
        const int key = vt_key(p);
        const hl16 sp = split_f16(tv[key][dim]);
        hb[e] = __builtin_bit_cast(uint16_t, sp.hi);
        lb[e] = __builtin_bit_cast(uint16_t, sp.lo);
      }
      hw[m] = hb[0] | (hb[1] << 16);
      lw[m] = lb[0] | (lb[1] << 16);
    }
    _Float16* o = vd + vfrag_piece(mt, 0) + (16 * c + ln) * 8;
    *reinterpret_cast<uint4*>(o) = uint4{hw[0], hw[1], hw[2], hw[3]};
    *reinterpret_cast<uint4*>(o + 512) = uint4{lw[0], lw[1], lw[2], lw[3]};
  }
}

}  // namespace sgd
