// k_attention.hip -- bidirectional MQA attention over packed variable-length
// sequences (MultiHeadAttentionChunked with mask=nil,
// internal/kernels/attention.go:88-363; GQA expansion model_int8.go:455-479).
//
// Reference semantics kept:
//   s_ij = (q_i . k_j) * scale                         (scale = 1/sqrt(head_dim))
//   m_i  = max_j s_ij                                  (before any exp)
//   e_ij = fastExp(s_ij - m_i)  -- 0 when s_ij - m_i < -10 (activation.go:104-106)
//   o_i  = sum_j e_ij v_j / sum_j e_ij
// fastExp is not multiplicative and clamps, so an online (running-max)
// softmax would change the weights; the kernel makes two passes over the
// keys: pass 1 finds the row max, pass 2 forms e, the row sum and P.V.
//
// Precision.  The attention output is re-quantized to int8 with a
// per-sequence scale right after this kernel, so an error of 2^-12 (plain
// fp16 operands) flips a few percent of the int8 codes by a whole quantum and
// the flips compound over 24 layers.  Both products therefore run as split
// fp16 on the matrix cores: x = hi + lo with hi = fp16(x), lo = fp16(x - hi),
// and a.b = ah.bh + ah.bl + al.bh accumulated in fp32 (about 2^-22 relative,
// the level of the reference's own fp32 rounding).  Q and K are scaled by 8
// before splitting (exact) to keep lo out of the fp16 subnormal range; the
// weights e are scaled by 2^10 for the same reason; both scalings are undone
// exactly.  Pass 1 computes the same split scores, so the max is the max of
// the scores pass 2 exponentiates (a max that is off by even 1e-4 moves every
// fastExp argument and, through fastExp's polynomial error, the weights by
// ~1e-5).
//
// Operands arrive already split, K and V in MFMA fragment order (sg_kv_prep.h),
// so every workgroup only copies fp16 tiles.
//
// Work split.  The G query heads that share a kv head are stacked into
// G*ceil(S/16) chunks of 16 (head, query) rows.  A workgroup is 8 waves, one
// chunk each, two waves per SIMD (so one wave's softmax VALU overlaps the
// other's MFMAs); all eight stream the same 32-key K and V^T tiles through
// LDS.  A wave holds its chunk's Q^T (split, 64 VGPRs) and its O^T
// accumulators (256 dims x 16 queries, 64 VGPRs) for the whole run.  Scores
// are computed transposed, S^T = K Q^T on v_mfma_f32_16x16x32_f16: a lane owns
// one query and 8 keys of the tile, so row max and row sum are lane-local
// plus two exchanges, and those 8 registers are exactly the B operand of
// O^T += V^T P^T (one 32-key MFMA step) once V^T's keys are stored in the
// matching order (sgd::vt_key; the V^T split writes that order).
#include "sg_device.h"
#include "sg_kernels.h"
#include "sg_kv_prep.h"

namespace {

constexpr int kHD = 256;            // head_dim
constexpr int kBK = 32;             // keys per tile
constexpr int kQW = 16;             // (head, query) rows per wave
constexpr int kWaves = sgk::kAttnChunks;
constexpr int kNT = kWaves * SG_WAVE;
constexpr float kQKScale = sgk::kAttnQKScale;
constexpr float kPScale = 1024.0f, kPUnscale = 1.0f / 1024.0f;

// split_f16(x * scale) of two values x0, x1, packed, for a power-of-two
// scale: hi = {fp16(p0), fp16(p1)}, lo = {fp16(p0 - hi.x), fp16(p1 - hi.y)}
// with p = x * scale.  p is exact and so is p - fp16(p) (fp16(p) is p rounded
// to 11 significant bits), so each half is one v_fma_mix{lo,hi}_f16 of x
// rounded once to fp16: the bits of rounding p and p - hi, in four
// instructions, the lo pair reading hi's halves through op_sel (the compiler
// forms p, packs hi and recomputes it instead).
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void split_pair(float x0, float x1, float scale, uint32_t& hi, uint32_t& lo) {
  asm("v_fma_mixlo_f16 %0, %2, %4, 0\n\t"
      "v_fma_mixhi_f16 %0, %3, %4, 0\n\t"
      "v_fma_mixlo_f16 %1, %2, %4, -%0 op_sel_hi:[0,0,1]\n\t"
      "v_fma_mixhi_f16 %1, %3, %4, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
      : "=&v"(hi), "=&v"(lo)
      : "v"(x0), "v"(x1), "s"(scale));
}

template <int I>
struct int_c {
  static constexpr int value = I;
};
static_assert(sgk::kAttnChunkRows == kQW, "host chunking must match the kernel");

__device__ __forceinline__ f32x4_t mfma16(half8_t a, half8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// V^T tiles hold their keys in sgd::vt_key order (sg_kv_prep.h), which makes
// the eight S^T registers a lane holds per 32-key tile the B operand of one
// O^T += V^T P^T step.

constexpr int kRegTiles = sgk::kAttnRegKeys / kBK;

// Offset of the Q fragments of rows q0 .. q0 + 15 of the sequence at padded key vo.
__device__ __forceinline__ int64_t q_subtile(int head, int n_tiles, int vo, int q0) {
  return ((int64_t)head * n_tiles + ((vo + q0) >> 5)) * sgd::kFragTile + sgd::kfrag_piece((q0 >> 4) & 1, 0, 0);
}

// Q^T as the B operand of one wave's 16 (head, query) rows: lane (query ln,
// group g4), k-step ks holds dims 32ks + 8g4 .. + 7 of row qr, scaled by 8
// and split hi/lo.  QPRE: Q arrives as the QKV GEMM's fp32 output and the wave
// applies attn_q_norm and RoPE to its 16 rows itself (the arithmetic of
// sgd::qk_split_group, so the operands are bit-identical), which saves writing
// Q's hi/lo operands and reading them back; tile: the wave's 16 x 40 floats
// of LDS for the norm, wtile its 256 floats for the norm weights.  Otherwise
// Q arrives split, qf the chunk's subtile of fragments.
template <bool QPRE>
__device__ __forceinline__ void q_operand(half8_t (&bqh)[kHD / 32], half8_t (&bql)[kHD / 32],
                                          const _Float16* __restrict__ qf, const sg_attn_qpre& qp, int qr, int pos,
                                          int head, int ln, int g4,
                                          int lane, float* tile, float* wtile) {
  if constexpr (QPRE) {
    // Every global load (the norm weights, Q, the RoPE table rows of the
    // row's position pos) is issued up front, so the prologue pays one memory
    // latency instead of one per phase; the registers are free this early.
    // Lane (ln, g4) holds elements e = 32ks + 8g4 + t of row ln.  The norm
    // weights, the same for every row, are one 16-byte load per lane (the
    // whole vector per wave) into wtile, read back as LDS broadcasts: loaded
    // per lane they took 16 of the wave's 48 load instructions, and the
    // prologue's time is its load instructions' (each wave's waits for the
    // other wave of its SIMD).
    float x[kHD / 32][8];
    const f32x4_t wl = qp.w ? reinterpret_cast<const f32x4_t*>(qp.w)[lane] : f32x4_t{0, 0, 0, 0};
    const float* src = qp.q + (int64_t)qr * qp.ldq + head * kHD + 8 * g4;
#pragma unroll
    for (int ks = 0; ks < kHD / 32; ks++) {
      // The fp32 Q row's last read: non-temporal, leaving L2 to the K/V tiles.
      const f32x4_t* s4 = reinterpret_cast<const f32x4_t*>(src + 32 * ks);
      *reinterpret_cast<f32x4_t*>(&x[ks][0]) = __builtin_nontemporal_load(s4);
      *reinterpret_cast<f32x4_t*>(&x[ks][4]) = __builtin_nontemporal_load(s4 + 1);
    }
    float cv[kHD / 64][8], sv[kHD / 64][8];
    const float* cr = qp.cos_t + (int64_t)pos * (kHD / 2) + 8 * g4;
    const float* sr = qp.sin_t + (int64_t)pos * (kHD / 2) + 8 * g4;
#pragma unroll
    for (int ks = 0; ks < kHD / 64; ks++) {
      *reinterpret_cast<f32x4_t*>(&cv[ks][0]) = *reinterpret_cast<const f32x4_t*>(cr + 32 * ks);
      *reinterpret_cast<f32x4_t*>(&cv[ks][4]) = *reinterpret_cast<const f32x4_t*>(cr + 32 * ks + 4);
      *reinterpret_cast<f32x4_t*>(&sv[ks][0]) = *reinterpret_cast<const f32x4_t*>(sr + 32 * ks);
      *reinterpret_cast<f32x4_t*>(&sv[ks][4]) = *reinterpret_cast<const f32x4_t*>(sr + 32 * ks + 4);
    }
    static_assert(kHD == 4 * SG_WAVE, "one float4 of the norm weights per lane");
    if (qp.w) reinterpret_cast<f32x4_t*>(wtile)[lane] = wl;
    if (qp.w) {
      // RMSNorm's sum of squares in the AVX2 lane order (sg_rmsnorm8): lane v
      // of a row chains element 8i + v over i.  Element e sits at i = 4ks + g4,
      // v = t here, so each 32-element chunk goes through the wave's 16 x
      // 40-float LDS tile; lane (row rA or rA + 8, v) then reads the chunk's
      // elements 8k + v, k = 0..3, in order.
      const int v = lane & 7, rA = lane >> 3;
      float accA = 0.0f, accB = 0.0f;
#pragma unroll
      for (int ks = 0; ks < kHD / 32; ks++) {
        asm volatile("" ::: "memory");
        *reinterpret_cast<f32x4_t*>(tile + ln * 40 + 8 * g4) = f32x4_t{x[ks][0], x[ks][1], x[ks][2], x[ks][3]};
        *reinterpret_cast<f32x4_t*>(tile + ln * 40 + 8 * g4 + 4) = f32x4_t{x[ks][4], x[ks][5], x[ks][6], x[ks][7]};
        asm volatile("" ::: "memory");
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const float a = tile[rA * 40 + 8 * k + v];
          accA = __builtin_fmaf(a, a, accA);
          const float b = tile[(rA + 8) * 40 + 8 * k + v];
          accB = __builtin_fmaf(b, b, accB);
        }
      }
      asm volatile("" ::: "memory");
      const float invA = 1.0f / sg_sqrt(sg_hsum8(accA) / (float)kHD + qp.eps);
      const float invB = 1.0f / sg_sqrt(sg_hsum8(accB) / (float)kHD + qp.eps);
      const float iA = __shfl(invA, 8 * (ln & 7)), iB = __shfl(invB, 8 * (ln & 7));
      const float inv = ln < 8 ? iA : iB;
#pragma unroll
      for (int ks = 0; ks < kHD / 32; ks++) {
        const float* wv = wtile + 32 * ks + 8 * g4;
#pragma unroll
        for (int t = 0; t < 8; t++) {
          const float u = x[ks][t] * inv;
          x[ks][t] = u * wv[t];
        }
      }
    }
    // RoPE (rope_cache.go:85-104): pairs (e, e + 128) are chunks ks and ks + 4
    // of the same lane and slot.
#pragma unroll
    for (int ks = 0; ks < kHD / 64; ks++) {
#pragma unroll
      for (int t = 0; t < 8; t++) {
        const float v0 = x[ks][t], v1 = x[ks + kHD / 64][t];
        const float a = v0 * cv[ks][t], b = v1 * sv[ks][t], cc = v0 * sv[ks][t], dd = v1 * cv[ks][t];
        x[ks][t] = a - b;
        x[ks + kHD / 64][t] = cc + dd;
      }
    }
#pragma unroll
    for (int ks = 0; ks < kHD / 32; ks++) {
      u32x4_t uh, ul;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        uint32_t h, l;
        split_pair(x[ks][2 * k], x[ks][2 * k + 1], kQKScale, h, l);
        uh[k] = h;
        ul[k] = l;
      }
      bqh[ks] = __builtin_bit_cast(half8_t, uh);
      bql[ks] = __builtin_bit_cast(half8_t, ul);
    }
  } else {
#pragma unroll
    for (int ks = 0; ks < kHD / 32; ks++) {
      bqh[ks] = *reinterpret_cast<const half8_t*>(qf + sgd::kfrag_piece(0, ks, 0) + 8 * lane);
      bql[ks] = *reinterpret_cast<const half8_t*>(qf + sgd::kfrag_piece(0, ks, 1) + 8 * lane);
    }
  }
}

constexpr int kTileBytes = 32 * 1024;  // one K or V tile, hi and lo halves
static_assert(kTileBytes == 2 * sgd::kFragTile && sgk::kAttnTileHalves == sgd::kFragTile, "tile layout");
constexpr int kRing = 3;               // tile stages in LDS
constexpr int kScoreBytes = sgk::kAttnSpillTileBytes;  // one tile's scores, 8 floats per lane and wave
static_assert(kScoreBytes == kWaves * 2048, "spill tile layout");

// Two passes over a sequence's 32-key tiles: pass 1 keeps each lane's scaled
// scores in registers (8 per tile, 128 VGPRs for the first kRegTiles tiles)
// and pass 2 reads them back instead of recomputing S^T, so K is streamed once
// and a third of the MFMAs and LDS reads go away.  SPILL (a launch with a
// sequence longer than kRegKeys keys): the tiles past kRegTiles write their
// scores to a per-workgroup spill range in pass 1 and read them back in pass 2
// through LDS, carried by the V^T item before their own.  The tiles reach LDS
// by buffer_load ... lds (no staging registers): one stream of 2 nt items, the
// nt K tiles then the nt V^T tiles, item i in ring stage i % 3, issued two
// items ahead; each wave issues four 1-KB copies per item (six when it also
// carries scores; past the last item it re-copies that one into the free
// stage), so a vmcnt of the next item's copy count says "item i has landed"
// and the barrier after it publishes every wave's copies and retires the
// stage the next copies overwrite.
//
// A tile's LDS stage is its 32 KB of fragments as they lie in memory, so a copy
// is 1 KB to 1 KB and a fragment read is the wave's lanes in order (no bank
// conflicts, an immediate offset per fragment).
//
// Split items.  A launch of fewer workgroups than CUs takes as long as its
// longest sequence's; `n_split` of its items (the first ones: the longest) then
// run as two workgroups of four chunks, a wave per SIMD each, and take 0.8 of
// an item's time (one K or V stream for half of the MFMAs, nothing to overlap a
// wave's softmax with).  us per launch, unsplit / split: 6 x 512 tokens 50 / 40,
// 5 x 1024 95 / 77, 2 x 2048 175 / 134, 40 x 128 20 / 17; more than 256 workgroups
// of halves lose (16 x 512: 55 / 77), so only as many items are split as there
// are idle CUs.
template <bool QPRE, bool SPILL, int W>
__device__ __forceinline__ void attn_rs_item(
    unsigned char* lds, unsigned char* slds, float* red, const sg_item& it, int half,
    const _Float16* __restrict__ qf, const _Float16* __restrict__ kf, const _Float16* __restrict__ vf, int n_tiles,
    float* __restrict__ out, int ldo, const int32_t* __restrict__ seq_off, const int32_t* __restrict__ voff, int G,
    float sscale, float* __restrict__ amax, const sg_attn_qpre& qp, const sg_attn_qout& qo, const sg_attn_spill& sp) {
  typedef __attribute__((address_space(3))) void* lds_ptr;

  const int kvh = blockIdx.y;
  const int r0 = seq_off[it.seq];
  const int S = seq_off[it.seq + 1] - r0;
  const int vo = voff[it.seq];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6) & (W - 1);
  const int wi = half * W + w;  // the wave's chunk of the item
  const int ln = lane & 15, g4 = lane >> 4;
  const int nqb = (S + kQW - 1) / kQW;
  const int nt = (S + kBK - 1) / kBK;  // <= kRegTiles unless SPILL (the host checks the longest sequence)
  if (W != kWaves && it.c0 + half * W >= G * nqb) return;  // workgroup-uniform, before any barrier
  const int c = it.c0 + wi;
  const bool active = c < G * nqb;  // wave-uniform
  const int hg = active ? c / nqb : 0;
  const int q0 = active ? (c % nqb) * kQW : 0;
  const int head = kvh * G + hg;
  const int qrow = q0 + ln;
  const bool qvalid = active && qrow < S;
  const int qr = r0 + min(qrow, S - 1);

  // ---- copies ----
  // Wave w's kCopies copies of an item: pieces kCopies * w .. of the tile.  Keys past
  // the sequence's end hold whatever the buffer held; their scores are masked
  // below (V's pad keys are zeros).
  const int64_t tile0 = (int64_t)kvh * n_tiles + (vo >> 5);
  const i32x4_t rk = sg_raw_rsrc(kf + tile0 * sgd::kFragTile);
  const i32x4_t rv = sg_raw_rsrc(vf + tile0 * sgd::kFragTile);
  constexpr int kCopies = 32 / W;
  auto copy_tile = [&](uint32_t dst, bool isk, int tile, uint32_t voff) {
    const uint32_t soff = (uint32_t)tile * kTileBytes + (uint32_t)w * (kCopies * 1024u);
#pragma unroll
    for (int i = 0; i < kCopies; i++) sg_lds_copy16(dst + 1024u * i, voff, isk ? rk : rv, soff + 1024u * i);
  };
  // SPILL: this workgroup's spilled scores, nt - kRegTiles tiles of
  // kScoreBytes (wave w's 2 KB at w * 2048: lane l's keys 4g4 + r at 16 l,
  // 16 + 4g4 + r at 1024 + 16 l).  V^T item nt + t - 1 also carries tile t's
  // scores when t >= kRegTiles, two more copies per wave into the item's
  // score stage.
  float* const wspill =
      SPILL && nt > kRegTiles
          ? sp.buf + ((size_t)kvh * sp.total + sp.off[it.seq] + (size_t)(it.c0 / kWaves) * (nt - kRegTiles)) *
                         (kScoreBytes / 4)
          : nullptr;
  const i32x4_t rsp = sg_raw_rsrc(wspill);
  const int last = 2 * nt - 1;
  auto carries = [&](int src) { return SPILL && src >= nt + kRegTiles - 1 && src < last; };
  auto issue_at = [&](int item, uint32_t voff) {
    const int src = item < last ? item : last;
    const uint32_t dst = (uint32_t)(uintptr_t)(lds_ptr)(lds + ((unsigned)item % kRing) * kTileBytes + w * (kCopies * 1024));
    copy_tile(dst, src < nt, src < nt ? src : src - nt, voff);
    if (carries(src)) {
      const uint32_t sd = (uint32_t)(uintptr_t)(lds_ptr)(slds + ((unsigned)item % kRing) * (W * 2048) + w * 2048);
      const uint32_t so = (uint32_t)((src - nt + 1 - kRegTiles) * kScoreBytes + wi * 2048);
      sg_lds_copy16(sd, 16u * lane, rsp, so);
      sg_lds_copy16(sd + 1024u, 16u * lane + 1024u, rsp, so);
    }
  };
  auto issue = [&](int item) { issue_at(item, 16u * lane); };
  // Wait until item i has landed, item i + 1 (kCopies copies per wave, or two more
  // when it carries scores) may still be in flight.
  auto wait_item = [&](int i) {
    if (carries(i + 1 < last ? i + 1 : last))
      sg_wait_vmcnt<kCopies + 2>();
    else
      sg_wait_vmcnt<kCopies>();
  };
  // A sequence of one tile (item 0 is all its K): for its pad keys a lane copies the
  // last key's fragment, which its neighbours read as well.  Reading the pad keys'
  // own made a forward of 4000 one-token sequences 8.75 ms, 8.45 now.
  const int key_last = nt == 1 ? max(S - 1 - kQW * (w / (W / 2)), 0) : kQW;  // in the wave's 16-key subtile
  issue_at(0, 16u * (lane - ln + min(ln, key_last)));
  issue(1);
  half8_t bqh[kHD / 32], bql[kHD / 32];
  // The Q prologue's LDS tiles sit in stage 2, which no copy touches before
  // the first barrier.
  static_assert(W * (16 * 40 + kHD) * 4 <= kTileBytes, "prologue tiles fit stage 2");
  // (Pre-split Q: rows past the end read the last one's fragments, as the keys.)
  q_operand<QPRE>(bqh, bql, QPRE ? nullptr : qf + q_subtile(head, n_tiles, vo, q0), qp, qr, qr - r0, head, ln, g4,
                  QPRE ? lane : lane - ln + min(ln, S - 1 - q0),
                  reinterpret_cast<float*>(lds + 2 * kTileBytes) + w * (16 * 40),
                  reinterpret_cast<float*>(lds + 2 * kTileBytes) + W * (16 * 40) + w * kHD);

  auto key_of = [&](int kt, int st, int r) { return kt + 16 * st + 4 * g4 + r; };
  // ---- pass 1: S^T = K Q^T per tile, kept in registers; row max ----
  auto scores2 = [&](const unsigned char* kb, f32x4_t& a0, f32x4_t& a1) {
    const _Float16* kp = reinterpret_cast<const _Float16*>(kb) + 8 * lane;
    auto rd = [&](int st, int ks, half8_t& h, half8_t& l) {
      h = *reinterpret_cast<const half8_t*>(kp + sgd::kfrag_piece(st, ks, 0));
      l = *reinterpret_cast<const half8_t*>(kp + sgd::kfrag_piece(st, ks, 1));
    };
    a0 = f32x4_t{0, 0, 0, 0};
    a1 = f32x4_t{0, 0, 0, 0};
    half8_t h0, l0, h1, l1;
    rd(0, 0, h0, l0);
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
    for (int ks = 0; ks < kHD / 32; ks++) {
      rd(1, ks, h1, l1);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      a0 = mfma16(h0, bqh[ks], a0);
      a0 = mfma16(h0, bql[ks], a0);
      a0 = mfma16(l0, bqh[ks], a0);
      __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
      if (ks + 1 < kHD / 32) {
        rd(0, ks + 1, h0, l0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      a1 = mfma16(h1, bqh[ks], a1);
      a1 = mfma16(h1, bql[ks], a1);
      a1 = mfma16(l1, bqh[ks], a1);
      __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
    }
  };
  float m = -INFINITY;
  f32x4_t sr[kRegTiles][2];
  // The scores are kept as s = raw * sscale (exact: sscale is a power of
  // two); a key past S (only in a sequence's last tile) keeps -inf, so pass
  // 2's fastExp clamp gives it a weight of exactly 0 without a per-key test
  // there.
#pragma unroll
  for (int t = 0; t < kRegTiles; t++) {
    if (t < nt) {
      wait_item(t);  // item t landed (item t + 1 may still be in flight)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      issue(t + 2);
      // Every wave computes (an inactive wave's results are never stored).
      scores2(lds + (t % kRing) * kTileBytes, sr[t][0], sr[t][1]);
      const int kt = t * kBK;
      if (kt + kBK <= S) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          sr[t][0][r] *= sscale;
          sr[t][1][r] *= sscale;
          m = fmaxf(m, fmaxf(sr[t][0][r], sr[t][1][r]));
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          sr[t][0][r] = key_of(kt, 0, r) < S ? sr[t][0][r] * sscale : -INFINITY;
          sr[t][1][r] = key_of(kt, 1, r) < S ? sr[t][1][r] * sscale : -INFINITY;
          m = fmaxf(m, fmaxf(sr[t][0][r], sr[t][1][r]));
        }
      }
    }
  }
  if constexpr (SPILL) {
    // Tiles past kRegTiles: their scores go to this wave's spill slots.
    for (int t = kRegTiles; t < nt; t++) {
      wait_item(t);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      issue(t + 2);
      f32x4_t s0, s1;
      scores2(lds + (t % kRing) * kTileBytes, s0, s1);
      const int kt = t * kBK;
      if (kt + kBK <= S) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          s0[r] *= sscale;
          s1[r] *= sscale;
          m = fmaxf(m, fmaxf(s0[r], s1[r]));
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          s0[r] = key_of(kt, 0, r) < S ? s0[r] * sscale : -INFINITY;
          s1[r] = key_of(kt, 1, r) < S ? s1[r] * sscale : -INFINITY;
          m = fmaxf(m, fmaxf(s0[r], s1[r]));
        }
      }
      float* sp = wspill + (size_t)(t - kRegTiles) * (kScoreBytes / 4) + wi * 512 + 4 * lane;
      *reinterpret_cast<f32x4_t*>(sp) = s0;
      *reinterpret_cast<f32x4_t*>(sp + 256) = s1;
    }
  }
  m = fmaxf(m, __shfl_xor(m, 16));
  m = fmaxf(m, __shfl_xor(m, 32));

  // ---- pass 2: e = fastExp(s - m), row sums, O^T += V^T P^T ----
  f32x4_t o[kHD / 16];
#pragma unroll
  for (int mt = 0; mt < kHD / 16; mt++) o[mt] = f32x4_t{0, 0, 0, 0};
  float lsum = 0.0f;
  auto pv = [&](const unsigned char* vb, const half8_t& ph, const half8_t& pl) {
    const _Float16* vp = reinterpret_cast<const _Float16*>(vb) + 8 * lane;
    half8_t fr[3][2];  // [buffer][hi, lo]
    auto rd = [&](int mt, half8_t(&f)[2]) {
      f[0] = *reinterpret_cast<const half8_t*>(vp + sgd::vfrag_piece(mt, 0));
      f[1] = *reinterpret_cast<const half8_t*>(vp + sgd::vfrag_piece(mt, 1));
    };
    rd(0, fr[0]);
    rd(1, fr[1]);
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int mt = 0; mt < kHD / 16; mt++) {
      if (mt + 2 < kHD / 16) {
        rd(mt + 2, fr[(mt + 2) % 3]);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      const half8_t(&f)[2] = fr[mt % 3];
      o[mt] = mfma16(f[0], ph, o[mt]);
      o[mt] = mfma16(f[0], pl, o[mt]);
      o[mt] = mfma16(f[1], ph, o[mt]);
      __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
    }
  };
  // One tile of pass 2: the weights from its scores, then P.V on its V^T item.
  auto tile2 = [&](const f32x4_t& s0, const f32x4_t& s1, int t) {
    const int item = nt + t;
    float e[8];  // slots 0..3: keys 4g4+r, slots 4..7: 16+4g4+r
#pragma unroll
    for (int r = 0; r < 4; r++) {
      e[r] = sg_fast_exp_nonpos(s0[r] - m);
      e[4 + r] = sg_fast_exp_nonpos(s1[r] - m);
    }
#pragma unroll
    for (int k = 0; k < 8; k++) lsum = lsum + e[k];
    u32x4_t uh, ul;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      uint32_t h, l;
      split_pair(e[2 * k], e[2 * k + 1], kPScale, h, l);
      uh[k] = h;
      ul[k] = l;
    }
    const half8_t ph = __builtin_bit_cast(half8_t, uh), pl = __builtin_bit_cast(half8_t, ul);
    wait_item(item);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(item + 2);
    pv(lds + ((unsigned)item % kRing) * kTileBytes, ph, pl);
  };
#pragma unroll
  for (int t = 0; t < kRegTiles; t++)
    if (t < nt) tile2(sr[t][0], sr[t][1], t);
  if constexpr (SPILL) {
    // Tile t's scores landed with item nt + t - 1 (published by its barrier);
    // the stage is overwritten only after the next barrier.
    for (int t = kRegTiles; t < nt; t++) {
      const unsigned char* sb = slds + ((unsigned)(nt + t - 1) % kRing) * (W * 2048) + w * 2048 + 16 * lane;
      tile2(*reinterpret_cast<const f32x4_t*>(sb), *reinterpret_cast<const f32x4_t*>(sb + 1024), t);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the re-copies past the last item have landed
  lsum = lsum + __shfl_xor(lsum, 16);
  lsum = lsum + __shfl_xor(lsum, 32);
  const float f = (1.0f / lsum) * kPUnscale;

  // O^T tile mt: lane holds query ln, dims 16mt + 4g4 + r.
  float mx = 0.0f;
  if (qvalid) {
    float* op = out + (int64_t)(r0 + qrow) * ldo + head * kHD + 4 * g4;
#pragma unroll
    for (int mt = 0; mt < kHD / 16; mt++) {
      f32x4_t y;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        y[j] = o[mt][j] * f;
        mx = fmaxf(mx, fabsf(y[j]));
      }
      *reinterpret_cast<f32x4_t*>(op + 16 * mt) = y;
    }
  }
  if (amax) {  // all chunks of a workgroup belong to one sequence
    mx = sg_wave_max(mx);
    if (lane == 0) red[w] = mx;
    __syncthreads();
    if (tid == 0) {
      float mm = red[0];
#pragma unroll
      for (int i = 1; i < W; i++) mm = fmaxf(mm, red[i]);
      sg_atomic_max_nonneg(amax + it.seq, mm);
    }
    // The workgroup holds the whole sequence (every row of every head; the
    // caller passes qo.q8 only then), so its maximum is the sequence's and
    // the output is quantized here, from the values just stored, as the
    // quantizer would quantize them: lane (query ln, group g4) codes dims
    // 16 mt + 4 g4 .. + 3 of its head, 4 bytes of K-block (head * 256 +
    // 16 mt) / 32 per mt.
    if (qo.q8 && qvalid) {
      float mm = red[0];
#pragma unroll
      for (int i = 1; i < W; i++) mm = fmaxf(mm, red[i]);
      float scale = 1.0f, inv = 0.0f;
      if (mm != 0.0f) {
        scale = mm / 127.0f;
        inv = 1.0f / scale;
      }
      const int row = r0 + qrow;
      if (hg == 0 && g4 == 0) qo.row_scale[row] = scale;
#pragma unroll
      for (int mt = 0; mt < kHD / 16; mt++) {
        const int col = head * kHD + 16 * mt + 4 * g4;
        uint32_t u = 0;
#pragma unroll
        for (int j = 0; j < 4; j++)
          u |= (uint32_t)(uint8_t)(int8_t)(int)sg_quant_code_nb(o[mt][j] * f, inv) << (8 * j);
        *reinterpret_cast<uint32_t*>(qo.q8 + ((int64_t)(col >> 5) * qo.a_rows + row) * 32 + (col & 31)) = u;
      }
    }
  }
}

template <bool QPRE, bool SPILL>
__global__ __launch_bounds__(kNT, 2) void k_attn_rs(
    const _Float16* __restrict__ qf, const _Float16* __restrict__ kf, const _Float16* __restrict__ vf, int n_tiles,
    float* __restrict__ out, int ldo, const int32_t* __restrict__ seq_off, const int32_t* __restrict__ voff,
    const sg_item* __restrict__ items, int n_items, int n_split, int G, float sscale, float* __restrict__ amax,
    sg_attn_qpre qp, sg_attn_qout qo, sg_attn_spill sp) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[kRing * kTileBytes];
  __shared__ __attribute__((aligned(16))) unsigned char slds[SPILL ? kRing * kScoreBytes : 16];
  __shared__ float red[kWaves];
  const int b = blockIdx.x;
  if (b < 2 * n_split) {  // n_split is a multiple of 8: the halves of an item on one XCD, like the items
    const int at = (b >> 4) * 8 + (b & 7);
    // Four waves stay (the others' end counts at barriers).
    if (at >= n_items || __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= kWaves / 2) return;
    attn_rs_item<QPRE, SPILL, kWaves / 2>(lds, slds, red, items[at], (b >> 3) & 1, qf, kf, vf, n_tiles, out, ldo,
                                          seq_off, voff, G, sscale, amax, qp, qo, sp);
  } else {
    attn_rs_item<QPRE, SPILL, kWaves>(lds, slds, red, items[b - n_split], 0, qf, kf, vf, n_tiles, out, ldo, seq_off,
                                      voff, G, sscale, amax, qp, qo, sp);
  }
}

// ---- small launches ----
//
// A launch of few workgroups leaves most CUs idle in k_attn_rs: its wave walks
// every key tile of its chunk alone, whatever else the GPU has to do (one
// 512-token sequence: 12 workgroups, 47 us; here 18 us, of which ~8 us are
// the megabyte of K and V fragments through each CU's 64 B/clk).  Here a workgroup's eight waves
// share C chunks of 16 (head, query) rows instead: pass 1 deals the 16-key
// subtiles to the waves, pass 2 the output dims, so a chunk's serial chain is
// an eighth as long and there are 8 / C times the workgroups.  Every sum keeps
// k_attn_rs's order -- a score's chain over the dims, a row sum's over the
// tiles, an output's over the tiles -- so the results are the same bits.
//   Pass 1: wave w scores subtiles w, w + 8, ...; K fragments come straight
//           from global memory (this wave alone uses them), one subtile ahead;
//           scores go to LDS (2 KB per tile), the row maximum is combined over
//           the waves.
//   exp:    each wave turns its own subtiles' scores into weights, in place.
//   Pass 2: wave w owns dims 32 w .. + 31; V fragments straight from global
//           memory, four to eight tiles ahead; every wave reads all weights,
//           splits them and keeps the row sums (identical in all waves).
// LDS holds every score (NT tiles), so nothing spills.  One workgroup per CU
// (two waves per SIMD, up to 256 VGPRs for the fragments in flight).
// The chunk maxima of |out| go to cmax (attn_cmax_base), not by atomics.
//
// Barrier over LDS only: loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int C, int NT>
__global__ __launch_bounds__(kNT, 2) void k_attn_small(
    const _Float16* __restrict__ qf, const _Float16* __restrict__ kf, const _Float16* __restrict__ vf,
    int n_tiles, float* __restrict__ out, int ldo,
    const int32_t* __restrict__ seq_off, const int32_t* __restrict__ voff, const sg_item* __restrict__ items,
    int n_items, int npad, int G, float sscale, float* __restrict__ cmax) {
  constexpr int NS = kHD / 32;  // k-steps
  constexpr int KN = NS / C;    // k-steps per fragment load group (the Q operands of C chunks leave room for that)
  __shared__ __attribute__((aligned(16))) f32x4_t sc[C][2 * NT][SG_WAVE];
  __shared__ float red[C][kWaves][kQW];
  static_assert(kHD == 32 * kWaves && (C == 1 || C == 2), "32 output dims per wave");
  // Item k's workgroups are blocks k, k + npad, ...: the same XCD each (npad
  // is a multiple of 8), so an item's K and V stay in one L2.
  const int k_it = blockIdx.x % npad, kvh = blockIdx.y;
  if (k_it >= n_items) return;
  const sg_item it = items[k_it];
  const int r0 = seq_off[it.seq];
  const int S = seq_off[it.seq + 1] - r0;
  const int vo = voff[it.seq];
  const int64_t tile0 = (int64_t)kvh * n_tiles + (vo >> 5);
  const int nqb = (S + kQW - 1) / kQW, nt = (S + kBK - 1) / kBK, nch = G * nqb;
  const int c0 = it.c0 + C * (int)(blockIdx.x / npad);
  if (c0 >= nch) return;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, g4 = lane >> 4;

  half8_t bqh[C][NS], bql[C][NS];
#pragma unroll
  for (int j = 0; j < C; j++) {  // past the last chunk: that one again, never stored
    const int c = min(c0 + j, nch - 1);
    const _Float16* qp = qf + q_subtile(kvh * G + c / nqb, n_tiles, vo, (c % nqb) * kQW) + 8 * lane;
#pragma unroll
    for (int ks = 0; ks < NS; ks++) {
      bqh[j][ks] = *reinterpret_cast<const half8_t*>(qp + sgd::kfrag_piece(0, ks, 0));
      bql[j][ks] = *reinterpret_cast<const half8_t*>(qp + sgd::kfrag_piece(0, ks, 1));
    }
  }

  // ---- pass 1 ----
  struct KFrag {
    half8_t h[KN], l[KN];
  };
  auto load_k = [&](KFrag& f, int u, int k0) {
    const _Float16* kp = kf + (tile0 + (u >> 1)) * sgd::kFragTile + sgd::kfrag_piece(u & 1, k0, 0) + 8 * lane;
#pragma unroll
    for (int ks = 0; ks < KN; ks++) {
      f.h[ks] = *reinterpret_cast<const half8_t*>(kp + sgd::kfrag_piece(0, ks, 0));
      f.l[ks] = *reinterpret_cast<const half8_t*>(kp + sgd::kfrag_piece(0, ks, 1));
    }
  };
  float m[C];
  f32x4_t a[C];
#pragma unroll
  for (int j = 0; j < C; j++) m[j] = -INFINITY;
  auto clear = [&]() {
#pragma unroll
    for (int j = 0; j < C; j++) a[j] = f32x4_t{0, 0, 0, 0};
  };
  auto dot = [&](const KFrag& f, auto k0c) {
    constexpr int K0 = decltype(k0c)::value;
#pragma unroll
    for (int ks = 0; ks < KN; ks++) {
#pragma unroll
      for (int j = 0; j < C; j++) a[j] = mfma16(f.h[ks], bqh[j][K0 + ks], a[j]);
#pragma unroll
      for (int j = 0; j < C; j++) a[j] = mfma16(f.h[ks], bql[j][K0 + ks], a[j]);
#pragma unroll
      for (int j = 0; j < C; j++) a[j] = mfma16(f.l[ks], bqh[j][K0 + ks], a[j]);
    }
  };
  auto keep = [&](int u) {
    const int k0 = 16 * u + 4 * g4;  // keys past S are masked
#pragma unroll
    for (int j = 0; j < C; j++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        a[j][r] = k0 + r < S ? a[j][r] * sscale : -INFINITY;
        m[j] = fmaxf(m[j], a[j][r]);
      }
      sc[j][u][lane] = a[j];
    }
  };
  // The prefetches are unconditional (past the last subtile they re-load it).
  KFrag f0, f1;
  const int last = 2 * nt - 1;
  load_k(f0, min(w, last), 0);
  if constexpr (C == 1) {
#pragma unroll 1
    for (int u = w; u <= last; u += 2 * kWaves) {
      load_k(f1, min(u + kWaves, last), 0);
      __builtin_amdgcn_sched_barrier(0);
      clear();
      dot(f0, int_c<0>{});
      keep(u);
      load_k(f0, min(u + 2 * kWaves, last), 0);
      __builtin_amdgcn_sched_barrier(0);
      if (u + kWaves <= last) {
        clear();
        dot(f1, int_c<0>{});
        keep(u + kWaves);
      }
    }
  } else {
#pragma unroll 1
    for (int u = w; u <= last; u += kWaves) {
      load_k(f1, u, KN);
      __builtin_amdgcn_sched_barrier(0);
      clear();
      dot(f0, int_c<0>{});
      load_k(f0, min(u + kWaves, last), 0);
      __builtin_amdgcn_sched_barrier(0);
      dot(f1, int_c<KN>{});
      keep(u);
    }
  }

  // V fragments of tiles t0 .. + 3: dim groups 2 w + i, hi (0) and lo (1).
  struct VFrag {
    half8_t v[4][2][2];
  };
  const _Float16* vp = vf + tile0 * sgd::kFragTile + sgd::vfrag_piece(2 * w, 0) + 8 * lane;
  auto load_v = [&](VFrag& f, int t0) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const _Float16* p = vp + (int64_t)min(t0 + u, nt - 1) * sgd::kFragTile;
#pragma unroll
      for (int i = 0; i < 2; i++) {
        f.v[u][i][0] = *reinterpret_cast<const half8_t*>(p + sgd::vfrag_piece(i, 0));
        f.v[u][i][1] = *reinterpret_cast<const half8_t*>(p + sgd::vfrag_piece(i, 1));
      }
    }
  };
  VFrag v0, v1;
  load_v(v0, 0);
#pragma unroll
  for (int j = 0; j < C; j++) {
    m[j] = fmaxf(m[j], __shfl_xor(m[j], 16));
    m[j] = fmaxf(m[j], __shfl_xor(m[j], 32));
    if (g4 == 0) red[j][w][ln] = m[j];
  }
  lds_barrier();
#pragma unroll
  for (int j = 0; j < C; j++)
#pragma unroll
    for (int i = 0; i < kWaves; i++) m[j] = fmaxf(m[j], red[j][i][ln]);

  // ---- weights: this wave's subtiles ----
#pragma unroll 1
  for (int u = w; u <= last; u += kWaves)
#pragma unroll
    for (int j = 0; j < C; j++) {
      f32x4_t e = sc[j][u][lane];
#pragma unroll
      for (int r = 0; r < 4; r++) e[r] = sg_fast_exp_nonpos(e[r] - m[j]);
      sc[j][u][lane] = e;
    }
  lds_barrier();

  // ---- pass 2 ----
  f32x4_t o[C][2];
  float lsum[C];
#pragma unroll
  for (int j = 0; j < C; j++) {
    o[j][0] = o[j][1] = f32x4_t{0, 0, 0, 0};
    lsum[j] = 0.0f;
  }
  auto group = [&](const VFrag& f, int t0) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (t0 + u >= nt) break;
#pragma unroll
      for (int j = 0; j < C; j++) {
        const f32x4_t e0 = sc[j][2 * (t0 + u)][lane], e1 = sc[j][2 * (t0 + u) + 1][lane];
        const float e[8] = {e0[0], e0[1], e0[2], e0[3], e1[0], e1[1], e1[2], e1[3]};
#pragma unroll
        for (int k = 0; k < 8; k++) lsum[j] = lsum[j] + e[k];
        u32x4_t uh, ul;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          uint32_t h, l;
          split_pair(e[2 * k], e[2 * k + 1], kPScale, h, l);
          uh[k] = h;
          ul[k] = l;
        }
        const half8_t ph = __builtin_bit_cast(half8_t, uh), pl = __builtin_bit_cast(half8_t, ul);
#pragma unroll
        for (int i = 0; i < 2; i++) o[j][i] = mfma16(f.v[u][i][0], ph, o[j][i]);
#pragma unroll
        for (int i = 0; i < 2; i++) o[j][i] = mfma16(f.v[u][i][0], pl, o[j][i]);
#pragma unroll
        for (int i = 0; i < 2; i++) o[j][i] = mfma16(f.v[u][i][1], ph, o[j][i]);
      }
    }
  };
#pragma unroll 1
  for (int t0 = 0; t0 < nt; t0 += 8) {
    load_v(v1, t0 + 4);
    __builtin_amdgcn_sched_barrier(0);
    group(v0, t0);
    load_v(v0, t0 + 8);
    __builtin_amdgcn_sched_barrier(0);
    group(v1, t0 + 4);
  }

  // O^T: lane holds query ln, dims 32 w + 16 i + 4 g4 + r.
#pragma unroll
  for (int j = 0; j < C; j++) {
    lsum[j] = lsum[j] + __shfl_xor(lsum[j], 16);
    lsum[j] = lsum[j] + __shfl_xor(lsum[j], 32);
    const float f = (1.0f / lsum[j]) * kPUnscale;
    const int c = min(c0 + j, nch - 1), qrow = (c % nqb) * kQW + ln;
    float mx = 0.0f;
    if (c0 + j < nch && qrow < S) {
      float* op = out + (int64_t)(r0 + qrow) * ldo + (kvh * G + c / nqb) * kHD + 32 * w + 4 * g4;
#pragma unroll
      for (int i = 0; i < 2; i++) {
        f32x4_t y;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          y[r] = o[j][i][r] * f;
          mx = fmaxf(mx, fabsf(y[r]));
        }
        *reinterpret_cast<f32x4_t*>(op + 16 * i) = y;
      }
    }
    if (cmax) {
      mx = sg_wave_max(mx);
      if (lane == 0) red[j][w][0] = mx;  // the row maxima were read before the weights' barrier
    }
  }
  if (!cmax) return;
  lds_barrier();
  if (threadIdx.x < C && c0 + (int)threadIdx.x < nch) {
    float mm = red[threadIdx.x][0][0];
#pragma unroll
    for (int i = 1; i < kWaves; i++) mm = fmaxf(mm, red[threadIdx.x][i][0]);
    cmax[sgk::attn_cmax_base(r0, it.seq, G * gridDim.y) + kvh * nch + c0 + threadIdx.x] = mm;
  }
}

// The fragments of already normed and rotated Q, K and of V in one launch: a
// workgroup per operand head (query heads, kv heads of K, of V) and 32-key tile,
// one row of workgroups (the grid's second dimension would end at 65535 heads).
// Q and K: a wave per 16-key subtile and half of the dims, lane l fragment lane
// l, so a whole subtile's stores are 1 KB contiguous; pad keys are not written
// (3000 sequences of 5 tokens: 93 us with the last key repeated there, 57 now).
__global__ __launch_bounds__(sgd::kKvThreads) void k_qkv_split(
    const float* __restrict__ q, int ldq, const float* __restrict__ k, const float* __restrict__ v, int ldkv, int H,
    int HKV, const int32_t* __restrict__ seq_off, const int32_t* __restrict__ voff,
    const sg_item* __restrict__ vtiles, int n_vtiles, _Float16* __restrict__ qf, _Float16* __restrict__ kf,
    _Float16* __restrict__ vf, int n_tiles) {
  __shared__ __attribute__((aligned(16))) float tv[kBK][sgd::kVtRowStride];
  const sg_item t = vtiles[blockIdx.x % n_vtiles];
  const int y = blockIdx.x / n_vtiles;
  if (y >= H + HKV) {  // workgroup-uniform
    sgd::v_split_tile(t, y - H - HKV, tv, v, ldkv, seq_off, voff, vf, n_tiles);
    return;
  }
  const int h = y < H ? y : y - H;
  const float* x0 = y < H ? q : k;
  const int ld = y < H ? ldq : ldkv;
  const int lane = threadIdx.x & 63, st = (threadIdx.x >> 6) & 1, k0 = 4 * (threadIdx.x >> 7);
  const int r0 = seq_off[t.seq], S = seq_off[t.seq + 1] - r0;
  const int key = t.c0 + 16 * st + (lane & 15);
  if (key >= S) return;  // no barrier below
  const float* src = x0 + (int64_t)(r0 + key) * ld + h * kHD + 32 * k0 + 8 * (lane >> 4);
  _Float16* dst = (y < H ? qf : kf) + ((int64_t)h * n_tiles + (voff[t.seq] + t.c0) / kBK) * sgd::kFragTile +
                  sgd::kfrag_piece(st, 0, 0) + k0 * 1024 + 8 * lane;
  f32x4_t x[4][2];
#pragma unroll
  for (int ks = 0; ks < 4; ks++) {
    x[ks][0] = *reinterpret_cast<const f32x4_t*>(src + 32 * ks);
    x[ks][1] = *reinterpret_cast<const f32x4_t*>(src + 32 * ks + 4);
  }
#pragma unroll
  for (int ks = 0; ks < 4; ks++) {
    u32x4_t uh, ul;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint32_t hi, lo;
      split_pair(x[ks][i >> 1][2 * (i & 1)], x[ks][i >> 1][2 * (i & 1) + 1], kQKScale, hi, lo);
      uh[i] = hi;
      ul[i] = lo;
    }
    *reinterpret_cast<u32x4_t*>(dst + sgd::kfrag_piece(0, ks, 0)) = uh;
    *reinterpret_cast<u32x4_t*>(dst + sgd::kfrag_piece(0, ks, 1)) = ul;
  }
}

// K's QK-norm/RoPE split and V's split in one launch: workgroups [0, nkb) take
// 32 (token, head) rows of K (and Q) each, the rest one (V tile, kv head)
// each, so the two halves' loads and stores overlap.
__global__ __launch_bounds__(sgd::kKvThreads) void k_kv_prep(
    const float* __restrict__ k, const float* __restrict__ v, int ldkv, const float* __restrict__ kw, int HKV, int T,
    const int32_t* __restrict__ row_pos, const float* __restrict__ cos_t, const float* __restrict__ sin_t, float eps,
    const int32_t* __restrict__ row_key, _Float16* __restrict__ kf, int nkb, const int32_t* __restrict__ seq_off,
    const int32_t* __restrict__ voff, const sg_item* __restrict__ vtiles, int n_vtiles, _Float16* __restrict__ vf,
    int n_tiles, sgk::sg_kv_q qp) {
  __shared__ __attribute__((aligned(16))) float tv[kBK][sgd::kVtRowStride];
  const int b = blockIdx.x;
  if (b < nkb) {  // workgroup-uniform
    const int64_t g = (int64_t)b * sgd::kKvRows + (threadIdx.x >> 3);
    float* tile = &tv[0][0] + (threadIdx.x / SG_WAVE) * (8 * 40);  // 8 x 40 floats per wave
    // (token, head) groups, query heads first.  With no query heads (qp.H =
    // 0) the Q arguments are never read; they then point at K (passing null
    // for them crashed this compiler's device pass).
    sgd::qk_split_group(g, threadIdx.x & 7, (threadIdx.x >> 3) & 7, tile, qp.q, qp.ldq, k, ldkv, qp.qw, kw, qp.H,
                        HKV, T, row_pos, cos_t, sin_t, eps, qp.qf, row_key, kf, n_tiles);
  } else {
    const int vb = b - nkb;
    sgd::v_split_tile(vtiles[vb % n_vtiles], vb / n_vtiles, tv, v, ldkv, seq_off, voff, vf, n_tiles);
  }
}

}  // namespace

namespace sgk {

hipError_t qkv_split(const float* q, int ldq, const float* k, const float* v, int ldkv, int H, int HKV,
                     const int32_t* seq_off, const int32_t* voff, const sg_item* vtiles, int n_vtiles, _Float16* qf,
                     _Float16* kf, _Float16* vf, int n_tiles, hipStream_t s) {
  if (n_vtiles <= 0) return hipSuccess;
  if ((ldq & 3) || (ldkv & 3) || H < 0 || HKV <= 0) return hipErrorInvalidValue;
  const int64_t nwg = (int64_t)n_vtiles * ((int64_t)H + 2 * (int64_t)HKV);
  if (nwg > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_qkv_split, dim3((unsigned)nwg), dim3(sgd::kKvThreads), 0, s, q, ldq, k, v, ldkv, H, HKV, seq_off,
                     voff, vtiles, n_vtiles, qf, kf, vf, n_tiles);
  return hipGetLastError();
}

hipError_t kv_prep(const float* k, const float* v, int ldkv, const float* kw, int HKV, int T, const int32_t* row_pos,
                   const float* cos_t, const float* sin_t, float eps, const int32_t* row_key, _Float16* kf,
                   const int32_t* seq_off, const int32_t* voff, const sg_item* vtiles, int n_vtiles, _Float16* vf,
                   int n_tiles, hipStream_t s, const sg_kv_q* qpart) {
  if (T <= 0 || n_vtiles < 0 || HKV <= 0) return hipSuccess;
  if ((ldkv & 3) || (reinterpret_cast<uintptr_t>(k) & 15) || (reinterpret_cast<uintptr_t>(v) & 15) ||
      (kw && (reinterpret_cast<uintptr_t>(kw) & 15)))
    return hipErrorInvalidValue;  // float4 loads of K and V rows and of the weights
  sgk::sg_kv_q qp{k, ldkv, kw, 0, kf};
  if (qpart && qpart->H > 0) {
    if (!qpart->q || !qpart->qf || (qpart->ldq & 3) || (reinterpret_cast<uintptr_t>(qpart->q) & 15) || (qpart->qw && (reinterpret_cast<uintptr_t>(qpart->qw) & 15)))
      return hipErrorInvalidValue;  // float4 loads of the Q rows and weights, 16-byte split stores
    qp = *qpart;
  }
  const int64_t nkb = ((int64_t)T * (qp.H + HKV) + sgd::kKvRows - 1) / sgd::kKvRows;
  const int64_t nb = nkb + (int64_t)n_vtiles * HKV;
  if (nb > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_kv_prep, dim3((unsigned)nb), dim3(sgd::kKvThreads), 0, s, k, v, ldkv, kw, HKV, T, row_pos, cos_t,
                     sin_t, eps, row_key, kf, (int)nkb, seq_off, voff, vtiles, n_vtiles, vf, n_tiles, qp);
  return hipGetLastError();
}

namespace {
template <int C, int NT>
void launch_small(int n_items, int HKV, hipStream_t s, const _Float16* qf, const _Float16* kf,
                  const _Float16* vf, int n_tiles, float* out, int ldo, const int32_t* seq_off,
                  const int32_t* voff, const sg_item* items, int G, float sscale, float* cmax) {
  const int npad = (n_items + 7) & ~7;
  hipLaunchKernelGGL((k_attn_small<C, NT>), dim3(npad * (kWaves / C), HKV), dim3(kNT), 0, s, qf, kf, vf, n_tiles, out, ldo,
                     seq_off, voff, items, n_items, npad, G, sscale, cmax);
}

template <bool QPRE, bool SPILL>
void launch_attn(int n_items, int HKV, int n_split, hipStream_t s, const _Float16* qf, const _Float16* kf,
                 const _Float16* vf, int n_tiles, float* out, int ldo, const int32_t* seq_off, const int32_t* voff,
                 const sg_item* items, int G, float sscale, float* amax, const sg_attn_qpre& qp, const sg_attn_qout& qo,
                 const sg_attn_spill& sp) {
  n_split = (n_split + 7) & ~7;  // past n_items: empty workgroups
  const int nwg = 2 * n_split + (n_items > n_split ? n_items - n_split : 0);
  hipLaunchKernelGGL((k_attn_rs<QPRE, SPILL>), dim3(nwg, HKV), dim3(kNT), 0, s, qf, kf, vf, n_tiles, out, ldo, seq_off,
                     voff, items, n_items, n_split, G, sscale, amax, qp, qo, sp);
}
}  // namespace

bool attn_small_form(int n_items, int HKV, int max_len) {
  return (int64_t)n_items * HKV <= kAttnSmallItems && max_len <= kAttnSmallKeys;
}

hipError_t attention_small(const _Float16* qf, const _Float16* kf, const _Float16* vf, int n_tiles,
                           float* out, int ldo, const int32_t* seq_off, const int32_t* voff,
                           const sg_item* items, int n_items, int H, int HKV, int hd, float scale,
                           float* cmax, int max_len, hipStream_t s) {
  if (n_items <= 0) return hipSuccess;
  if (hd != kHD || HKV <= 0 || H % HKV || max_len <= 0 || !attn_small_form(n_items, HKV, max_len))
    return hipErrorInvalidValue;
  if (!qf || (ldo & 3)) return hipErrorInvalidValue;  // float4 stores
  const float sscale = scale / (kQKScale * kQKScale);
  using fn = void (*)(int, int, hipStream_t, const _Float16*, const _Float16*, const _Float16*, int, float*, int, const int32_t*, const int32_t*, const sg_item*, int, float, float*);
  const bool two = max_len <= 1024 && (int64_t)n_items * HKV > kAttnSmallOneItems;
  const fn f = max_len <= 512    ? (two ? launch_small<2, 16> : launch_small<1, 16>)
               : max_len <= 1024 ? (two ? launch_small<2, 32> : launch_small<1, 32>)
                                 : launch_small<1, 64>;
  f(n_items, HKV, s, qf, kf, vf, n_tiles, out, ldo, seq_off, voff, items, H / HKV, sscale, cmax);
  return hipGetLastError();
}

hipError_t attention(const _Float16* qf, const _Float16* kf, const _Float16* vf, int n_tiles,
                     float* out, int ldo, const int32_t* seq_off, const int32_t* voff, const sg_item* items, int n_items, int H, int HKV, int hd, float scale,
                     float* amax, int max_len, hipStream_t s, const sg_attn_qpre* qpre,
                     const sg_attn_qout* qout, const sg_attn_spill* spill, int n_split) {
  if (n_items <= 0) return hipSuccess;
  if (n_split < 0 || n_split > n_items) return hipErrorInvalidValue;
  if (hd != kHD || HKV <= 0 || H % HKV || max_len <= 0) return hipErrorInvalidValue;
  // The quantizing epilogue needs the register-scores kernel, one workgroup per
  // sequence (one kv head, every chunk of the sequence in one item) and amax.
  if (qout && (!qout->q8 || !qout->row_scale || HKV != 1 || max_len > kAttnRegKeys || !amax ||
               (H / HKV) * ((max_len + kQW - 1) / kQW) > kWaves))
    return hipErrorInvalidValue;
  const sg_attn_qout qo = qout ? *qout : sg_attn_qout{nullptr, 0, nullptr};
  if (ldo & 3) return hipErrorInvalidValue;
  static_assert(kBK == 32 && kRegTiles == sgk::kAttnRegKeys / 32, "attention_spill_tiles");
  const bool spills = attention_spill_tiles(max_len) > 0;
  if (spills && (!spill || !spill->buf || !spill->off || spill->total <= 0 ||
                 (reinterpret_cast<uintptr_t>(spill->buf) & 15)))
    return hipErrorInvalidValue;
  const sg_attn_spill sp = spills ? *spill : sg_attn_spill{nullptr, nullptr, 0};
  const float sscale = scale / (kQKScale * kQKScale);
  sg_attn_qpre qp{};
  if (qpre) {
    if (!qpre->q || !qpre->cos_t || !qpre->sin_t || (qpre->ldq & 3) ||
        (reinterpret_cast<uintptr_t>(qpre->q) & 15) || (reinterpret_cast<uintptr_t>(qpre->w) & 15) ||
        (reinterpret_cast<uintptr_t>(qpre->cos_t) & 15) || (reinterpret_cast<uintptr_t>(qpre->sin_t) & 15))
      return hipErrorInvalidValue;  // float4 loads of Q rows, weights and table rows
    qp = *qpre;
  } else if (!qf) {
    return hipErrorInvalidValue;
  }
  using fn = void (*)(int, int, int, hipStream_t, const _Float16*, const _Float16*, const _Float16*, int, float*, int,
                      const int32_t*, const int32_t*, const sg_item*, int, float, float*, const sg_attn_qpre&,
                      const sg_attn_qout&, const sg_attn_spill&);
  static const fn table[2][2] = {{launch_attn<false, false>, launch_attn<false, true>},
                                 {launch_attn<true, false>, launch_attn<true, true>}};
  if (qout) n_split = 0;  // one workgroup per sequence
  table[qpre != nullptr][spills](n_items, HKV, n_split, s, qf, kf, vf, n_tiles, out, ldo, seq_off, voff, items, H / HKV,
                                 sscale, amax, qp, qo, sp);
  return hipGetLastError();
}

}  // namespace sgk
