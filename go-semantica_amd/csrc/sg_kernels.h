// sg_kernels.h -- host-side launchers for the gfx950 kernels (internal to the
// library; the public surface is include/semantica_gpu.h).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// One unit of per-sequence work: attention workgroup (sequence, first 32-row
// chunk) or V^T split tile (sequence, first key).
struct sg_item { int32_t seq, c0; };
// Q's QK-norm + RoPE done inside the attention kernel: fp32 q [T][ldq] as the
// QKV GEMM wrote it, attn_q_norm weights (null: no norm) and the RoPE tables
// [pos][128].  A row's position is its index within its sequence (positions
// restart at 0 in every sequence, as the forward's row_pos holds them).
struct sg_attn_qpre {
  const float* q;
  int ldq;
  const float* w;
  const float* cos_t;
  const float* sin_t;
  float eps;
};

// Optional attention epilogue: the attention output quantized per sequence
// into the block-major GEMM operand q8[H*hd/32][a_rows][32] and row_scale
// (quantize's arithmetic on the values written to out), for launches in which
// one workgroup holds every row and head of its sequence (one work item per
// sequence and a single kv head); the caller checks.
struct sg_attn_qout {
  int8_t* q8;
  int a_rows;
  float* row_scale;
};

// Where attention() keeps the scores of the tiles past its register-held ones
// (sequences longer than sgk::kAttnRegKeys keys): per kv head, `total` tiles of
// sgk::kAttnSpillTileBytes at buf (16-byte aligned); sequence i's workgroups
// at tile off[i] + (c0 / sgk::kAttnChunks) * sgk::attention_spill_tiles(S_i).
struct sg_attn_spill {
  float* buf;
  const int32_t* off;
  int total;
};

namespace sgk {

// GEMM operands are block-major int8 [K/32][rows][32]; activation buffers hold
// gemm_pad_rows(M) rows per K-block so that every workgroup tile reads
// allocated memory (rows past M are never stored).
constexpr int kGemmRowPad = 256;
inline int gemm_pad_rows(int M) { return (M + kGemmRowPad - 1) / kGemmRowPad * kGemmRowPad; }

// ---- load-time repack (k_rows.hip) ----
// Raw Q8_0 rows [rows][cols/32][34 B] -> block-major int8 weights
// w8[b][dst(r)][32] (ld rows per block) and fp32 block scales (IEEE
// converter) st[b][dst(r)] (ld per block), dst(r) = row_off + (r / grp) *
// gstride + r % grp (grp = rows, gstride = 0: plain row_off + r).
hipError_t repack_q8_0(const uint8_t* raw, int rows, int cols, int8_t* w8, float* st, int ld, int row_off, int grp,
                       int gstride, hipStream_t s);
// token_embd: int8 values q[v][d] and per-block scales (gguf halving converter) sc[v][d/32].
hipError_t repack_embd(const uint8_t* raw, int vocab, int d, int8_t* q, float* sc, hipStream_t s);
// int8 x[M][K] -> block-major int8 y[K/32][a_rows][32] (the GEMM operand).
hipError_t i8_blocked(const int8_t* x, int M, int K, int8_t* y, int a_rows, hipStream_t s);
hipError_t fill_f32(float* p, float v, int64_t n, hipStream_t s);
hipError_t fill_i32(int32_t* p, int32_t v, int64_t n, hipStream_t s);
// The first row r < T with tokens[r] outside [0, vocab), folded into *first by
// atomicMin (the embedding kernels record theirs the same way).
hipError_t first_bad_token(const int32_t* tokens, int T, int vocab, int32_t* first, hipStream_t s);

// ---- per-row kernels (k_rows.hip) ----
// Small launches (row_max_form(T, d)) can pass the rows' maxima on instead of
// the sequences': embed_norm and post_res_norm with rmax != null write each
// row's max|xn| to rmax[T] (amax null or unused), and norm_quantize with rmax
// (and the CSR seq_off) takes each sequence's maximum over its rows.  The
// atomics on amax cost ~13 ns each, one after another (the sequences' maxima
// share a cache line): with a wave per row they were most of the kernel.
// The fused GEMM + post-norm writes only amax: it serves none of these launches.
constexpr int kWaveRows = 8192;  // the form's launches have fewer rows
bool row_max_form(int T, int d);
// Embedding gather * sqrt(d) -> h; then RMSNorm(w) -> xn (stored when xn != null) and
// per-sequence max|xn| -> amax.  A token outside [0, vocab) is read as token 0
// and its row folded into *err by atomicMin (*err starts at INT32_MAX).
hipError_t embed_norm(const int32_t* tokens, int T, const int8_t* eq, const float* es, int vocab, int d,
                      float sqrt_d, const float* w, float eps, const int32_t* row_seq, float* h, float* xn,
                      float* amax, int32_t* err, hipStream_t s, float* rmax = nullptr);
// Per-sequence symmetric quantization of x[rows][cols] (stride ldx) using amax[row_seq[r]].
// Writes the int8 codes block-major q8[cols/32][a_rows][32] (the GEMM operand)
// and row_scale[rows].
// cmax (with the CSR seq_off, H heads; rows < kWaveRows):
// the sequence's maximum is taken over attention_small's chunk maxima instead
// of amax.
hipError_t quantize(const float* x, int ldx, int rows, int cols, const int32_t* row_seq, const float* amax,
                    int8_t* q8, int a_rows, float* row_scale, hipStream_t s, const float* cmax = nullptr,
                    const int32_t* seq_off = nullptr, int H = 0);
// xn = RMSNorm(h; w) recomputed row by row exactly as post_res_norm / embed_norm
// formed it, quantized with amax[row_seq[r]] into the block-major int8 GEMM
// operand q8[d/32][a_rows][32] and row_scale[T] (quantize's arithmetic).
hipError_t norm_quantize(const float* h, const float* w, float eps, int T, int d, const int32_t* row_seq,
                         const float* amax, int8_t* q8, int a_rows, float* row_scale, hipStream_t s,
                         const float* rmax = nullptr, const int32_t* seq_off = nullptr);
// Per-sequence symmetric quantization of x[rows][cols] from scratch: codes
// row-major q[rows][cols], scales seq_scale[n_seq].  amax [n_seq]: zeros on
// entry, the sequences' max|x| on return.
hipError_t quantize_seqs(const float* x, int rows, int cols, const int32_t* row_seq, int n_seq, float* amax, int8_t* q,
                         float* seq_scale, hipStream_t s);
// RMSNorm rows in the reference's order; amax (optional) collects per-sequence max|y|.
hipError_t rmsnorm(float* dst, const float* src, const float* w, int rows, int n, float eps,
                   const int32_t* row_seq, float* amax, hipStream_t s);
// QK-norm + RoPE in place (fp32); head_dim 256.
hipError_t qknorm_rope(float* q, int ldq, float* k, int ldk, const float* qw, const float* kw, int H, int HKV,
                       int T, const int32_t* row_pos, const float* cos_t, const float* sin_t, float eps,
                       hipStream_t s);
// h = RMSNorm(o; w_post) + h ; xn = RMSNorm(h; w_next) (stored when xn != null) ;
// amax (optional) per sequence of max|xn|.
hipError_t post_res_norm(const float* o, float* h, const float* w_post, const float* w_next, float eps, int T,
                         int d, float* xn, const int32_t* row_seq, float* amax, hipStream_t s,
                         float* rmax = nullptr);
// g = geluquick(gate)*up over rows x cols; amax (optional) per sequence of max|g|.
hipError_t gelu_mul(float* g, int ldd, const float* gate, int ldg, const float* up, int ldu, int rows, int cols,
                    const int32_t* row_seq, float* amax, hipStream_t s);
hipError_t pool_l2(float* out, const float* x, int ldx, int out_dim, const int32_t* seq_off, int n_seq,
                   hipStream_t s);
hipError_t embed_only(const int32_t* tokens, int T, const int8_t* eq, const float* es, int vocab, int d,
                      float sqrt_d, float* h, int32_t* err, hipStream_t s);
// Streaming yardsticks over n floats (n % 4 == 0, 16-byte aligned): kind 0
// c = a + b (fp32), kind 1 c = int8 codes of a (b unused).
hipError_t stream_probe(int kind, const float* a, const float* b, void* c, int64_t n, hipStream_t s);
// k_issue_probe<kind> on `blocks` workgroups of 4 waves: sink [blocks * 256]
// floats, clk [blocks * 4 * 2] (per wave: shader cycles, wall-clock ticks).
hipError_t issue_probe(int kind, int blocks, float* sink, long long* clk, int iters, hipStream_t s);

// ---- GEMM (k_gemm.hip) ----
// Y[M][N] = (sum_b float(P_b) * St[b][n]) * row_scale[m] with A int8 [M][K]
// block-major [K/32][a_rows][32] (a_rows >= gemm_pad_rows(M)), W int8 [N][K]
// block-major [K/32][N][32], St [K/32][N].  sums != null additionally dumps
// the exact block sums int32 [M][N][K/32].  cold_weights: W is not expected
// in L2 (the forward, one layer after another), which selects deeper load
// pipelines for small grids; the results are the same either way.
// The V columns [col0, N) of the QKV GEMM written straight as attention's V
// fragments (vf, n_tiles 32-key tiles per kv head, as k_kv_prep's V half
// writes them: sequence s from tile voff[s] / 32 on) instead of fp32 into Y;
// the bits are the same.  Positions past a sequence's end are not written.
struct sg_vt_out {
  _Float16* vf;
  int n_tiles;
  int col0;
  const int32_t* row_seq;
  const int32_t* seq_off;
  const int32_t* voff;
};
// Whether gemm_q8 takes an sg_vt_out at M rows (the direct-to-LDS kernels).
bool gemm_writes_vt(int M);
hipError_t gemm_q8(const int8_t* A, int a_rows, const int8_t* W, const float* St, const float* row_scale, float* Y,
                   int32_t* sums, int M, int N, int K, hipStream_t s, bool cold_weights = false,
                   const sg_vt_out* vto = nullptr);
// FFN gate/up GEMM with GELUQuick(gate) * up in the epilogue: W holds 2*Nh rows,
// gate and up interleaved in groups of kGeluGroup (see repack_q8_0's grouping);
// G[M][Nh] is bit-identical to the unfused GEMMs + gelu_mul; amax (optional,
// with row_seq) collects the sequences' max|g|.
hipError_t gemm_q8_gelu(const int8_t* A, int a_rows, const int8_t* W, const float* St, const float* row_scale,
                        float* G, int M, int Nh, int K, const int32_t* row_seq, float* amax, hipStream_t s,
                        bool cold_weights = false);
// gemm_q8 followed by post_res_norm on its output (N = d): o = the GEMM, then
// h = RMSNorm(o; w_post) + h, xn = RMSNorm(h; w_next) (stored when xn !=
// null), amax (optional, with row_seq) per sequence of max|xn|.  For N = 768
// and large M one launch computes whole rows and norms them without storing o
// (o is then left untouched); h, xn and amax are bit-identical either way.
hipError_t gemm_q8_res_norm(const int8_t* A, int a_rows, const int8_t* W, const float* St, const float* row_scale,
                            float* o, int M, int N, int K, float* h, const float* w_post, const float* w_next, float eps,
                            float* xn, const int32_t* row_seq, float* amax, hipStream_t s);
// Whether gemm_q8_res_norm runs as one launch for these arguments.
bool gemm_res_norm_fused(int M, int N, const float* w_post, const float* w_next);
// Gate/up interleaving used by gemm_q8_gelu: source row r of a matrix goes to
// row row_off + (r / 32) * 64 + r % 32 (gate: row_off 0, up: row_off 32).
constexpr int kGeluGroup = 32;

// ---- attention (k_attention.hip) ----
constexpr float kAttnQKScale = 8.0f;  // Q and K are split after scaling by 8 (exact)
constexpr int kAttnChunkRows = 16;    // (head, query) rows per attention chunk (one wave)
constexpr int kAttnChunks = 8;        // chunks per attention workgroup
constexpr int kAttnRegKeys = 512;     // longest sequence whose scores pass 1 keeps in registers
// Keys a sequence of S keys occupies in the padded numbering (whole 32-key tiles).
inline int attn_key_pad(int S) { return (S + 31) / 32 * 32; }
// Padded key numbering: sequence s holds keys voff[s] .. voff[s] + S - 1 of
// Tp = sum of attn_key_pad(S), row_key[row] its row's key.  K and V are held in
// MFMA fragment order (sg_kv_prep.h), kf and vf [HKV][n_tiles] tiles of
// kAttnTileHalves, n_tiles = Tp / 32.
constexpr int kAttnTileHalves = 16384;
// The kernel seam's operands: Q and K (already normed and rotated) and V split
// into qf [H][n_tiles], kf and vf; vtiles: (seq, key0) per 32 keys.
hipError_t qkv_split(const float* q, int ldq, const float* k, const float* v, int ldkv, int H, int HKV,
                     const int32_t* seq_off, const int32_t* voff, const sg_item* vtiles, int n_vtiles, _Float16* qf,
                     _Float16* kf, _Float16* vf, int n_tiles, hipStream_t s);
// K's QK-norm, RoPE and split, and V's split, in one launch: K and V share the
// row stride ldkv (columns of the QKV output).  n_vtiles = 0: K only (V written
// by the QKV GEMM, sg_vt_out).
// Optional Q part of kv_prep: the H query heads' norm (qw), RoPE and hi/lo
// split as well, into Q's
// fragments qf [H][n_tiles], for launches that run the attention on pre-split Q.
struct sg_kv_q {
  const float* q;
  int ldq;
  const float* qw;
  int H;
  _Float16* qf;
};
hipError_t kv_prep(const float* k, const float* v, int ldkv, const float* kw, int HKV, int T, const int32_t* row_pos,
                   const float* cos_t, const float* sin_t, float eps, const int32_t* row_key, _Float16* kf,
                   const int32_t* seq_off, const int32_t* voff, const sg_item* vtiles, int n_vtiles, _Float16* vf,
                   int n_tiles, hipStream_t s, const sg_kv_q* qpart = nullptr);
// out[T][ldo] = attention over the split operands; items: (seq, first chunk)
// per workgroup, chunk c of a sequence = (head c / ceil(S/16), rows 16*(c % ceil(S/16))).
// qpre != null: Q is taken from qpre (fp32, normed and rotated in the kernel
// with qknorm_rope's arithmetic) and qf is ignored.  max_len: the
// longest sequence of the launch.  Pass 1's scores stay in registers up to
// kAttnRegKeys keys; a longer sequence keeps the rest in spill (required
// when max_len exceeds kAttnRegKeys).  The first n_split items run as two
// workgroups of half the chunks (not with qout), the same bits.  A sequence gives the same bits
// whatever the launch's max_len.
hipError_t attention(const _Float16* qf, const _Float16* kf, const _Float16* vf, int n_tiles, float* out, int ldo, const int32_t* seq_off, const int32_t* voff, const sg_item* items, int n_items, int H, int HKV, int hd, float scale,
                     float* amax, int max_len, hipStream_t s, const sg_attn_qpre* qpre = nullptr,
                     const sg_attn_qout* qout = nullptr, const sg_attn_spill* spill = nullptr, int n_split = 0);
// The same for launches too small to fill the GPU (attn_small_form), with Q
// pre-split: the same bits as attention(), no spill buffer.  cmax (optional)
// receives each chunk's max|out|, sequence i's chunks (kv head by kv head) from
// attn_cmax_base(seq_off[i], i, H) on; it holds attn_cmax_base(T, n_seq, H)
// floats.
// Where the lines lie (us per launch on MI355X, k_attn_rs / one chunk per
// workgroup / two; 512 tokens unless said): 12 items 47 / 18 / -, 24 items
// 47 / 19 / -, 48 items 47 / 33 / 23, 72 items 48 / - / 44; 128 tokens, 48 items
// 21 / - / 13; 1024 tokens, 24 items 88 / 30 / -, 48 items 88 / - / 37; 2048
// tokens, 48 items 166 / 96 / -, 144 items 170 / 245 / -.  The small form wins
// while its workgroups (8 or 4 per item, one per CU) make about one round.
constexpr int kAttnSmallItems = 64;     // up to this many (items x kv heads): the small form
constexpr int kAttnSmallKeys = 2048;    // ... for sequences of up to this many keys (scores in LDS)
constexpr int kAttnSmallOneItems = 32;  // up to this many: one chunk per workgroup, above: two (to 1024 keys)
bool attn_small_form(int n_items, int HKV, int max_len);
__host__ __device__ inline int64_t attn_cmax_base(int row0, int seq, int H) {
  return ((int64_t)row0 / kAttnChunkRows + seq) * H;  // >= H * (chunks of 16 rows of the sequences before)
}
hipError_t attention_small(const _Float16* qf, const _Float16* kf, const _Float16* vf, int n_tiles, float* out, int ldo, const int32_t* seq_off, const int32_t* voff,
                           const sg_item* items, int n_items, int H, int HKV, int hd, float scale,
                           float* cmax, int max_len, hipStream_t s);
// Score tiles a sequence of S keys spills per attention workgroup (one 32-key
// tile of one workgroup: kAttnSpillTileBytes).
constexpr int kAttnSpillTileBytes = kAttnChunks * 2048;
inline int attention_spill_tiles(int S) {
  const int t = (S + 31) / 32 - kAttnRegKeys / 32;
  return t > 0 ? t : 0;
}

// ---- attention in the reference's float32 order (k_attn_exact.hip) ----
// out[T][ldo] (head h at h*hd) from q[T][ldq], k/v[T][ldkv] (kv head h / (H/HKV)),
// every operation in attention.go's order; P: attention_exact_scratch bytes;
// amax (optional) collects each sequence's max|out| (atomic max, >= 0).
// hd must be 256, max_len <= 2048, q/k rows 16-byte aligned; n_seq * H <= 65535.
size_t attention_exact_scratch(int T, int H, int max_len);
hipError_t attention_exact(const float* q, int ldq, const float* k, const float* v, int ldkv, float* out, int ldo,
                           const int32_t* seq_off, const int32_t* row_seq, int n_seq, int T, int H, int HKV, int hd,
                           float scale, int max_len, float* P, float* amax, hipStream_t s);

// ---- brute-force search (k_search.hip) ----
// Storage modes, the values of brute.QuantizationMode (search/brute/quant.go:8-15).
constexpr int kBfF32 = 0, kBfI8 = 1, kBfI16 = 2;
// Index layout: grp [dim/8][N][8] elements, tail [N][dim%8] elements.
// Rows row0..row0+n of the index from float vectors src[n][ld]: normalized
// (builder.go:131-141) when `normalize`, then quantized (quant.go:17-41).
hipError_t bf_build(int mode, const float* src, int64_t ld, int n, int dim, int row0, int N, void* grp, void* tail,
                    bool normalize, hipStream_t s);
// builder.go:131-141 in place on n rows [n][dim].
hipError_t bf_normalize(float* x, int n, int dim, hipStream_t s);
// Stored rows (row-major [n][dim], as serialized) -> rows row0.. of the layout.
hipError_t bf_relayout(int mode, const void* rows, int n, int dim, int row0, int N, void* grp, void* tail,
                       hipStream_t s);
// Rows row0..row0+n of the layout -> row-major [n][dim].
hipError_t bf_unpack(int mode, const void* grp, const void* tail, int row0, int n, int dim, int N, void* rows,
                     hipStream_t s);
// scores[q][ld_scores] for nq normalized queries [nq][dim] against all N vectors.
hipError_t bf_score(int mode, const void* grp, const void* tail, int N, int dim, const float* queries, int nq,
                    float* scores, int64_t ld_scores, hipStream_t s);
// The reference's top-k of every query's scores (k <= N): out_idx/out_dist [nq][k]
// in arbitrary order (positions, not ids).  state: int32 [nq][8]; hist: [nq][256].
hipError_t bf_select(const float* scores, int64_t ld_scores, int N, int nq, int k, int32_t* state, uint32_t* hist,
                     int32_t* out_idx, float* out_dist, hipStream_t s);

// ---- prefiltered search (k_search.hip, "prefiltering") ----
// Largest L2 norm of the stored vectors (dequantized units), as float bits in
// *vmax (device); +inf when one is not finite.
hipError_t bf_vnorm(int mode, const void* grp, const void* tail, int N, int dim, uint32_t* vmax, hipStream_t s);
constexpr int kBfBlock = 64;            // vectors per block
constexpr size_t kBfPfLds = 144 << 10;  // LDS for the queries' fragments
constexpr int bf_prefilter_cap(int k) { return 4 * k + 64; }  // listed blocks per query
bool bf_prefilter_ok(int N, int dim, int k, float vnorm);
// A query's listed blocks and candidates grow with k and are one workgroup's
// work at two of the four steps, so few queries for many vectors are better off
// with the full path's grid-wide passes.  us a search, full / prefiltered:
//   10^6 x 768 int8, 1 query    k 500 284 / 243   700 290 / 267   1000 306 / 338
//   4,000,000 x 64 int8, 1      k 500 213 / 158   1000 237 / 249  4000 440 / 646
//   300,000 x 256 float32, 1    k 500 153 / 142
//   4,000,000 x 256 float32, 4  k 1000 1229 / 1074 4000 1942 / 2085
//   10^6 x 256 float32, 16      k 1000 1290 / 1125; 4,000,000: k 4000 5752 / 4929
constexpr int kBfMostK = 512;    // k up to here for any number of queries
constexpr int kBfManyQueries = 16;  // any k from this many on
int bf_prefilter_queries(int dim);  // queries per call
// Why a query was not decided: the query itself is not one for the prefilter, or
// the stored vectors leave it open (too many blocks, a tie at the k-th place).
constexpr int kBfUnfit = 1, kBfOpen = 2;
struct sg_bf_work {
  _Float16* qfrag;   // 64 x (dim rounded up to 32) + 1024
  float* eps;        // [nq][2]: the bound (then the score that the k best reach), its unit
  float* blockmax;   // [nq][blocks]
  int32_t* list;     // [nq][cap]
  int32_t* count;    // [nq]
  float* cand;       // [nq][cap * kBfBlock]
  int32_t* out_idx;  // [nq][k]
  float* out_dist;   // [nq][k]
  int32_t* flags;    // [nq]: not 0 = not decided, run the query through bf_score / bf_select
};
// queries [nq][dim]: normalized in place when `normalize` (bf_normalize's
// arithmetic).  out_idx / out_dist as bf_select's, for the unflagged queries.
hipError_t bf_prefilter(int mode, const void* grp, const void* tail, int N, int dim, float vnorm, float* queries,
                        int nq, bool normalize, int k, const sg_bf_work& w, hipStream_t s);

}  // namespace sgk
