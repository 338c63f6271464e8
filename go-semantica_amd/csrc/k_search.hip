// k_search.hip -- brute-force vector search (search/brute) for gfx950: index
// build (normalize + quantize), scoring of every stored vector against a
// batch of queries, and the exact top-k selection.
//
// Index layout in HBM.  The reference stores vectors row-major [N][dim]
// (index.go:11-25).  Here the first 8*G elements of every vector (G = dim/8)
// are stored as [G][N][8] -- group g of all vectors contiguous -- so the lane
// that scores vector n reads its group g with one 8/16/32-byte load and a
// wave's loads are 512 contiguous bytes (int8).  The last R = dim % 8
// elements of each vector sit in a tail array [N][R].  Groups follow the
// reference's 8-lane split exactly: lane j of the AVX2 loop owns elements
// 8g + j, and the tail is what its scalar loop handles.
//
// Arithmetic (bit-exact to the amd64 AVX2 path of the reference):
//   int8/int16  d = float(q) * inv  (inv = float32(1/127) / float32(1/32767)),
//               acc_j = acc_j + d * x  (three roundings, dot_amd64.s:24-34,52-62)
//   float32     acc_j = fma(v, x, acc_j)  (dot_amd64.s:85-95)
//   reduction   ((l0+l4)+(l1+l5)) + ((l2+l6)+(l3+l7))  (VEXTRACTF128/VADDPS/2xVHADDPS)
//   tail        int modes: one unrolled group of 4 partial sums, then singles,
//               through the clamping lookup tables (quant.go:57-135);
//               float32: sum += a*b (index.go:209-212)
#include "sg_device.h"
#include "sg_kernels.h"

namespace {

constexpr int kBfThreads = 256;

template <typename T>
struct BfElem;
template <>
struct BfElem<int8_t> {
  static constexpr bool kQuant = true;
  static constexpr int kLo = -127;
  __device__ static float inv() { return (float)(1.0 / 127.0); }
  __device__ static float scale() { return 127.0f; }
};
template <>
struct BfElem<int16_t> {
  static constexpr bool kQuant = true;
  static constexpr int kLo = -32767;
  __device__ static float inv() { return (float)(1.0 / 32767.0); }
  __device__ static float scale() { return 32767.0f; }
};
template <>
struct BfElem<float> {
  static constexpr bool kQuant = false;
};

// One group of 8 stored elements as loaded (8, 16 or 32 bytes), and its
// conversion to the AVX2 loop's per-lane operand (no clamp: VPMOVSX +
// VCVTDQ2PS take the code as it is; then the scale multiply, rounded).
template <typename T>
struct BfRaw;
template <>
struct BfRaw<int8_t> {
  uint2 w;
  __device__ void load(const int8_t* p) { w = *reinterpret_cast<const uint2*>(p); }
  __device__ void get(float (&v)[8]) const {
#pragma unroll
    for (int l = 0; l < 4; l++) {
      v[l] = (float)(int8_t)(w.x >> (8 * l)) * BfElem<int8_t>::inv();
      v[4 + l] = (float)(int8_t)(w.y >> (8 * l)) * BfElem<int8_t>::inv();
    }
  }
};
template <>
struct BfRaw<int16_t> {
  uint4 w;
  __device__ void load(const int16_t* p) { w = *reinterpret_cast<const uint4*>(p); }
  __device__ void get(float (&v)[8]) const {
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int l = 0; l < 4; l++) {
      v[2 * l] = (float)(int16_t)(u[l] & 0xffffu) * BfElem<int16_t>::inv();
      v[2 * l + 1] = (float)(int16_t)(u[l] >> 16) * BfElem<int16_t>::inv();
    }
  }
};
template <>
struct BfRaw<float> {
  float4 a, b;
  __device__ void load(const float* p) {
    a = *reinterpret_cast<const float4*>(p);
    b = *reinterpret_cast<const float4*>(p + 4);
  }
  __device__ void get(float (&v)[8]) const {
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
};

// Tail element through the lookup table of quant.go:57-77 (the most negative
// code clamps to -127 / -32767).
template <typename T>
__device__ __forceinline__ float bf_lut(T c) {
  int v = (int)c;
  v = v < BfElem<T>::kLo ? BfElem<T>::kLo : v;
  return (float)v * BfElem<T>::inv();
}

// ------------------------------------------------------------------ build --

// builder.go:131-141 on each row: float64 sum of the float32 squares in index
// order, norm = float32(1/sqrt(sum)), v *= norm (a zero vector stays as is);
// then quant.go:17-41: clamp to [-1, 1] and math.Round(float64(v) * 127 or
// 32767) (sg_round_prod_f_nb: the product rounded once, half away from zero).
// A workgroup takes 64 vectors, staged through LDS 64 dimensions at a time with
// coalesced loads (the next chunk's in flight meanwhile), twice: one lane per
// vector runs the sums, then a thread per (vector, group) quantizes, a wave's
// stores covering one group of 64 vectors.  (A lane per vector reading its own
// row from memory moved 0.2 TB/s: 21.9 ms for 10^6 x 768 to int8; now 1.14.)
constexpr int kBuildDims = 64, kBuildRows = 64;
template <typename T>
__global__ __launch_bounds__(kBfThreads) void k_bf_build(const float* __restrict__ src, int64_t ld, int n, int dim,
                                                        int row0, int N, T* __restrict__ grp, T* __restrict__ tail,
                                                        int normalize) {
  __shared__ float tile[kBuildRows][kBuildDims + 1];
  __shared__ float norms[kBuildRows];
  __shared__ int scales[kBuildRows];
  constexpr int L = kBuildRows * kBuildDims / kBfThreads;  // loads per thread and chunk
  const int tid = threadIdx.x, v0 = blockIdx.x * kBuildRows;
  const int lc = tid % kBuildDims, lrow = tid / kBuildDims;  // column, first row of this thread's loads
  const int chunks = (dim + kBuildDims - 1) / kBuildDims;
  float r[L];
  auto fetch = [&](int c) {
    const int col = min(c * kBuildDims + lc, dim - 1);
#pragma unroll
    for (int u = 0; u < L; u++)
      r[u] = src[(int64_t)min(v0 + lrow + (kBfThreads / kBuildDims) * u, n - 1) * ld + col];
  };
  auto stage = [&]() {
#pragma unroll
    for (int u = 0; u < L; u++) tile[lrow + (kBfThreads / kBuildDims) * u][lc] = r[u];
  };
  double sum = 0.0;
  fetch(0);
  if (normalize) {
    for (int c = 0; c < chunks; c++) {
      __syncthreads();
      stage();
      __syncthreads();
      fetch(c + 1 < chunks ? c + 1 : 0);
      if (tid < kBuildRows) {
        const int cn = min(kBuildDims, dim - c * kBuildDims);
        for (int i0 = 0; i0 < cn; i0 += 16) {
          float v[16];
#pragma unroll
          for (int u = 0; u < 16; u++) v[u] = tile[tid][min(i0 + u, kBuildDims - 1)];
#pragma unroll
          for (int u = 0; u < 16; u++) {
            const float sq = v[u] * v[u];
            if (i0 + u < cn) sum += (double)sq;
          }
        }
      }
    }
    if (tid < kBuildRows) {
      scales[tid] = sum != 0.0;
      norms[tid] = sum != 0.0 ? (float)(1.0 / sqrt(sum)) : 1.0f;
    }
  }
  const int G = dim >> 3, R = dim & 7;
  const int vec = tid % kBuildRows;
  const bool live = v0 + vec < n;
  const int64_t row = row0 + v0 + vec;
  for (int c = 0; c < chunks; c++) {
    __syncthreads();
    stage();
    __syncthreads();
    if (c + 1 < chunks) fetch(c + 1);
    const float norm = normalize ? norms[vec] : 1.0f;
    const bool scale = normalize && scales[vec];
#pragma unroll
    for (int u = 0; u < kBuildDims / 8 * kBuildRows / kBfThreads; u++) {
      const int gl = tid / kBuildRows + (kBfThreads / kBuildRows) * u, g = c * (kBuildDims / 8) + gl;
      T q[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        float x = tile[vec][8 * gl + e];
        if (scale) x = x * norm;
        if constexpr (BfElem<T>::kQuant) {
          x = x > 1.0f ? 1.0f : (x < -1.0f ? -1.0f : x);
          q[e] = (T)(int)sg_round_prod_f_nb(x, BfElem<T>::scale());
        } else {
          q[e] = x;
        }
      }
      if (live && g < G) {
        __builtin_memcpy(__builtin_assume_aligned(grp + ((int64_t)g * N + row) * 8, 8 * sizeof(T)), q, sizeof q);
      } else if (live && g == G) {
#pragma unroll
        for (int e = 0; e < 8; e++)
          if (e < R) tail[row * R + e] = q[e];
      }
    }
  }
}

// builder.go:131-141 in place on rows of x (the queries of SearchVector,
// index.go:36-38).  One wave per row: the row is staged in LDS with
// coalesced loads, lane 0 runs the float64 sum in index order, and all lanes
// scale.
constexpr int kNormChunk = 1024;

__global__ __launch_bounds__(64) void k_bf_normalize(float* __restrict__ x, int dim) {
  __shared__ float buf[kNormChunk];
  __shared__ float norm;
  __shared__ int scale;
  float* v = x + (int64_t)blockIdx.x * dim;
  const int lane = threadIdx.x;
  double sum = 0.0;
  for (int c0 = 0; c0 < dim; c0 += kNormChunk) {
    const int cn = min(kNormChunk, dim - c0);
    for (int i = lane; i < cn; i += 64) buf[i] = v[c0 + i];
    __syncthreads();
    if (lane == 0)
      for (int i = 0; i < cn; i++) {
        const float sq = buf[i] * buf[i];
        sum += (double)sq;
      }
    __syncthreads();
  }
  if (lane == 0) {
    scale = sum != 0.0;
    norm = sum != 0.0 ? (float)(1.0 / sqrt(sum)) : 1.0f;
  }
  __syncthreads();
  if (!scale) return;
  for (int i = lane; i < dim; i += 64) v[i] = v[i] * norm;
}

// Stored rows (row-major, as serialized) -> the grouped layout, and back.
template <typename T>
__global__ void k_bf_relayout(const T* __restrict__ rows, int64_t n_elems, int dim, int row0, int N,
                              T* __restrict__ grp, T* __restrict__ tail) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n_elems) return;
  const int64_t row = row0 + e / dim;
  const int i = (int)(e % dim);
  const int G = dim >> 3, R = dim & 7;
  const int g = i >> 3;
  if (g < G)
    grp[((int64_t)g * N + row) * 8 + (i & 7)] = rows[e];
  else
    tail[row * R + (i & 7)] = rows[e];
}

template <typename T>
__global__ void k_bf_unpack(const T* __restrict__ grp, const T* __restrict__ tail, int64_t n_elems, int dim,
                            int row0, int N, T* __restrict__ rows) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n_elems) return;
  const int64_t row = row0 + e / dim;
  const int i = (int)(e % dim);
  const int G = dim >> 3, R = dim & 7;
  const int g = i >> 3;
  rows[e] = g < G ? grp[((int64_t)g * N + row) * 8 + (i & 7)] : tail[row * R + (i & 7)];
}

// ---------------------------------------------------------------- scoring --

// The eight lane sums' reduction and the scalar tail (x, tp: the query's and the
// vector's last R elements).
template <typename T>
__device__ __forceinline__ float bf_finish(const float (&l)[8], int G, int R, const float* __restrict__ x,
                                           const T* __restrict__ tp) {
  float sum = 0.0f;
  if (G > 0) sum += ((l[0] + l[4]) + (l[1] + l[5])) + ((l[2] + l[6]) + (l[3] + l[7]));
  if constexpr (BfElem<T>::kQuant) {
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
    int i = 0;
    if (R >= 4) {
      s0 += x[0] * bf_lut<T>(tp[0]);
      s1 += x[1] * bf_lut<T>(tp[1]);
      s2 += x[2] * bf_lut<T>(tp[2]);
      s3 += x[3] * bf_lut<T>(tp[3]);
      i = 4;
    }
    sum += s0 + s1 + s2 + s3;
    for (; i < R; i++) sum += x[i] * bf_lut<T>(tp[i]);
  } else {
    for (int i = 0; i < R; i++) {
      const float p = (float)tp[i] * x[i];
      sum += p;
    }
  }
  return sum;
}

// scores[q][n] for QB queries (rows q0 + QB * blockIdx.y .. of `queries`, already normalized)
// against every stored vector; lane = vector.  The workgroup stages the
// queries in LDS, kQChunk dimensions at a time, and every lane reads them by
// broadcast; each lane issues the loads of kBfBatch groups before using them.
constexpr int kQChunk = 256;
// Groups loaded together per lane: 32 bytes of int8 / int16, 64 of float32.
template <typename T>
constexpr int kBfBatch = sizeof(T) == 1 ? 4 : 2;

template <typename T, int QB>
__global__ __launch_bounds__(kBfThreads) void k_bf_score(const T* __restrict__ grp, const T* __restrict__ tail,
                                                        int N, int dim, const float* __restrict__ queries, int q0,
                                                        int nq, float* __restrict__ scores, int64_t ld_scores) {
  __shared__ __attribute__((aligned(16))) float qs[QB][kQChunk];
  q0 += QB * blockIdx.y;
  const int n = blockIdx.x * kBfThreads + threadIdx.x;
  const bool live = n < N;
  const int nn = live ? n : N - 1;  // lanes past the end load a valid vector and store nothing
  const int G = dim >> 3, R = dim & 7;

  float acc[QB][8];
#pragma unroll
  for (int j = 0; j < QB; j++)
#pragma unroll
    for (int l = 0; l < 8; l++) acc[j][l] = 0.0f;

  const T* gp = grp + (int64_t)nn * 8;
  const int64_t gstride = (int64_t)N * 8;
  for (int c0 = 0; c0 < 8 * G; c0 += kQChunk) {
    const int cn = min(kQChunk, 8 * G - c0);
    __syncthreads();  // the previous chunk's reads are done
    for (int e = threadIdx.x; e < QB * cn; e += kBfThreads) {
      const int j = e / cn, i = e - j * cn;
      qs[j][i] = queries[(int64_t)min(q0 + j, nq - 1) * dim + c0 + i];
    }
    __syncthreads();
    const int g0 = c0 >> 3, gn = cn >> 3;
    for (int g = 0; g < gn; g += kBfBatch<T>) {
      BfRaw<T> raw[kBfBatch<T>];  // all of a batch's loads in flight at once
#pragma unroll
      for (int u = 0; u < kBfBatch<T>; u++)
        if (g + u < gn) raw[u].load(gp + (g0 + g + u) * gstride);
#pragma unroll
      for (int u = 0; u < kBfBatch<T>; u++) {
        if (g + u >= gn) break;
        float v[8];
        raw[u].get(v);
#pragma unroll
        for (int j = 0; j < QB; j++) {
          const float4 xa = *reinterpret_cast<const float4*>(&qs[j][8 * (g + u)]);
          const float4 xb = *reinterpret_cast<const float4*>(&qs[j][8 * (g + u) + 4]);
          const float x[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
          for (int l = 0; l < 8; l++) {
            if constexpr (BfElem<T>::kQuant) {
              const float p = v[l] * x[l];
              acc[j][l] = acc[j][l] + p;
            } else {
              acc[j][l] = __builtin_fmaf(v[l], x[l], acc[j][l]);
            }
          }
        }
      }
    }
  }
  if (!live) return;

  const T* tp = tail + (int64_t)n * R;
#pragma unroll
  for (int j = 0; j < QB; j++) {
    if (q0 + j >= nq) break;
    scores[(int64_t)(q0 + j) * ld_scores + n] =
        bf_finish<T>(acc[j], G, R, queries + (int64_t)(q0 + j) * dim + 8 * G, tp);
  }
}

// -------------------------------------------------------------- selection --
//
// The reference keeps a k-slot list while streaming the scores in stored
// order (index.go:84-131): the first k fill it; later ones replace the
// current minimum (its first slot) only when strictly larger.  The list
// always holds the k largest values seen, so at the end it holds every score
// above the k-th largest value v_k plus some scores equal to v_k.  When
// exactly k scores are >= v_k the result is that set, whatever the order;
// only a tie straddling the k-th place makes the slot history matter.
// Hence: an exact radix select finds v_k and the counts above / at it; the
// common case collects the >= v_k set in parallel; a query with a straddling
// tie replays the reference's streaming loop (one wave, exact).
//
// Per-query state, int32[8]: 0 prefix (key bits fixed so far), 1 mask,
// 2 k_rem (places left inside the prefix), 3 above (count with key > prefix
// bits decided), 4 at (count in the final bin), 5 done-blocks counter,
// 6 collected, 7 tie flag.

// Order-preserving key of a score; -0 maps with +0 (they compare equal).
__device__ __forceinline__ uint32_t bf_key(float d) {
  const uint32_t u = __float_as_uint(d == 0.0f ? 0.0f : d);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr int kSelPerThread = 16;
constexpr int kSelBlock = kBfThreads * kSelPerThread;  // scores per workgroup

// One 8-bit digit of the radix select (digit 0 = bits 31..24).  Every
// workgroup histograms its range of one query's scores among the keys that
// match the prefix, adds it to hist[q]; the last workgroup to finish picks the
// bin holding the k-th largest key, updates the state and clears hist[q].
__global__ __launch_bounds__(kBfThreads) void k_bf_radix(const float* __restrict__ scores, int64_t ld_scores,
                                                        int N, int digit, int32_t* __restrict__ state,
                                                        uint32_t* __restrict__ hist) {
  const int q = blockIdx.y;
  const float* s = scores + (int64_t)q * ld_scores;
  int32_t* st = state + 8 * q;
  uint32_t* hq = hist + 256 * q;
  __shared__ uint32_t h[256];
  __shared__ uint32_t suf[256];
  __shared__ int last;
  h[threadIdx.x] = 0;
  const uint32_t prefix = (uint32_t)st[0], mask = (uint32_t)st[1];
  const int shift = 24 - 8 * digit;
  __syncthreads();
  const int base = blockIdx.x * kSelBlock;
  // Scores crowd into a few bins (the top digit holds sign and exponent), so
  // each wave adds its lanes bin by bin: one LDS atomic per distinct bin.
  const int lane = threadIdx.x & 63;
#pragma unroll 4
  for (int t = 0; t < kSelPerThread; t++) {
    const int i = base + t * kBfThreads + threadIdx.x;
    int bin = -1;
    if (i < N) {
      const uint32_t k = bf_key(s[i]);
      if ((k & mask) == prefix) bin = (int)((k >> shift) & 255u);
    }
    uint64_t todo = __ballot(bin >= 0);
    while (todo) {
      const int leader = __builtin_ctzll(todo);
      const int lb = __shfl(bin, leader);
      const uint64_t same = __ballot(bin == lb);
      if (lane == leader) atomicAdd(&h[lb], (uint32_t)__popcll(same));
      todo &= ~same;
    }
  }
  __syncthreads();
  // Every value shared between workgroups here is read and written with
  // device-scope atomics, so ordering needs no cache maintenance: each wave
  // waits until its bin additions are performed before the workgroup counts
  // itself done, and the last workgroup reads the bins with atomic loads.
  // (A __threadfence() per workgroup would write back and invalidate the L2
  // thousands of times per pass.)
  if (h[threadIdx.x]) atomicAdd(&hq[threadIdx.x], h[threadIdx.x]);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) last = atomicAdd(&st[5], 1) == (int)gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  // suffix sums over the bins, highest first
  const uint32_t c = __hip_atomic_load(&hq[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  suf[threadIdx.x] = c;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const uint32_t add = threadIdx.x + off < 256 ? suf[threadIdx.x + off] : 0u;
    __syncthreads();
    suf[threadIdx.x] += add;
    __syncthreads();
  }
  const int k_rem = st[2];
  // the bin b with suf[b+1] < k_rem <= suf[b]
  const uint32_t above = threadIdx.x < 255 ? suf[threadIdx.x + 1] : 0u;
  if ((int64_t)above < k_rem && (int64_t)suf[threadIdx.x] >= k_rem) {
    st[0] = (int32_t)(prefix | ((uint32_t)threadIdx.x << shift));
    st[1] = (int32_t)(mask | (255u << shift));
    st[2] = k_rem - (int)above;
    st[3] += (int)above;
    st[4] = (int)c;
  }
  hq[threadIdx.x] = 0u;
  if (threadIdx.x == 0) st[5] = 0;
}

// Common case (exactly k scores >= v_k): every such score's position and
// value go to out[q][0..k) in arbitrary order.  With a straddling tie the
// query is flagged for k_bf_stream instead.
__global__ __launch_bounds__(kBfThreads) void k_bf_collect(const float* __restrict__ scores, int64_t ld_scores,
                                                          int N, int k, int32_t* __restrict__ state,
                                                          int32_t* __restrict__ out_idx, float* __restrict__ out_dist) {
  const int q = blockIdx.y;
  int32_t* st = state + 8 * q;
  const int above = st[3], at = st[4];
  if (above + at != k) {  // tie straddles the k-th place
    if (blockIdx.x == 0 && threadIdx.x == 0) st[7] = 1;
    return;
  }
  const uint32_t kk = (uint32_t)st[0];
  const float* s = scores + (int64_t)q * ld_scores;
  const int base = blockIdx.x * kSelBlock;
  for (int t = 0; t < kSelPerThread; t++) {
    const int i = base + t * kBfThreads + threadIdx.x;
    if (i < N) {
      const float d = s[i];
      if (bf_key(d) >= kk) {
        const int slot = atomicAdd(&st[6], 1);
        if (slot < k) {
          out_idx[(int64_t)q * k + slot] = i;
          out_dist[(int64_t)q * k + slot] = d;
        }
      }
    }
  }
}

// The reference's streaming loop (index.go:84-131) for the flagged queries,
// one wave each.  The k slots live in out[q]; (min, first slot of the min) is
// kept in registers and recomputed after each replacement.  Scores are read
// 64 at a time; a ballot of "score > min" skips the rejected ones.
__device__ __forceinline__ void bf_min_slot(const float* dist, int k, float& mn, int& mi) {
  const int lane = threadIdx.x;
  float m = __builtin_inff();
  int idx = 0x7fffffff;
  for (int j = lane; j < k; j += 64) {
    const float d = dist[j];
    if (d < m) {  // first slot of the minimum within this lane's slots
      m = d;
      idx = j;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float m2 = __shfl_xor(m, o);
    const int i2 = __shfl_xor(idx, o);
    if (m2 < m || (m2 == m && i2 < idx)) {
      m = m2;
      idx = i2;
    }
  }
  mn = m;
  mi = idx;
}

__device__ void bf_stream(const float* __restrict__ s, int N, int k, int32_t* oi, float* od) {
  const int lane = threadIdx.x;
  for (int j = lane; j < k; j += 64) {  // the first k fill the list
    oi[j] = j;
    od[j] = s[j];
  }
  __threadfence_block();
  float mn;
  int mi;
  bf_min_slot(od, k, mn, mi);
  for (int base = k; base < N; base += 64) {
    const int i = base + lane;
    const float d = i < N ? s[i] : -__builtin_inff();
    uint64_t live = __ballot(i < N && d > mn);
    while (live) {
      const int b = __builtin_ctzll(live);
      const float db = __shfl(d, b);
      if (lane == 0) {
        oi[mi] = base + b;
        od[mi] = db;
      }
      __threadfence_block();
      bf_min_slot(od, k, mn, mi);
      live &= ~((2ull << b) - 1ull);  // later lanes only
      live &= __ballot(i < N && d > mn);
    }
  }
}

__global__ __launch_bounds__(64) void k_bf_stream(const float* __restrict__ scores, int64_t ld_scores, int N, int k,
                                                 const int32_t* __restrict__ state, int32_t* __restrict__ out_idx,
                                                 float* __restrict__ out_dist) {
  const int q = blockIdx.x;
  if (state[8 * q + 7] == 0) return;
  bf_stream(scores + (int64_t)q * ld_scores, N, k, out_idx + (int64_t)q * k, out_dist + (int64_t)q * k);
}

// ------------------------------------------------------------- prefiltering --
//
// Scoring every (query, vector) pair in the reference's float32 order costs two
// VALU operations per dimension that no matrix core can do, and the scores are
// then written and re-read by the selection.  For the indexes and batches
// bf_prefilter_ok accepts, the search instead
//   1. k_bf_approx: scores blocks of 64 vectors against up to 64 queries on the
//      fp16 matrix cores and keeps only each block's maximum per query;
//   2. k_bf_blocks: per query, takes a value T that at least k block maxima reach
//      and lists the blocks whose maximum reaches T - 2 eps;
//   3. k_bf_rescore: scores the listed blocks' vectors in the reference's order;
//   4. k_bf_top: selects the exact top k of those scores.
// eps bounds |approximate - reference-order| score for every stored vector
// (bf_prep: fp16 rounding of both operands, the accumulation on either side,
// against the largest stored norm; the operands are the reference's: whole
// groups' codes as they are, the tail's clamped).  At least k vectors have an exact score of
// T - eps or more, so the k-th best exact score v_k is at least that and every
// vector that reaches v_k has an approximate score of at least T - 2 eps: it is
// in a listed block, and the result is the exact top k.  A query for which this
// does not decide -- a tie straddling the k-th place, more than `cap` listed
// blocks, a query that is zero, tiny, huge or not finite, scores that could leave
// float32's normal range (kPfScoreLeast) -- is flagged, and the caller runs it
// through bf_score / bf_select.
// 64 queries x 10^6 x 768 int8, top 10, MI355X: 151 us for step 1 (5.1 TB/s, the
// rate of a large copy) and 76 for the rest, against 2796 for the reference-order
// scores of every pair and 870 for selecting among them.
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

constexpr int kPfBlock = sgk::kBfBlock;  // vectors per block: two 32-row MFMA tiles
// Least and largest product of the query's norm and the largest stored one.  No
// partial sum of the reference's order exceeds it (Cauchy-Schwarz, and roundings
// of under 1e-3 in all), so below 1e37 none is infinite.  What eps leaves out is
// the absolute error of results below float32's normal range, 2^-150 each (2^-126
// were they flushed to zero): at most 2 dim + 48 of them, 5.6e-35, against a
// slack in eps of 2.4e-5 times the product, 2.4e-30 from 1e-25 on.
constexpr float kPfScoreLeast = 1.0e-25f, kPfScoreMost = 1.0e37f;
// Least stored norm.  k_bf_vnorm sums float32 squares, whose absolute error is
// 2^-126 each at most where they underflow: 2.8e-35 over the 2304 dimensions a
// prefiltered index has, 1.4e-5 of a norm of 1e-15 (its user allows for 1e-2).
// Below, a vector of many tiny elements can seem shorter than one of few, and the
// largest norm come out too small.  (Norms past 1.8e19 come out infinite.)
constexpr float kPfNormLeast = 1.0e-15f;
// Threads per workgroup: two column tiles' fragments fill much of the LDS (one
// workgroup per CU); one leaves room for several smaller workgroups, which
// share a short index out more evenly.
template <int CT>
constexpr int kPfThreads = CT == 2 ? 512 : 256;

// 8 stored elements as fp16 (exact for int8; int16 and v * vscale rounded).
template <typename T>
__device__ __forceinline__ half8 pf_half8(const BfRaw<T>& r, float vscale);
template <>
__device__ __forceinline__ half8 pf_half8<int8_t>(const BfRaw<int8_t>& r, float) {
  // c + 128 as the low mantissa bits of 1024: 0x6400 | u is 1024 + u exactly.
  const half2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
  half8 h;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t u = (i ? r.w.y : r.w.x) ^ 0x80808080u;
    const half2_t a = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x05010500u)) - off;
    const half2_t b = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x05030502u)) - off;
    h[4 * i] = a[0];
    h[4 * i + 1] = a[1];
    h[4 * i + 2] = b[0];
    h[4 * i + 3] = b[1];
  }
  return h;
}
template <>
__device__ __forceinline__ half8 pf_half8<int16_t>(const BfRaw<int16_t>& r, float) {
  const uint32_t u[4] = {r.w.x, r.w.y, r.w.z, r.w.w};
  half8 h;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    h[2 * i] = (_Float16)(int16_t)(u[i] & 0xffffu);
    h[2 * i + 1] = (_Float16)(int16_t)(u[i] >> 16);
  }
  return h;
}
template <>
__device__ __forceinline__ half8 pf_half8<float>(const BfRaw<float>& r, float vscale) {
  float v[8];
  r.get(v);
  half8 h;
#pragma unroll
  for (int i = 0; i < 8; i++) h[i] = (_Float16)(v[i] * vscale);
  return h;
}

// Largest L2 norm of the stored vectors in stored units (codes, or floats),
// as float bits folded by atomicMax; +inf when any is not finite.
template <typename T>
__global__ __launch_bounds__(kBfThreads) void k_bf_vnorm(const T* __restrict__ grp, const T* __restrict__ tail, int N,
                                                        int dim, uint32_t* __restrict__ vmax) {
  const int n = blockIdx.x * kBfThreads + threadIdx.x;
  const int nn = min(n, N - 1);
  const int G = dim >> 3, R = dim & 7;
  float ss = 0.0f;
  for (int g = 0; g < G; g += 8) {
    BfRaw<T> raw[8];
#pragma unroll
    for (int u = 0; u < 8; u++) raw[u].load(grp + ((int64_t)min(g + u, G - 1) * N + nn) * 8);
#pragma unroll
    for (int u = 0; u < 8; u++) {
      float v[8], sq = 0.0f;
      raw[u].get(v);
#pragma unroll
      for (int l = 0; l < 8; l++) sq += v[l] * v[l];
      ss += g + u < G ? sq : 0.0f;
    }
  }
  for (int i = 0; i < R; i++) {
    float t = (float)tail[(int64_t)nn * R + i];
    if constexpr (BfElem<T>::kQuant) t = t * BfElem<T>::inv();
    ss += t * t;
  }
  float m = sqrtf(ss);
  if (!(m <= 3.0e38f)) m = __builtin_inff();
  // One atomic per workgroup, and only if it would raise the maximum: on one
  // address they go one after another, 13 ns each (one per wave: 25 us for
  // 100,000 x 256 int16, 11 us now).
  __shared__ float red[kBfThreads / 64];
  m = sg_wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 1; i < kBfThreads / 64; i++) m = fmaxf(m, red[i]);
    const uint32_t u = __float_as_uint(m);
    if (u > __hip_atomic_load(vmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(vmax, u);
  }
}

// Queries of one pass: normalized in place when asked (builder.go:131-141, as
// k_bf_normalize), then scaled by a power of two to a largest element in
// [256, 512) and rounded to fp16 in the MFMA B operand's order, qfrag [k-step
// of two 8-element groups][col_tiles][64 lanes][8] (lane 32 h + c: query c of
// the tile, group 2 s + h; the last k-step's first half holds the tail when
// dim % 8; zeros elsewhere and for queries past nq).  eps[2 q] = the bound above
// in k_bf_approx's units, eps[2 q + 1] what takes these to scores.
// A workgroup per query: one wave took 19 us for 64 queries of 768 dims, four 13.
constexpr int kPrepThreads = 256;
__global__ __launch_bounds__(kPrepThreads) void k_bf_prep(float* __restrict__ queries, int nq, int dim, int normalize,
                                               float vnorm_s, float vunit, int exact_v, int col_tiles, _Float16* __restrict__ qfrag,
                                               float* __restrict__ eps, int32_t* __restrict__ flags) {
  extern __shared__ __attribute__((aligned(16))) float buf[];  // dim rounded up to 16, floats then doubles
  __shared__ float norm;
  __shared__ int scale;
  __shared__ float red[2][kPrepThreads / 64];
  __shared__ int bad;
  const int q = blockIdx.x, tid = threadIdx.x, wave = tid >> 6;
  const bool live = q < nq;
  const int dimp = (dim + 15) & ~15;
  float* x = queries + (int64_t)q * dim;
  double* sqs = reinterpret_cast<double*>(buf + dimp);
  if (tid == 0) bad = 0;
  for (int i = tid; i < dimp; i += kPrepThreads) {
    const float v = live && i < dim ? x[i] : 0.0f;
    const float sq = v * v;
    buf[i] = v;
    sqs[i] = (double)sq;
  }
  __syncthreads();
  if (normalize && live) {
    if (tid == 0) {
      // The float64 sum in index order (the pad's zeros add nothing): a chain of
      // additions, the next 16 squares read under the current 16.
      double sum = 0.0;
      double2 cur[8], nxt[8];
#pragma unroll
      for (int u = 0; u < 8; u++) cur[u] = reinterpret_cast<const double2*>(sqs)[u];
      for (int i = 0; i < dimp; i += 16) {
        const int j = min(i + 16, dimp - 16);
#pragma unroll
        for (int u = 0; u < 8; u++) nxt[u] = reinterpret_cast<const double2*>(sqs + j)[u];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; u++) {
          sum += cur[u].x;
          sum += cur[u].y;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) cur[u] = nxt[u];
      }
      scale = sum != 0.0;  // a zero vector stays as it is
      norm = sum != 0.0 ? (float)(1.0 / sqrt(sum)) : 1.0f;
    }
    __syncthreads();
    const float n = norm;
    if (scale)
      for (int i = tid; i < dim; i += kPrepThreads) {
        buf[i] = buf[i] * n;
        x[i] = buf[i];
      }
    __syncthreads();
  }
  float m = 0.0f, ss = 0.0f;
  bool finite = true;
  for (int i = tid; i < dim; i += kPrepThreads) {
    const float a = fabsf(buf[i]);
    finite = finite && a <= 1.0e30f;
    m = fmaxf(m, a);
  }
  if (!finite) bad = 1;
  m = sg_wave_max(m);
  if ((tid & 63) == 0) red[0][wave] = m;
  __syncthreads();
  finite = bad == 0;
#pragma unroll
  for (int i = 0; i < kPrepThreads / 64; i++) m = fmaxf(m, red[0][i]);
  const bool ok = live && finite && m >= 1.0e-30f;
  int e = 0;
  if (ok) (void)frexpf(m, &e);  // m = f * 2^e, f in [0.5, 1)
  const float sc = ok ? ldexpf(1.0f, 9 - e) : 0.0f;
  for (int i = tid; i < dim; i += kPrepThreads) {
    const float t = buf[i] * sc;
    ss += t * t;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  if ((tid & 63) == 0) red[1][wave] = ss;
  __syncthreads();
  if (tid == 0 && live) {
    ss = 0.0f;
#pragma unroll
    for (int i = 0; i < kPrepThreads / 64; i++) ss += red[1][i];
    // Per product: fp16 rounding of x (2^-11) and of v unless exact; the two
    // accumulations: at most dim + 32 float32 roundings of up to an ulp (2^-23)
    // each on the matrix cores, dim / 8 + 24 (2^-24) in the reference's order;
    // sums of |x v| bounded by the norms' product (Cauchy-Schwarz).  fp16
    // subnormals: 2^-25 per element on either side.
    const float xn = sqrtf(ss) * 1.001f;
    const float rel = 4.8829e-4f * (exact_v ? 1.0f : 2.0f) + (float)(dim + 32) * 1.2e-7f +
                      (float)(dim / 8 + 24) * 6.0e-8f + 1.0e-6f;
    const float rd = sqrtf((float)dim) * 3.0e-8f;
    const float unit = (1.0f / sc) * (1.0f / vunit);  // k_bf_approx's units to scores
    const float most = xn * vnorm_s * unit;  // bounds |score|; 0 or infinite where unit leaves the range
    eps[2 * q] = 1.05f * (rel * xn * vnorm_s + rd * (xn + vnorm_s));
    eps[2 * q + 1] = unit;
    flags[q] = ok && most >= kPfScoreLeast && most <= kPfScoreMost ? 0 : sgk::kBfUnfit;
  }
  const int G = dim >> 3, R = dim & 7, ct = q >> 5, c = q & 31;
  const int ks_main = (G + 1) >> 1, ks = ks_main + (R ? 1 : 0);
  for (int i = tid; i < ks * 2; i += kPrepThreads) {  // one 8-element piece per thread
    const int s = i >> 1, h = i & 1;
    int src = -1, cnt = 8;
    if (s < ks_main) {
      if (2 * s + h < G) src = 8 * (2 * s + h);
    } else if (h == 0) {
      src = 8 * G;
      cnt = R;
    }
    half8 v;
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = src >= 0 && u < cnt ? (_Float16)(buf[src + u] * sc) : (_Float16)0.0f;
    *reinterpret_cast<half8*>(qfrag + (((int64_t)s * col_tiles + ct) * 64 + 32 * h + c) * 8) = v;
  }
}

// blockmax[q][nb]: the largest approximate score of each block's 64 vectors,
// in scaled units.  Bound by reading the index once per pass (HBM): the fp16
// MFMAs of 64 queries take about a third of that time.  A wave walks blocks
// b, b + waves, ... with PF k-steps of loads in flight (the ring runs on from
// block to block); lane (row, h) of a 32-row tile loads group 2 s + h of its
// vector: 8, 16 or 32 contiguous bytes, 32 vectors side by side.  The queries'
// fragments sit in LDS.
template <typename T, int CT, int PF>
__global__ __launch_bounds__(kPfThreads<CT>, 2) void k_bf_approx(const T* __restrict__ grp, const T* __restrict__ tail,
                                                            int N, int dim, float vscale,
                                                            const _Float16* __restrict__ qfrag, int nq,
                                                            float* __restrict__ blockmax, int nb) {
  extern __shared__ __attribute__((aligned(16))) _Float16 qs[];  // [ks][CT][64][8]
  const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = dim >> 3, R = dim & 7;
  const int ks_main = (G + 1) >> 1, ks = ks_main + (R ? 1 : 0);
  for (int i = threadIdx.x; i < ks * CT * 64; i += kPfThreads<CT>)
    reinterpret_cast<uint4*>(qs)[i] = reinterpret_cast<const uint4*>(qfrag)[i];
  __syncthreads();
  const int nwaves = gridDim.x * (kPfThreads<CT> / 64);
  const int b0 = blockIdx.x * (kPfThreads<CT> / 64) + wave;
  if (b0 >= nb) return;
  const int nblk = (nb - b0 + nwaves - 1) / nwaves;  // this wave's blocks
  const int64_t steps = (int64_t)nblk * ks_main;

  // Load stream: block lb, k-step ls (past the last step the last one again).
  int lb = b0, ls = 0;
  auto fetch = [&](BfRaw<T>(&r)[2]) {
    const int64_t g = min(2 * ls + lh, G - 1);
#pragma unroll
    for (int t = 0; t < 2; t++)
      r[t].load(grp + (g * N + min(lb * kPfBlock + 32 * t + lr, N - 1)) * 8);
    if (ls + 1 < ks_main) {
      ls++;
    } else if (lb + nwaves < nb) {
      ls = 0;
      lb += nwaves;
    }
  };
  BfRaw<T> ring[PF][2];
#pragma unroll
  for (int i = 0; i < PF; i++) fetch(ring[i]);

  f32x16_t acc[2][CT];
  auto clear = [&]() {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int c = 0; c < CT; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][c][r] = 0.0f;
  };
  auto mul = [&](int s, const half8 (&a)[2]) {
#pragma unroll
    for (int c = 0; c < CT; c++) {
      const half8 b = *reinterpret_cast<const half8*>(qs + ((s * CT + c) * 64 + lane) * 8);
#pragma unroll
      for (int t = 0; t < 2; t++) acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t], b, acc[t][c], 0, 0, 0);
    }
  };
  clear();
  int b = b0, s = 0;
  for (int64_t st = 0; st < steps; st += PF) {
#pragma unroll
    for (int i = 0; i < PF; i++) {
      if (st + i < steps) {
        half8 a[2];
#pragma unroll
        for (int t = 0; t < 2; t++) a[t] = pf_half8<T>(ring[i][t], vscale);
        fetch(ring[i]);
        __builtin_amdgcn_sched_barrier(0);
        mul(s, a);
        if (++s == ks_main) {  // wave-uniform: the block is complete
          if (R) {
            half8 tl[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
              const T* tp = tail + (int64_t)min(b * kPfBlock + 32 * t + lr, N - 1) * R;
#pragma unroll
              for (int u = 0; u < 8; u++) {
                float v = u < R ? (float)tp[min(u, R - 1)] : 0.0f;
                if constexpr (BfElem<T>::kQuant)
                  v = fmaxf(v, (float)BfElem<T>::kLo);  // bf_lut's clamp
                else
                  v = v * vscale;
                tl[t][u] = lh == 0 ? (_Float16)v : (_Float16)0.0f;
              }
            }
            mul(ks_main, tl);
          }
#pragma unroll
          for (int c = 0; c < CT; c++) {
            float m = acc[0][c][0];
#pragma unroll
            for (int r = 0; r < 16; r++) m = fmaxf(m, fmaxf(acc[0][c][r], acc[1][c][r]));
            m = fmaxf(m, __shfl_xor(m, 32));
            const int q = 32 * c + lr;
            if (lh == 0 && q < nq) blockmax[(int64_t)q * nb + b] = m;
          }
          clear();
          s = 0;
          b += nwaves;
        }
      }
    }
  }
}

// The value T of a workgroup's radix select over the keys that visit(f) hands to
// f(valid, key), a whole wave at a time: the k-th largest key's top 11 bits a
// pass (10 in the third) with the rest zero; above = keys above T's bin, at =
// keys in it.  hist: 2048 + 64 words of LDS.  Every thread of the workgroup calls
// this.
constexpr int kTopThreads = 1024;
template <int PASSES, typename F>
__device__ __forceinline__ void wg_select(F visit, int k, uint32_t* hist, uint32_t& T, int& above, int& at) {
  __shared__ uint32_t sh_prefix;
  __shared__ int sh_above, sh_at;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t prefix = 0;
  int gone = 0, in_bin = 0;
#pragma unroll
  for (int p = 0; p < PASSES; p++) {
    const int bits = p < 2 ? 11 : 10, shift = p == 0 ? 21 : p == 1 ? 10 : 0;
    const uint32_t mask = p == 0 ? 0u : ~0u << (p == 1 ? 21 : 10);
    for (int i = tid; i < 2048; i += kTopThreads) hist[i] = 0;
    __syncthreads();
    visit([&](bool valid, uint32_t u) {
      int bin = -1;
      if (valid && (u & mask) == prefix) bin = (int)((u >> shift) & ((1u << bits) - 1u));
      // Scores crowd into a few bins of the top digit: one addition per
      // distinct bin of the wave there.
      if (p == 0) {
        uint64_t todo = __ballot(bin >= 0);
        while (todo) {
          const int lb = __shfl(bin, __builtin_ctzll(todo));
          const uint64_t same = __ballot(bin == lb);
          if (lane == 0) atomicAdd(&hist[lb], (uint32_t)__popcll(same));
          todo &= ~same;
        }
      } else if (bin >= 0) {
        atomicAdd(&hist[bin], 1u);
      }
    });
    __syncthreads();
    // Suffix counts: thread t owns bins 2t, 2t + 1.
    uint32_t* wsum = hist + 2048;
    const uint32_t c0 = hist[2 * tid], c1 = hist[2 * tid + 1];
    uint32_t run = c0 + c1;  // inclusive suffix over the wave's lanes >= this one
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t v = __shfl_down(run, o);
      if (lane + o < 64) run += v;
    }
    if (lane == 0) wsum[wave] = run;
    __syncthreads();
    uint32_t after = run - c0 - c1;
    for (int w2 = wave + 1; w2 < kTopThreads / 64; w2++) after += wsum[w2];
    const uint32_t need = (uint32_t)(k - gone);
    // bin b with (keys in higher bins) < need <= (those + its own)
    if (after < need && need <= after + c1) {
      sh_prefix = prefix | ((uint32_t)(2 * tid + 1) << shift);
      sh_above = gone + (int)after;
      sh_at = (int)c1;
    } else if (after + c1 < need && need <= after + c1 + c0) {
      sh_prefix = prefix | ((uint32_t)(2 * tid) << shift);
      sh_above = gone + (int)(after + c1);
      sh_at = (int)c0;
    }
    __syncthreads();
    prefix = sh_prefix;
    gone = sh_above;
    in_bin = sh_at;
    __syncthreads();
  }
  T = prefix;
  above = gone;
  at = in_bin;
}

// visit of n keys key(i), i < n, the loads of B of a thread's keys in flight
// together (a workgroup alone on its CU waits for each of them otherwise; where a
// thread has few keys, the loads past the last one cost more than that).
constexpr int kKeyBatch = 8;
template <int B, typename K>
__device__ __forceinline__ auto each_key(K key, int n) {
  return [=](auto f) {
    for (int i0 = 0; i0 < n; i0 += B * kTopThreads) {
      uint32_t u[B];
#pragma unroll
      for (int b = 0; b < B; b++) u[b] = key(min(i0 + b * kTopThreads + (int)threadIdx.x, n - 1));
#pragma unroll
      for (int b = 0; b < B; b++) {
        if (i0 + b * kTopThreads >= n) break;  // workgroup-uniform
        f(i0 + b * kTopThreads + (int)threadIdx.x < n, u[b]);
      }
    }
  };
}

// The float whose bf_key is u.
__device__ __forceinline__ float bf_unkey(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? u & 0x7fffffffu : ~u);
}

// list[q][0 .. count[q]): the blocks that can hold one of query q's k best.
// Leaves in eps[2 q] the score T - 2 eps, which each of the k best reaches.
__global__ __launch_bounds__(kTopThreads) void k_bf_blocks(const float* __restrict__ blockmax, int nb, int k,
                                                          float* __restrict__ eps, int cap,
                                                          int32_t* __restrict__ list, int32_t* __restrict__ count,
                                                          int32_t* __restrict__ flags) {
  __shared__ uint32_t hist[2048 + 64];
  __shared__ int cnt;
  const int q = blockIdx.x;
  const float* bm = blockmax + (int64_t)q * nb;
  if (flags[q]) {  // workgroup-uniform
    if (threadIdx.x == 0) count[q] = 0;
    return;
  }
  uint32_t T;
  int above, at;
  // The k-th largest maximum of four blocks each: at least k blocks reach it,
  // for a quarter of the keys.  Its low bits are zero, and the cut's own
  // rounding is covered by eps' slack.
  wg_select<2>(
      each_key<1>(
          [=](int i) {
            float m = bm[4 * i];
#pragma unroll
            for (int u = 1; u < 4; u++) m = fmaxf(m, bm[min(4 * i + u, nb - 1)]);
            return bf_key(m);
          },
          (nb + 3) / 4),
      k, hist, T, above, at);
  const float cut = bf_unkey(T) - 2.0f * eps[2 * q];
  if (threadIdx.x == 0) cnt = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += kTopThreads)
    if (bm[i] >= cut) {
      const int slot = atomicAdd(&cnt, 1);
      if (slot < cap) list[(int64_t)q * cap + slot] = i;
    }
  __syncthreads();
  if (threadIdx.x == 0) {
    eps[2 * q] = cut * eps[2 * q + 1];
    count[q] = cnt <= cap ? cnt : 0;
    if (cnt > cap) flags[q] = sgk::kBfOpen;
  }
}

// Half a stored group: four elements as loaded, and as the AVX2 loop's operands.
template <typename T>
struct BfHalf;
template <>
struct BfHalf<int8_t> {
  uint32_t w;
  __device__ void load(const int8_t* p) { w = *reinterpret_cast<const uint32_t*>(p); }
  __device__ void get(float (&v)[4]) const {
#pragma unroll
    for (int l = 0; l < 4; l++) v[l] = (float)(int8_t)(w >> (8 * l)) * BfElem<int8_t>::inv();
  }
};
template <>
struct BfHalf<int16_t> {
  uint2 w;
  __device__ void load(const int16_t* p) { w = *reinterpret_cast<const uint2*>(p); }
  __device__ void get(float (&v)[4]) const {
    v[0] = (float)(int16_t)(w.x & 0xffffu) * BfElem<int16_t>::inv();
    v[1] = (float)(int16_t)(w.x >> 16) * BfElem<int16_t>::inv();
    v[2] = (float)(int16_t)(w.y & 0xffffu) * BfElem<int16_t>::inv();
    v[3] = (float)(int16_t)(w.y >> 16) * BfElem<int16_t>::inv();
  }
};
template <>
struct BfHalf<float> {
  float4 w;
  __device__ void load(const float* p) { w = *reinterpret_cast<const float4*>(p); }
  __device__ void get(float (&v)[4]) const {
    v[0] = w.x; v[1] = w.y; v[2] = w.z; v[3] = w.w;
  }
};

// cand[q][64 i + l]: the score of vector 64 list[q][i] + l in the reference's
// order (k_bf_score's arithmetic).  Bound by memory latency: a few dozen blocks
// per query.  So a wave takes half a block, two lanes a vector -- lane 2 v + h
// keeps the lane sums 4 h .. 4 h + 3 of vector v -- with B groups in flight and
// the next B behind them; a workgroup takes two blocks and holds its query in
// LDS.  (A lane per vector with 8 to 16 groups in flight: 14 us for one query
// over float32 x 512, 32 for 64 over int8 x 768; 7.5 and 22 now.)  Vectors past N: NaN
// bits 0xffffffff, whose key is 0.
template <typename T>
__global__ __launch_bounds__(kBfThreads) void k_bf_rescore(const T* __restrict__ grp, const T* __restrict__ tail, int N,
                                                          int dim, const float* __restrict__ queries,
                                                          const int32_t* __restrict__ list,
                                                          const int32_t* __restrict__ count, int cap,
                                                          float* __restrict__ cand) {
  constexpr int B = sizeof(T) == 4 ? 16 : 32;  // half groups in flight per lane
  extern __shared__ __attribute__((aligned(16))) float xs[];  // the query's whole groups
  const int q = blockIdx.y, lane = threadIdx.x & 63, h = lane & 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // The wave's entry is read along with the count (cap is even: in bounds); a
  // second block past the list repeats the first one.
  const int i0 = blockIdx.x * (kBfThreads / 128);
  const int e0 = list[(int64_t)q * cap + i0], e1 = list[(int64_t)q * cap + i0 + 1];
  const int n_list = count[q];
  if (i0 >= n_list) return;  // workgroup-uniform
  const bool second = (wave >> 1) && i0 + 1 < n_list;
  const int i = i0 + (second ? 1 : 0);
  const int l = 32 * (wave & 1) + (lane >> 1);  // vector of the block
  const int n = (second ? e1 : e0) * kPfBlock + l;
  const int nn = min(n, N - 1);
  const int G = dim >> 3, R = dim & 7;
  const float* x = queries + (int64_t)q * dim;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const T* gp = grp + (int64_t)nn * 8 + 4 * h;
  const int64_t gs = (int64_t)N * 8;
  // No branch between a load and its use: it would sink the loads.
  BfHalf<T> cur[B], nxt[B];
#pragma unroll
  for (int u = 0; u < B; u++) cur[u].load(gp + min(u, G - 1) * gs);
  for (int e = threadIdx.x; e < 8 * G; e += kBfThreads) xs[e] = x[e];
  __syncthreads();
  auto add = [&](const BfHalf<T>& raw, int g) {
    float v[4];
    raw.get(v);
    const float4 xv4 = *reinterpret_cast<const float4*>(xs + 8 * g + 4 * h);
    const float xv[4] = {xv4.x, xv4.y, xv4.z, xv4.w};
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if constexpr (BfElem<T>::kQuant) {
        const float p = v[t] * xv[t];
        acc[t] = acc[t] + p;
      } else {
        acc[t] = __builtin_fmaf(v[t], xv[t], acc[t]);
      }
    }
  };
  int g = 0;
  for (; g + B <= G; g += B) {
#pragma unroll
    for (int u = 0; u < B; u++) nxt[u].load(gp + min(g + B + u, G - 1) * gs);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < B; u++) add(cur[u], g + u);
#pragma unroll
    for (int u = 0; u < B; u++) cur[u] = nxt[u];
  }
#pragma unroll
  for (int u = 0; u < B; u++)
    if (g + u < G) add(cur[u], g + u);
  float s8[8];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const float o = __shfl_xor(acc[t], 1);
    s8[t] = h ? o : acc[t];
    s8[4 + t] = h ? acc[t] : o;
  }
  const float sum = bf_finish<T>(s8, G, R, x + 8 * G, tail + (int64_t)nn * R);
  if (h == 0) cand[((int64_t)q * cap + i) * kPfBlock + l] = n < N ? sum : __uint_as_float(0xffffffffu);
}

// The exact top k of the candidates: out_idx/out_dist [q][k] in arbitrary
// order; a tie straddling the k-th place flags the query.  The candidates that
// reach cut[2 q] (at least k of them: k_bf_blocks) are few as a rule: gathered in
// LDS, each is ranked against the others.  (With k or more of them the k best are
// among them whatever the cut.)  Three radix passes over all
// candidates, a chain of barriers, took 9.6 us for one query of 150,000 vectors, 5.0 now; they are
// left for more than kTopRank of them.  Bound by the latency of a workgroup's
// reads, so kKeyBatch of a thread's go out together (one at a time, a query for
// 1000 of 10^6 x 768 int8: 574 us a search, 338 now), and what is below the cut
// shares one bin.
constexpr int kTopRank = kTopThreads, kTopAhead = 2;
__global__ __launch_bounds__(kTopThreads) void k_bf_top(const float* __restrict__ cand,
                                                       const int32_t* __restrict__ list,
                                                       const int32_t* __restrict__ count, int cap, int k,
                                                       const float* __restrict__ cut, int32_t* __restrict__ out_idx,
                                                       float* __restrict__ out_dist, int32_t* __restrict__ flags) {
  __shared__ uint32_t hist[2048 + 64];
  __shared__ __attribute__((aligned(16))) uint32_t keys[kTopRank];
  __shared__ float score[kTopRank];
  __shared__ int from[kTopRank];
  __shared__ int cnt, tie;
  const int q = blockIdx.x;
  // The first candidates are read along with their number (the buffer holds at
  // least 68 blocks per query).
  static_assert(sgk::bf_prefilter_cap(1) * kPfBlock >= kTopAhead * kTopThreads, "reads ahead in bounds");
  float ahead[kTopAhead];
  int block[kTopAhead];
#pragma unroll
  for (int u = 0; u < kTopAhead; u++) {
    const int i = threadIdx.x + u * kTopThreads;
    ahead[u] = cand[(int64_t)q * cap * kPfBlock + i];
    block[u] = list[(int64_t)q * cap + i / kPfBlock];
  }
  const int n = count[q] * kPfBlock;
  if (flags[q] || n < k) {
    if (threadIdx.x == 0 && flags[q] == 0) flags[q] = sgk::kBfOpen;
    return;
  }
  const float* cs = cand + (int64_t)q * cap * kPfBlock;
  if (threadIdx.x == 0) cnt = tie = 0;
  keys[threadIdx.x] = 0u;  // below every score's key
  __syncthreads();
  const float least = cut[2 * q];
  auto take = [&](float d, int at) {
    if (d >= least) {  // not the NaN past the last vector
      const int slot = atomicAdd(&cnt, 1);
      if (slot < kTopRank) {
        keys[slot] = bf_key(d);
        score[slot] = d;
        from[slot] = at;
      }
    }
  };
#pragma unroll
  for (int u = 0; u < kTopAhead; u++) {
    const int i = threadIdx.x + u * kTopThreads;
    if (i < n) take(ahead[u], block[u] * kPfBlock + i % kPfBlock);
  }
  for (int i0 = threadIdx.x + kTopAhead * kTopThreads; i0 < n; i0 += kKeyBatch * kTopThreads) {
    float d[kKeyBatch];
#pragma unroll
    for (int b = 0; b < kKeyBatch; b++) d[b] = cs[min(i0 + b * kTopThreads, n - 1)];
#pragma unroll
    for (int b = 0; b < kKeyBatch; b++) {
      const int i = i0 + b * kTopThreads;
      if (i < n && d[b] >= least) take(d[b], list[(int64_t)q * cap + i / kPfBlock] * kPfBlock + i % kPfBlock);
    }
  }
  __syncthreads();
  const int m = cnt;
  if (m >= k && m <= kTopRank) {
    if ((int)threadIdx.x < m) {
      const uint32_t u = keys[threadIdx.x];
      int gt = 0, eq = 0, before = 0;
      for (int j = 0; j < m; j += 4) {
        const uint4 o4 = *reinterpret_cast<const uint4*>(&keys[j]);
        const uint32_t o[4] = {o4.x, o4.y, o4.z, o4.w};
#pragma unroll
        for (int t = 0; t < 4; t++) {
          gt += o[t] > u;
          eq += o[t] == u;
          before += o[t] == u && j + t < (int)threadIdx.x;
        }
      }
      if (gt < k) {
        if (gt + eq > k) {
          tie = 1;
        } else {
          out_idx[(int64_t)q * k + gt + before] = from[threadIdx.x];
          out_dist[(int64_t)q * k + gt + before] = score[threadIdx.x];
        }
      }
    }
    __syncthreads();
    if (threadIdx.x == 0 && tie) flags[q] = sgk::kBfOpen;
    return;
  }
  // Below the cut: key 0, as past the last vector (one addition to one bin).
  const float low = m >= k ? least : -__builtin_inff();
  auto key = [=](float d) { return d >= low ? bf_key(d) : 0u; };
  uint32_t T;
  int above, at;
  wg_select<3>(each_key<kKeyBatch>([=](int i) { return key(cs[i]); }, n), k, hist, T, above, at);
  if (above + at != k) {
    if (threadIdx.x == 0) flags[q] = sgk::kBfOpen;
    return;
  }
  if (threadIdx.x == 0) cnt = 0;
  __syncthreads();
  for (int i0 = threadIdx.x; i0 < n; i0 += kKeyBatch * kTopThreads) {
    float d[kKeyBatch];
#pragma unroll
    for (int b = 0; b < kKeyBatch; b++) d[b] = cs[min(i0 + b * kTopThreads, n - 1)];
#pragma unroll
    for (int b = 0; b < kKeyBatch; b++) {
      const int i = i0 + b * kTopThreads;
      if (i < n && key(d[b]) >= T) {
        const int slot = atomicAdd(&cnt, 1);
        if (slot < k) {
          out_idx[(int64_t)q * k + slot] = list[(int64_t)q * cap + i / kPfBlock] * kPfBlock + i % kPfBlock;
          out_dist[(int64_t)q * k + slot] = d[b];
        }
      }
    }
  }
}

// The whole selection over N <= R * 1024 scores in one launch, a workgroup per
// query with its keys in registers: the radix select, then the scores >= v_k, or
// (a straddling tie) the first wave's replay of the streaming loop.  The
// general path is ten launches, four of them grid-wide passes: a
// query over 2000 x 256 int8 took 91 us with it, 40 with this; 4 over 10,000 x 512
// 147 and 71; 8 over 30,000 x 256 (k = 100) 174 and 137.  From about 45,000 (64 queries:
// 440 and 457) the grid-wide passes are the faster ones.
constexpr int kSelMost = 32;  // keys per thread of the largest instance
template <int R>
__global__ __launch_bounds__(kTopThreads) void k_bf_select_wg(const float* __restrict__ scores, int64_t ld_scores, int N,
                                                             int k, int32_t* __restrict__ out_idx,
                                                             float* __restrict__ out_dist) {
  __shared__ uint32_t hist[2048 + 64];
  __shared__ int cnt;
  const int q = blockIdx.x, tid = threadIdx.x;
  const float* s = scores + (int64_t)q * ld_scores;
  int32_t* oi = out_idx + (int64_t)q * k;
  float* od = out_dist + (int64_t)q * k;
  float d[R];
#pragma unroll
  for (int u = 0; u < R; u++) d[u] = s[min(u * kTopThreads + tid, N - 1)];
  if (tid == 0) cnt = 0;
  uint32_t T;
  int above, at;
  wg_select<3>(
      [&](auto f) {
#pragma unroll
        for (int u = 0; u < R; u++) f(u * kTopThreads + tid < N, bf_key(d[u]));
      },
      k, hist, T, above, at);
  if (above + at != k) {  // a tie straddles the k-th place (workgroup-uniform)
    if (tid < 64) bf_stream(s, N, k, oi, od);
    return;
  }
#pragma unroll
  for (int u = 0; u < R; u++) {
    const int i = u * kTopThreads + tid;
    if (i < N && bf_key(d[u]) >= T) {
      const int slot = atomicAdd(&cnt, 1);
      if (slot < k) {
        oi[slot] = i;
        od[slot] = d[u];
      }
    }
  }
}

__global__ void k_bf_fill_i32(int32_t* p, int64_t n, int32_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// state initial values: prefix 0, mask 0, k_rem k, above 0, at 0, 0, 0, 0.
__global__ void k_bf_state_init(int32_t* state, int nq, int k) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nq * 8) state[i] = (i & 7) == 2 ? k : 0;
}

unsigned nblocks(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

template <typename T>
hipError_t score_t(const void* grp, const void* tail, int N, int dim, const float* queries, int nq, float* scores,
                   int64_t ld, hipStream_t s) {
  const T* g = static_cast<const T*>(grp);
  const T* t = static_cast<const T*>(tail);
  const unsigned nb = nblocks(N, kBfThreads);
  // Queries per lane: 8 use a loaded vector best.  A launch of few workgroups is
  // bound by one workgroup's time instead (a vector's loads and sums in a row),
  // so there the queries go to as many workgroups as two a CU (the sums are
  // the same).  With the selection in one launch below: 16 queries over 3000 x 768
  // int8 168 -> 70 us, 32 over 13,000 x 300 182 -> 92.
  int most = 8;
  while (most > 1 && (int64_t)nb * ((nq + most - 1) / most) < 512) most /= 2;
  if (most < 8 && (int64_t)nb * ((nq + most - 1) / most) > 512) most *= 2;
  for (int q0 = 0; q0 < nq;) {
    const int left = nq - q0;
    int qb = most;
    while (qb > left) qb /= 2;
    const int groups = left / qb < 65535 ? left / qb : 65535;
    const auto f = qb == 8 ? k_bf_score<T, 8> : qb == 4 ? k_bf_score<T, 4> : qb == 2 ? k_bf_score<T, 2> : k_bf_score<T, 1>;
    hipLaunchKernelGGL(f, dim3(nb, groups), dim3(kBfThreads), 0, s, g, t, N, dim, queries, q0, nq, scores, ld);
    q0 += qb * groups;
  }
  return hipGetLastError();
}

}  // namespace

namespace sgk {

hipError_t bf_build(int mode, const float* src, int64_t ld, int n, int dim, int row0, int N, void* grp, void* tail,
                    bool normalize, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const unsigned nb = nblocks(n, kBuildRows);
  const int nz = normalize ? 1 : 0;
  switch (mode) {
    case kBfF32:
      hipLaunchKernelGGL(k_bf_build<float>, dim3(nb), dim3(kBfThreads), 0, s, src, ld, n, dim, row0, N,
                         static_cast<float*>(grp), static_cast<float*>(tail), nz);
      break;
    case kBfI8:
      hipLaunchKernelGGL(k_bf_build<int8_t>, dim3(nb), dim3(kBfThreads), 0, s, src, ld, n, dim, row0, N,
                         static_cast<int8_t*>(grp), static_cast<int8_t*>(tail), nz);
      break;
    case kBfI16:
      hipLaunchKernelGGL(k_bf_build<int16_t>, dim3(nb), dim3(kBfThreads), 0, s, src, ld, n, dim, row0, N,
                         static_cast<int16_t*>(grp), static_cast<int16_t*>(tail), nz);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t bf_normalize(float* x, int n, int dim, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_bf_normalize, dim3(n), dim3(64), 0, s, x, dim);
  return hipGetLastError();
}

hipError_t bf_relayout(int mode, const void* rows, int n, int dim, int row0, int N, void* grp, void* tail,
                       hipStream_t s) {
  const int64_t ne = (int64_t)n * dim;
  if (ne <= 0) return hipSuccess;
  const unsigned nb = nblocks(ne, 256);
  switch (mode) {
    case kBfF32:
      hipLaunchKernelGGL(k_bf_relayout<float>, dim3(nb), dim3(256), 0, s, static_cast<const float*>(rows), ne, dim,
                         row0, N, static_cast<float*>(grp), static_cast<float*>(tail));
      break;
    case kBfI8:
      hipLaunchKernelGGL(k_bf_relayout<int8_t>, dim3(nb), dim3(256), 0, s, static_cast<const int8_t*>(rows), ne,
                         dim, row0, N, static_cast<int8_t*>(grp), static_cast<int8_t*>(tail));
      break;
    case kBfI16:
      hipLaunchKernelGGL(k_bf_relayout<int16_t>, dim3(nb), dim3(256), 0, s, static_cast<const int16_t*>(rows), ne,
                         dim, row0, N, static_cast<int16_t*>(grp), static_cast<int16_t*>(tail));
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t bf_unpack(int mode, const void* grp, const void* tail, int row0, int n, int dim, int N, void* rows,
                     hipStream_t s) {
  const int64_t ne = (int64_t)n * dim;
  if (ne <= 0) return hipSuccess;
  const unsigned nb = nblocks(ne, 256);
  switch (mode) {
    case kBfF32:
      hipLaunchKernelGGL(k_bf_unpack<float>, dim3(nb), dim3(256), 0, s, static_cast<const float*>(grp),
                         static_cast<const float*>(tail), ne, dim, row0, N, static_cast<float*>(rows));
      break;
    case kBfI8:
      hipLaunchKernelGGL(k_bf_unpack<int8_t>, dim3(nb), dim3(256), 0, s, static_cast<const int8_t*>(grp),
                         static_cast<const int8_t*>(tail), ne, dim, row0, N, static_cast<int8_t*>(rows));
      break;
    case kBfI16:
      hipLaunchKernelGGL(k_bf_unpack<int16_t>, dim3(nb), dim3(256), 0, s, static_cast<const int16_t*>(grp),
                         static_cast<const int16_t*>(tail), ne, dim, row0, N, static_cast<int16_t*>(rows));
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t bf_score(int mode, const void* grp, const void* tail, int N, int dim, const float* queries, int nq,
                    float* scores, int64_t ld_scores, hipStream_t s) {
  if (N <= 0 || nq <= 0) return hipSuccess;
  switch (mode) {
    case kBfF32: return score_t<float>(grp, tail, N, dim, queries, nq, scores, ld_scores, s);
    case kBfI8: return score_t<int8_t>(grp, tail, N, dim, queries, nq, scores, ld_scores, s);
    case kBfI16: return score_t<int16_t>(grp, tail, N, dim, queries, nq, scores, ld_scores, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t bf_select(const float* scores, int64_t ld_scores, int N, int nq, int k, int32_t* state, uint32_t* hist,
                     int32_t* out_idx, float* out_dist, hipStream_t s) {
  if (N <= 0 || nq <= 0 || k <= 0) return hipSuccess;
  if (k > N) return hipErrorInvalidValue;
  if (N <= kSelMost * kTopThreads) {
    const auto f = N <= 4 * kTopThreads    ? k_bf_select_wg<4>
                   : N <= 16 * kTopThreads ? k_bf_select_wg<16>
                                           : k_bf_select_wg<kSelMost>;
    hipLaunchKernelGGL(f, dim3(nq), dim3(kTopThreads), 0, s, scores, ld_scores, N, k, out_idx, out_dist);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_bf_state_init, dim3(nblocks((int64_t)nq * 8, 256)), dim3(256), 0, s, state, nq, k);
  hipLaunchKernelGGL(k_bf_fill_i32, dim3(nblocks((int64_t)nq * 256, 256)), dim3(256), 0, s,
                     reinterpret_cast<int32_t*>(hist), (int64_t)nq * 256, 0);
  hipLaunchKernelGGL(k_bf_fill_i32, dim3(nblocks((int64_t)nq * k, 256)), dim3(256), 0, s, out_idx, (int64_t)nq * k,
                     -1);
  const dim3 grid(nblocks(N, kSelBlock), nq);
  for (int digit = 0; digit < 4; digit++)
    hipLaunchKernelGGL(k_bf_radix, grid, dim3(kBfThreads), 0, s, scores, ld_scores, N, digit, state, hist);
  hipLaunchKernelGGL(k_bf_collect, grid, dim3(kBfThreads), 0, s, scores, ld_scores, N, k, state, out_idx, out_dist);
  hipLaunchKernelGGL(k_bf_stream, dim3(nq), dim3(64), 0, s, scores, ld_scores, N, k, state, out_idx, out_dist);
  return hipGetLastError();
}

hipError_t bf_vnorm(int mode, const void* grp, const void* tail, int N, int dim, uint32_t* vmax, hipStream_t s) {
  if (N <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_bf_fill_i32, dim3(1), dim3(64), 0, s, reinterpret_cast<int32_t*>(vmax), (int64_t)1, 0);
  const dim3 grid(nblocks(N, kBfThreads)), blk(kBfThreads);
  switch (mode) {
    case kBfF32:
      hipLaunchKernelGGL(k_bf_vnorm<float>, grid, blk, 0, s, static_cast<const float*>(grp),
                         static_cast<const float*>(tail), N, dim, vmax);
      break;
    case kBfI8:
      hipLaunchKernelGGL(k_bf_vnorm<int8_t>, grid, blk, 0, s, static_cast<const int8_t*>(grp),
                         static_cast<const int8_t*>(tail), N, dim, vmax);
      break;
    case kBfI16:
      hipLaunchKernelGGL(k_bf_vnorm<int16_t>, grid, blk, 0, s, static_cast<const int16_t*>(grp),
                         static_cast<const int16_t*>(tail), N, dim, vmax);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

namespace {
int pf_ksteps(int dim) { return ((dim >> 3) + 1) / 2 + ((dim & 7) ? 1 : 0); }

template <typename T, int CT>
hipError_t approx_t(const void* grp, const void* tail, int N, int dim, float vscale, const _Float16* qfrag, int nq,
                    float* blockmax, int nb, hipStream_t s) {
  constexpr int PF = sizeof(T) == 1 ? 12 : sizeof(T) == 2 ? 8 : 6;
  constexpr int waves = kPfThreads<CT> / 64, most = 256 * (CT == 2 ? 1 : 3);
  const int wgs = (nb + waves - 1) / waves;
  const size_t lds = (size_t)pf_ksteps(dim) * CT * 1024;
  hipLaunchKernelGGL((k_bf_approx<T, CT, PF>), dim3(wgs < most ? wgs : most), dim3(kPfThreads<CT>), lds, s,
                     static_cast<const T*>(grp), static_cast<const T*>(tail), N, dim, vscale, qfrag, nq, blockmax, nb);
  return hipGetLastError();
}
}  // namespace

bool bf_prefilter_ok(int N, int dim, int k, float vnorm) {
  const int nb = (N + kBfBlock - 1) / kBfBlock;
  return N <= (1 << 30) && dim >= 16 && (size_t)pf_ksteps(dim) * 1024 <= kBfPfLds && nb >= 2 * bf_prefilter_cap(k) &&
         vnorm >= kPfNormLeast && vnorm <= 1.0e30f;
}

int bf_prefilter_queries(int dim) { return (size_t)pf_ksteps(dim) * 2048 <= kBfPfLds ? 64 : 32; }

hipError_t bf_prefilter(int mode, const void* grp, const void* tail, int N, int dim, float vnorm, float* queries,
                        int nq, bool normalize, int k, const sg_bf_work& w, hipStream_t s) {
  if (nq <= 0 || nq > bf_prefilter_queries(dim) || !bf_prefilter_ok(N, dim, k, vnorm)) return hipErrorInvalidValue;
  const int ct = nq > 32 ? 2 : 1, nb = (N + kBfBlock - 1) / kBfBlock, cap = bf_prefilter_cap(k);
  // Stored norm in the units of the fp16 operand: codes as they are (the norm
  // is in dequantized units), floats scaled by a power of two to a largest
  // norm in [128, 256).
  float vscale = 1.0f, vs = vnorm;
  if (mode == kBfF32) {
    int e = 0;
    (void)frexpf(vnorm, &e);
    vscale = ldexpf(1.0f, 8 - e);
    vs = vnorm * vscale;
  } else {
    vs = vnorm * (mode == kBfI8 ? 127.0f : 32767.0f);
  }
  hipLaunchKernelGGL(k_bf_prep, dim3(32 * ct), dim3(kPrepThreads), (sizeof(float) + sizeof(double)) * (size_t)((dim + 15) & ~15), s, queries, nq, dim,
                     normalize ? 1 : 0, vs * 1.01f, vs / vnorm, mode == kBfI8 ? 1 : 0, ct, w.qfrag, w.eps, w.flags);
  hipError_t e = hipErrorInvalidValue;
  switch (mode) {
#define SG_PF(MODE, T)                                                                                           \
  case MODE:                                                                                                     \
    e = ct == 2 ? approx_t<T, 2>(grp, tail, N, dim, vscale, w.qfrag, nq, w.blockmax, nb, s)                      \
                : approx_t<T, 1>(grp, tail, N, dim, vscale, w.qfrag, nq, w.blockmax, nb, s);                     \
    if (e != hipSuccess) return e;                                                                               \
    hipLaunchKernelGGL(k_bf_blocks, dim3(nq), dim3(kTopThreads), 0, s, w.blockmax, nb, k, w.eps, cap, w.list,    \
                       w.count, w.flags);                                                                        \
    hipLaunchKernelGGL(k_bf_rescore<T>, dim3(nblocks(cap, kBfThreads / 128), nq), dim3(kBfThreads),               \
                       sizeof(float) * (size_t)(dim & ~7), s,                                                     \
                       static_cast<const T*>(grp), static_cast<const T*>(tail), N, dim, queries, w.list, w.count, \
                       cap, w.cand);                                                                             \
    break;
    SG_PF(kBfF32, float)
    SG_PF(kBfI8, int8_t)
    SG_PF(kBfI16, int16_t)
#undef SG_PF
    default:
      return e;
  }
  hipLaunchKernelGGL(k_bf_top, dim3(nq), dim3(kTopThreads), 0, s, w.cand, w.list, w.count, cap, k, w.eps,
                     w.out_idx, w.out_dist, w.flags);
  return hipGetLastError();
}

}  // namespace sgk
