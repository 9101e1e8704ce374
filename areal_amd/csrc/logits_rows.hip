// Logits-in label log-probabilities and entropy: the forward one workgroup per row, the backward one per 8 KiB of a
// row. Bound by HBM. Rows of any start and length are read in 16-byte steps: with 2-byte accesses for vocabularies
// that are no multiple of 8, 4000 x 50257 bf16 took 232 us forward and 302 backward, now 71 and 132.
//
// Follows areal/utils/functional/vocab_parallel.py:16-30: log_softmax(logits.float() / T),
// gather at the label, entropy = -sum p log p; row chunking (:42-82) does not change values.
// The forward reads each logit once (online max / sum-exp); the backward reads it once more
// and writes d loss / d logits in the dtype of the logits:
//     d lp_label / d x_j = (1[j == label] - p_j) / T
//     d entropy  / d x_j = -p_j (log p_j + entropy) / T
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace {

constexpr float LOG2E_F = 1.4426950408889634f;
constexpr float LN2_F = 0.6931471805599453f;

// Vector accesses carry the non-temporal hint: every logit is read once per kernel (and every
// dlogit written once), and a plain read of a [4096, 151936] bf16 array in this access pattern
// measures 6.15 TB/s without the hint, 7.04 TB/s with it. `Vec` loads from any element (gfx950 runs
// with unaligned access enabled: still one 16-byte instruction); stores are aligned by their caller.
template <typename T> struct Elem;
template <> struct Elem<float> {
  typedef f32x4 Vec __attribute__((aligned(4)));
  static constexpr int VEC = 4;
  static DEVI float load(const float* p) { return *p; }
  static DEVI void widen(const f32x4& v, float* o) { o[0] = v[0]; o[1] = v[1]; o[2] = v[2]; o[3] = v[3]; }
  static DEVI void store(float* p, float v) { *p = v; }
  static DEVI void storev(float* p, const float* o) {
    f32x4 v = {o[0], o[1], o[2], o[3]};
    __builtin_nontemporal_store(v, (f32x4*)p);
  }
};
template <> struct Elem<u16> {  // bf16 bit patterns
  typedef u32x4 Vec __attribute__((aligned(2)));
  static constexpr int VEC = 8;
  static DEVI float load(const u16* p) { return bf16_bits_to_f32(*p); }
  static DEVI void widen(const u32x4& v, float* o) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = __builtin_bit_cast(float, v[i] << 16);
      o[2 * i + 1] = __builtin_bit_cast(float, v[i] & 0xffff0000u);
    }
  }
  static DEVI void store(u16* p, float v) { *p = f32_to_bf16_bits(v); }
  static DEVI void storev(u16* p, const float* o) {
    u32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = (uint32_t)f32_to_bf16_bits(o[2 * i]) | ((uint32_t)f32_to_bf16_bits(o[2 * i + 1]) << 16);
    __builtin_nontemporal_store(v, (u32x4*)p);
  }
};

// U vectors, `step` vectors apart: all loads before the first use.
template <typename T, int U, bool KEEP = false>
DEVI void load_group(const T* p, int64_t step, float (&z)[U * Elem<T>::VEC]) {
  typename Elem<T>::Vec v[U];  // KEEP: without the non-temporal hint
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const auto* const at = (const typename Elem<T>::Vec*)(p + u * step * Elem<T>::VEC);
    v[u] = KEEP ? *at : __builtin_nontemporal_load(at);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) Elem<T>::widen(v[u], z + u * Elem<T>::VEC);
}

// A row of V elements at p: `head` elements up to the first 16-byte boundary, `vecs` whole vectors, the rest.
template <typename T> struct RowSplit {
  int head, vecs, edge;  // edge: elements in front of and behind the vectors (fewer than two vectors)
  DEVI RowSplit(const T* p, int V) {
    const int h = (int)((16 - ((uintptr_t)p & 15)) & 15) / (int)sizeof(T);
    head = h < V ? h : V;
    vecs = (V - head) / Elem<T>::VEC;
    edge = V - vecs * Elem<T>::VEC;
  }
  DEVI int edge_index(int e) const { return e < head ? e : vecs * Elem<T>::VEC + e; }
};

// Vectors a thread loads before it uses the first. Forward, 4096 x 151936 bf16: 1, 2, 4 and 8 are alike (189 to
// 191 us: eight blocks of 256 threads a CU keep enough in flight); one block of 1024 per row at 300 rows 31.7 us with
// one, 28.2 with two or four, 32.3 with eight.
constexpr int FWD_GROUP = 2;
// Below this many rows a row gets 1024 threads instead of 256: at 1024 x 151936 bf16 four blocks of 256 a CU
// take 52.2 us and blocks of 1024 62.1; at 300 rows blocks of 256 took 53.3 us, of 1024 28.2; at 16 28.1 and 16.6.
constexpr int64_t FWD_FEW_ROWS = 1024;
// A block of the backward takes one run of BWD_GROUP * BWD_THREADS vectors of a row (8 KiB), so that the blocks in
// flight read and write one stretch of memory in order: a block per row, 2048 places at once, took 485 us at
// 4096 x 151936 bf16 (5.1 TB/s), this 401 (6.2 TB/s); one vector per thread 417, three 405, four 399 (and 140.9 us
// against 131.9 at 4000 x 50257). At 16 rows a block per row left the chip idle: 31.9 us, this 6.9.
constexpr int BWD_GROUP = 2;
constexpr int BWD_THREADS = 256;
constexpr int64_t BWD_MAX_BLOCKS = 1 << 23;  // a launch is limited to 2^32 threads

struct Online {
  float m, s, q;  // max of z2 = x*c2, sum 2^(z2-m), sum (z2-m) 2^(z2-m)
};
// Sums of a part without a finite logit are 0, or NaN where it met a NaN or (the entropy's) a -inf, and stay so.
DEVI void online_merge(Online& a, const Online& b) {
  const float m = fmaxf(a.m, b.m);
  float s = 0.f, q = 0.f;
  auto part = [&](const Online& o) {
    const float d = o.m > neg_inf() ? o.m - m : 0.f, al = fast_exp2(d);
    s += al * o.s;
    q += al * fmaf(d, o.s, o.q);
  };
  part(a);
  part(b);
  a.m = m; a.s = s; a.q = q;
}
// x: raw logits; the exponents are z2 = x * c2 (c2 > 0). The running maximum is kept as the
// rounded product of the largest logit and every exponent is taken relative to it with one fused
// multiply-subtract, as the backward evaluates them against lse2.
template <int N>
DEVI void online_add(Online& st, const float (&x)[N], float c2) {
  float xm = x[0];
#pragma unroll
  for (int i = 1; i < N; ++i) xm = fmaxf(xm, x[i]);
  const float vm = xm * c2;
  if (vm > st.m) {
    if (st.m > neg_inf()) {
      const float d = st.m - vm, al = fast_exp2(d);
      st.q = al * fmaf(d, st.s, st.q);
      st.s = al * st.s;
    }
    st.m = vm;
  }
  // Nothing but -inf so far: exponentials of 0, not of inf - inf. A logit of -inf leaves the log-probabilities
  // alone and makes the entropy NaN, as p log p = 0 x -inf does.
  const float m = st.m > neg_inf() ? st.m : 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float t = fmaf(x[i], c2, -m);
    const float e = fast_exp2(t);
    st.s += e;
    st.q = fmaf(t, e, st.q);
  }
}

DEVI Online block_merge(Online st, Online* smem) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    Online other;
    other.m = __shfl_xor(st.m, o, 64); other.s = __shfl_xor(st.s, o, 64);
    other.q = __shfl_xor(st.q, o, 64);
    online_merge(st, other);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) smem[w] = st;
  __syncthreads();
  Online r = smem[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) online_merge(r, smem[i]);
  return r;
}

// Where a backward follows (lse2 is asked for) the last rows are read without the non-temporal hint, as much as the memory-side cache
// of 256 MB holds, or twice that of more than 900 MB, so that part of the backward's reads come from there. Forward and
// backward, inputs new to the caches, us, all under the hint / last 256 MB without / 512 MB / all: bf16 4096 x 151936 588 / 568 /
// 557 / 574, 3300 x 151936 477 / 457 / 454, 3500 x 128256 427 / 415 / 424 / 435, 2000 x 151936 289 / 274 / 273 / 277, 1500 x 128256 183 /
// 176 / 187 / 187, 1200 x 151936 174 / 165 / 167 / 168, 9500 x 50257 463 / 445 / 443, 9000 x 32000 278 / 269 / 271 / 272; fp32 2000 x
// 151936 576 / 560 / 546 / 566, 1800 x 128256 441 / 425 / 414, 4000 x 50257 390 / 377 / 375 / 379, 4000 x 32000 245 / 236 / 244 / 244. The rows
// read from the last to the first, so that the ones kept are those that the backward starts with, give less: 562 with 320 MB at
// 4096 x 151936, and they lose with rows of up to 128 KB (9000 x 32000 289, fp32 570 for 545) and at 128256 (3500 rows 444 with 320 MB). A
// forward that no backward follows keeps the hint: 2000 x 151936 190, 193 to 203 without.
constexpr int64_t KEEP_LAST = (int64_t)256 << 20, KEEP_MORE = (int64_t)512 << 20, KEEP_MORE_FROM = (int64_t)900 << 20;
// lse2[t] = max + log2(sum) in base-2 units of z2 = x * inv_temp * log2(e).
template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void rows_fwd_kernel(const T* __restrict__ logits, int64_t ld,
                                                           const int64_t* __restrict__ labels, int V,
                                                           float inv_temp, float* __restrict__ logprobs,
                                                           float* __restrict__ entropy,
                                                           float* __restrict__ lse2_out, unsigned keep_from) {
  __shared__ Online smem[THREADS / 64];
  const int64_t row = blockIdx.x;
  const T* x = logits + row * ld;
  const float c2 = inv_temp * LOG2E_F;
  Online st{neg_inf(), 0.f, 0.f};
  constexpr int VEC = Elem<T>::VEC, U = FWD_GROUP;
  const RowSplit<T> rs(x, V);
  const T* body = x + rs.head;
  auto sweep = [&](auto keep) {
    constexpr bool KEEP = decltype(keep)::value;
    int v = threadIdx.x;
    for (; v + (U - 1) * THREADS < rs.vecs; v += U * THREADS) {
      float z[U * VEC];
      load_group<T, U, KEEP>(body + (int64_t)v * VEC, THREADS, z);
      online_add(st, z, c2);
    }
    for (; v < rs.vecs; v += THREADS) {
      float z[VEC];
      load_group<T, 1, KEEP>(body + (int64_t)v * VEC, 0, z);
      online_add(st, z, c2);
    }
  };
  if (blockIdx.x >= keep_from) sweep(std::true_type{});
  else sweep(std::false_type{});
  if ((int)threadIdx.x < rs.edge) {
    float z[1] = {Elem<T>::load(x + rs.edge_index(threadIdx.x))};
    online_add(st, z, c2);
  }
  const Online r = block_merge(st, smem);
  if (threadIdx.x == 0) {
    const float log2s = fast_log2(r.s);
    const float lse2 = r.m + log2s;
    const int64_t lab = labels[row];
    float lp = 0.f;
    if (lab >= 0 && lab < V) {
      // the label's exponent as the sums saw it: relative to the running maximum, by one fused
      // multiply-subtract
      const float tl = fmaf(Elem<T>::load(x + lab), c2, -r.m);
      lp = (tl - log2s) * LN2_F;
      lp = lp > 0.f ? 0.f : lp;  // (NaN stays)
    }
    if (logprobs) logprobs[row] = lp;
    if (entropy) entropy[row] = (log2s - r.q / r.s) * LN2_F;
    if (lse2_out) lse2_out[row] = lse2;
  }
}

// Block (row, part) writes part `part` of `parts` equal runs of vectors of the row.
template <typename T, bool ENT>
__global__ __launch_bounds__(BWD_THREADS) void rows_bwd_kernel(
    const T* __restrict__ logits, int64_t ld, const int64_t* __restrict__ labels, int V,
    float inv_temp, const float* __restrict__ lse2, const float* __restrict__ entropy,
    const float* __restrict__ grad_lp, const float* __restrict__ grad_ent, T* __restrict__ dlogits,
    int64_t ldd, unsigned parts, unsigned part_vecs) {
  const int64_t row = blockIdx.x / parts;
  const unsigned part = blockIdx.x % parts;
  const T* x = logits + row * ld;
  T* d = dlogits + row * ldd;
  const float c2 = inv_temp * LOG2E_F;
  const float l2 = lse2[row];
  const float glp = (grad_lp ? grad_lp[row] : 0.f) * inv_temp;
  const float gen = ENT ? grad_ent[row] * inv_temp : 0.f;
  const float ent = ENT ? entropy[row] : 0.f;
  const int64_t lab64 = labels[row];
  const int lab = (lab64 >= 0 && lab64 < V) ? (int)lab64 : -1;
  auto gradient = [&](float z, bool label) {
    const float t = fmaf(z, c2, -l2);
    const float p = fast_exp2(t);
    float g = -p * glp;
    if (label) g += glp;
    if (ENT) g -= gen * p * (t * LN2_F + ent);
    return g;
  };
  constexpr int VEC = Elem<T>::VEC, U = BWD_GROUP;
  const RowSplit<T> rs(d, V);
  // vectors of this part: [v, end)
  const int begin = (int)(part * part_vecs);
  const int end = rs.vecs - begin < (int)part_vecs ? rs.vecs : begin + (int)part_vecs;
  auto group = [&](auto n, int v) {
    constexpr int N = decltype(n)::value;
    float z[N * VEC];
    const int at = rs.head + v * VEC;
    load_group<T, N>(x + at, BWD_THREADS, z);
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int to_label = lab - (at + u * BWD_THREADS * VEC);
#pragma unroll
      for (int i = 0; i < VEC; ++i) z[u * VEC + i] = gradient(z[u * VEC + i], to_label == i);
      Elem<T>::storev(d + at + u * BWD_THREADS * VEC, z + u * VEC);
    }
  };
  int v = begin + threadIdx.x;
  for (; v + (U - 1) * BWD_THREADS < end; v += U * BWD_THREADS) group(std::integral_constant<int, U>{}, v);
  for (; v < end; v += BWD_THREADS) group(std::integral_constant<int, 1>{}, v);
  if (part == 0 && (int)threadIdx.x < rs.edge) {
    const int at = rs.edge_index(threadIdx.x);
    Elem<T>::store(d + at, gradient(Elem<T>::load(x + at), at == lab));
  }
}

template <typename T>
int launch_rows_fwd(const void* logits, int64_t ld, const int64_t* labels, int64_t T_, int64_t V,
                    float inv_temp, float* lp, float* ent, float* lse2, hipStream_t stream) {
  const int64_t row_bytes = V * (int64_t)sizeof(T);
  const int64_t keep_bytes = T_ * row_bytes <= KEEP_MORE_FROM ? KEEP_LAST : KEEP_MORE;
  const unsigned keep_from = (unsigned)(lse2 == nullptr ? T_ : std::max<int64_t>(T_ - keep_bytes / row_bytes, 0));
  auto launch = [&](auto threads) {
    constexpr int THREADS = decltype(threads)::value;
    hipLaunchKernelGGL((rows_fwd_kernel<T, THREADS>), dim3((unsigned)T_), dim3(THREADS), 0, stream,
                       (const T*)logits, ld, labels, (int)V, inv_temp, lp, ent, lse2, keep_from);
  };
  if (T_ < FWD_FEW_ROWS)
    launch(std::integral_constant<int, 1024>{});
  else
    launch(std::integral_constant<int, 256>{});
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

template <typename T>
int launch_rows_bwd(const void* logits, int64_t ld, const int64_t* labels, int64_t T_, int64_t V,
                    float inv_temp, const float* lse2, const float* ent, const float* glp,
                    const float* gent, void* dlogits, int64_t ldd, hipStream_t stream) {
  const int64_t vecs = V / Elem<T>::VEC, per = BWD_GROUP * BWD_THREADS;
  int64_t parts = std::max<int64_t>(ceil_div_i64(vecs, per), 1);
  parts = std::min(parts, std::max<int64_t>(BWD_MAX_BLOCKS / T_, 1));
  const int64_t part_vecs = round_up_i64(ceil_div_i64(vecs, parts), per);
  auto launch = [&](auto with_entropy) {
    hipLaunchKernelGGL((rows_bwd_kernel<T, decltype(with_entropy)::value>), dim3((unsigned)(T_ * parts)),
                       dim3(BWD_THREADS), 0, stream, (const T*)logits, ld, labels, (int)V, inv_temp, lse2, ent, glp,
                       gent, (T*)dlogits, ldd, (unsigned)parts, (unsigned)part_vecs);
  };
  if (gent)
    launch(std::true_type{});
  else
    launch(std::false_type{});
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

}  // namespace

extern "C" {

// dtype: 0 = fp32 logits, 1 = bf16 logits. logits [T, V] with row pitch ld (elements).
// Outputs fp32 [T]: logprobs, entropy (nullable), lse2 (nullable; log-sum-exp in base-2 units,
// the only state the backward needs besides entropy).
int areal_logits_logprobs_entropy_fwd(const void* logits, int dtype, int64_t ld,
                                      const int64_t* labels, int64_t T, int64_t V,
                                      float inv_temperature, float* logprobs, float* entropy,
                                      float* lse2, hipStream_t stream) {
  if (T < 0 || V <= 0 || ld < V || !(inv_temperature > 0.f)) return AREAL_ERR_BAD_ARG;
  if (T == 0) return AREAL_OK;
  if (!logits || !labels) return AREAL_ERR_BAD_ARG;
  if (V > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  if (dtype == 0)
    return launch_rows_fwd<float>(logits, ld, labels, T, V, inv_temperature, logprobs, entropy, lse2,
                                  stream);
  if (dtype == 1)
    return launch_rows_fwd<u16>(logits, ld, labels, T, V, inv_temperature, logprobs, entropy, lse2,
                                stream);
  return AREAL_ERR_BAD_ARG;
}

// dlogits [T, V] (same dtype as logits, row pitch ldd) = grad_logprobs * d lp / d logits
// + grad_entropy * d entropy / d logits; either upstream gradient may be null.
int areal_logits_logprobs_entropy_bwd(const void* logits, int dtype, int64_t ld,
                                      const int64_t* labels, int64_t T, int64_t V,
                                      float inv_temperature, const float* lse2,
                                      const float* entropy, const float* grad_logprobs,
                                      const float* grad_entropy, void* dlogits, int64_t ldd,
                                      hipStream_t stream) {
  if (T < 0 || V <= 0 || ld < V || ldd < V || !(inv_temperature > 0.f)) return AREAL_ERR_BAD_ARG;
  if (T == 0) return AREAL_OK;
  if (!logits || !labels || !lse2 || !dlogits) return AREAL_ERR_BAD_ARG;
  if (grad_entropy != nullptr && entropy == nullptr) return AREAL_ERR_BAD_ARG;
  if (V > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  if (dtype == 0)
    return launch_rows_bwd<float>(logits, ld, labels, T, V, inv_temperature, lse2, entropy,
                                  grad_logprobs, grad_entropy, dlogits, ldd, stream);
  if (dtype == 1)
    return launch_rows_bwd<u16>(logits, ld, labels, T, V, inv_temperature, lse2, entropy,
                                grad_logprobs, grad_entropy, dlogits, ldd, stream);
  return AREAL_ERR_BAD_ARG;
}

}  // extern "C"
